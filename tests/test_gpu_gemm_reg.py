"""The exact products with the weights made in the operand registers (gemm_i8r_kernel) against the oracle's matmul!, bit for bit."""
import numpy as np
import pytest

import oracle_lib as orc
from illatio_amd import synth

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.fixture(scope="module")
def dev():
    from illatio_amd import hip
    return hip.open_hip(0)


# rows around tiles of 32, 64 and 128, tokens around patches of 32 and tiles of 128, one super-block, two, an odd number
@pytest.mark.parametrize("rows_a_tile", ["64", "128"])
@pytest.mark.parametrize("qtype,rows,cols,n", [
    (synth.Q4_K, 1, 256, 17), (synth.Q4_K, 127, 512, 33), (synth.Q4_K, 129, 768, 128), (synth.Q4_K, 300, 2560, 130),
    (synth.Q6_K, 31, 256, 64), (synth.Q6_K, 128, 512, 127), (synth.Q6_K, 65, 1280, 129), (synth.Q6_K, 257, 2816, 250)])
def test_operands_in_registers_bit_for_bit(dev, monkeypatch, rows_a_tile, qtype, rows, cols, n):
    from illatio_amd import dense, hip
    monkeypatch.setenv("ILT_I8_FEW", "0")
    monkeypatch.setenv("ILT_I8_TM", rows_a_tile)
    rng = synth.make_rng(rows + cols + n)
    w = synth.weights(qtype, rows, cols, rng).copy()
    # a row of the largest scales and quants, tokens of one sign: the largest integer sums there are
    blk = w.reshape(rows, -1, synth.BLOCK_BYTES[qtype])[rows // 2]
    if qtype == synth.Q4_K:
        blk[:, 4:] = 0xFF
    else:
        blk[:, :192] = 0
        blk[:, 192:208] = 0x80
    x = synth.activations((n, cols), rng)
    x[n // 2] = 1.0
    x[n // 3, :256] = 0.0
    bias = synth.activations(rows, rng)
    m = dense.upload_gmat(dev, "w", qtype, rows, cols, w)
    act = dense.QAct(dev, n, cols, ("q8k",))
    xb, bb, y, y2 = hip.hip_upload_new(dev, x), hip.hip_upload_new(dev, bias), hip.hip_alloc(dev, 4 * n * rows), hip.hip_alloc(dev, 4 * n * rows)
    dense.quantize_act(dev, xb, act)
    want = orc.matmul(qtype, w, rows, cols, x, nthreads=8).reshape(n, rows)
    dense.cmat_mul(dev, m, act, y, n)
    got = hip.hip_floats(y, n * rows).reshape(n, rows)
    assert np.array_equal(bits(got), bits(want)), np.argwhere(bits(got) != bits(want))[:5]
    dense.cmat_mul(dev, m, act, y, n, bias=bb, acc=True)
    assert np.array_equal(bits(hip.hip_floats(y, n * rows).reshape(n, rows)), bits(want + (want + bias[None, :])))
    dense.cmat_mul_n(dev, [(m, y, None), (m, y2, bb)], act, n)       # two matrices a launch
    assert np.array_equal(bits(hip.hip_floats(y, n * rows).reshape(n, rows)), bits(want))
    assert np.array_equal(bits(hip.hip_floats(y2, n * rows).reshape(n, rows)), bits(want + bias[None, :]))
    for b in (xb, bb, y, y2):
        hip.hip_free(b)
    act.free()
    m.free()
