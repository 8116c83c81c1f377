"""The exact products of a few tokens (gemm_i8_few_kernel) against the oracle's matmul!, bit for bit."""
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


# rows around tiles of 16 and 32, tokens around tiles of 16 and 32, columns of fewer units than waves, of a whole and of a
# broken number of rounds (a round: what LDS holds the terms of), Q8_0 rows that end in half a unit
SHAPES = [
    (synth.Q4_K, 1, 256, 2), (synth.Q4_K, 33, 2560, 16), (synth.Q4_K, 48, 4608, 17), (synth.Q4_K, 130, 1024, 95),
    (synth.Q6_K, 17, 256, 1), (synth.Q6_K, 32, 2816, 33), (synth.Q6_K, 47, 9728, 32), (synth.Q6_K, 160, 512, 130),
    (synth.Q8_0, 15, 32, 3), (synth.Q8_0, 64, 896, 31), (synth.Q8_0, 31, 1888, 40), (synth.Q8_0, 16, 4864, 15)]


# (the cut over eight waves: Q8_0's alone)
@pytest.mark.parametrize("cut,qtype,rows,cols,n", [(cut,) + s for cut in ("2", "4", "8") for s in SHAPES if cut != "8" or s[0] == synth.Q8_0])
def test_few_tokens_bit_for_bit(dev, monkeypatch, cut, qtype, rows, cols, n):
    from illatio_amd import dense, hip
    monkeypatch.setenv("ILT_I8_FEW", cut)
    rng = synth.make_rng(rows + cols + n)
    w = synth.weights(qtype, rows, cols, rng)
    x = synth.activations((n, cols), rng)
    x[n // 2, :min(256, cols)] = 0.0
    bias = synth.activations(rows, rng)
    m = dense.upload_gmat(dev, "w", qtype, rows, cols, w)
    act = dense.QAct(dev, n, cols, ("q8",) if qtype == synth.Q8_0 else ("q8k",))
    xb, bb, y = hip.hip_upload_new(dev, x), hip.hip_upload_new(dev, bias), hip.hip_alloc(dev, 4 * n * rows)
    dense.quantize_act(dev, xb, act)
    code = [dense.KQUANT_CODE[qtype]] if qtype != synth.Q8_0 else []
    mm = "mm_q8" if qtype == synth.Q8_0 else "mm_k"
    wa = [m.qs, m.d, act.xq, act.xs] if qtype == synth.Q8_0 else code + [m.qs, act.kq, act.kd, act.ksum]
    hip.launch(dev, mm, 1, 256, wa + [y, None, rows, cols, n, 0])
    want = orc.matmul(qtype, w, rows, cols, x, nthreads=8).reshape(n, rows)
    got = hip.hip_floats(y, n * rows).reshape(n, rows)
    assert np.array_equal(bits(got), bits(want)), np.argwhere(bits(got) != bits(want))[:5]
    hip.launch(dev, mm, 1, 256, wa + [y, bb, rows, cols, n, 1])
    assert np.array_equal(bits(hip.hip_floats(y, n * rows).reshape(n, rows)), bits(want + (want + bias[None, :])))
    for b in (xb, bb, y):
        hip.hip_free(b)
    act.free()
    m.free()
