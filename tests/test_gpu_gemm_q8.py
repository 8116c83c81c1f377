"""The exact Q8_0 products in register tiles (gemm_q8_kernel) against the oracle's matmul!, bit for bit."""
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


# rows and tokens around each tile's edges, fewer steps than the ring has stages, columns of half a step of 128; one matrix with
# bias and accumulation, then three in a launch
@pytest.mark.parametrize("tile", ["1", "2", "3", "4"])
@pytest.mark.parametrize("rows,cols,n", [(1, 64, 1), (33, 128, 31), (31, 192, 33), (129, 896, 65), (300, 256, 17), (127, 1024, 130)])
def test_q8_tiles_bit_for_bit(dev, monkeypatch, tile, rows, cols, n):
    from illatio_amd import dense, hip
    monkeypatch.setenv("ILT_Q8_TILE", tile)
    monkeypatch.setenv("ILT_I8_FEW", "0")
    rng = synth.make_rng(rows + cols + n)
    x = synth.activations((n, cols), rng)
    x[n // 2, :32] = 0.0
    shapes = [rows, 16, rows + 5]
    ws = [synth.weights(synth.Q8_0, r, cols, rng) for r in shapes]
    bias = synth.activations(rows, rng)
    ms = [dense.upload_gmat(dev, "w", synth.Q8_0, r, cols, w) for r, w in zip(shapes, ws)]
    act = dense.QAct(dev, n, cols, ("q8",))
    xb, bb = hip.hip_upload_new(dev, x), hip.hip_upload_new(dev, bias)
    ys = [hip.hip_alloc(dev, 4 * n * r) for r in shapes]
    dense.quantize_act(dev, xb, act)
    want = [orc.matmul(synth.Q8_0, w, r, cols, x, nthreads=8).reshape(n, r) for r, w in zip(shapes, ws)]
    hip.launch(dev, "mm_q8", 1, 256, [ms[0].qs, ms[0].d, act.xq, act.xs, ys[0], None, rows, cols, n, 0])
    hip.launch(dev, "mm_q8", 1, 256, [ms[0].qs, ms[0].d, act.xq, act.xs, ys[0], bb, rows, cols, n, 1])
    assert np.array_equal(bits(hip.hip_floats(ys[0], n * rows).reshape(n, rows)), bits(want[0] + (want[0] + bias[None, :])))
    monkeypatch.delenv("ILT_I8_FEW")
    args = []
    for m, y, r in zip(ms, ys, shapes):
        args += [m.qs, m.d, y, None, r]
    hip.launch(dev, "mm_q8_mma2", 1, 256, args + [act.xq, act.xs, cols, n, 0])
    for y, r, w in zip(ys, shapes, want):
        got = hip.hip_floats(y, n * r).reshape(n, r)
        assert np.array_equal(bits(got), bits(w)), np.argwhere(bits(got) != bits(w))[:5]
    for b in [xb, bb] + ys:
        hip.hip_free(b)
    act.free()
    for m in ms:
        m.free()
