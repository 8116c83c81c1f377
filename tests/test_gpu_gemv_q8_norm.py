"""Q8_0 decode products with rmsnorm! inside the streamed launch against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib as orc
from illatio_amd import synth
from test_gpu_gemv import bits, norm_rows, tie_row

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from illatio_amd import hip
    return hip.open_hip(0)


# one float4 a thread and the last of them, more of them with a remainder, the widest, and one past it (the looping variant)
@pytest.mark.parametrize("cols,streamed", [(896, 2), (1024, 2), (1088, 2), (3008, 2), (4096, 2), (4160, 0)])
def test_q8_norm_inside_the_streamed_product(dev, cols, streamed):
    from illatio_amd import dense, hip
    rng = synth.make_rng(cols)
    rows, eps = 1200, 1e-6
    ws = [synth.weights(synth.Q8_0, rows, cols, rng) for _ in range(2)]
    ms = [dense.upload_gmat(dev, "w", synth.Q8_0, rows, cols, w) for w in ws]
    nw, bias = synth.activations(cols, rng) * np.float32(0.1) + np.float32(1.0), synth.activations(rows, rng)
    nwb, bb, y = hip.hip_upload_new(dev, nw), hip.hip_upload_new(dev, bias), hip.hip_alloc(dev, 4 * rows)
    for x in (synth.activations(cols, rng), tie_row(cols), norm_rows(cols, 1, rng)[0], np.zeros(cols, np.float32)):
        h, xb = orc.rmsnorm(x, nw, eps), hip.hip_upload_new(dev, np.ascontiguousarray(x, np.float32))
        want = [orc.matmul(synth.Q8_0, w, rows, cols, h) for w in ws]
        before = hip.lib().ilt_streamed_launches()
        dense.mv_multi(dev, [(ms[0], y, bb)], xf=xb, norm=(nwb, eps))
        assert np.array_equal(bits(hip.hip_floats(y, rows)), bits(want[0] + bias))
        dense.glu_mul(dev, ms[0], ms[1], None, y, xf=xb, norm=(nwb, eps))
        assert np.array_equal(bits(hip.hip_floats(y, rows)), bits(orc.swiglu(want[0], want[1])))
        assert hip.lib().ilt_streamed_launches() - before == streamed
        hip.hip_free(xb)
    for b in (nwb, bb, y):
        hip.hip_free(b)
    for m in ms:
        m.free()
