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
@pytest.mark.parametrize("rows_a_tile", ["64", "128", "1", "2", "3"])
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


# the super-blocks shared out over four waves, a workgroup and two a CU: fewer of them than waves, a last round that is not whole, whole rounds; rows and
# tokens around tiles of 32 and 64
@pytest.mark.parametrize("tile", ["6", "7"])
@pytest.mark.parametrize("qtype,rows,cols,n", [
    (synth.Q4_K, 1, 256, 17), (synth.Q4_K, 33, 512, 33), (synth.Q4_K, 64, 1024, 32), (synth.Q4_K, 95, 1280, 65), (synth.Q4_K, 300, 2560, 40),
    (synth.Q6_K, 31, 256, 64), (synth.Q6_K, 32, 768, 31), (synth.Q6_K, 65, 1024, 97), (synth.Q6_K, 128, 9728, 21), (synth.Q6_K, 257, 2816, 50)])
def test_super_blocks_shared_out_bit_for_bit(dev, monkeypatch, tile, qtype, rows, cols, n):
    test_operands_in_registers_bit_for_bit(dev, monkeypatch, tile, qtype, rows, cols, n)


# the same over eight waves, tiles of 16 rows and of 32 and 16 tokens
@pytest.mark.parametrize("tile", ["8", "9"])
@pytest.mark.parametrize("qtype,rows,cols,n", [
    (synth.Q4_K, 1, 256, 2), (synth.Q4_K, 17, 2048, 33), (synth.Q4_K, 33, 2304, 16), (synth.Q4_K, 300, 4096, 21),
    (synth.Q6_K, 15, 256, 31), (synth.Q6_K, 16, 1792, 17), (synth.Q6_K, 47, 4352, 9), (synth.Q6_K, 128, 9728, 64)])
def test_super_blocks_shared_out_over_eight_waves_bit_for_bit(dev, monkeypatch, tile, qtype, rows, cols, n):
    test_operands_in_registers_bit_for_bit(dev, monkeypatch, tile, qtype, rows, cols, n)


# four waves of 16 rows on the same tokens, 16, 32 and 64 of them: fewer blocks than buffers, rows and tokens around the tiles
@pytest.mark.parametrize("tile", ["10", "11", "12"])
@pytest.mark.parametrize("qtype,rows,cols,n", [
    (synth.Q4_K, 1, 256, 2), (synth.Q4_K, 63, 512, 33), (synth.Q4_K, 65, 768, 16), (synth.Q4_K, 300, 2560, 65),
    (synth.Q6_K, 15, 256, 31), (synth.Q6_K, 64, 512, 17), (synth.Q6_K, 129, 1024, 64), (synth.Q6_K, 200, 2816, 130)])
def test_sixteen_rows_a_wave_bit_for_bit(dev, monkeypatch, tile, qtype, rows, cols, n):
    test_operands_in_registers_bit_for_bit(dev, monkeypatch, tile, qtype, rows, cols, n)


# Q, K and V of mixed formats in one launch of such tiles, against the products for few tokens
@pytest.mark.parametrize("tile", ["6", "7", "8", "9", "10", "11", "12"])
def test_mixed_formats_with_super_blocks_shared_out(dev, monkeypatch, tile):
    from illatio_amd import hip, model
    host = model.synth_model(12, d=768, ffn=1024, nh=12, nkv=4, hd=64, nl=2, vocab=700)
    c = host["config"]
    prompt = synth.make_rng(91).integers(0, c["vocab"], 37).tolist()
    res = []
    for one in (True, False):
        monkeypatch.setenv("ILT_I8_FEW", "0" if one else "1")
        monkeypatch.setenv("ILT_I8_TM", tile)
        m = model.DenseModel(dev, host, nctx=40)
        m.forward_n(prompt)
        res.append([hip.hip_floats(m.logits, c["vocab"])] + [hip.hip_floats(m.layers[1][k], 37 * c["nkv"] * c["hd"]) for k in ("kc", "vc")])
        m.free()
    for a, b in zip(*res):
        assert np.isfinite(a).all() and np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("rows_a_tile", ["64", "128"])
@pytest.mark.parametrize("qtype,rows,cols,n", [(synth.Q2_K, 129, 768, 33), (synth.Q2_K, 64, 256, 130), (synth.IQ2_XXS, 129, 256, 65), (synth.IQ2_XXS, 100, 1280, 128)])
def test_expert_formats_on_a_dense_matrix_bit_for_bit(dev, monkeypatch, rows_a_tile, qtype, rows, cols, n):
    from illatio_amd import ds4f, hip
    monkeypatch.setenv("ILT_I8_TM", rows_a_tile)
    rng = synth.make_rng(rows + cols + n)
    w, x = synth.weights(qtype, rows, cols, rng), synth.activations((n, cols), rng)
    x[n // 2] = 1.0
    wb, xb, y = hip.hip_upload_new(dev, w), hip.hip_upload_new(dev, x), hip.hip_alloc(dev, 4 * n * rows)
    ds4f.dk_mm(dev, "d4_mm_q2_k" if qtype == synth.Q2_K else "d4_mm_iq2_xxs", wb, None, synth.row_bytes(qtype, cols), rows, cols, xb, y, n)
    want = orc.matmul(qtype, w, rows, cols, x, nthreads=8).reshape(n, rows)
    got = hip.hip_floats(y, n * rows).reshape(n, rows)
    assert np.array_equal(bits(got), bits(want)), np.argwhere(bits(got) != bits(want))[:5]
    for b in (wb, xb, y):
        hip.hip_free(b)


# groups around patches of 32 and tiles of 128, one without rows
@pytest.mark.parametrize("qtype,rows,cols", [(synth.Q2_K, 128, 256), (synth.Q2_K, 161, 1280), (synth.IQ2_XXS, 128, 256), (synth.IQ2_XXS, 200, 768)])
def test_groups_bit_for_bit(dev, qtype, rows, cols):
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(rows + cols)
    counts = np.array([1, 32, 0, 33, 64, 65, 128, 129, 260], np.uint32)
    ne, total = len(counts), int(counts.sum())
    bases = (np.cumsum(counts) - counts).astype(np.uint32)
    rb = synth.row_bytes(qtype, cols)
    w = synth.weights(qtype, ne * rows, cols, rng).reshape(ne, rows, rb)
    x = synth.activations((total, cols), rng)
    wb, xb, y = hip.hip_upload_new(dev, w), hip.hip_upload_new(dev, x), hip.hip_alloc(dev, 4 * total * rows)
    ptrs = hip.hip_upload_new(dev, np.array([wb.ptr + z * rows * rb for z in range(ne)], np.uint64))
    cb, bb = hip.hip_upload_new(dev, counts), hip.hip_upload_new(dev, bases)
    xq, xd, xs = ds4f._q8k(dev, xb, total * cols)
    hip.launch(dev, "d4_mm_id_q2_k" if qtype == synth.Q2_K else "d4_mm_id_iq2_xxs", (1, 1, ne), 128,
               [cols, rows, rb, cols, rows, hip.I64(0), ptrs, cb, bb, xq, y, xd, xs, hip.I64(total)])
    got = hip.hip_floats(y, total * rows).reshape(total, rows)
    for z in range(ne):
        if counts[z] == 0:
            continue
        at = slice(int(bases[z]), int(bases[z] + counts[z]))
        want = orc.matmul(qtype, w[z], rows, cols, x[at], nthreads=8).reshape(-1, rows)
        assert np.array_equal(bits(got[at]), bits(want)), (z, np.argwhere(bits(got[at]) != bits(want))[:5])
    for b in (wb, xb, y, ptrs, cb, bb, xq, xd, xs):
        hip.hip_free(b)


# which expert and which of its rows a workgroup takes: as many experts as a launch has and a number that is no multiple of four,
# most without rows, the first and the last with some, whole tiles and a row more
@pytest.mark.parametrize("ne,some", [(256, [0, 3, 4, 63, 64, 127, 200, 255]), (253, [2, 7, 128, 252]), (5, [4]), (3, [0])])
def test_groups_far_apart_bit_for_bit(dev, ne, some):
    from illatio_amd import hip, ds4f
    rng = synth.make_rng(ne)
    rows, cols = 128, 256
    counts = np.zeros(ne, np.uint32)
    counts[some] = [(1, 129, 128, 257)[i % 4] for i in range(len(some))]
    total = int(counts.sum())
    bases = (np.cumsum(counts) - counts).astype(np.uint32)
    rb = synth.row_bytes(synth.Q2_K, cols)
    w = synth.weights(synth.Q2_K, 3 * rows, cols, rng).reshape(3, rows, rb)
    x = synth.activations((total, cols), rng)
    wb, xb, y = hip.hip_upload_new(dev, w), hip.hip_upload_new(dev, x), hip.hip_alloc(dev, 4 * total * rows)
    ptrs = hip.hip_upload_new(dev, np.array([wb.ptr + z % 3 * rows * rb for z in range(ne)], np.uint64))
    cb, bb = hip.hip_upload_new(dev, counts), hip.hip_upload_new(dev, bases)
    xq, xd, xs = ds4f._q8k(dev, xb, total * cols)
    hip.launch(dev, "d4_mm_id_q2_k", (1, 1, ne), 128, [cols, rows, rb, cols, rows, hip.I64(0), ptrs, cb, bb, xq, y, xd, xs, hip.I64(total)])
    got = hip.hip_floats(y, total * rows).reshape(total, rows)
    for z in some:
        at = slice(int(bases[z]), int(bases[z] + counts[z]))
        want = orc.matmul(synth.Q2_K, w[z % 3], rows, cols, x[at], nthreads=8).reshape(-1, rows)
        assert np.array_equal(bits(got[at]), bits(want)), (z, np.argwhere(bits(got[at]) != bits(want))[:5])
    for b in (wb, xb, y, ptrs, cb, bb, xq, xd, xs):
        hip.hip_free(b)


# experts' matrices on two-byte boundaries: by the slot's address, by the offset into it, and both (together a multiple of four)
@pytest.mark.parametrize("rows,cols", [(128, 256), (161, 1280)])
@pytest.mark.parametrize("at,add", [(2, 0), (0, 2), (2, 2), (6, 8)])
def test_groups_of_q2_k_on_even_addresses_bit_for_bit(dev, rows, cols, at, add):
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(rows + cols + at + add)
    counts = np.array([1, 0, 33, 64, 65, 129], np.uint32)
    ne, total = len(counts), int(counts.sum())
    bases = (np.cumsum(counts) - counts).astype(np.uint32)
    rb = synth.row_bytes(synth.Q2_K, cols)
    w = synth.weights(synth.Q2_K, ne * rows, cols, rng).reshape(ne, rows, rb)
    x = synth.activations((total, cols), rng)
    step = rows * rb + 16                             # (a slot ends 16 bytes before the next one: a multiple of four)
    host = np.zeros(at + add + ne * step, np.uint8)
    for z in range(ne):
        host[at + add + z * step:][:rows * rb] = w[z].ravel()
    wb, xb, y = hip.hip_upload_new(dev, host), hip.hip_upload_new(dev, x), hip.hip_alloc(dev, 4 * total * rows)
    ptrs = hip.hip_upload_new(dev, np.array([wb.ptr + at + z * step for z in range(ne)], np.uint64))
    cb, bb = hip.hip_upload_new(dev, counts), hip.hip_upload_new(dev, bases)
    xq, xd, xs = ds4f._q8k(dev, xb, total * cols)
    hip.launch(dev, "d4_mm_id_q2_k", (1, 1, ne), 128, [cols, rows, rb, cols, rows, hip.I64(add), ptrs, cb, bb, xq, y, xd, xs, hip.I64(total)])
    got = hip.hip_floats(y, total * rows).reshape(total, rows)
    for z in range(ne):
        if counts[z] == 0:
            continue
        part = slice(int(bases[z]), int(bases[z] + counts[z]))
        want = orc.matmul(synth.Q2_K, w[z], rows, cols, x[part], nthreads=8).reshape(-1, rows)
        assert np.array_equal(bits(got[part]), bits(want)), (z, np.argwhere(bits(got[part]) != bits(want))[:5])
    for b in (wb, xb, y, ptrs, cb, bb, xq, xd, xs):
        hip.hip_free(b)
