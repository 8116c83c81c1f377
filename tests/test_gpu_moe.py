"""GPU parity of the MoE expert path's kernels against the CPU oracle: routing (indices
and weights bit for bit), the grouping of (token, slot) rows by expert, the gather, the
gated activation, and one token's whole routed + shared FFN (DK-FFN-TAIL's sequence)."""
import numpy as np
import pytest

import oracle_lib as orc
from illatio_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from illatio_amd import hip
    return hip.open_hip(0)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("ne,nu,n", [(256, 6, 64), (16, 3, 5), (64, 8, 33)])
def test_route_indices_and_weights_bit_exact(dev, ne, nu, n):
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(ne + n)
    logits = synth.zipf_router_logits(n, ne, rng)
    logits[1, :] = 0.25                                    # every expert equal: the first nu win, in order
    logits[2, ne // 2:] = logits[2, 0]                     # many exact ties
    logits[3, :4] = [30.0, -30.0, 21.0, -21.0]             # softplus's outer branches
    for bias in (None, (rng.standard_normal(ne) * 0.05).astype(np.float32)):
        lb = hip.hip_upload_new(dev, logits)
        bb = None if bias is None else hip.hip_upload_new(dev, bias)
        sel, w = ds4f.route(dev, lb, n, ne, nu, 1.5, bb)
        gs = hip.hip_download(sel, np.uint32, n * nu).reshape(n, nu)
        gw = hip.hip_floats(w, n * nu).reshape(n, nu)
        for t in range(n):
            ws, ww = orc.route(logits[t], nu, 1.5, bias)
            assert gs[t].tolist() == ws.tolist(), (t, gs[t], ws)
            assert np.array_equal(bits(gw[t]), bits(ww)), t
        if bias is None:
            assert gs[1].tolist() == list(range(nu))
        for b in (lb, bb, sel, w):
            hip.hip_free(b)


@pytest.mark.parametrize("ne,nu,n,vocab", [(256, 6, 70, 500), (16, 3, 5, 9), (64, 8, 33, 129280)])
def test_route_from_the_hash_table_bit_exact(dev, ne, nu, n, vocab):
    """A hash layer's routing (d4-route's tid2eid branch, ds4f.lisp:961-963; d4_route with hash = 1,
    cuda/ds4f_chunk.cu:439-440): each token's experts are its row of the table as it stands -- unsorted, an expert
    named twice staying twice, the bias ignored -- and the weights are the oracle's bit for bit."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(ne + n + 5)
    logits = synth.zipf_router_logits(n, ne, rng)
    logits[1, :] = -40.0                                   # the sum of the probabilities under its floor
    logits[2, :4] = [30.0, -30.0, 21.0, -21.0]             # softplus's outer branches
    table = np.stack([rng.permutation(ne)[:nu] for _ in range(vocab)]).astype(np.int32)
    table[vocab - 1, :] = ne - 1                           # one expert in every slot
    table[0, :] = np.arange(nu)[::-1]
    table[1, :4 if nu > 3 else nu] = [0, 1, 2, 3][:4 if nu > 3 else nu]
    tokens = rng.integers(0, vocab, n).astype(np.uint32)
    tokens[0], tokens[1], tokens[2] = vocab - 1, 0, 1
    lb, tb, kb = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, table), hip.hip_upload_new(dev, tokens)
    bias = (rng.standard_normal(ne) * 0.5).astype(np.float32)
    bb = hip.hip_upload_new(dev, bias)
    for b in (None, bb):                                   # the bias plays no part on a hash layer
        sel, w = ds4f.route(dev, lb, n, ne, nu, 1.5, b, tid2eid=tb, tokens=kb)
        gs = hip.hip_download(sel, np.uint32, n * nu).reshape(n, nu)
        gw = hip.hip_floats(w, n * nu).reshape(n, nu)
        for t in range(n):
            ws, ww = orc.route_table(logits[t], table, tokens[t], nu, 1.5)
            assert gs[t].tolist() == ws.tolist() == table[tokens[t]].tolist(), (t, gs[t], ws)
            assert np.array_equal(bits(gw[t]), bits(ww)), t
        hip.hip_free(sel); hip.hip_free(w)
    # the slot-block launch by the reference's name refuses a hash layer without its table
    with pytest.raises(hip.HipError):
        hip.launch(dev, "d4_route", n, ne, [ne, nu, 1, 1.5, 0, lb, None, None, None, lb, lb], shared=0)
    with pytest.raises(ValueError):
        ds4f.route(dev, lb, n, ne, nu, 1.5, tid2eid=tb)
    for b in (lb, tb, kb, bb):
        hip.hip_free(b)


def test_hash_layer_decode_step_bit_exact(dev):
    """One token's FFN on a hash layer with nothing going through the host: d4_route leaves the token's table row on
    the device, the experts' launches index the slot table by it, and the step has the bits of d4-routed! +
    d4-shared! on the oracle's table row."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(77)
    ne, nu, d, ff, clamp, vocab = 16, 3, 512, 256, 7.0, 40
    gate, up, down, sg, su, sd = _moe_weights(rng, ne, d, ff)
    pool = ds4f.ExpertPool(dev, ne, d, ff, gate, up, down)
    sh = ds4f.SharedExpert(dev, d, ff, sg, su, sd)
    logits, norm = synth.activations(ne, rng), synth.activations(d, rng)
    table = np.stack([rng.permutation(ne)[:nu] for _ in range(vocab)]).astype(np.int32)
    token = np.array([23], np.uint32)
    lb, tb, kb, nb = (hip.hip_upload_new(dev, a) for a in (logits, table, token, norm))
    wsel, ww = orc.route_table(logits, table, 23, nu, 1.5)
    assert sorted(wsel.tolist()) != sorted(orc.route(logits, nu, 1.5)[0].tolist())
    routed, _ = orc.moe_routed(gate, up, down, d, ff, wsel, ww, clamp, norm)
    shared = orc.moe_shared(sg, su, sd, d, ff, clamp, norm)
    want = (routed + shared).astype(np.float32)           # d4-ffn's last step (ds4f.lisp:980-992): the ordered sum, then the shared row
    moe = ds4f.ffn_step_device(dev, pool, sh, lb, nb, ne, nu, 1.5, clamp, tid2eid=tb, tokens=kb)
    got = hip.hip_floats(moe, d)
    assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()
    for b in (lb, tb, kb, nb, moe):
        hip.hip_free(b)
    pool.free(); sh.free()


def test_route_with_nan_and_masked_scores(dev):
    """Scores that are NaN (an overflow upstream) and experts masked by a bias of minus infinity: the
    CPU's insertion (ds4f.lisp:966-972) compares NaNs false both ways, so its result depends on the
    insertion order; the kernel gives the same indices (NU different experts below NE in every
    case, which the kernels downstream index tables with) and the same weights, NaN where the CPU's
    are NaN."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(99)
    ne, nu, n = 256, 6, 12
    logits = synth.activations((n, ne), rng)
    logits[0, :] = np.nan                                  # every score NaN: the first nu experts, in order
    logits[1, 3] = np.nan                                  # one NaN among the first nu inserted
    logits[2, 100] = np.nan                                # one NaN later on: never inserted
    logits[3, ::2] = np.nan
    logits[4, :ne - 3] = np.nan                            # fewer numbers than slots
    logits[5, [0, 1, 2, 3, 4, 5]] = [np.nan, 9.0, np.nan, 8.0, 7.0, np.nan]
    logits[6, 7] = np.inf
    logits[7, :] = -200.0                                  # softplus underflows to zero: all tied at 0, the sum floored
    bias = np.zeros(ne, np.float32)
    bias[10:200] = -np.inf                                 # masked experts
    for b in (None, bias):
        lb = hip.hip_upload_new(dev, logits)
        bb = None if b is None else hip.hip_upload_new(dev, b)
        sel, w = ds4f.route(dev, lb, n, ne, nu, 1.5, bb)
        gs = hip.hip_download(sel, np.uint32, n * nu).reshape(n, nu)
        gw = hip.hip_floats(w, n * nu).reshape(n, nu)
        for t in range(n):
            ws, ww = orc.route(logits[t], nu, 1.5, b)
            assert gs[t].tolist() == ws.tolist(), (t, gs[t], ws)
            assert len(set(gs[t].tolist())) == nu and int(gs[t].max()) < ne
            assert np.array_equal(np.isnan(gw[t]), np.isnan(ww)), t
            ok = ~np.isnan(ww)
            assert np.array_equal(bits(gw[t][ok]), bits(ww[ok])), t
        if b is None:
            assert gs[0].tolist() == list(range(nu)) and gs[7].tolist() == list(range(nu))
        for x in (lb, bb, sel, w):
            hip.hip_free(x)


@pytest.mark.parametrize("n,ne,nu", [(1, 1, 1), (1, 1024, 64), (16, 64, 64), (341, 5, 3), (1025, 256, 1), (1366, 1000, 3), (8192, 2, 8), (8193, 256, 8)])
def test_rows_grouped_and_quantized_into_their_places(dev, n, ne, nu):
    """The grouping's one launch (the last size takes the four: as many rows more than 65,536), around a workgroup's 1,024 rows, with
    experts that nobody chose; and the tokens' blocks in each of their rows against quant_q8k's, gathered."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(n + ne + nu)
    rows, d = n * nu, 512
    sh = np.sort(rng.integers(0, max(1, ne * 3 // 4), rows)).astype(np.uint32) if n == 341 else (rng.random(rows) ** 3 * ne).astype(np.uint32)
    wh, xh = rng.standard_normal(rows).astype(np.float32), synth.activations((n, d), rng)
    xh[0, :256] = 0.0
    sel, w, x = hip.hip_upload_new(dev, sh), hip.hip_upload_new(dev, wh), hip.hip_upload_new(dev, xh)
    g = ds4f.group_rows(dev, sel, w, n, ne, nu)
    get = lambda k, c: hip.hip_download(g[k], np.uint32, c)
    counts, bases, rmap, smap = get("counts", ne), get("bases", ne), get("rmap", rows), get("smap", rows)
    assert np.array_equal(counts, np.bincount(sh, minlength=ne)) and np.array_equal(bases, np.cumsum(counts) - counts)
    assert np.array_equal(np.sort(smap), np.arange(rows)) and np.array_equal(rmap[smap], np.arange(rows) // nu)
    assert np.array_equal(smap, bases[sh] + get("rank", rows)) and ((smap >= bases[sh]) & (smap < bases[sh] + counts[sh])).all()
    assert np.array_equal(hip.hip_floats(g["wrow"], rows)[smap], wh)
    xq, xd, xs = ds4f._q8k(dev, x, n * d)
    oq, od = hip.hip_alloc(dev, rows * d), hip.hip_alloc(dev, 4 * rows * d // 256)
    hip.launch(dev, "d4_quant_q8k_rows", (n * d // 256 + 3) // 4, 256, [d, n, nu, x, g["smap"], oq, od])
    assert np.array_equal(hip.hip_download(oq, np.int8, rows * d).reshape(rows, d), hip.hip_download(xq, np.int8, n * d).reshape(n, d)[rmap])
    assert np.array_equal(hip.hip_floats(od, rows * d // 256).reshape(rows, -1), hip.hip_floats(xd, n * d // 256).reshape(n, -1)[rmap])
    for b in [sel, w, x, xq, xd, xs, oq, od] + list(g.values()):
        hip.hip_free(b)


def test_group_rows_invariants_and_gather(dev):
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(5)
    n, ne, nu, d = 300, 256, 6, 64
    logits = synth.zipf_router_logits(n, ne, rng)
    lb = hip.hip_upload_new(dev, logits)
    sel, w = ds4f.route(dev, lb, n, ne, nu, 1.5)
    g = ds4f.group_rows(dev, sel, w, n, ne, nu)
    rows = n * nu
    hs = hip.hip_download(sel, np.uint32, rows)
    hw = hip.hip_floats(w, rows)
    counts = hip.hip_download(g["counts"], np.uint32, ne)
    bases = hip.hip_download(g["bases"], np.uint32, ne)
    rmap = hip.hip_download(g["rmap"], np.uint32, rows)
    smap = hip.hip_download(g["smap"], np.uint32, rows)
    wrow = hip.hip_floats(g["wrow"], rows)
    assert np.array_equal(counts, np.bincount(hs, minlength=ne))
    assert np.array_equal(bases, np.concatenate([[0], np.cumsum(counts)[:-1]]))
    assert sorted(smap.tolist()) == list(range(rows))                      # a permutation
    assert np.array_equal(rmap[smap], np.arange(rows) // nu)               # row -> its token
    assert np.array_equal(bits(wrow[smap]), bits(hw))
    e_of_row = np.searchsorted(np.cumsum(counts), np.arange(rows), side="right")
    assert np.array_equal(e_of_row[smap], hs)                              # each row inside its expert's range
    src = synth.activations((n, d), rng)
    sb = hip.hip_upload_new(dev, src)
    x = hip.hip_alloc(dev, 4 * rows * d)
    hip.launch(dev, "d4_gather_rows", (rows * d + 255) // 256, 256, [d, rows, sb, g["rmap"], x])
    assert np.array_equal(bits(hip.hip_floats(x, rows * d).reshape(rows, d)), bits(src[rmap]))
    # the slot-ordered sum over rows, with the shared expert's rows added after
    down = synth.activations((rows, d), rng)
    shared = synth.activations((n, d), rng)
    db, shb, moe = hip.hip_upload_new(dev, down), hip.hip_upload_new(dev, shared), hip.hip_alloc(dev, 4 * n * d)
    hip.launch(dev, "d4_moe_sum_rows", (n * d + 255) // 256, 256, [d, nu, n, db, g["smap"], shb, moe])
    want = np.zeros((n, d), np.float32)
    for s in range(nu):
        want = want + down[smap.reshape(n, nu)[:, s]]
    want = want + shared
    assert np.array_equal(bits(hip.hip_floats(moe, n * d).reshape(n, d)), bits(want))
    for b in [lb, sel, w, sb, x, db, shb, moe] + list(g.values()):
        hip.hip_free(b)


@pytest.mark.parametrize("clamp", [0.0, 0.7])
def test_swiglu_w_matches_cpu_silu(dev, clamp):
    from illatio_amd import hip
    rng = synth.make_rng(9)
    n, ff = 6, 512
    g = (synth.activations((n, ff), rng) * 3).astype(np.float32)
    u = synth.activations((n, ff), rng)
    g[0, :6] = [0.0, -0.0, 25.0, -25.0, 88.0, -100.0]
    w = (rng.random(n, dtype=np.float32) + 0.1).astype(np.float32)
    gb, ub, wb = (hip.hip_upload_new(dev, a) for a in (g, u, w))
    mid, xq, xs = hip.hip_alloc(dev, 4 * n * ff), hip.hip_alloc(dev, n * ff), hip.hip_alloc(dev, 4 * n * ff // 32)
    hip.launch(dev, "d4_swiglu_w", (n * ff + 255) // 256, 256, [n, ff, float(clamp), gb, ub, wb, mid, xq, xs])
    got = hip.hip_floats(mid, n * ff).reshape(n, ff)
    want = np.empty_like(got)
    for r in range(n):
        for j in range(ff):
            gv, uv = g[r, j], u[r, j]
            if clamp > 1e-6:
                gv = min(gv, np.float32(clamp)); uv = max(np.float32(-clamp), min(uv, np.float32(clamp)))
            want[r, j] = (np.float32(orc.silu(gv)) * uv) * w[r]
    assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()
    wq, ws = orc.quantize_q8(want, f16_scale=False)
    assert np.array_equal(hip.hip_download(xq, np.int8, n * ff), wq)
    assert np.array_equal(bits(hip.hip_floats(xs, n * ff // 32)), bits(ws))
    for b in (gb, ub, wb, mid, xq, xs):
        hip.hip_free(b)


def _moe_weights(rng, ne, d, ff):
    gate = synth.weights(synth.IQ2_XXS, ne * ff, d, rng)
    up = synth.weights(synth.IQ2_XXS, ne * ff, d, rng)
    down = synth.weights(synth.Q2_K, ne * d, ff, rng)
    sg = synth.weights(synth.Q8_0, ff, d, rng)
    su = synth.weights(synth.Q8_0, ff, d, rng)
    sd = synth.weights(synth.Q8_0, d, ff, rng)
    return gate, up, down, sg, su, sd


@pytest.mark.parametrize("ne,d,ff,nu,clamp", [(8, 512, 256, 3, 0.0), (8, 512, 256, 3, 0.05), (12, 4096, 2048, 6, 0.0),
                                                (12, 2048, 1024, 9, 0.0),       # (nine slots: the sum as a launch of its own)
                                                (12, 2048, 1024, 8, 0.05)])     # (eight: the most the last product adds itself)
def test_moe_decode_step_bit_exact(dev, ne, d, ff, nu, clamp):
    """the benchmark's config 4's sequence at a reduced expert count (12 resident experts of the
    full 4096 x 2048 shape), and a small shape with the clamp on: route -> gate/up -> gated
    activation -> per-slot Q8_K -> down -> ordered sum + shared expert.  In the one-call step the sum rides on the
    shared expert's down launch at the large shape; the small one and the one with nine slots launch it."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(ne * 1000 + d)
    gate, up, down, sg, su, sd = _moe_weights(rng, ne, d, ff)
    pool = ds4f.ExpertPool(dev, ne, d, ff, gate, up, down)
    sh = ds4f.SharedExpert(dev, d, ff, sg, su, sd)
    for trial in range(2):
        norm = synth.activations(d, rng)
        logits = synth.activations(ne, rng)
        want, wsel, ww = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, clamp, logits, norm)
        lb, nb = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, norm)
        sel, w = ds4f.route(dev, lb, 1, ne, nu, 1.5)
        hsel, hw = hip.hip_download(sel, np.uint32, nu), hip.hip_floats(w, nu)
        assert hsel.tolist() == wsel.tolist() and np.array_equal(bits(hw), bits(ww))
        sout = ds4f.ffn_shared(dev, sh, nb, clamp)
        assert np.array_equal(bits(hip.hip_floats(sout, d)), bits(orc.moe_shared(sg, su, sd, d, ff, clamp, norm)))
        keep = {}
        moe = ds4f.ffn_tail(dev, pool, hsel, hw, nb, sout, clamp, keep)
        _, wmid = orc.moe_routed(gate, up, down, d, ff, wsel, ww, clamp, norm)
        assert np.array_equal(bits(keep["mid"]), bits(wmid)), np.abs(keep["mid"] - wmid).max()
        got = hip.hip_floats(moe, d)
        assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()
        # the same step in five launches (activations quantized inside the product kernels, gate/up/gated activation fused)
        fused = ds4f.ffn_step_fused(dev, pool, sh, hsel, hw, nb, clamp)
        got = hip.hip_floats(fused, d)
        assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()
        # and with the routing left on the device (six launches, no host round trip)
        ondev = ds4f.ffn_step_device(dev, pool, sh, lb, nb, ne, nu, 1.5, clamp)
        got = hip.hip_floats(ondev, d)
        assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()
        # the same step queued by one call into the library (the routing carried along by the shared expert's gate/up
        # launch at the large shape), its intermediates in a caller's workspace
        out = hip.hip_alloc(dev, 4 * d)
        ds4f.ffn_step_call(dev, pool, sh, lb, nb, out, ne, nu, 1.5, clamp)
        got = hip.hip_floats(out, d)
        assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()
        for b in (lb, nb, sel, w, sout, moe, fused, ondev, out):
            hip.hip_free(b)
    # a bias on the scores, a workspace used twice, and one that is too small
    bias = (rng.standard_normal(ne) * 0.5).astype(np.float32)
    norm, logits = synth.activations(d, rng), synth.activations(ne, rng)
    want, wsel, _ = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, clamp, logits, norm, bias=bias)
    assert wsel.tolist() != orc.route(logits, nu, 1.5)[0].tolist()          # the bias changes the choice
    lb, nb, bb, out = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, norm), hip.hip_upload_new(dev, bias), hip.hip_alloc(dev, 4 * d)
    ws = hip.hip_alloc(dev, ds4f.step_workspace_bytes(nu, d, ff), zero=False)
    for _ in range(2):
        ds4f.ffn_step_call(dev, pool, sh, lb, nb, out, ne, nu, 1.5, clamp, bias=bb, wsbuf=ws)
        assert np.array_equal(bits(hip.hip_floats(out, d)), bits(want))
    small = hip.DBuf(ws.ptr, ws.bytes - 256, dev)
    with pytest.raises(hip.HipError):
        ds4f.ffn_step_call(dev, pool, sh, lb, nb, out, ne, nu, 1.5, clamp, wsbuf=small)
    # scores that are NaN (the routing's slow branch, here inside the launch that carries the routing along at the
    # large shape): the step ends normally, NaN where the CPU path's result is NaN and its bits elsewhere
    for where in ([1], list(range(0, ne, 2)), list(range(ne))):
        lg = logits.copy(); lg[where] = np.nan
        want, _, _ = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, clamp, lg, norm)
        hip.hip_upload_vector(lb, lg)
        ds4f.ffn_step_call(dev, pool, sh, lb, nb, out, ne, nu, 1.5, clamp, wsbuf=ws)
        got = hip.hip_floats(out, d)
        assert np.array_equal(np.isnan(got), np.isnan(want)), where
        ok = ~np.isnan(want)
        assert np.array_equal(bits(got[ok]), bits(want[ok])), where
    for b in (lb, nb, bb, out, ws):
        hip.hip_free(b)
    pool.free(); sh.free()


def test_experts_read_through_from_pinned_host_memory(dev):
    """Experts without a place in HBM: their matrices stay in pinned, mapped host memory and the table of slots points
    there (the reference's read-through, ds4f.cu:742-760, cuda-ds4f.lisp:553-640); their device slots are zeroed, so the
    decode step's bits -- equal to the all-resident pool's and the oracle's -- can only come from host memory."""
    from illatio_amd import ds4f, hip
    ne, d, ff, nu, clamp = 8, 512, 256, 3, 0.05
    rng = synth.make_rng(77)
    gate, up, down, sg, su, sd = _moe_weights(rng, ne, d, ff)
    sh = ds4f.SharedExpert(dev, d, ff, sg, su, sd)
    norm, logits = synth.activations(d, rng), synth.activations(ne, rng)
    want, wsel, _ = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, clamp, logits, norm)
    on_host = [int(wsel[0]), int(wsel[2]), int(next(e for e in range(ne) if e not in wsel.tolist()))]      # two that are chosen, one that is not
    pool = ds4f.ExpertPool(dev, ne, d, ff, gate, up, down, host_experts=on_host)
    lb, nb, out = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, norm), hip.hip_alloc(dev, 4 * d)
    ds4f.ffn_step_call(dev, pool, sh, lb, nb, out, ne, nu, 1.5, clamp)
    assert np.array_equal(bits(hip.hip_floats(out, d)), bits(want))
    for b in (lb, nb, out):
        hip.hip_free(b)
    pool.free(); sh.free()


@pytest.mark.parametrize("ne,d,ff,nu,n,clamp", [(8, 512, 256, 3, 9, 0.05), (12, 4096, 2048, 6, 4, 0.0)])
def test_moe_short_pass_of_a_few_tokens_bit_exact(dev, ne, d, ff, nu, n, clamp):
    """A speculative step's verification (cuda-ds4f-spec.lisp:30-100): the FFN of up to nine tokens
    at once, experts shared between tokens, every token with the bits of its own decode step."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(ne * 77 + n)
    gate, up, down, sg, su, sd = _moe_weights(rng, ne, d, ff)
    pool = ds4f.ExpertPool(dev, ne, d, ff, gate, up, down)
    sh = ds4f.SharedExpert(dev, d, ff, sg, su, sd)
    norm = synth.activations((n, d), rng)
    logits = synth.activations((n, ne), rng)
    logits[1] = logits[0]                     # two tokens on the same experts
    lb, nb = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, norm)
    # a launch slot per (token, slot) row in token order; the rows grouped by expert; the reference's own launches
    # with counts and bases (cuda-ds4f-spec.lisp:82-88)
    for grouped in (False, True, "counts"):
        moe = ds4f.ffn_small(dev, pool, sh, lb, nb, n, ne, nu, 1.5, clamp, grouped=grouped)
        got = hip.hip_floats(moe, n * d).reshape(n, d)
        for t in range(n):
            want, _, _ = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, clamp, logits[t], norm[t])
            assert np.array_equal(bits(got[t]), bits(want)), (grouped, t, np.abs(got[t] - want).max())
        hip.hip_free(moe)
    for b in (lb, nb):
        hip.hip_free(b)
    pool.free(); sh.free()


# an expert's rows from one to nine (groups of three and of two of them, whole and broken), more than 64 rows in all, every
# width that the shared decoding takes at its ends, steps with lanes left over, fewer weight rows than a workgroup's, and widths
# past it that take a row at a time, more experts than one launch routes beside the rounding
@pytest.mark.parametrize("ne,d,ff,nu,n", [(3, 256, 1024, 3, 9), (16, 512, 512, 8, 9), (70, 1024, 256, 1, 9), (8, 256, 256, 2, 1),
                                          (9, 4096, 256, 4, 5), (5, 256, 4096, 4, 7), (8, 768, 2816, 2, 4), (6, 2304, 1536, 3, 4),
                                          (4, 4352, 256, 2, 3), (4, 256, 4352, 2, 3), (600, 256, 256, 3, 2)])
def test_moe_short_pass_over_groups_and_widths(dev, ne, d, ff, nu, n):
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(ne * 131 + d + ff + n)
    gate, up, down, sg, su, sd = _moe_weights(rng, ne, d, ff)
    pool = ds4f.ExpertPool(dev, ne, d, ff, gate, up, down)
    sh = ds4f.SharedExpert(dev, d, ff, sg, su, sd)
    norm = synth.activations((n, d), rng)
    norm[0, 3::64] = 0.0
    norm[-1, 17], norm[-1, 40] = 50.0, -50.0            # a block's largest magnitude with both signs
    if n > 2:
        norm[1] = 0.0
    logits = synth.activations((n, ne), rng)
    lb, nb = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, norm)
    moe = ds4f.ffn_small(dev, pool, sh, lb, nb, n, ne, nu, 1.5, 0.0)
    got = hip.hip_floats(moe, n * d).reshape(n, d)
    for t in range(n):
        want, _, _ = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, 0.0, logits[t], norm[t])
        assert np.array_equal(bits(got[t]), bits(want)), (t, np.abs(got[t] - want).max())
    for b in (lb, nb, moe):
        hip.hip_free(b)
    pool.free(); sh.free()


# the shared expert's rows beside the routed experts': two rows a wave at their last number of tokens, one at its first, a last step
# of columns that is a quarter and three quarters of one
@pytest.mark.parametrize("ne,d,ff,nu,n", [(4, 1280, 512, 2, 6), (5, 512, 1792, 2, 6), (4, 1280, 768, 3, 7), (3, 3840, 256, 1, 2)])
def test_moe_short_pass_with_the_shared_expert_beside(dev, ne, d, ff, nu, n):
    test_moe_short_pass_over_groups_and_widths(dev, ne, d, ff, nu, n)


@pytest.mark.parametrize("d,ff,n,clamp", [(512, 256, 37, 0.05), (4096, 2048, 130, 0.0)])
def test_shared_expert_over_a_chunk_bit_exact(dev, d, ff, n, clamp):
    """The shared expert of a chunk through d4_mm_q8_0 (DK-FFN-HEAD-CHUNK, cuda-ds4f-prefill.lisp:294-298): every
    token's row has d4-shared!'s bits (ds4f.lisp:1039-1048), and the chunk's routed experts summed with it give
    each token its own decode step."""
    from illatio_amd import ds4f, hip
    rng = synth.make_rng(d + n)
    ne, nu = 8, 3
    gate, up, down, sg, su, sd = _moe_weights(rng, ne, d, ff)
    pool = ds4f.ExpertPool(dev, ne, d, ff, gate, up, down)
    sh = ds4f.SharedExpert(dev, d, ff, sg, su, sd)
    norms = synth.activations((n, d), rng)
    logits = synth.zipf_router_logits(n, ne, rng)
    lb, nb = hip.hip_upload_new(dev, logits), hip.hip_upload_new(dev, norms)
    sout = ds4f.ffn_shared_chunk(dev, sh, nb, n, clamp)
    got = hip.hip_floats(sout, n * d).reshape(n, d)
    sample = sorted({0, 1, n // 2, n - 1})
    for t in sample:
        want = orc.moe_shared(sg, su, sd, d, ff, clamp, norms[t], nthreads=8)
        assert np.array_equal(bits(got[t]), bits(want)), (t, np.abs(got[t] - want).max())
    moe = ds4f.ffn_routed_chunk(dev, pool, lb, nb, sout, n, ne, nu, 1.5, clamp)
    out = hip.hip_floats(moe, n * d).reshape(n, d)
    for t in sample:
        want, _, _ = orc.moe_token(gate, up, down, sg, su, sd, d, ff, ne, nu, 1.5, clamp, logits[t], norms[t], nthreads=8)
        assert np.array_equal(bits(out[t]), bits(want)), (t, np.abs(out[t] - want).max())
    for b in (lb, nb, sout, moe):
        hip.hip_free(b)
    pool.free(); sh.free()
