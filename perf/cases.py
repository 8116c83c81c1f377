"""The work that a user of this package has it do, as cases that can be measured: a decoder's turns (a prompt, greedy
tokens) at the two model shapes the benchmark names, single quantized products, and the MoE layer's decode step, short
pass and prompt chunk -- each through the functions of illatio_amd that a program calls for it.

listed() is the cases themselves and draw() gives more of the same ranges; prepare() makes what a program holds before the
call (weights on the device, inputs, a workspace), run() is one pass, work() what a pass cannot do without and
tolerance() how far another correct implementation may be from it.  Weights and inputs are synthetic and seeded.
"""
import numpy as np
import torch

from illatio_amd import dense, ds4f, hip, model, synth

FORMATS = {"q8_0": synth.Q8_0, "q4_k": synth.Q4_K, "q6_k": synth.Q6_K}

# The benchmark's two decoders: hidden width, feed-forward width, query heads, key/value heads, head width, layers, vocabulary.
SHAPES = {
    "qwen3-4b": {"d": 2560, "ffn": 9728, "nh": 32, "nkv": 8, "hd": 128, "nl": 36, "vocab": 151936, "q8": False},
    "qwen2.5-0.5b": {"d": 896, "ffn": 4864, "nh": 14, "nkv": 2, "hd": 64, "nl": 24, "vocab": 151936, "q8": True},
}
ROUTE_SCALE = 1.5          # the routed experts' weight scale of the benchmark's MoE configurations


def listed():
    return [
        # one decode product on one token's floats: the smallest call a host makes by itself, over as soon as it is queued
        {"name": "product-q8_0-896x4864", "kind": "product", "fmt": "q8_0", "rows": 896, "cols": 4864, "glu": False, "norm": False},
        # an answer being written, a conversation of ordinary length behind it: what a chat spends its time on
        {"name": "decode-4b-600", "kind": "turn", "model": "qwen3-4b", "ctx": 600, "prompt": 1, "tokens": 16},
        # the same far into a long document
        {"name": "decode-4b-4100", "kind": "turn", "model": "qwen3-4b", "ctx": 4100, "prompt": 1, "tokens": 16},
        # a whole turn on the small Q8_0 model: a prompt of a paragraph and the first words of the answer
        {"name": "turn-0.5b-301", "kind": "turn", "model": "qwen2.5-0.5b", "ctx": 0, "prompt": 301, "tokens": 16},
        # the user's next message in a conversation: a sentence on top of what the caches hold
        {"name": "prompt-4b-21", "kind": "turn", "model": "qwen3-4b", "ctx": 300, "prompt": 21, "tokens": 0},
        # the benchmark's prompt
        {"name": "prompt-4b-512", "kind": "turn", "model": "qwen3-4b", "ctx": 0, "prompt": 512, "tokens": 0},
        # a document: more than one chunk of tokens, and not a whole number of any tile
        {"name": "prompt-4b-2500", "kind": "turn", "model": "qwen3-4b", "ctx": 0, "prompt": 2500, "tokens": 0},
        # a prefill product on the bf16 matrix cores from the quantized matrix, the float activations rounded inside the pass
        {"name": "gemm-bf16-q6_k-4096", "kind": "gemm", "fmt": "q6_k", "rows": 17408, "cols": 5120, "tokens": 4096, "path": "bf16"},
        # one token through a MoE layer past its router, 256 experts resident
        {"name": "moe-step-256", "kind": "moe", "op": "step", "ne": 256, "nu": 6, "d": 4096, "ff": 2048, "tokens": 1, "clamp": 0.0},
        # a speculative step's tokens verified together
        {"name": "moe-small-5", "kind": "moe", "op": "small", "ne": 256, "nu": 6, "d": 4096, "ff": 2048, "tokens": 5, "clamp": 7.0},
        # a prompt's chunk through the layer with the CPU path's bits, an ordinary number of tokens
        {"name": "moe-chunk-exact-1000", "kind": "moe", "op": "chunk", "ne": 256, "nu": 6, "d": 4096, "ff": 2048, "tokens": 1000, "clamp": 0.0},
        # the largest chunk, on the bf16 matrix cores
        {"name": "moe-chunk-bf16-4096", "kind": "moe", "op": "chunk-bf16", "ne": 256, "nu": 6, "d": 4096, "ff": 2048, "tokens": 4096, "clamp": 0.0},
    ]


def _log(rng, lo, hi):
    """A whole number from LO to HI, spread over the logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["product", "decode", "decode", "prompt", "prompt", "turn", "gemm", "moe", "moe"])
    if kind == "product":
        fmt = rng.choice(sorted(FORMATS))
        unit = 32 if fmt == "q8_0" else 256
        cols = max(unit, _log(rng, 512, 9728) // unit * unit)
        return {"kind": "product", "fmt": fmt, "rows": _log(rng, 128, 20000), "cols": cols, "glu": rng.random() < 0.3, "norm": rng.random() < 0.3}
    if kind in ("decode", "prompt", "turn"):
        m = rng.choice(sorted(SHAPES))
        if kind == "decode":
            return {"kind": "turn", "model": m, "ctx": _log(rng, 16, 8000), "prompt": 1, "tokens": rng.randint(8, 16)}
        n = _log(rng, 2, 2500)
        ctx = _log(rng, 16, 2000) if n < 500 and rng.random() < 0.5 else 0
        return {"kind": "turn", "model": m, "ctx": ctx, "prompt": n, "tokens": 0 if kind == "prompt" else rng.randint(4, 16)}
    if kind == "gemm":
        fmt = rng.choice(["q4_k", "q6_k"])
        path = rng.choice(["exact", "bf16", "bf16-resident"])
        return {"kind": "gemm", "fmt": fmt, "rows": _log(rng, 512, 17408), "cols": _log(rng, 1024, 9728) // 256 * 256, "tokens": _log(rng, 8, 4096), "path": path}
    op = rng.choice(["step", "small", "chunk", "chunk-bf16"])
    tokens = {"step": 1, "small": rng.randint(2, 9)}.get(op) or _log(rng, 24, 4096)
    return {"kind": "moe", "op": op, "ne": rng.choice([32, 64, 128, 256]), "nu": rng.randint(2, 8), "d": rng.choice([2048, 4096]),
            "ff": rng.choice([1024, 1536, 2048]), "tokens": tokens, "clamp": rng.choice([0.0, 7.0])}


# ---- what a program holds ---------------------------------------------------------------------------------------------


class _Held:
    """The device memory of one state, given back with its last reference: a result that lies in it keeps it."""

    def __init__(self, dev):
        self.dev, self.frees = dev, []

    def own(self, thing, free=None):
        self.frees.append(free or (lambda: hip.hip_free(thing)))
        return thing

    def __del__(self):
        hip.hip_sync(self.dev)
        for f in self.frees:
            f()


class _Array:
    def __init__(self, held, ptr, shape, kind):
        self.held = held
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (ptr, False), "version": 3}


def _tensor(held, ptr, shape, kind="<f4"):
    """The device memory at PTR as a torch tensor, in place."""
    return torch.as_tensor(_Array(held, ptr, shape, kind), device="cuda")


class _Blocks:
    """Quantized matrices of one format and scale of their blocks: runs of one seeded supply of blocks, each from a place of its
    own (a supply of more blocks than a row has, of a number that no row's divides, so that no two rows of a matrix are alike)."""

    def __init__(self, rng, qtype, dscale, most, nblocks):
        per = synth.BLOCK_WEIGHTS[qtype]
        self.rng, self.bb, self.per, self.n = rng, synth.BLOCK_BYTES[qtype], per, nblocks
        base = synth.weights(qtype, nblocks, per, rng, dscale=dscale).ravel()
        self.bytes = np.tile(base, (most // per + 2 * nblocks - 1) // nblocks) if most else base

    def take(self, rows, cols):
        nbytes = rows * cols // self.per * self.bb
        at = int(self.rng.integers(0, self.n)) * self.bb
        return self.bytes[at:at + nbytes].reshape(rows, -1)

    def experts(self, ne, rows, cols):
        """NE matrices, from places a fixed number of blocks apart."""
        nbytes = rows * cols // self.per * self.bb
        step = (self.bytes.size - nbytes) // self.bb // ne * self.bb
        return np.lib.stride_tricks.as_strided(self.bytes, (ne, nbytes), (step, 1))


def _host_model(name, rng):
    """A seeded random-init decoder of the named shape, its layers adding a fraction of the stream as a trained model's do."""
    c = SHAPES[name]
    d, ffn, nh, nkv, hd = c["d"], c["ffn"], c["nh"], c["nkv"], c["hd"]
    qd, kvd = nh * hd, nkv * hd
    norm = lambda n: (synth.activations(n, rng) * 0.1 + 1.0).astype(np.float32)
    layers = []
    if c["q8"]:
        w = _Blocks(rng, synth.Q8_0, None, max(ffn * d, c["vocab"] * d), 300007)
        q8 = lambda rows, cols: (synth.Q8_0, w.take(rows, cols))
        bias = lambda n: (synth.activations(n, rng) * 0.5).astype(np.float32)
        for _ in range(c["nl"]):
            layers.append({"wq": q8(qd, d), "wk": q8(kvd, d), "wv": q8(kvd, d), "wo": q8(d, qd), "gate": q8(ffn, d), "up": q8(ffn, d), "down": q8(d, ffn),
                           "bq": bias(qd), "bk": bias(kvd), "bv": bias(kvd), "attn_norm": norm(d), "ffn_norm": norm(d), "q_norm": None, "k_norm": None})
        embd = q8(c["vocab"], d)
    else:
        w4, wo = _Blocks(rng, synth.Q4_K, None, ffn * d, 50021), _Blocks(rng, synth.Q4_K, 0.0002 * 0.005, d * qd, 20011)
        w6, wd = _Blocks(rng, synth.Q6_K, None, kvd * d, 10007), _Blocks(rng, synth.Q6_K, 0.002 / 32.0 * 0.005, d * ffn, 50021)
        we = _Blocks(rng, synth.Q6_K, 0.01 * 8.0 / 32.0, c["vocab"] * d, 160001)
        for _ in range(c["nl"]):
            layers.append({"wq": (synth.Q4_K, w4.take(qd, d)), "wk": (synth.Q4_K, w4.take(kvd, d)), "wv": (synth.Q6_K, w6.take(kvd, d)),
                           "wo": (synth.Q4_K, wo.take(d, qd)), "gate": (synth.Q4_K, w4.take(ffn, d)), "up": (synth.Q4_K, w4.take(ffn, d)),
                           "down": (synth.Q6_K, wd.take(d, ffn)), "attn_norm": norm(d), "ffn_norm": norm(d), "q_norm": norm(hd), "k_norm": norm(hd)})
        embd = (synth.Q6_K, we.take(c["vocab"], d))
    return {"config": {**{k: c[k] for k in ("d", "ffn", "nh", "nkv", "hd", "nl", "vocab")}, "eps": 1e-6, "rope_base": 1e6, "neox": True},
            "embd": embd, "output": embd, "output_norm": norm(d), "layers": layers}


def _prepare_turn(case, rng, dev, held):
    c = SHAPES[case["model"]]
    ctx, n = case["ctx"], case["prompt"]
    nctx = ctx + n + case["tokens"]
    m = model.DenseModel(dev, _host_model(case["model"], rng), nctx=nctx)
    held.own(m, m.free)
    words = rng.integers(0, c["vocab"], ctx + n).tolist()
    if ctx:
        m.eval_tokens(words[:ctx], logits=False)       # the conversation so far
    last = m.layers[-1]
    caches = [_tensor(held, last[k].ptr, (nctx, c["nkv"] * c["hd"])) for k in ("kc", "vc")]
    return {"model": m, "ctx": ctx, "words": words[ctx:], "tokens": case["tokens"], "logits": _tensor(held, m.logits.ptr, (c["vocab"],)), "caches": caches}


def _run_turn(s):
    m = s["model"]
    m.pos = s["ctx"]                                   # the turn again, from the same place in the conversation
    m.eval_tokens(s["words"])
    out = {"logits": s["logits"], "k": s["caches"][0], "v": s["caches"][1]}
    if s["tokens"]:
        out["ids"] = np.array(m.decode_greedy(s["tokens"]), np.int64)
    return out


def _prepare_product(case, rng, dev, held):
    fmt, rows, cols = FORMATS[case["fmt"]], case["rows"], case["cols"]
    nmat = 2 if case["glu"] else 1
    w = _Blocks(rng, fmt, None, rows * cols, 50021)
    mats = [dense.upload_gmat(dev, "w%d" % i, fmt, rows, cols, w.take(rows, cols)) for i in range(nmat)]
    for m in mats:
        held.own(m, m.free)
    x = held.own(hip.hip_upload_new(dev, synth.activations(cols, rng)))
    norm = (held.own(hip.hip_upload_new(dev, (synth.activations(cols, rng) * 0.1 + 1.0).astype(np.float32))), 1e-6) if case["norm"] else None
    y = held.own(hip.hip_alloc(dev, 4 * rows))
    return {"dev": dev, "mats": mats, "x": x, "norm": norm, "y": y, "out": _tensor(held, y.ptr, (rows,))}


def _run_product(s):
    if len(s["mats"]) == 2:
        dense.glu_mul(s["dev"], s["mats"][0], s["mats"][1], None, s["y"], xf=s["x"], norm=s["norm"])
    else:
        dense.mv_multi(s["dev"], [(s["mats"][0], s["y"], None)], xf=s["x"], norm=s["norm"])
    return s["out"]


TWO_PASS_FROM = 1536       # tokens from which the bf16 product goes through a bf16 copy of the matrix (as the benchmark's prefill product does)


def _prepare_gemm(case, rng, dev, held):
    fmt, rows, cols, n, path = FORMATS[case["fmt"]], case["rows"], case["cols"], case["tokens"], case["path"]
    w = dense.upload_gmat(dev, "w", fmt, rows, cols, _Blocks(rng, fmt, None, rows * cols, 50021).take(rows, cols))
    held.own(w, w.free)
    x = held.own(hip.hip_upload_new(dev, synth.activations((n, cols), rng)))
    y = held.own(hip.hip_alloc(dev, 4 * n * rows))
    s = {"dev": dev, "w": w, "x": x, "y": y, "n": n, "path": path, "out": _tensor(held, y.ptr, (n, rows))}
    if path == "exact":
        s["act"] = dense.QAct(dev, n, cols, ("q8k",))
        held.own(s["act"], s["act"].free)
    elif path == "bf16" and n < TWO_PASS_FROM:
        s["xb"] = held.own(hip.hip_alloc(dev, 2 * n * cols))
    else:
        s["xb"] = held.own(hip.hip_alloc(dev, dense.slabs_bytes(n, cols)))
        s["wb"] = held.own(hip.hip_alloc(dev, dense.slabs_bytes(rows, cols)))
        if path == "bf16-resident":
            dense.dequant_bf16(dev, w, s["wb"])
    return s


def _run_gemm(s):
    dev, w, n = s["dev"], s["w"], s["n"]
    if s["path"] == "exact":
        dense.cmat_mul(dev, w, dense.quantize_act(dev, s["x"], s["act"]), s["y"], n)
    elif "wb" not in s:
        dense.cmat_mul_bf16(dev, w, dense.cvt_bf16(dev, s["x"], n * w.cols, s["xb"]), s["y"], n)
    else:
        if s["path"] == "bf16":
            dense.dequant_bf16(dev, w, s["wb"])
        dense.mat_mul_bf16(dev, s["wb"], w.rows, w.cols, dense.cvt_bf16_slabs(dev, s["x"], n, w.cols, s["xb"]), s["y"], n)
    return s["out"]


def _prepare_moe(case, rng, dev, held):
    ne, nu, d, ff, n = (case[k] for k in ("ne", "nu", "d", "ff", "tokens"))
    w, wd = _Blocks(rng, synth.IQ2_XXS, None, 4 * ff * d, 50021), _Blocks(rng, synth.Q2_K, None, 4 * ff * d, 50021)
    pool = ds4f.ExpertPool(dev, ne, d, ff, w.experts(ne, ff, d), w.experts(ne, ff, d)[::-1], wd.experts(ne, d, ff))
    held.own(pool, pool.free)
    w8 = _Blocks(rng, synth.Q8_0, None, ff * d, 50021)
    sh = ds4f.SharedExpert(dev, d, ff, w8.take(ff, d), w8.take(ff, d), w8.take(d, ff))
    held.own(sh, sh.free)
    x = held.own(hip.hip_upload_new(dev, synth.activations((n, d), rng)))
    # a router's logits: some experts are chosen far more often than others
    logits = held.own(hip.hip_upload_new(dev, synth.zipf_router_logits(n, ne, rng)))
    s = {"dev": dev, "pool": pool, "sh": sh, "x": x, "logits": logits, "case": case, "held": held, "last": [None]}
    if case["op"] == "step":
        s["moe"] = held.own(hip.hip_alloc(dev, 4 * d))
        s["ws"] = held.own(hip.hip_alloc(dev, ds4f.step_workspace_bytes(nu, d, ff), zero=False))
        s["out"] = _tensor(held, s["moe"].ptr, (d,))
    elif case["op"] != "small":
        rows = n * nu
        s["ws"] = hip.Workspace(dev, rows * (4 * d * 2 + 2 * d + 4 * ff * 3 + 2 * ff + d + ff + 4096) + n * (8 * d + 12 * ff) + (16 << 20))
        held.own(s["ws"], s["ws"].free)
    else:
        last = held.own(s["last"], lambda: hip.hip_free(last[0]))
    return s


def _run_moe(s):
    c, dev, pool, sh = s["case"], s["dev"], s["pool"], s["sh"]
    ne, nu, n, clamp = c["ne"], c["nu"], c["tokens"], c["clamp"]
    if c["op"] == "step":
        ds4f.ffn_step_call(dev, pool, sh, s["logits"], s["x"], s["moe"], ne, nu, ROUTE_SCALE, clamp, wsbuf=s["ws"])
        return s["out"]
    if c["op"] == "small":
        hip.hip_free(s["last"][0])                     # the result of the pass before, which its caller is done with
        s["last"][0] = moe = ds4f.ffn_small(dev, pool, sh, s["logits"], s["x"], n, ne, nu, ROUTE_SCALE, clamp, grouped=True)
    else:
        ws = s["ws"]
        ws.reset()
        sout = ds4f.ffn_shared_chunk(dev, sh, s["x"], n, clamp, ws=ws)
        routed = ds4f.ffn_routed_chunk_bf16 if c["op"] == "chunk-bf16" else ds4f.ffn_routed_chunk
        moe = routed(dev, pool, s["logits"], s["x"], sout, n, ne, nu, ROUTE_SCALE, clamp, ws=ws)
    return _tensor(s["held"], moe.ptr, (n, c["d"]))


PREPARE = {"turn": _prepare_turn, "product": _prepare_product, "gemm": _prepare_gemm, "moe": _prepare_moe}
RUN = {"turn": _run_turn, "product": _run_product, "gemm": _run_gemm, "moe": _run_moe}


def prepare(case, seed):
    dev = hip.open_hip(0)
    s = PREPARE[case["kind"]](case, synth.make_rng(seed), dev, _Held(dev))
    s["kind"] = case["kind"]
    hip.hip_sync(dev)
    return s


def run(state):
    return RUN[state["kind"]](state)


# ---- what a pass cannot do without ------------------------------------------------------------------------------------


def _bytes(fmt, rows, cols):
    return rows * synth.row_bytes(fmt, cols)


def _work_turn(case):
    c = SHAPES[case["model"]]
    d, ffn, nl, qd, kvd = c["d"], c["ffn"], c["nl"], c["nh"] * c["hd"], c["nkv"] * c["hd"]
    f4, f6 = (synth.Q8_0, synth.Q8_0) if c["q8"] else (synth.Q4_K, synth.Q6_K)
    layer = _bytes(f4, qd + kvd + 2 * ffn, d) + _bytes(f4, d, qd) + _bytes(f6, kvd, d) + _bytes(f6, d, ffn)
    weights = nl * (d * (2 * qd + 2 * kvd) + 3 * d * ffn)
    head = _bytes(f6, c["vocab"], d)
    # every pass over the matrices is one token's, or the whole prompt's; the caches are read up to each pass's last position
    nbytes = flops = 0
    for n, ctx in [(case["prompt"], case["ctx"])] + [(1, case["ctx"] + case["prompt"] + i) for i in range(case["tokens"])]:
        nbytes += nl * (layer + 8 * kvd * (ctx + n)) + head + 4 * c["vocab"] + n * synth.row_bytes(f6, d)
        flops += 2 * weights * n + 2 * c["vocab"] * d + nl * 4 * qd * (n * ctx + n * (n + 1) // 2)
    return nbytes, flops


def _work_moe(case):
    ne, nu, d, ff, n = (case[k] for k in ("ne", "nu", "d", "ff", "tokens"))
    expert = _bytes(synth.IQ2_XXS, 2 * ff, d) + _bytes(synth.Q2_K, d, ff)
    shared = _bytes(synth.Q8_0, 2 * ff, d) + _bytes(synth.Q8_0, d, ff)
    # (of a chunk's experts, those that no token chose are not read: a token's choices are nearly independent given the
    # router's preferences, so the number chosen is counted on logits drawn as the inputs are)
    if n == 1:
        used = nu
    else:
        used = len(np.unique(np.argsort(-synth.zipf_router_logits(n, ne, synth.make_rng(1)), axis=1)[:, :nu]))
    return used * expert + shared + 8 * n * d + 4 * n * ne, 2 * n * (nu + 1) * 3 * d * ff


def work(case):
    if case["kind"] == "turn":
        nbytes, flops = _work_turn(case)
    elif case["kind"] == "moe":
        nbytes, flops = _work_moe(case)
    else:
        rows, cols, n = case["rows"], case["cols"], case.get("tokens", 1)
        nmat = 2 if case.get("glu") else 1
        nbytes = nmat * _bytes(FORMATS[case["fmt"]], rows, cols) + 4 * n * (cols + rows)
        if case.get("path") == "bf16-resident":
            nbytes = 2 * rows * cols + 4 * n * (cols + rows)
        flops = 2 * nmat * rows * cols * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # the bf16 products round both operands to 8 bits of mantissa and add in single precision in an order of their own
    if case.get("path", "").startswith("bf16") or case.get("op") == "chunk-bf16":
        return {"rel": 1e-2, "max": 5e-2}
    # everything else promises the CPU path's bits
    return "exact"
