"""Every launch with more dynamic LDS than the 64 KB that a kernel gets by itself asks for it first (hipFuncSetAttribute), and which
kernels a chunk's attention takes.  The library's host code runs here on a stand-in for the HIP runtime that notes what it is
asked for and launches nothing (no GPU)."""
import os
import re
import subprocess
import sys

RUNTIME = r"""
#include <stdio.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim3_;
static struct { const void* f; const char* name; long asked; } k[2048];
static int nk;
static __thread struct { dim3_ g, b; size_t lds; void* st; } cfg;
void** __hipRegisterFatBinary(const void* d) { static void* h; return &h; }
void __hipUnregisterFatBinary(void** h) {}
void __hipRegisterVar(void** m, void* v, char* n, char* d, int e, size_t s, int c, int g) {}
void __hipRegisterFunction(void** m, const void* f, char* n, const char* d, unsigned t, void* a, void* b, void* c, void* e, int* w) {
  if (nk < 2048) { k[nk].f = f; k[nk].name = d; k[nk].asked = 65536; nk++; }
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void* st) { cfg.g = g; cfg.b = b; cfg.lds = lds; cfg.st = st; return 0; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* lds, void** st) { *g = cfg.g; *b = cfg.b; *lds = cfg.lds; *st = cfg.st; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* f, int attr, int v) {
  for (int i = 0; i < nk; i++) if (k[i].f == f && attr == 8 && v > k[i].asked) k[i].asked = v;
  return 0;
}
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** args, size_t lds, void* st) {
  for (int i = 0; i < nk; i++) if (k[i].f == f) printf("%s %s %zu of %ld\n", (long)lds > k[i].asked ? "UNASKED" : "ok", k[i].name, lds, k[i].asked);
  return 0;
}
"""

CALLS = r"""
import ctypes as C, os, sys
C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
P, Z, I, S = C.c_uint64(1 << 40), C.c_uint64(0), C.c_int, C.c_uint64(0)
def ok(e, *what):
    assert e == 0, (e,) + what
for cols in (256, 2560, 4096, 9728, 16384):
    for rows in (32, 2560, 19456):
        for n in (2, 16, 17, 40, 130, 512, 2048):
            for t in (0, 2):
                ok(L.ilt_mm_k(S, I(t), P, P, P, P, P, Z, I(rows), I(cols), I(n), I(0)), "mm_k", t, rows, cols, n)
            ok(L.ilt_mm_k_n(S, I(2), P, P, Z, I(rows), P, P, Z, I(rows), Z, Z, Z, I(0), P, P, P, I(cols), I(n), I(0)), "mm_k_n", rows, cols, n)
            ok(L.ilt_mm_q8(S, P, P, P, P, P, Z, I(rows), I(cols), I(n), I(0)), "mm_q8", rows, cols, n)
            ok(L.ilt_mm_q8_mma2(S, P, P, P, Z, I(rows), P, P, P, Z, I(rows), Z, Z, Z, Z, I(0), P, P, I(cols), I(n), I(0)), "mm_q8_mma2", rows, cols, n)
            ok(L.ilt_cvt_bf16(S, P, P, C.c_int64(n * cols)), "cvt")
            for t in (12, 14):
                ok(L.ilt_mm_k_bf16(S, I(t), P, P, P, Z, I(rows), I(cols), I(n), I(0)), "mm_k_bf16", t, rows, cols, n)
            if rows % 256 == 0:
                ok(L.ilt_mm_bf16(S, P, P, P, Z, I(rows), I(cols), I(n), I(0)), "mm_bf16", rows, cols, n)
for total in (8, 300, 24576):
    for d, ff in ((512, 256), (4096, 2048)):
        grb, drb = d // 256 * 66, ff // 256 * 84
        add, T = C.c_int64, C.c_int64(total)
        ok(L.ilt_d4_mm_id2_iq2_xxs(S, I(d), I(ff), I(grb), add(0), add(ff * grb), P, P, P, I(64), T, P, P, P, P), "id2")
        ok(L.ilt_d4_mm_id_q2_k(S, I(ff), I(d), I(drb), add(2 * ff * grb), P, P, P, I(64), T, P, P, P, P), "id")
        ok(L.ilt_d4_mm_id_bf16(S, I(10), I(ff), I(d), I(drb), add(2 * ff * grb), P, P, P, I(64), T, P, Z, P), "id_bf16")
        ok(L.ilt_d4_mm_id_glu_bf16(S, I(16), I(d), I(ff), I(grb), add(0), add(ff * grb), P, P, P, I(64), T, P, P, C.c_float(0), P, P), "id_glu_bf16")
for nh, nkv, hd in ((32, 8, 128), (14, 2, 64), (32, 8, 96)):
    for pos in (0, 500, 1000, 1500, 4000, 8000):
        ok(L.ilt_attn_step(S, P, P, P, Z, Z, P, P, P, P, I(nh), I(nkv), I(hd), I(hd), I(pos), C.c_float(1e-6), I(1), P, I(8192)), "attn_step", hd, pos)
        for n in (1, 33, 130):
            for scratch in (P, Z):
                ok(L.ilt_attn_rows(S, P, P, P, P, I(nh), I(nkv), I(hd), I(pos), I(n), scratch), "attn_rows", hd, pos, n)
"""


def launched(tmp_path, calls, **env):
    """The lines that the stand-in printed for CALLS: a launch each."""
    from illatio_amd import hip
    (tmp_path / "runtime.c").write_text(RUNTIME)
    so = str(tmp_path / "runtime.so")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-w", "-o", so, str(tmp_path / "runtime.c")])
    r = subprocess.run([sys.executable, "-c", calls, so, hip.LIB_PATH], env={**os.environ, **env}, capture_output=True, text=True)
    lines = r.stdout.splitlines()
    assert r.returncode == 0, (r.stderr[-2000:], lines[-3:])
    return lines


def test_no_launch_takes_more_lds_than_it_asked_for(tmp_path):
    lines = launched(tmp_path, CALLS, ILT_ATTN_SPLIT="0")
    assert len(lines) > 500 and sum("gemm_i8_few" in x for x in lines) > 50
    assert any(int(x.split()[-3]) > 65536 for x in lines)
    assert not sorted({x for x in lines if x.startswith("UNASKED")})


CHUNKS = r"""
import ctypes as C, sys
C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
I = C.c_int
at = lambda off=0: C.c_uint64((1 << 40) + off)
for hd in (64, 128):
    for ctx in (100, 1000, 3000):
        assert L.ilt_attn_rows(C.c_uint64(0), at(QUERY), at(), at(), at(), I(16), I(4), I(hd), I(ctx - 40), I(40), at()) == 0
"""


def kernels(lines):
    """The attention kernels of the launches, and in brackets the template's first number and whether it leaves quantized rows."""
    found = (re.search(r"\d(attn_[a-z_]+?)_kernel(?:I((?:L[ib]\d+E)+))?", x) for x in lines)
    return [(m.group(1), m.group(2) or "") for m in found if m]


def test_which_kernels_a_chunks_attention_takes(tmp_path):
    names = lambda lines: {n for n, _ in kernels(lines)} - {"attn_softmax"}
    mm = {"attn_short_mm", "attn_scores_mm", "attn_values_mm_row"}
    assert names(launched(tmp_path, "QUERY = 0" + CHUNKS, ILT_ATTN_MM="1")) == mm
    assert names(launched(tmp_path, "QUERY = 0" + CHUNKS, ILT_ATTN_MM="0")) == {"attn_scores", "attn_values_chunk"}
    assert names(launched(tmp_path, "QUERY = 4" + CHUNKS)) == {"attn_scores", "attn_values_chunk"}
    assert names(launched(tmp_path, "QUERY = 0" + CHUNKS, ILT_ATTN_CHUNK="0")) == {"attn_scores", "attn_values", "attn_values_tiled"}


SHORT = r"""
import ctypes as C, sys
C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
P, I = C.c_uint64(1 << 40), C.c_int
for nh, nkv, hd, pos, n in %s:
    print("at", nh, nkv, hd, pos, n, flush=True)
    assert L.ilt_attn_rows(C.c_uint64(0), P, P, P, P, I(nh), I(nkv), I(hd), I(pos), I(n), P) == 0
    C.CDLL(None).fflush(None)
"""


def test_one_launch_of_two_rounds_of_values_only_for_few_positions(tmp_path):
    """Groups of more heads than a round of attn_short_mm_kernel's waves takes the values of: one launch up to 96 or 64 positions."""
    one = [(20, 4, 128, 94, 2), (24, 4, 128, 88, 8), (28, 4, 128, 62, 2), (32, 4, 128, 48, 16), (28, 4, 128, 64, 32), (64, 8, 128, 64, 32), (16, 4, 128, 254, 2), (32, 4, 64, 254, 2)]
    three = [(20, 4, 128, 95, 2), (24, 4, 128, 200, 8), (28, 4, 128, 63, 2), (32, 4, 128, 49, 16), (28, 4, 128, 65, 32), (64, 8, 128, 65, 32), (16, 4, 128, 255, 2), (32, 4, 64, 255, 2)]
    assert [k[0] for k in chunk_kernels(tmp_path, one + three)] == ["attn_short_mm"] * len(one) + ["attn_scores_mm"] * len(three)


def chunk_kernels(tmp_path, shapes):
    """A shape's attention kernels, one after another."""
    calls = []
    for x in launched(tmp_path, SHORT % (shapes,)):
        if x.startswith("at "):
            calls.append([])
        else:
            calls[-1].append(kernels([x])[0])
    return [[n + (re.match(r"Li(\d+)E", t).group(1) if n == "attn_values_mm" else "") for n, t in c] for c in calls]


def test_a_chunks_attention_on_each_side_of_its_lines(tmp_path):
    """One launch: groups of 3 to 8 heads, up to 256 workgroups (KV heads x tokens), 256 positions, 448 from 128 workgroups on.  Three: values of
    a row a wave up to 1,400 waves (rows x KV heads x 64-column parts), of sixteen rows from 1,600 waves on, or fewer where the chunk
    lies further in than it is long; else of four.  (nh, nkv, hd, first position, tokens.)"""
    short = ["attn_short_mm"]
    three = lambda values: ["attn_scores_mm", "attn_softmax", values]
    row, r4, r16 = three("attn_values_mm_row"), three("attn_values_mm4"), three("attn_values_mm16")
    for shape, want in {
            (3, 1, 64, 0, 2): short, (2, 1, 64, 0, 2): row, (8, 1, 64, 0, 2): short, (9, 1, 64, 0, 2): row,
            (32, 8, 128, 0, 32): short, (32, 8, 128, 0, 33): r4, (12, 4, 128, 0, 64): short, (12, 4, 128, 0, 65): r4,
            (8, 2, 128, 239, 17): short, (8, 2, 128, 239, 18): row, (14, 2, 64, 193, 63): short, (14, 2, 64, 193, 64): short, (14, 2, 64, 194, 63): row,
            (32, 8, 128, 432, 16): short, (32, 8, 128, 433, 16): row, (32, 8, 128, 433, 15): row, (16, 4, 128, 416, 32): short, (16, 4, 128, 417, 32): row,
            # the shapes of test_gpu_model's runs in one launch, and of those with a row and with four rows a wave
            (12, 4, 128, 61, 3): short, (40, 5, 128, 15, 49): short, (15, 3, 64, 63, 2): short, (24, 4, 64, 412, 36): short, (7, 1, 128, 0, 64): short,
            (24, 3, 128, 40, 44): short, (10, 2, 128, 80, 16): short, (4, 4, 64, 14, 2): row, (8, 2, 64, 15, 175): row, (8, 2, 64, 15, 176): r4,
            (10, 2, 128, 507, 6): row, (6, 6, 64, 2047, 3): row, (32, 8, 128, 301, 33): r4, (4, 4, 128, 3, 177): r4, (14, 2, 64, 2, 130): r4,
            (16, 16, 128, 0, 799): r16, (8, 8, 128, 0, 1584): r4, (8, 8, 128, 0, 1585): r16,
            (32, 8, 128, 600, 256): r16, (32, 8, 128, 256, 256): r4, (32, 8, 128, 600, 128): r4}.items():
        assert chunk_kernels(tmp_path, [shape])[0] == want, shape


MANY_ROWS = r"""
import ctypes as C, sys
C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
P, Z, I = C.c_uint64(1 << 40), C.c_uint64(0), C.c_int
for t, rows, cols, n in %s:
    assert L.ilt_mm_k(C.c_uint64(0), I(t), P, P, P, P, P, Z, I(rows), I(cols), I(n), I(0)) == 0
"""


def test_few_tokens_stay_where_the_other_kernel_takes_not_so_many_rows(tmp_path):
    """Up to 16 tokens of Q6_K (2) and Q4_K (0) on 2^21 rows, which the kernel with operands in registers refuses, and on one less."""
    shapes = [(t, (1 << 21) - less, cols, n) for t, cols, n in ((2, 1024, 2), (2, 1024, 16), (0, 256, 12), (0, 1536, 16)) for less in (0, 1)]
    lines = launched(tmp_path, MANY_ROWS % shapes)
    assert ["few" if "gemm_i8_few" in x else "reg" if any(k in x for k in ("gemm_i8h", "gemm_i8w", "gemm_i8s", "gemm_i8r")) else x for x in lines] == ["few", "reg"] * 4


QUANT_ROWS = r"""
import ctypes as C, sys
C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
P, I = C.c_uint64(1 << 40), C.c_int
for x, xq in ((0, 0), (4, 0), (8, 0), (12, 0), (0, 1), (0, 2), (16, 4)):
    at = lambda off: C.c_uint64((1 << 40) + off)
    print(x, xq, L.ilt_d4_quant_q8k_rows(C.c_uint64(0), I(512), I(3), I(2), at(x), P, at(xq), P))
"""


def test_quantizing_into_rows_wants_the_addresses_that_its_loads_and_stores_do(tmp_path):
    """ilt_d4_quant_q8k_rows on floats off 16 bytes or quants off 4: an error and no launch, as ilt_quant_q8k."""
    lines = launched(tmp_path, QUANT_ROWS)
    assert sum("quant_q8k_rows" in x for x in lines) == 2
    codes = [int(x.split()[2]) for x in lines if "quant_q8k_rows" not in x]
    assert [c == 0 for c in codes] == [True, False, False, False, False, False, True]
