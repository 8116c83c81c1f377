// A few tokens' routed experts: an expert's blocks decoded once for up to R of its rows of activations (the FFN of a short
// pass, DK-FFN-SMALL, cuda-ds4f-spec.lisp:30-100), every result with the CPU path's bits (kquant.lisp:180-236).
#include "ilt_device.h"
#include "ilt_kernels.h"
#include "ilt_iq2xxs_tables.h"
#include "ilt_route.h"
#include <algorithm>

namespace {

__device__ const u64 iq2_grid_share[256] = { ILT_IQ2XXS_GRID_VALUES };

struct ShareArgs {
  const u64* ptrs;             // an expert's matrices
  const u32* rexp;             // row i of the n grouped rows works on expert rexp[i]; an expert's rows one after another
  const u32* xrow;             // ... and on row xrow[i] of the activations (null: row i)
  const i8* xq; const float* xd; const int* bsums;
  long long add, add2;         // the matrix at ptrs[e] + add (IQ2_XXS: the gate, its up at add2)
  const float* wts; float clamp;
  float* y;                    // n rows of `rows` results
  int rows, row_bytes, S, n;
  IltShareBeside beside; int by;        // the shared expert's product in the same launch: the grid's first by rows of workgroups
};

constexpr int kAhead = 2;      // steps loaded ahead

template <int FMT> struct ShareFmt;
// R rows of activations at once, STEPS of 16 blocks a wave and matrix
template <> struct ShareFmt<ILT_IQ2_XXS> { static constexpr int MATS = 2, TERMS = 1, R = 3, STEPS = 4; };
template <> struct ShareFmt<ILT_Q2_K> { static constexpr int MATS = 1, TERMS = 2, R = 2, STEPS = 8; };

template <int FMT> struct ShareRaw;        // a lane's quarter of a block as it is in memory
template <> struct ShareRaw<ILT_IQ2_XXS> { int4 q; u16 d; };
template <> struct ShareRaw<ILT_Q2_K> { int4 q, sb; u32 dd; };
template <int FMT> struct ShareX;          // ... and the activations it meets
template <> struct ShareX<ILT_IQ2_XXS> { int4 x[4]; float d; };
template <> struct ShareX<ILT_Q2_K> { int4 x[4]; int bs[2]; float d; };

__device__ __forceinline__ void share_load(ShareRaw<ILT_IQ2_XXS>& r, __amdgpu_buffer_rsrc_t w, u32 blk, int j) {
  r.q = ilt_bld16(w, blk * 66 + 2 + 16 * j);
  r.d = ilt_bld2(w, blk * 66);
}
__device__ __forceinline__ void share_load(ShareRaw<ILT_Q2_K>& r, __amdgpu_buffer_rsrc_t w, u32 blk, int j) {
  r.q = ilt_bld16(w, blk * 84 + 16 + 16 * j);
  r.sb = ilt_bld16(w, blk * 84);
  r.dd = ilt_bld4(w, blk * 84 + 80);
}
__device__ __forceinline__ void share_load_x(ShareX<ILT_IQ2_XXS>& X, const ShareArgs& p, long blk, int j) {
#pragma unroll
  for (int k = 0; k < 4; k++) X.x[k] = ilt_ld16((const u8*)p.xq + blk * 256 + 64 * j + 16 * k);
  X.d = p.xd[blk];
}
__device__ __forceinline__ void share_load_x(ShareX<ILT_Q2_K>& X, const ShareArgs& p, long blk, int j) {
#pragma unroll
  for (int k = 0; k < 4; k++) X.x[k] = ilt_ld16((const u8*)p.xq + blk * 256 + 128 * (j >> 1) + 16 * (j & 1) + 32 * k);
  const int4 b = ilt_ld16((const u8*)(p.bsums + blk * 16 + 4 * j));         // (at most 16 * 127: 16 bits)
  X.bs[0] = (b.x & 0xFFFF) | (b.z << 16);
  X.bs[1] = (b.y & 0xFFFF) | (b.w << 16);
  X.d = p.xd[blk];
}

// What a step makes of its blocks once, for all the rows of activations.  IQ2_XXS: the codebook as eight 2-bit magnitudes in the
// nibbles of a dword and the signs as bit 2 of them, so a table is 4 bytes an entry and a byte permutation gives four signed
// weights (entries of 8 bytes with masks to negate by: twice the LDS reads' conflicts, 16 registers more).
template <int FMT> struct ShareW;
template <> struct ShareW<ILT_IQ2_XXS> { int w[16]; float s0, s1, d; };
template <> struct ShareW<ILT_Q2_K> { int4 q[4]; int sc[4], mn[2]; float d, dmin; };
__device__ __forceinline__ void share_decode(ShareW<ILT_IQ2_XXS>& W, const ShareRaw<ILT_IQ2_XXS>& r, int) {
  const u32 g[2] = {(u32)r.q.x, (u32)r.q.z}, aux[2] = {(u32)r.q.y, (u32)r.q.w};
  u32 c[8];
#pragma unroll
  for (int l = 0; l < 8; l++) {
    // (the tables begin LDS -- the kernel has no other --, so an index times four is the address)
    const u32 a = aux[l >> 2];
    const int sh = 7 * (l & 3) - 2;
    c[l] = *(ILT_LDS const u32*)(uintptr_t)(((g[l >> 2] >> (8 * (l & 3))) & 0xFF) << 2) |
           *((ILT_LDS const u32*)(uintptr_t)((sh < 0 ? a << -sh : a >> sh) & 0x1FC) + 256);
  }
#pragma unroll
  for (int l = 0; l < 8; l++) {                        // the bytes of the codebook, and what they are negated
    W.w[2 * l] = (int)__builtin_amdgcn_perm(0x00D5E7F8, 0x002B1908, c[l] & 0x07070707);
    W.w[2 * l + 1] = (int)__builtin_amdgcn_perm(0x00D5E7F8, 0x002B1908, (c[l] >> 4) & 0x07070707);
  }
  W.s0 = 0.5f + (float)(aux[0] >> 28);
  W.s1 = 0.5f + (float)(aux[1] >> 28);
  W.d = ilt_h2f(r.d);
}
__device__ __forceinline__ void share_decode(ShareW<ILT_Q2_K>& W, const ShareRaw<ILT_Q2_K>& r, int j) {
  const int h = j >> 1, half = j & 1;
  const u32 wa = (u32)(h ? r.sb.z : r.sb.x) >> (8 * half), wb = (u32)(h ? r.sb.w : r.sb.y) >> (8 * half);
  const u32 wj = (u32)(j == 0 ? r.sb.x : j == 1 ? r.sb.y : j == 2 ? r.sb.z : r.sb.w);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    W.q[k] = make_int4((r.q.x >> (2 * k)) & 0x03030303, (r.q.y >> (2 * k)) & 0x03030303, (r.q.z >> (2 * k)) & 0x03030303,
                       (r.q.w >> (2 * k)) & 0x03030303);
    W.sc[k] = (int)(((k < 2 ? wa : wb) >> (16 * (k & 1))) & 0xF);
  }
  W.mn[0] = (int)(wj >> 4) & 0x000F000F;              // sub-blocks 4j and 4j + 2, 4j + 1 and 4j + 3
  W.mn[1] = (int)(wj >> 12) & 0x000F000F;
  W.d = ilt_h2f((u16)(r.dd & 0xFFFF));
  W.dmin = ilt_h2f((u16)(r.dd >> 16));
}
typedef short share_v2s __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int share_dot2(int a, int b, int c) {
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(share_v2s, a), __builtin_bit_cast(share_v2s, b), c, false);
}
// One row's term of the block, from its four lanes to lane 0 of them, in the order of block_terms (kernels_gemv.hip).
__device__ __forceinline__ void share_terms(const ShareW<ILT_IQ2_XXS>& W, const ShareX<ILT_IQ2_XXS>& X, int, bool puts, float* t) {
  int a0 = 0, a1 = 0;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    a0 = ilt_dot16(make_int4(W.w[4 * k], W.w[4 * k + 1], W.w[4 * k + 2], W.w[4 * k + 3]), X.x[k], a0);
    a1 = ilt_dot16(make_int4(W.w[4 * k + 8], W.w[4 * k + 9], W.w[4 * k + 10], W.w[4 * k + 11]), X.x[k + 2], a1);
  }
  const float te = (float)a0 * W.s0, to = (float)a1 * W.s1;
  float a = te, b = to;                                // (the CPU's leading 0 + shows in a zero's sign alone, which the row's sum drops)
  a = a + ilt_dppf<ILT_DPP_SHL(1)>(te); b = b + ilt_dppf<ILT_DPP_SHL(1)>(to);
  a = a + ilt_dppf<ILT_DPP_SHL(2)>(te); b = b + ilt_dppf<ILT_DPP_SHL(2)>(to);
  a = a + ilt_dppf<ILT_DPP_SHL(3)>(te); b = b + ilt_dppf<ILT_DPP_SHL(3)>(to);
  float v = (W.d * X.d) * (a + b);
  asm volatile("" : "+v"(v));
  if (puts) ilt_lds_stf(t, v);
}
__device__ __forceinline__ void share_terms(const ShareW<ILT_Q2_K>& W, const ShareX<ILT_Q2_K>& X, int j, bool puts, float* t) {
  int isum = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) isum = ilt_mad24(W.sc[k], ilt_dot16(W.q[k], X.x[k], 0), isum);
  int mins = share_dot2(W.mn[0], X.bs[0], share_dot2(W.mn[1], X.bs[1], 0));
  isum = ilt_sum4(isum);
  mins = ilt_sum4(mins);
  // lane 0 the minimums' term, lane 1 the other: one multiplication and one store for both
  const float v = ((j ? X.d : -X.d) * (j ? W.d : W.dmin)) * (float)(j ? isum : mins);
  if (puts) ilt_lds_stf(t + j, v);
}

__device__ __forceinline__ float share_sum(const float* t, int n) {        // ((0 + t[0]) + t[1]) + ...
  float o = 0.0f;
  int k = 0;
  for (; k + 8 <= n; k += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = ilt_lds_ldf(t + k + i);
#pragma unroll
    for (int i = 0; i < 8; i++) o = o + v[i];
  }
  for (; k < n; k++) o = o + ilt_lds_ldf(t + k);
  return o;
}

// The shared expert's Q8_0 rows on the pass's tokens: a wave takes one row of a matrix (two up to six tokens), 32 blocks a step, two
// lanes a block; the blocks' float terms in LDS, then a lane a row and token adds them in order.
// Why here: as launches of their own these products wait for memory, 13 and 8 us of five tokens', and the routed experts' for their
// instructions, 26 and 14, one after the other; as the first workgroups of the same launch they are over before it (the pass 97 -> 84 us, waiting for it
// included).
constexpr int kBesideTokens = 9;
__device__ __forceinline__ void share_beside(const IltShareBeside& q, int at, u8* smem) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 1;
  const int nb = q.cols >> 5, rw = q.ntok <= 6 ? 2 : 1, r0 = (at * 4 + wave) * rw;
  if (r0 >= q.nmat * q.rows) return;                   // (whole waves; no barrier below)
  const int m = r0 >= q.rows ? 1 : 0, row = r0 - m * q.rows;       // (an even number of rows a matrix)
  const i8* const w = (const i8*)ilt_uniform_ptr(m ? q.w[1] : q.w[0]) + (long)row * q.cols;
  const u16* const wd = (const u16*)ilt_uniform_ptr(m ? q.wd[1] : q.wd[0]) + (long)row * nb;
  const int pitch = nb + 1;                            // (a float between rows: the sums' lanes on different banks)
  float* const terms = (float*)smem + (long)wave * rw * q.ntok * pitch;
  const int steps = (q.cols + 1023) >> 10;             // at most four
  int4 wv[2][4]; u16 dv[2][4];
#pragma unroll
  for (int r = 0; r < 2; r++)
#pragma unroll
    for (int s = 0; s < 4; s++)
      if (r < rw && s < steps) {
        const int c = min(1024 * s + 16 * lane, q.cols - 16);
        wv[r][s] = *(const int4*)(w + (long)r * q.cols + c);
        dv[r][s] = wd[(long)r * nb + (c >> 5)];
      }
#pragma unroll
  for (int s = 0; s < 4; s++)
    if (s < steps) {
      const int c = min(1024 * s + 16 * lane, q.cols - 16), b = c >> 5;
      const bool live = 1024 * s + 16 * lane < q.cols;
      const float d0 = ilt_h2f(dv[0][s]), d1 = ilt_h2f(dv[1][s]);
#pragma unroll
      for (int t0 = 0; t0 < kBesideTokens; t0 += 2)
        if (t0 < q.ntok) {
          int4 x[2]; float dx[2];
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const int tk = min(t0 + t, q.ntok - 1);
            x[t] = *(const int4*)(q.xq + (long)tk * q.cols + c);
            dx[t] = q.xs[(long)tk * nb + b];
          }
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const int i0 = ilt_sum2(ilt_dot16(wv[0][s], x[t], 0)), i1 = rw > 1 ? ilt_sum2(ilt_dot16(wv[1][s], x[t], 0)) : 0;
            const float v = (float)(j ? i1 : i0) * ((j ? d1 : d0) * dx[t]);      // lane 0 of a block the first row's term, lane 1 the second's
            if (live && j < rw && t0 + t < q.ntok) ilt_lds_stf(terms + (j * q.ntok + t0 + t) * pitch + b, v);
          }
        }
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (lane < rw * q.ntok) {
    const int r = lane / q.ntok, t = lane - r * q.ntok;
    (m ? q.y[1] : q.y[0])[(long)t * q.rows + row + r] = share_sum(terms + lane * pitch, nb);
  }
}

// Grid y: up to R rows of an expert (as many workgroups as rows: those past the last group end at once).  A wave: STEPS steps of
// whole rows of up to 16 blocks (four lanes a block) of each matrix.  A step's blocks lie at the same place in their rows in every
// step, so a lane's share of the R rows of activations stays in registers.
// Bound by its instructions: a step of IQ2_XXS takes about 105 ns of a SIMD to decode and 45 for each row of activations (the
// instructions of three operands, the dot products and the DPP adds issue at half the rate of an and, a shift or an add), and
// by the 66-byte blocks' loads, which lie on no dword (17 ns a load and CU against 7).  Three rows and four steps a wave for
// IQ2_XXS, two and eight for Q2_K: what 96 registers hold, five waves a SIMD, no second round of workgroups for five tokens.
// Five tokens of six of 256 experts, 4,096 x 2,048 (30 rows, 14 experts): gate and up 26 us (a row at a time, the matrix
// decoded for each and the activations read from LDS: 55; two rows 27.7, four 26.8), down 14 (25; three rows 14.3); nine
// tokens 39 and 20.
template <int FMT>
__global__ __launch_bounds__(256, 5) void share_kernel(ShareArgs p) {
  using F = ShareFmt<FMT>;
  constexpr int R = F::R;
  extern __shared__ __align__(16) unsigned char smem[];
  if ((int)blockIdx.y < p.by) { share_beside(p.beside, blockIdx.y * gridDim.x + blockIdx.x, smem); return; }
  const int group = (int)blockIdx.y - p.by;
  u32* const tab = (u32*)smem;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 3;
  int y0 = -1;
  for (int c = 0, groups = 0, run = 0; c < p.n; c += 64) {      // (the same in every wave)
    const int i = c + lane;
    const u32 v = p.rexp[min(i, p.n - 1)], pv = p.rexp[max(min(i, p.n - 1) - 1, 0)];
    const u64 upto = ~0ull >> (63 - lane), starts = __ballot(i < p.n && (i == 0 || v != pv)), mine = starts & upto;
    const bool first = i < p.n && (i - (mine ? c + 63 - __builtin_clzll(mine) : run)) % R == 0;
    const u64 firsts = __ballot(first), hit = __ballot(first && groups + __builtin_popcountll(firsts & upto) - 1 == group);
    if (hit) { y0 = c + __builtin_ctzll(hit); break; }
    groups += __builtin_popcountll(firsts);
    if (starts) run = c + 63 - __builtin_clzll(starts);
  }
  if (y0 < 0) return;
  y0 = __builtin_amdgcn_readfirstlane(y0);
  const u32 e = p.rexp[y0];
  int nr = 1;
#pragma unroll
  for (int r = 1; r < R; r++) nr += p.rexp[min(y0 + r, p.n - 1)] == e && y0 + r < p.n;      // (an expert's rows lie side by side)
  nr = __builtin_amdgcn_readfirstlane(nr);

  const int S = p.S, rps = 16 / S, rb = F::STEPS * rps;      // rows a step, rows a wave
  // this lane's block of a step (lanes past the last whole row: block 0 once more, and no terms), its row of the step, its place there
  const int blk = lane >> 2 < rps * S ? lane >> 2 : 0, brow = blk / S, bpos = blk - brow * S;
  const bool puts = j < F::TERMS && lane >> 2 < rps * S;
  const int row0 = (blockIdx.x * 4 + wave) * rb, left = min(rb, p.rows - row0);
  const u8* const w = (const u8*)ilt_uniform_ptr((const void*)p.ptrs[e]);
  const u32 bytes = __builtin_amdgcn_readfirstlane((u32)(max(left, 0) * p.row_bytes));
  const __amdgpu_buffer_rsrc_t w0 = ilt_rsrc(w + p.add + (long)row0 * p.row_bytes, bytes);
  const __amdgpu_buffer_rsrc_t w1 = F::MATS > 1 ? ilt_rsrc(w + p.add2 + (long)row0 * p.row_bytes, bytes) : w0;
  ShareRaw<FMT> raw[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; u++) share_load(raw[u], F::MATS > 1 && (u & 1) ? w1 : w0, u / F::MATS * rps * S + blk, j);
  ShareX<FMT> X[R];
#pragma unroll
  for (int r = 0; r < R; r++)
    if (r < nr) share_load_x(X[r], p, (long)(p.xrow ? p.xrow[y0 + r] : (u32)(y0 + r)) * S + bpos, j);
  if (FMT == ILT_IQ2_XXS) {
    const int t = threadIdx.x;
    const u64 g = iq2_grid_share[t];
    tab[t] = ((u32)(g >> 4) & 0x03030303) | ((u32)(g >> 32) & 0x30303030);
    if (t < 128) {                                     // the bytes that sign pattern t negates
      const u32 s = t | ((__popc(t) & 1) << 7);
      const u32 lo = ((s & 0xF) * 0x00204081u) & 0x01010101u, hi = ((s >> 4) * 0x00204081u) & 0x01010101u;
      tab[256 + t] = lo << 2 | hi << 6;
    }
    __syncthreads();
  }
  if (left <= 0) return;

  // terms: per row of activations and matrix, rb rows of S * TERMS, a float between rows (else the sums' lanes meet in a bank)
  const int pitch = (S << (F::TERMS - 1)) + 1, tile = rb * pitch;
  float* const terms = (float*)(tab + (FMT == ILT_IQ2_XXS ? 384 : 0)) + (long)wave * R * F::MATS * tile;
  float* t = terms + brow * pitch + bpos * F::TERMS;
#pragma unroll 1
  for (int k = 0; k < F::STEPS * F::MATS; k += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
      ShareW<FMT> W;
      share_decode(W, raw[u], j);
      share_load(raw[u], F::MATS > 1 && (u & 1) ? w1 : w0, (k + u + kAhead) / F::MATS * rps * S + blk, j);     // (past the end: zeros)
      float* const tu = t + (F::MATS > 1 ? (u & 1) * tile : 0) + (k + u) / F::MATS * rps * pitch;
#pragma unroll
      for (int r = 0; r < R; r++)
        if (r < nr) share_terms(W, X[r], j, puts, tu + r * F::MATS * tile);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int i = lane; i < nr * rb; i += 64) {
    const int r = i / rb, row = i - r * rb;
    if (row >= left) continue;
    const float* tr = terms + r * F::MATS * tile + row * pitch;
    float v = share_sum(tr, S * F::TERMS);
    if constexpr (FMT == ILT_IQ2_XXS) {                // the experts' gated activation, as d4_swiglu_w computes it
      float g = 0.25f * v, up = 0.25f * share_sum(tr + tile, S);
      if (p.clamp > 1e-6f) { g = fminf(g, p.clamp); up = fmaxf(-p.clamp, fminf(up, p.clamp)); }
      v = ilt_silu(g) * up * p.wts[y0 + r];
    }
    p.y[(long)(y0 + r) * p.rows + row0 + row] = v;
  }
}

// A block of 256 floats by a wave, lane l's values 4l .. 4l+3 in v.
__device__ __forceinline__ u32 share_pack(const int* q) {
  return (u32)(q[0] & 0xFF) | ((u32)(q[1] & 0xFF) << 8) | ((u32)(q[2] & 0xFF) << 16) | ((u32)(q[3] & 0xFF) << 24);
}
// quantize-q8!, d not rounded
__device__ __forceinline__ void share_q8(const float* v, u32 b, i8* __restrict__ xq, float* __restrict__ xs) {
  const int lane = threadIdx.x & 63;
  float m = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  m = fmaxf(m, ilt_dppf<ILT_DPP_XOR1>(m));
  m = fmaxf(m, ilt_dppf<ILT_DPP_XOR2>(m));
  m = fmaxf(m, ilt_dppf<ILT_DPP_HALF_MIRROR>(m));
  const float d = m / 127.0f, id = d == 0.0f ? 0.0f : 1.0f / d;
  int q[4];
#pragma unroll
  for (int k = 0; k < 4; k++) q[k] = (int)rintf(v[k] * id);
  ((u32*)(xq + (long)b * 256))[lane] = share_pack(q);
  if ((lane & 7) == 0) xs[b * 8 + (lane >> 3)] = d;
}
// quantize-q8k!.  A NaN is no block's largest (the CPU's comparisons with it fail), its quant is 0.
__device__ __forceinline__ void share_q8k(const float* v, u32 b, i8* __restrict__ kq, float* __restrict__ kd, int* __restrict__ bsums) {
  const int lane = threadIdx.x & 63;
  float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  // the first value of the largest magnitude: the first lane that holds the maximum, its first value
  int at = 4;
#pragma unroll
  for (int k = 3; k >= 0; k--) at = fabsf(v[k]) == amax ? k : at;
  const u64 hit = __ballot(at < 4);
  const float mine = at == 0 ? v[0] : at == 1 ? v[1] : at == 2 ? v[2] : v[3];
  const float mx = hit ? __shfl(mine, __builtin_ctzll(hit)) : 0.0f;              // (nothing but NaNs: no value is the largest)
  const bool any = amax != 0.0f;
  const float iscale = any ? -127.0f / mx : 0.0f;
  int q[4];
#pragma unroll
  for (int k = 0; k < 4; k++) q[k] = any ? min(127, (int)rintf(iscale * v[k])) : 0;
  ((u32*)(kq + (long)b * 256))[lane] = share_pack(q);
  const int s = ilt_sum4((q[0] + q[1]) + (q[2] + q[3]));
  if ((lane & 3) == 0) bsums[b * 16 + (lane >> 2)] = s;
  if (lane == 0) kd[b] = any ? 1.0f / iscale : 0.0f;
}
__device__ __forceinline__ float4 share_ld(const float* __restrict__ x, u32 b) { return ((const float4*)(x + (long)b * 256))[threadIdx.x & 63]; }

constexpr int kOpenWaves = 9;  // a wave a token
// A pass's first launch: workgroup 0 routes and groups (one token a wave, a serial chain of 8 us: everything else a pass starts
// with fits beside it), the others quantize the tokens, a block a wave.  K 0: routed by a launch before.
template <int K>
__global__ __launch_bounds__(64 * kOpenWaves) void share_open_kernel(int ntok, int ne, int nu, float scale, const float* __restrict__ logits,
                                                          const float* __restrict__ bias, u32* __restrict__ rexp, u32* __restrict__ xrow,
                                                          float* __restrict__ wrow, u32* __restrict__ smap, const float* __restrict__ x, u32 nblocks,
                                                          i8* __restrict__ xq, float* __restrict__ xs, i8* __restrict__ kq, float* __restrict__ kd,
                                                          int* __restrict__ bsums) {
  if (blockIdx.x == 0) {
    if constexpr (K > 0) small_route<K>(ntok, ne, nu, scale, logits, bias, rexp, xrow, wrow, smap);
    return;
  }
  const u32 b = (blockIdx.x - 1) * kOpenWaves + (threadIdx.x >> 6);
  if (b >= nblocks) return;
  const float4 x4 = share_ld(x, b);
  const float v[4] = {x4.x, x4.y, x4.z, x4.w};
  share_q8(v, b, xq, xs);
  share_q8k(v, b, kq, kd, bsums);
}

// Between the products: the shared expert's gated activation in Q8_0 (nshared blocks of 256), the routed experts' in Q8_K, in
// one launch (5 us for 9).
__global__ __launch_bounds__(256) void share_mid_kernel(u32 nshared, const float* __restrict__ g, const float* __restrict__ u, float clamp,
                                                        i8* __restrict__ mq, float* __restrict__ ms, u32 nblocks, const float* __restrict__ x,
                                                        i8* __restrict__ kq, float* __restrict__ kd, int* __restrict__ bsums) {
  const u32 b = blockIdx.x * 4 + (threadIdx.x >> 6);
  float v[4];
  if (b < nshared) {                                   // d4_swiglu_w without weights
    const float4 g4 = share_ld(g, b), u4 = share_ld(u, b);
    const float gs[4] = {g4.x, g4.y, g4.z, g4.w}, us[4] = {u4.x, u4.y, u4.z, u4.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      float gk = gs[k], uk = us[k];
      if (clamp > 1e-6f) { gk = fminf(gk, clamp); uk = fmaxf(-clamp, fminf(uk, clamp)); }
      v[k] = ilt_silu(gk) * uk;
    }
    share_q8(v, b, mq, ms);
  } else if (b - nshared < nblocks) {
    const float4 x4 = share_ld(x, b - nshared);
    v[0] = x4.x; v[1] = x4.y; v[2] = x4.z; v[3] = x4.w;
    share_q8k(v, b - nshared, kq, kd, bsums);
  }
}

template <int FMT>
hipError_t launch_share(ShareArgs& p, const IltShareBeside* beside, hipStream_t st) {
  using F = ShareFmt<FMT>;
  const int S = p.S, rb = F::STEPS * (16 / S), gx = (p.rows + 4 * rb - 1) / (4 * rb);
  size_t lds = (FMT == ILT_IQ2_XXS ? 384 * 4 : 0) + 4ull * F::R * F::MATS * rb * (S * F::TERMS + 1) * 4;
  if (beside) {
    const IltShareBeside& q = *beside;
    if (q.ntok < 1 || q.ntok > kBesideTokens || q.cols < 256 || q.cols > 4096 || q.cols % 256 || q.rows < 2 || q.rows % 2 || q.nmat < 1 || q.nmat > 2) return hipErrorInvalidValue;
    const int rw = q.ntok <= 6 ? 2 : 1, tiles = (q.nmat * q.rows + 4 * rw - 1) / (4 * rw);
    p.beside = q; p.by = (tiles + gx - 1) / gx;
    lds = std::max(lds, (size_t)16 * rw * q.ntok * (q.cols / 32 + 1));      // (25 KB at most)
  }
  if (p.n + p.by > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(share_kernel<FMT>, dim3(gx, p.n + p.by), dim3(256), lds, st, p);
  return hipGetLastError();
}

}  // namespace

int ilt_k_share_takes(int d, int ff) {
  auto ok = [](int cols) { return cols > 0 && cols % 256 == 0 && cols <= 4096; };
  return ok(d) && ok(ff);
}

hipError_t ilt_k_share_open(int ne, int nu, float scale, const float* logits, const float* bias, int ntok, uint32_t* rexp, uint32_t* xrow, float* wrow,
                            uint32_t* smap, const float* x, int d, int8_t* xq, float* xs, int8_t* kq, float* kd, int* bsums, hipStream_t st) {
  if (ntok < 1 || ntok > kOpenWaves || ne < 1 || ne > 1024 || nu < 1 || nu > 64 || nu > ne || ntok * nu > 1024 || d < 256 || d % 256) return hipErrorInvalidValue;
  const u32 nblocks = (u32)ntok * (d / 256);
#define OPEN(K) hipLaunchKernelGGL(share_open_kernel<K>, dim3(1 + (nblocks + kOpenWaves - 1) / kOpenWaves), dim3(64 * kOpenWaves), 0, st, ntok, ne, nu, scale, logits, bias, rexp, xrow, \
                                   wrow, smap, x, nblocks, xq, xs, kq, kd, bsums)
  if (ne <= 64) OPEN(1);
  else if (ne <= 128) OPEN(2);
  else if (ne <= 256) OPEN(4);
  else if (ne <= 512) OPEN(8);
  else {                                               // (16 experts a lane spill their registers: once, in the kernel on its own)
    const hipError_t e = ilt_k_small_route(ne, nu, scale, logits, bias, ntok, rexp, xrow, wrow, smap, st);
    if (e != hipSuccess) return e;
    OPEN(0);
  }
#undef OPEN
  return hipGetLastError();
}

hipError_t ilt_k_share_mid(int ntok, int rows, int ff, float clamp, const float* g, const float* u, int8_t* mq, float* ms, const float* x, int8_t* kq,
                           float* kd, int* bsums, hipStream_t st) {
  if (ntok < 1 || rows < 1 || ff < 256 || ff % 256 || (long long)(ntok + rows) * ff > (1LL << 32)) return hipErrorInvalidValue;
  const u32 ns = (u32)ntok * (ff / 256), nr = (u32)rows * (ff / 256);
  hipLaunchKernelGGL(share_mid_kernel, dim3((ns + nr + 3) / 4), dim3(256), 0, st, ns, g, u, clamp, mq, ms, nr, x, kq, kd, bsums);
  return hipGetLastError();
}

hipError_t ilt_k_share_gate_up(const uint64_t* ptrs, long long gate, long long up, int d, int ff, int n, const uint32_t* rexp, const uint32_t* xrow,
                               const int8_t* kq, const float* kd, const float* wts, float clamp, float* y, const IltShareBeside* beside, hipStream_t st) {
  if (n < 1 || n > 65535) return hipErrorInvalidValue;
  ShareArgs p = {};
  p.ptrs = (const u64*)ptrs; p.rexp = rexp; p.xrow = xrow; p.xq = kq; p.xd = kd; p.add = gate; p.add2 = up; p.wts = wts; p.clamp = clamp; p.y = y;
  p.rows = ff; p.row_bytes = d / 256 * 66; p.S = d / 256; p.n = n;
  return launch_share<ILT_IQ2_XXS>(p, beside, st);
}

hipError_t ilt_k_share_down(const uint64_t* ptrs, long long add, int ff, int d, int n, const uint32_t* rexp, const int8_t* kq, const float* kd,
                            const int* bsums, float* y, const IltShareBeside* beside, hipStream_t st) {
  if (n < 1 || n > 65535) return hipErrorInvalidValue;
  ShareArgs p = {};
  p.ptrs = (const u64*)ptrs; p.rexp = rexp; p.xq = kq; p.xd = kd; p.bsums = bsums; p.add = add; p.y = y;
  p.rows = d; p.row_bytes = ff / 256 * 84; p.S = ff / 256; p.n = n;
  return launch_share<ILT_Q2_K>(p, beside, st);
}
