// Prefill products of a few tokens (2 to about a hundred), exact: Y[t][r] = W[r].x_t with the decode kernel's bits, W in
// GGUF Q4_K / Q6_K / Q8_0 blocks.
//
// What bounds such a product is the matrix's way from memory and a launch's latency: 32 tokens on a Qwen3-4B layer are 57 MB
// of blocks (12 us at the rate a large copy reaches) and 6 GFLOP.  A tile of 64 or 128 rows, staged in LDS between barriers,
// leaves most of the CUs without a tile (1,024 rows: 16 of 256) and every tile a chain of load, wait, unpack, wait.  Here
// nothing is shared: a wave takes 16 rows (RT of them: 32) and 16 NT tokens through whole super-blocks by itself, its loads a
// super-block ahead in registers, straight into the operands of v_mfma_i32_16x16x32_i8 -- no LDS, no barrier on the way.
// The four waves of a workgroup share a tile's super-blocks out among them (super-block u to wave u mod 4), leave each
// block's float terms in LDS, and add them in the CPU's order at the end, so that even a matrix of 1,024 rows is 64
// workgroups of four waves.
//
// The operands.  Lane (r, q) = (lane & 15, lane >> 4) holds of row (or token) r eight bytes of a group of 32 columns; which
// eight does not matter to the integer sum as long as weights and tokens agree.  Both come as 16-byte loads of 64
// consecutive bytes a row (lanes q = 0, 1 the first group, 2, 3 the second), and v_permlane32_swap_b32 on the halves of the
// two registers pairs deals each group to all four q: bytes 16 (q & 1) + 8 (q >> 1) of it.  Q6_K scales every 16 columns:
// v_permlane16_swap_b32 then leaves the group's first 16 columns in one register (bytes 4 q) and the second in the other, and
// a second product with the weights' operand {w, 0} has the first 16's sum alone.  Tokens are the product's M side and rows its N side, so a
// lane's results all belong to its own row and the row's scales never leave the lane.  The minimums (Q4_K) and the offset
// of 32 (Q6_K) are one f16 product of the sums of 16 quants (at most 2,032) with the 6- or 8-bit scales: whole
// numbers below 2^23, so exact in its single-precision accumulators.
#include "ilt_device.h"
#include "ilt_kernels.h"
#include <stdlib.h>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));


struct FewMat {
  const u8* w; const u16* wd;            // Q8_0: quants and f16 scales
  float* y; const float* bias;
  long long row_bytes, ldy;
  int rows, fmt, tile0;                  // tile0: the matrix's first row tile among the launch's
};
struct FewParams {
  FewMat mat[4];
  int nmat, cols, ntok, ttiles, acc;
  int units, uround;                     // units of columns in all, and in a round (what LDS holds the terms of)
  const i8* xq; const float* xs; const int* bsums;
};

// columns a unit has, float terms a unit leaves, activation scales a unit has
template <int FMT> struct FF;
template <> struct FF<ILT_Q4_K> { static constexpr int COLS = 256, TERMS = 2, SCALES = 1, XL = 4; };
template <> struct FF<ILT_Q6_K> { static constexpr int COLS = 256, TERMS = 1, SCALES = 1, XL = 4; };
template <> struct FF<ILT_Q8_0> { static constexpr int COLS = 64, TERMS = 2, SCALES = 2, XL = 1; };

__device__ __forceinline__ void swap32(int& a, int& b) {      // lanes 32..63 of a for lanes 0..31 of b
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0]; b = r[1];
}
__device__ __forceinline__ void swap16(int& a, int& b) {      // lanes 16..31 and 48..63 of a for lanes 0..15 and 32..47 of b
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0]; b = r[1];
}
__device__ __forceinline__ long pair(int lo, int hi) { return (long)((u64)(u32)lo | ((u64)(u32)hi << 32)); }
// 16 bytes of each of 64 consecutive ones a row: v.x, v.y the lane's share of the first 32, v.z, v.w of the second
__device__ __forceinline__ void deal(int4& v) { swap32(v.x, v.z); swap32(v.y, v.w); }

// ---- the weights of 16 rows, one unit -----------------------------------------------------------------
template <int FMT> struct FewW;
template <> struct FewW<ILT_Q4_K> { int4 hdr, q[2]; };
template <> struct FewW<ILT_Q6_K> { int4 l[2], sc; int2 h[2]; u16 d; };
template <> struct FewW<ILT_Q8_0> { int4 q; u16 d[2]; };

// (w: the matrix, the same in every lane, and 32-bit offsets: half the registers that a pointer a row takes)
__device__ __forceinline__ void few_load(FewW<ILT_Q4_K>& r, const u8* __restrict__ w, u32 row, const u16* __restrict__, u32, int u, int q, int) {
  const u8* b = w + (size_t)(row + (u32)u * 144u);
  r.hdr = *(const int4*)b;
  const u8* c = w + (size_t)(row + (u32)u * 144u + 16u * q);
  r.q[0] = *(const int4*)(c + 16);
  r.q[1] = *(const int4*)(c + 80);
}
__device__ __forceinline__ void few_load(FewW<ILT_Q6_K>& r, const u8* __restrict__ w, u32 row, const u16* __restrict__, u32, int u, int q, int) {
  const u32 o = row + (u32)u * (u32)ILT_Q6K_STRIDE;
  const u8 *b = w + (size_t)o, *c = w + (size_t)(o + 16u * q), *h = w + (size_t)(o + 16u * (q & 1) + 8u * (q >> 1));
  r.l[0] = ilt_ld16(c);
  r.l[1] = ilt_ld16(c + 64);
  r.h[0] = ilt_ld8(h + 128);
  r.h[1] = ilt_ld8(h + 160);
  r.sc = ilt_ld16(b + 192);
  r.d = ilt_ld2(b + 208);
}
// (a row's last unit may be half a one: what lies past the row is read from its last 64 bytes' place and masked)
__device__ __forceinline__ void few_load(FewW<ILT_Q8_0>& r, const u8* __restrict__ w, u32 row, const u16* __restrict__ wd, u32 drow, int u, int q, int cols) {
  r.q = *(const int4*)(w + (size_t)(row + (u32)min(64 * u + 16 * q, cols - 16)));
  const int nb = cols >> 5;
  r.d[0] = wd[(size_t)(drow + 2u * u)];
  r.d[1] = wd[(size_t)(drow + (u32)min(2 * u + 1, nb - 1))];
}

// ---- the tokens' quants (and sums of 16) of one unit ---------------------------------------------------
template <int FMT, int NT> struct FewX { int4 x[NT][FF<FMT>::XL], bs[NT]; };
template <int FMT, int NT>
__device__ __forceinline__ void few_load_x(FewX<FMT, NT>& r, const i8* __restrict__ xq, const int* __restrict__ bsums, const u32 (&xrow)[NT], int u, int q, int cols) {
#pragma unroll
  for (int np = 0; np < NT; np++) {
    if constexpr (FMT == ILT_Q8_0) r.x[np][0] = *(const int4*)(xq + (size_t)(xrow[np] + (u32)min(64 * u + 16 * q, cols - 16)));
    else {
#pragma unroll
      for (int s = 0; s < 4; s++) r.x[np][s] = *(const int4*)(xq + (size_t)(xrow[np] + 256u * u + 16u * q) + 64 * s);
      r.bs[np] = *(const int4*)(bsums + (size_t)((xrow[np] >> 4) + 16u * u + 4u * q));
    }
  }
}

__device__ __forceinline__ v4h halves(float a, float b, float c, float d) { return v4h{(_Float16)a, (_Float16)b, (_Float16)c, (_Float16)d}; }
__device__ __forceinline__ int sbyte(int v, int i) { return (v << (24 - 8 * i)) >> 24; }
__device__ __forceinline__ int ubyte(int v, int i) { return (u32)(v << (24 - 8 * i)) >> 24; }

// One unit's float terms of 16 RT rows x 16 NT tokens: t[k][rp][np], k < TERMS; yd: the activation scales of the unit,
// tokens 4q .. 4q+3 of each patch.  The expressions are the CPU kernels' (kquant.lisp:180-236, tensor.lisp:329-336).
template <int NT, int RT>
__device__ __forceinline__ void few_unit(const FewW<ILT_Q4_K> (&w)[RT], FewX<ILT_Q4_K, NT>& x, const float* yd, int q, v4f (&t)[2][RT][NT]) {
  v4i isum[RT][NT];
#pragma unroll
  for (int rp = 0; rp < RT; rp++)
#pragma unroll
    for (int np = 0; np < NT; np++) isum[rp][np] = v4i{0, 0, 0, 0};
  int sc[RT][2], mn[RT][2];
#pragma unroll
  for (int rp = 0; rp < RT; rp++) {
    const u32 a = (u32)w[rp].hdr.y, b = (u32)w[rp].hdr.z, c = (u32)w[rp].hdr.w;       // get_scale_min_k4, four groups a word
    sc[rp][0] = (int)(a & 0x3F3F3F3F); mn[rp][0] = (int)(b & 0x3F3F3F3F);
    sc[rp][1] = (int)((c & 0x0F0F0F0F) | ((a >> 2) & 0x30303030));
    mn[rp][1] = (int)(((c >> 4) & 0x0F0F0F0F) | ((b >> 2) & 0x30303030));
  }
#pragma unroll
  for (int m = 0; m < 2; m++) {
    int4 wq[RT];
#pragma unroll
    for (int rp = 0; rp < RT; rp++) { wq[rp] = w[rp].q[m]; deal(wq[rp]); }
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int s = 2 * m + e;
#pragma unroll
      for (int np = 0; np < NT; np++) deal(x.x[np][s]);
#pragma unroll
      for (int rp = 0; rp < RT; rp++) {
        const int w0 = e ? wq[rp].z : wq[rp].x, w1 = e ? wq[rp].w : wq[rp].y;
        const long lo = pair(w0 & 0x0F0F0F0F, w1 & 0x0F0F0F0F), hi = pair((int)((u32)w0 >> 4) & 0x0F0F0F0F, (int)((u32)w1 >> 4) & 0x0F0F0F0F);
        const int s0 = ubyte(sc[rp][m], 2 * e), s1 = ubyte(sc[rp][m], 2 * e + 1);
#pragma unroll
        for (int np = 0; np < NT; np++) {
          const v4i z = {0, 0, 0, 0};
          const v4i d0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pair(x.x[np][s].x, x.x[np][s].y), lo, z, 0, 0, 0);
          const v4i d1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pair(x.x[np][s].z, x.x[np][s].w), hi, z, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; i++) isum[rp][np][i] = ilt_mad24(s0, d0[i], isum[rp][np][i]);
          asm("" : "+v"(isum[rp][np]));       // (added up here: a sum put off to the end keeps every product in a register)
#pragma unroll
          for (int i = 0; i < 4; i++) isum[rp][np][i] = ilt_mad24(s1, d1[i], isum[rp][np][i]);
          asm("" : "+v"(isum[rp][np]));
        }
      }
    }
  }
#pragma unroll
  for (int rp = 0; rp < RT; rp++) {
    const int mw = q < 2 ? mn[rp][0] : mn[rp][1], mq = (u32)mw >> (16 * (q & 1));       // the minimums of groups 2q and 2q + 1
    const float m0 = (float)(mq & 0xFF), m1 = (float)((mq >> 8) & 0xFF);
    const v4h mh = halves(m0, m0, m1, m1);
    const float dd = ilt_h2f((u16)(w[rp].hdr.x & 0xFFFF)), dm = ilt_h2f((u16)((u32)w[rp].hdr.x >> 16));
#pragma unroll
    for (int np = 0; np < NT; np++) {
      const v4h bh = halves((float)x.bs[np].x, (float)x.bs[np].y, (float)x.bs[np].z, (float)x.bs[np].w);
      const v4f imin = __builtin_amdgcn_mfma_f32_16x16x16f16(bh, mh, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
      const float4 y4 = *(const float4*)(yd + 16 * np + 4 * q);
      const float yv[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        t[0][rp][np][i] = -((yv[i] * dm) * imin[i]);
        t[1][rp][np][i] = (yv[i] * dd) * (float)isum[rp][np][i];
      }
    }
  }
}

template <int NT, int RT>
__device__ __forceinline__ void few_unit(const FewW<ILT_Q6_K> (&w)[RT], FewX<ILT_Q6_K, NT>& x, const float* yd, int q, v4f (&t)[1][RT][NT]) {
  v4i isum[RT][NT];
  // -32 * sum of scale * (sum of 16 quants): the quants' offset
#pragma unroll
  for (int rp = 0; rp < RT; rp++) {
    const int sw = q == 0 ? w[rp].sc.x : q == 1 ? w[rp].sc.y : q == 2 ? w[rp].sc.z : w[rp].sc.w;
    const v4h sh = halves((float)sbyte(sw, 0), (float)sbyte(sw, 1), (float)sbyte(sw, 2), (float)sbyte(sw, 3));
#pragma unroll
    for (int np = 0; np < NT; np++) {
      const v4h bh = halves((float)x.bs[np].x, (float)x.bs[np].y, (float)x.bs[np].z, (float)x.bs[np].w);
      const v4f im = __builtin_amdgcn_mfma_f32_16x16x16f16(bh, sh, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) isum[rp][np][i] = (int)im[i] * -32;
    }
  }
#pragma unroll
  for (int c = 0; c < 2; c++) {
    int4 l[RT]; int2 h[RT];
#pragma unroll
    for (int rp = 0; rp < RT; rp++) {
      l[rp] = w[rp].l[c]; h[rp] = w[rp].h[c];
      deal(l[rp]);
      swap16(l[rp].x, l[rp].y); swap16(l[rp].z, l[rp].w); swap16(h[rp].x, h[rp].y);
    }
#pragma unroll
    for (int hi = 0; hi < 2; hi++) {
      const int s = 2 * c + hi;
#pragma unroll
      for (int np = 0; np < NT; np++) { deal(x.x[np][s]); swap16(x.x[np][s].x, x.x[np][s].y); swap16(x.x[np][s].z, x.x[np][s].w); }
#pragma unroll
      for (int rp = 0; rp < RT; rp++) {
#pragma unroll
        for (int g = 0; g < 2; g++) {                  // the groups of 32 columns 4c + 2hi + g; top bits 2 (2hi + g) of the qh bytes
          const int la = g ? l[rp].z : l[rp].x, lb = g ? l[rp].w : l[rp].y, sh = 4 * hi + 2 * g;
          const int na = hi ? (int)((u32)la >> 4) : la, nb = hi ? (int)((u32)lb >> 4) : lb;
          const int ta = sh <= 4 ? h[rp].x << (4 - sh) : (int)((u32)h[rp].x >> (sh - 4)), tb = sh <= 4 ? h[rp].y << (4 - sh) : (int)((u32)h[rp].y >> (sh - 4));
          const int wa = (na & 0x0F0F0F0F) | (ta & 0x30303030), wb = (nb & 0x0F0F0F0F) | (tb & 0x30303030);
          const int k = 8 * c + 4 * hi + 2 * g, scw = (k >> 2) == 0 ? w[rp].sc.x : (k >> 2) == 1 ? w[rp].sc.y : (k >> 2) == 2 ? w[rp].sc.z : w[rp].sc.w;
          // sa * a + sb * b with the sum of the two from one product of the whole group: sb * (a + b) + (sa - sb) * a
          const int sb = sbyte(scw, (k & 3) + 1), sa = sbyte(scw, k & 3) - sb;
#pragma unroll
          for (int np = 0; np < NT; np++) {
            const long xv = g ? pair(x.x[np][s].z, x.x[np][s].w) : pair(x.x[np][s].x, x.x[np][s].y);
            const v4i z = {0, 0, 0, 0};
            const v4i da = __builtin_amdgcn_mfma_i32_16x16x32_i8(xv, pair(wa, 0), z, 0, 0, 0);
            const v4i db = __builtin_amdgcn_mfma_i32_16x16x32_i8(xv, pair(wa, wb), z, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) isum[rp][np][i] = ilt_mad24(sa, da[i], isum[rp][np][i]);
            asm("" : "+v"(isum[rp][np]));
#pragma unroll
            for (int i = 0; i < 4; i++) isum[rp][np][i] = ilt_mad24(sb, db[i], isum[rp][np][i]);
            asm("" : "+v"(isum[rp][np]));
          }
        }
      }
    }
  }
#pragma unroll
  for (int rp = 0; rp < RT; rp++) {
    const float dd = ilt_h2f(w[rp].d);
#pragma unroll
    for (int np = 0; np < NT; np++) {
      const float4 y4 = *(const float4*)(yd + 16 * np + 4 * q);
      const float yv[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
      for (int i = 0; i < 4; i++) t[0][rp][np][i] = (dd * yv[i]) * (float)isum[rp][np][i];
    }
  }
}

template <int NT, int RT>
__device__ __forceinline__ void few_unit(const FewW<ILT_Q8_0> (&w)[RT], FewX<ILT_Q8_0, NT>& x, const float* yd, int q, v4f (&t)[2][RT][NT]) {
#pragma unroll
  for (int np = 0; np < NT; np++) deal(x.x[np][0]);
#pragma unroll
  for (int rp = 0; rp < RT; rp++) {
    int4 wq = w[rp].q;
    deal(wq);
    const float d0 = ilt_h2f(w[rp].d[0]), d1 = ilt_h2f(w[rp].d[1]);
#pragma unroll
    for (int np = 0; np < NT; np++) {
      const v4i z = {0, 0, 0, 0};
      const v4i i0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pair(x.x[np][0].x, x.x[np][0].y), pair(wq.x, wq.y), z, 0, 0, 0);
      const v4i i1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pair(x.x[np][0].z, x.x[np][0].w), pair(wq.z, wq.w), z, 0, 0, 0);
      const float4 a4 = *(const float4*)(yd + 16 * np + 4 * q), b4 = *(const float4*)(yd + 16 * NT + 16 * np + 4 * q);
      const float av[4] = {a4.x, a4.y, a4.z, a4.w}, bv[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        t[0][rp][np][i] = (float)i0[i] * (d0 * av[i]);
        t[1][rp][np][i] = (float)i1[i] * (d1 * bv[i]);
      }
    }
  }
}

// One tile: rows row0 .. of the matrix m, tokens tok0 .. tok0 + ntok - 1 (at most 16 NT).  LDS: a round's activation scales
// [scale][token], then its terms [unit][term][patch][lane].
template <int FMT, int NT, int RT, int NW>
__device__ __forceinline__ void few_tile(const FewParams& p, const FewMat& m, int row0, long tok0, int ntok, unsigned char* smem) {
  using F = FF<FMT>;
  constexpr int TW = 16 * NT, OUTS = 256 * RT * NT;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, q = lane >> 4;
  const int units = (p.cols + F::COLS - 1) / F::COLS, nscale = FMT == ILT_Q8_0 ? p.cols >> 5 : p.cols >> 8;
  const int uround = p.uround;
  float* const xls = (float*)smem;
  float* const terms = xls + uround * F::SCALES * TW;
  u32 wrow[RT], drow[RT], xrow[NT];
#pragma unroll
  for (int rp = 0; rp < RT; rp++) {
    const u32 row = (u32)min(row0 + 16 * rp + r, m.rows - 1);
    wrow[rp] = row * (u32)m.row_bytes;
    drow[rp] = row * (u32)nscale;
  }
#pragma unroll
  for (int np = 0; np < NT; np++) xrow[np] = (u32)min(16 * np + r, ntok - 1) * (u32)p.cols;
  const i8* const xq = p.xq + tok0 * p.cols;
  const int* const bsums = FMT == ILT_Q8_0 ? nullptr : p.bsums + tok0 * (p.cols >> 4);
  FewW<FMT> wa[RT], wb[RT];
  FewX<FMT, NT> xa, xb;
  auto load = [&](FewW<FMT> (&w)[RT], FewX<FMT, NT>& x, int u) {
    u = min(u, units - 1);
#pragma unroll
    for (int rp = 0; rp < RT; rp++) few_load(w[rp], m.w, wrow[rp], m.wd, drow[rp], u, q, p.cols);
    few_load_x<FMT, NT>(x, xq, bsums, xrow, u, q, p.cols);
  };
  constexpr int NS = (OUTS + 64 * NW - 1) / (64 * NW);      // results a thread adds up
  float sum[NS];
#pragma unroll
  for (int j = 0; j < NS; j++) sum[j] = 0.0f;
  load(wa, xa, wave);
  for (int u0 = 0; u0 < units; u0 += uround) {
    const int u1 = min(u0 + uround, units);
    if (u0) __syncthreads();                            // the round before has been added
    for (int i = tid; i < (u1 - u0) * F::SCALES * TW; i += 64 * NW) {
      const int s = i / TW, tk = i % TW, g = u0 * F::SCALES + s;
      xls[i] = g < nscale ? p.xs[(tok0 + min(tk, ntok - 1)) * nscale + g] : 0.0f;
    }
    __syncthreads();
    auto unit = [&](const FewW<FMT> (&w)[RT], FewX<FMT, NT>& x, int u) {
      v4f t[F::TERMS][RT][NT];
      few_unit<NT, RT>(w, x, xls + (u - u0) * F::SCALES * TW, q, t);
#pragma unroll
      for (int k = 0; k < F::TERMS; k++)
#pragma unroll
        for (int rp = 0; rp < RT; rp++)
#pragma unroll
          for (int np = 0; np < NT; np++) *(v4f*)(terms + ((u - u0) * F::TERMS + k) * OUTS + (rp * NT + np) * 256 + 4 * lane) = t[k][rp][np];
    };
    // (uround is a multiple of 2 NW or all the units: a round starts with the wave's unit in wa)
    for (int u = u0 + wave; u < u1; u += 2 * NW) {
      load(wb, xb, u + NW);
      unit(wa, xa, u);
      load(wa, xa, u + 2 * NW);
      if (u + NW < u1) unit(wb, xb, u + NW);
    }
    __syncthreads();
    // the terms in the CPU's order, a result a thread and patch (a last half unit of Q8_0 leaves one term, not two)
    const int nt = FMT == ILT_Q8_0 ? min(2 * u1, nscale) - 2 * u0 : (u1 - u0) * F::TERMS;
#pragma unroll
    for (int j = 0; j < NS; j++) {
      const float* t = terms + 64 * NW * j + tid;
      if (64 * NW * j + tid >= OUTS) break;
      float o = sum[j];
      int k = 0;
      for (; k + 8 <= nt; k += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = t[(k + i) * OUTS];
#pragma unroll
        for (int i = 0; i < 8; i++) o = o + v[i];
      }
      for (; k < nt; k++) o = o + t[k * OUTS];
      sum[j] = o;
    }
  }
#pragma unroll
  for (int j = 0; j < NS; j++) {
    const int f = 64 * NW * j + tid, pt = f >> 8, rp = pt / NT, np = pt % NT, l = (f >> 2) & 63;
    const int row = row0 + 16 * rp + (l & 15), tk = 16 * np + 4 * (l >> 4) + (f & 3);
    if (f < OUTS && row < m.rows && tk < ntok) {
      float v = sum[j];
      if (m.bias) v = v + m.bias[row];
      float* yo = m.y + (tok0 + tk) * m.ldy + row;
      if (p.acc) v = *yo + v;
      *yo = v;
    }
  }
}

// FSET: the matrices' format, or 0 where Q4_K and Q6_K meet in a launch.  Registers: a Q6_K tile of two patches, alone or beside
// Q4_K, spills in the 168 that three workgroups a CU leave (a mixed launch of 1024 + 512 + 512 rows x 1024 on 17 tokens 7.1 us
// with twelve spilled, 6.3 with two workgroups; 2048 + 512 + 512 x 2560 10.2 and 9.5).
template <int FSET, int NT, int RT, int NW>
__global__ __launch_bounds__(64 * NW, (NW == 8 ? (NT == 1 ? 2 : 1) : RT * NT == 1 ? 4 : RT * NT == 2 && FSET != ILT_Q6_K && FSET != 0 ? 3 : 2)) void gemm_i8_few_kernel(FewParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  // the token tiles of a row tile next to one another on a die, so that its blocks come into that die's L2 once
  const int ntile = gridDim.x / p.ttiles, per = (ntile + 7) >> 3;
  int rt, tt;
  if ((ntile & 7) == 0) { const int k = blockIdx.x >> 3; rt = (blockIdx.x & 7) * per + k / p.ttiles; tt = k % p.ttiles; }
  else { rt = blockIdx.x / p.ttiles; tt = blockIdx.x % p.ttiles; }
  int mi = 0;
  while (mi + 1 < p.nmat && rt >= p.mat[mi + 1].tile0) mi++;
  const FewMat& m = p.mat[mi];
  const int row0 = (rt - m.tile0) * 16 * RT;
  const long tok0 = (long)tt * 16 * NT;
  const int ntok = min(16 * NT, p.ntok - (int)tok0);
  if constexpr (FSET != 0) few_tile<FSET, NT, RT, NW>(p, m, row0, tok0, ntok, smem);
  else if (m.fmt == ILT_Q4_K) few_tile<ILT_Q4_K, NT, RT, NW>(p, m, row0, tok0, ntok, smem);
  else few_tile<ILT_Q6_K, NT, RT, NW>(p, m, row0, tok0, ntok, smem);
}

template <int FSET, int NT, int RT, int NW>
hipError_t few_launch(FewParams& p, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < p.nmat; i++) { p.mat[i].tile0 = tiles; tiles += (p.mat[i].rows + 16 * RT - 1) / (16 * RT); }
  constexpr int terms = FSET == ILT_Q6_K ? 1 : 2, scales = FSET == ILT_Q8_0 ? 2 : 1, ucols = FSET == ILT_Q8_0 ? 64 : 256;
  constexpr int per = terms * 1024 * RT * NT + scales * 64 * NT;
  const int units = (p.cols + ucols - 1) / ucols;
  constexpr int room = 76 * 1024;                                // two workgroups a CU at least
  const int most = room / per / (2 * NW) * (2 * NW);
  p.uround = units <= most ? units : most;
  static bool attr_set[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!attr_set[dev]) {            // more dynamic LDS than the default 64 KB: asked for once per device
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_i8_few_kernel<FSET, NT, RT, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, room);
    if (e != hipSuccess) return e;
    attr_set[dev] = true;
  }
  static_assert(room / per >= 2 * NW, "a round is whole turns of the four waves' two register sets");
  hipLaunchKernelGGL((gemm_i8_few_kernel<FSET, NT, RT, NW>), dim3(tiles * p.ttiles), dim3(64 * NW), (size_t)p.uround * per, st, p);
  return hipGetLastError();
}

// How a launch is cut: 32 tokens a tile from 17 on; tiles of 16 rows with the columns shared out over four waves, or (Q8_0) over
// eight where a row is long and the launch has no more tiles than CUs (896 x 4864 on 21 tokens 20.6 -> 16.4 us); tiles of 32 rows, which read the tokens half as often, once tiles of 16 are more than the CUs
// take at a time (Q4_K 2560 x 4096 on 48 tokens, 320 tiles: 17.8 -> 14.2 us; on 32 tokens, 160: 10.5 against 14.1; Q8_0,
// whose units are short, from 600 tiles on: 4864 x 896 on 32 tokens, 304: 7.5 against 8.5, on 48, 608: 11.6 -> 10.5).
template <int FSET>
hipError_t few_dispatch(FewParams& p, int forced, hipStream_t st) {
  const int nt = p.ntok <= 16 ? 1 : 2;
  p.ttiles = (p.ntok + 16 * nt - 1) / (16 * nt);
  long tiles = 0;
  for (int i = 0; i < p.nmat; i++) tiles += (p.mat[i].rows + 15) / 16;
  tiles *= p.ttiles;
  const bool wide = tiles > (FSET == ILT_Q8_0 || nt == 1 ? 600 : 256), deep = tiles <= 256 && p.cols >= 2048;
  const int v = forced > 1 ? forced : wide ? 2 : deep ? 8 : 4;
  if constexpr (FSET == ILT_Q8_0) { if (v == 8) return nt == 1 ? few_launch<FSET, 1, 1, 8>(p, st) : few_launch<FSET, 2, 1, 8>(p, st); }      // (K-quants: four waves)
  if (nt == 1) return v == 2 ? few_launch<FSET, 1, 2, 4>(p, st) : few_launch<FSET, 1, 1, 4>(p, st);
  return v == 2 ? few_launch<FSET, 2, 2, 4>(p, st) : few_launch<FSET, 2, 1, 4>(p, st);
}

// Whether kernels_gemm_reg.hip's waves of 16 rows are the better ones (rows16: tiles of 16 rows; nsb: super-blocks of a row)
bool halves_take(bool q4, long long rows16, int ntok, int nsb) {
  const long long t16 = rows16 * ((ntok + 15) / 16), t32 = rows16 * ((ntok + 31) / 32);
  if (ntok <= 16) return t16 <= 512 ? nsb >= (q4 ? 14 : 4) : q4 ? ntok >= 12 && t16 >= 1024 : nsb >= 4;
  return t16 <= 256 ? !q4 || nsb >= 4 : t32 <= 256 && (!q4 || nsb >= 12);
}

}  // namespace

// Up to four matrices (all Q8_0, or Q4_K and Q6_K in any mix) on the same quantized tokens in one launch.
// hipErrorNotSupported (nothing launched) where the shapes are not this kernel's.  K-quants against the kernels with the weights in
// operand registers (kernels_gemm_reg.hip): those from 17 tokens on where the launch is more than 128 tiles of 32 x 32 (us here and there: Q4_K
// 6144 x 2560 on 21, 192 tiles: 12.1 and 11.5, 2560 x 4096 on 40, 160: 16.6 and 12.5), and their tiles of 16 rows, eight waves' each, where those fit the
// chip and their rounds of eight super-blocks have enough to do.  Up to 16 tokens (512 tiles of 16 tokens): Q4_K from fourteen on (2560 x 3072, twelve, on
// 16 6.6 and 6.8, x 3584 7.3 and 6.7; 8192 x 4096 13.0 and 11.8), else four (2560 x 512 5.0 and 5.1, x 1024 5.8 and 5.2; 8192 x 2560 11.0 and 10.6); past those tiles
// Q6_K as before (12288 x 4096 on 8 20.8 and 16.3), Q4_K from 1,024 tiles and twelve tokens on (19456 x 2560 on 4 13.2 and 13.6, 16 15.5 and 14.4).  More
// tokens, 256 tiles of 16: Q4_K from four on (1024 x 512 on 24 5.2 and 5.0, x 1024 5.6 and 5.2), Q6_K always (1024 x 256 5.4 and 4.9); 256 tiles of 32:
// Q4_K from twelve (4096 x 2560, ten, on 21 8.2 and 8.6; 2560 x 3072 on 24 8.8 and 8.3), Q6_K always (2560 x 512 6.3 and 5.6).  Q8_0 against its own kernel (kernels_gemm_q8.hip),
// whose waves make a tile's terms and sums in registers: up to 16 tokens here, unless the tiles of 16 rows fill the chip (896 x 4864
// on 16 tokens 12.7 us against 16.1, on 24 17.1 against 16.1; 4096 x 2048 on 16, 256 tiles: 8.1 against 8.3; 9728 x 896, 608:
// 7.7 against 5.8); where its smallest tile does not go (cols no multiple of 128) from 640 tiles of 32 x 32 and 96 tokens on.
// ILT_I8_FEW (tests): "0" never, "1" always, "2", "4" always, that cut, "8" Q8_0's over eight waves (K-quants: "4").
hipError_t ilt_k_gemm_i8_few(int nmat, const int* fmts, const uint8_t* const* ws, const uint16_t* const* wds, const int* rows, float* const* ys,
                             const float* const* biases, int cols, const int8_t* xq, const float* xs, const int* bsums, int ntok, int acc,
                             hipStream_t st, long long ldy) {
  const char* const f = getenv("ILT_I8_FEW");
  const int forced = f ? atoi(f) : -1;
  if (nmat < 1 || nmat > 4 || ntok < 1 || forced == 0 || (forced < 0 && getenv("ILT_I8_PLANES"))) return hipErrorNotSupported;
  FewParams p = {};
  p.nmat = nmat; p.cols = cols; p.ntok = ntok; p.acc = acc; p.xq = xq; p.xs = xs; p.bsums = bsums;
  int fset = fmts[0];
  long long tiles32 = 0, tiles16 = 0;
  bool small = false;                       // a matrix of less than a tile of the registers' kernel
  bool reg = nmat <= 3 && (nmat == 1 || !ldy) && cols < ILT_REG_COLS;      // what that kernel takes at all
  for (int i = 0; i < nmat; i++) {
    const int fm = fmts[i];
    if (fm != ILT_Q4_K && fm != ILT_Q6_K && fm != ILT_Q8_0) return hipErrorNotSupported;
    if (cols % (fm == ILT_Q8_0 ? 32 : 256)) return hipErrorNotSupported;
    if (fm != fset) { if (fm == ILT_Q8_0 || fset == ILT_Q8_0) return hipErrorNotSupported; fset = 0; }
    FewMat& m = p.mat[i];
    m.w = ws[i]; m.wd = wds ? wds[i] : nullptr; m.y = ys[i]; m.bias = biases ? biases[i] : nullptr; m.rows = rows[i]; m.fmt = fm;
    m.ldy = ldy ? ldy : rows[i];
    m.row_bytes = fm == ILT_Q8_0 ? cols : (long long)(cols / 256) * (fm == ILT_Q4_K ? 144 : ILT_Q6K_STRIDE);
    if (m.ldy < rows[i] || (long long)rows[i] * m.row_bytes >= 0x7FFFFFFFLL || (((uintptr_t)ws[i]) & 15)) return hipErrorNotSupported;   // 32-bit offsets
    tiles32 += (rows[i] + 31) / 32;
    tiles16 += (rows[i] + 15) / 16;
    small |= rows[i] < 128;
    reg &= rows[i] < ILT_REG_ROWS && m.ldy < ILT_REG_ROWS;
  }
  tiles32 *= (ntok + 31) / 32;
  if (tiles32 > 0x3FFFFFFF) return hipErrorNotSupported;
  if (forced < 0 && fset == ILT_Q8_0) {
    if (cols % 128 == 0 ? ntok > 16 || tiles32 > 128 : ntok >= 96 && tiles32 > 640) {
      const hipError_t e = ilt_k_gemm_q8(nmat, ws, wds, rows, ys, biases, cols, xq, xs, ntok, acc, st, ldy);
      if (e != hipErrorNotSupported) return e;
    }
  } else if (forced < 0 && ((!small && ntok > 16 && tiles32 > 128) || (reg && halves_take(fset != ILT_Q6_K, tiles16, ntok, cols / 256))))
    return hipErrorNotSupported;
  switch (fset) {
    case ILT_Q8_0: return few_dispatch<ILT_Q8_0>(p, forced, st);
    case ILT_Q4_K: return few_dispatch<ILT_Q4_K>(p, forced, st);
    case ILT_Q6_K: return few_dispatch<ILT_Q6_K>(p, forced, st);
    default: return few_dispatch<0>(p, forced, st);
  }
}
