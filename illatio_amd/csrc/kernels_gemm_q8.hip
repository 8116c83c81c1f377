// The exact prefill product of Q8_0 rows: Y[t][r] = W[r].x_t with the CPU path's bits (tensor.lisp:329-336), for up to four
// matrices on the same quantized tokens in a launch.
//
// Q8_0 scales every block of 32 in float on either side, sum += float(isum) * (dw * dx), block after block, so there is nothing
// to fold into integers and what bounds the product is the vector ALU: four operations a block and result -- the two scales'
// product, the integer as a float, the term and the sum.  The integer costs a subtraction, not a conversion: the matrix core adds
// to 0x4B400000, the bits of 12582912.0f, and a block's integer is below 2^22 (a conversion takes as long as 1.6 of the
// additions).  A wave takes RP x TP patches of 16 rows x 16 tokens: v_mfma_i32_16x16x32_i8 is one block deep, and its four results
// a lane want four tokens' scales from LDS where the 32 x 32 form wants sixteen (of LDS's traffic that was half).
//
// Both operands' slabs of 64 columns, and the scales of their two blocks, come by direct loads into a ring of ST stages; a step is
// one wait and one barrier.  Where a wave's results lie in registers over the whole row, a small product is a chain of steps: the
// ring's depth hides the memory's latency, and the smaller the tile the more waves share the chip.
#include "ilt_device.h"
#include "ilt_kernels.h"
#include <stdlib.h>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

struct Q8Mat { const u8* w; const u16* wd; float* y; const float* bias; long long ldy; int rows, tile0; };
struct Q8Params {
  Q8Mat mat[4];
  int nmat, cols, ntok, acc, rtiles, ttiles;      // tiles of rows (all matrices'), of tokens
  const i8* xq; const float* xs;
};

template <int MS, int RP, int TP, int WR, int WT, int KB> struct Q8Tile {
  static constexpr int TR = MS * RP * WR, TT = MS * TP * WT, THREADS = 64 * WR * WT;
  static constexpr int RB = 32 * KB, PC = 2 * KB;                      // bytes and 16-byte pieces of a row a step
  static constexpr int NP = (TR + TT) * PC / THREADS;                   // 16-byte pieces a thread sends for a step
  static constexpr int NS = (TR * KB / 2 + KB * TT + THREADS - 1) / THREADS;     // words of scales
  static constexpr int SLAB = (TR + TT) * RB, STAGE = SLAB + NS * THREADS * 4;
};

// where piece pk of a row lies in its slab: the rows a read takes together on different banks
template <int KB> __device__ __forceinline__ int q8_swz(int row) { return KB == 2 ? (row >> 2) & 3 : (row >> 1) & 7; }

template <int MS> struct Q8Acc;
template <> struct Q8Acc<16> {
  typedef v4f F; typedef v4i I; typedef long O;
  static __device__ __forceinline__ O load(const void* p) { const int2 v = ilt_lds_ld8(p); return (long)((u64)(u32)v.x | ((u64)(u32)v.y << 32)); }
  static __device__ __forceinline__ I mul(O x, O w, I c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(x, w, c, 0, 0, 0); }
};
template <> struct Q8Acc<32> {
  typedef v16f F; typedef v16i I; typedef v4i O;
  static __device__ __forceinline__ O load(const void* p) { const int4 v = ilt_lds_ld16(p); return v4i{v.x, v.y, v.z, v.w}; }
  static __device__ __forceinline__ I mul(O x, O w, I c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(x, w, c, 0, 0, 0); }
};

template <int MS, int RP, int TP, int WR, int WT, int KB, int ST, int OCC>
__global__ __launch_bounds__(64 * WR * WT, OCC) void gemm_q8_kernel(Q8Params p) {
  using T = Q8Tile<MS, RP, TP, WR, WT, KB>;
  constexpr int TR = T::TR, TT = T::TT, NTH = T::THREADS;
  extern __shared__ __align__(16) unsigned char smem[];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), r = lane & (MS - 1), q = lane / MS;
  // each die walks a run of tiles, eight row tiles of one token tile after another (both operands' slabs stay in its L2)
  const int total = p.rtiles * p.ttiles, per = (total + 7) >> 3, s = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || s >= total) return;
  const int rg = s / (8 * p.ttiles), rem = s - rg * 8 * p.ttiles, nr = min(8, p.rtiles - 8 * rg), tt = rem / nr, rt = 8 * rg + rem - tt * nr;
  int mi = 0;
  while (mi + 1 < p.nmat && rt >= p.mat[mi + 1].tile0) mi++;
  const Q8Mat& m = p.mat[mi];
  const int r0 = (rt - m.tile0) * TR, tok0 = tt * TT, rows = min(TR, m.rows - r0), ntok = min(TT, p.ntok - tok0);
  const int nk = p.cols / (32 * KB), nb = p.cols / 32;

  const u8* const wbase = (const u8*)ilt_uniform_ptr((const i8*)m.w + (long)r0 * p.cols);
  const u8* const xbase = (const u8*)ilt_uniform_ptr(p.xq + (long)tok0 * p.cols);
  const u8* const dwbase = (const u8*)ilt_uniform_ptr((const i8*)(m.wd + (long)r0 * nb));
  const u8* const dxbase = (const u8*)ilt_uniform_ptr((const i8*)(p.xs + (long)tok0 * nb));
  // (rows and tokens past the tile's are its last: loaded, never stored)
  u32 off[T::NP], soff[T::NS], sstep[T::NS];
#pragma unroll
  for (int k = 0; k < T::NP; k++) {
    const int i = k * NTH + t, row = i / T::PC, pk = (i % T::PC) ^ q8_swz<KB>(row);        // a wave's rows: of one operand
    off[k] = (u32)(row < TR ? min(row, rows - 1) : min(row - TR, ntok - 1)) * (u32)p.cols + 16 * pk;
  }
  // (words: pairs of row scales [pair][row], then the tokens' [block][token])
#pragma unroll
  for (int k = 0; k < T::NS; k++) {
    const int i = k * NTH + t, j = i - TR * KB / 2;
    soff[k] = j < 0 ? (u32)min(i % TR, rows - 1) * (u32)nb * 2 + 4 * (i / TR) : ((u32)min(j % TT, ntok - 1) * (u32)nb + min(j / TT, KB - 1)) * 4;
    sstep[k] = j < 0 ? 2 * KB : 4 * KB;
  }
  auto issue = [&](unsigned char* stage, int ks) {
#pragma unroll
    for (int k = 0; k < T::NP; k++) {
      const bool isw = (k * NTH + wave * 64) / T::PC < TR;
      ilt_g2lds16((isw ? wbase : xbase) + (off[k] + (u32)T::RB * ks), stage + (k * NTH + wave * 64) * 16);
    }
#pragma unroll
    for (int k = 0; k < T::NS; k++) {
      const bool isw = k * NTH + t < TR * KB / 2;
      __builtin_amdgcn_global_load_lds((const ILT_GLOBAL void*)((isw ? dwbase : dxbase) + (soff[k] + sstep[k] * ks)),
                                       (ILT_LDS void*)(stage + T::SLAB + (k * NTH + wave * 64) * 4), 4, 0, 0);
    }
  };

  constexpr int NR = MS * MS / 64;                  // results a lane and patch: tokens 8 (i / 4) + 4 q + i % 4 (16: 4 q + i), row r
  typedef typename Q8Acc<MS>::F vf;
  typedef typename Q8Acc<MS>::I vi;
  typedef typename Q8Acc<MS>::O O;
  const int wr0 = MS * RP * (wave % WR), wt0 = MS * TP * (wave / WR);
  // a lane's part of a block: 8 bytes (16: 16 x 16 patches) or 16
  auto part = [&](int row, int b) {
    const int sw = q8_swz<KB>(row);
    return MS == 16 ? (u32)row * T::RB + 16 * ((2 * b + (q >> 1)) ^ sw) + 8 * (q & 1) : (u32)row * T::RB + 16 * ((2 * b + q) ^ sw);
  };
  u32 roff[RP][KB], toff[TP][KB];
#pragma unroll
  for (int b = 0; b < KB; b++) {
#pragma unroll
    for (int i = 0; i < RP; i++) roff[i][b] = part(wr0 + MS * i + r, b);
#pragma unroll
    for (int i = 0; i < TP; i++) toff[i][b] = part(TR + wt0 + MS * i + r, b);
  }
  const u32 dwoff = T::SLAB + (u32)(wr0 + r) * 4, dxoff = T::SLAB + (u32)(TR * KB / 2 + wt0 + 4 * q) * 4;

  vf sum[TP][RP];
#pragma unroll
  for (int a = 0; a < TP; a++)
#pragma unroll
    for (int b = 0; b < RP; b++)
#pragma unroll
      for (int i = 0; i < NR; i++) sum[a][b][i] = 0.0f;
  constexpr int NL = T::NP + T::NS;
#pragma unroll
  for (int i = 0; i < ST - 1; i++) issue(smem + i * T::STAGE, min(i, nk - 1));
  vi magic;
#pragma unroll
  for (int i = 0; i < NR; i++) magic[i] = 0x4B400000;
  unsigned char *cur = smem, *fill = smem + (ST - 1) * T::STAGE;
  for (int ks = 0; ks < nk; ks++) {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"((ST - 2) * NL) : "memory");
    ilt_barrier_lds();                             // the step's slabs are in, and the stage to be filled has been read by all
    issue(fill, min(ks + ST - 1, nk - 1));
    __builtin_amdgcn_sched_barrier(0);
    float dw[RP][KB];
#pragma unroll
    for (int b = 0; b < RP; b++)
#pragma unroll
      for (int j = 0; j < KB / 2; j++) {
        const u32 d2 = *ILT_LDS_PTR(const u32, cur + dwoff + 4 * MS * b + 4 * TR * j);
        dw[b][2 * j] = ilt_h2f((u16)d2); dw[b][2 * j + 1] = ilt_h2f((u16)(d2 >> 16));
      }
    auto load_dx = [&](int a, int kk, float (&dx)[NR]) {
#pragma unroll
      for (int g = 0; g < NR / 4; g++) {
        const int4 d4 = ilt_lds_ld16(cur + dxoff + 4 * MS * a + 32 * g + 4 * TT * kk);
        dx[4 * g] = __int_as_float(d4.x); dx[4 * g + 1] = __int_as_float(d4.y); dx[4 * g + 2] = __int_as_float(d4.z); dx[4 * g + 3] = __int_as_float(d4.w);
      }
    };
    if constexpr (RP * TP == 1) {                    // one patch a wave: a block's operands as they are wanted (all of them first: 3 % slower)
#pragma unroll
      for (int kk = 0; kk < KB; kk++) {
        const O wv = Q8Acc<MS>::load(cur + roff[0][kk]), xv = Q8Acc<MS>::load(cur + toff[0][kk]);
        float dx[NR];
        load_dx(0, kk, dx);
        const vi d = Q8Acc<MS>::mul(xv, wv, magic);
#pragma unroll
        for (int i = 0; i < NR; i++) sum[0][0][i] = sum[0][0][i] + (__int_as_float(d[i]) - 12582912.0f) * (dw[0][kk] * dx[i]);
      }
    } else {
      // a patch's products are made while the one before it is scaled and added, four results side by side: one after another every
      // instruction waited for the one before it (4096 x 4096 on 1,000 tokens: tiles of 64 x 64 90.8 -> 84.4 us, on 100, where a CU has
      // one of them, 44.4 -> 33.2; of 128 x 128 98 -> 90)
      constexpr int N = KB * TP * RP;
      O wv[KB][RP], xv[KB][TP];
#pragma unroll
      for (int kk = 0; kk < KB; kk++) {
#pragma unroll
        for (int b = 0; b < RP; b++) wv[kk][b] = Q8Acc<MS>::load(cur + roff[b][kk]);
#pragma unroll
        for (int a = 0; a < TP; a++) xv[kk][a] = Q8Acc<MS>::load(cur + toff[a][kk]);
      }
      float dx[2][NR];
      load_dx(0, 0, dx[0]);
      vi d[2];
      d[0] = Q8Acc<MS>::mul(xv[0][0], wv[0][0], magic);
#pragma unroll
      for (int k = 0; k < N; k++) {
        const int kk = k / (TP * RP), a = k / RP % TP, b = k % RP, n = k + 1;
        if (n < N) {
          if (n % RP == 0) load_dx(n / RP % TP, n / (TP * RP), dx[n / RP & 1]);
          d[n & 1] = Q8Acc<MS>::mul(xv[n / (TP * RP)][n / RP % TP], wv[n / (TP * RP)][n % RP], magic);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NR; i += 4) {
          float u[4], m[4];
#pragma unroll
          for (int j = 0; j < 4; j++) { u[j] = __int_as_float(d[k & 1][i + j]) - 12582912.0f; m[j] = dw[b][kk] * dx[k / RP & 1][i + j]; }
          asm volatile("" : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]), "+v"(m[0]), "+v"(m[1]), "+v"(m[2]), "+v"(m[3]));
#pragma unroll
          for (int j = 0; j < 4; j++) u[j] = u[j] * m[j];
          asm volatile("" : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
#pragma unroll
          for (int j = 0; j < 4; j++) sum[a][b][i + j] = sum[a][b][i + j] + u[j];
        }
        asm volatile("" : "+v"(sum[a][b]));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    fill = cur;
    cur += T::STAGE;
    if (cur == smem + ST * T::STAGE) cur = smem;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the tail's redundant loads: nothing may land in LDS after the workgroup ends

  const u32 ldy4 = (u32)m.ldy * 4;
  const __amdgpu_buffer_rsrc_t ry = ilt_rsrc(ilt_uniform_ptr(m.y + (long)tok0 * m.ldy), (u32)(ntok - 1) * ldy4 + (u32)m.rows * 4);
#pragma unroll
  for (int b = 0; b < RP; b++) {
    const int row = wr0 + MS * b + r;
    const bool ok = row < rows;
    const u32 base = ok ? (u32)(wt0 + 4 * q) * ldy4 + (u32)(r0 + row) * 4 : 0x80000000u;
    const float bv = m.bias && ok ? m.bias[r0 + row] : 0.0f;
#pragma unroll
    for (int a = 0; a < TP; a++)
#pragma unroll
      for (int i = 0; i < NR; i++) {
        float v = sum[a][b][i];
        const u32 o = base + (u32)(MS * a + 8 * (i >> 2) + (i & 3)) * ldy4;
        if (m.bias) v = v + bv;
        if (p.acc) v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ry, o, 0, 0)) + v;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(u32, v), ry, o, 0, 0);
      }
  }
}

template <int MS, int RP, int TP, int WR, int WT, int KB, int ST, int OCC>
hipError_t q8_launch(Q8Params& p, hipStream_t st) {
  using T = Q8Tile<MS, RP, TP, WR, WT, KB>;
  p.rtiles = 0;
  for (int i = 0; i < p.nmat; i++) { p.mat[i].tile0 = p.rtiles; p.rtiles += (p.mat[i].rows + T::TR - 1) / T::TR; }
  p.ttiles = (p.ntok + T::TT - 1) / T::TT;
  const long long per = ((long long)p.rtiles * p.ttiles + 7) / 8;
  if (per * 8 > 0x7FFFFFFFLL) return hipErrorNotSupported;
  constexpr int bytes = ST * T::STAGE;
  static_assert((T::TR + T::TT) * T::PC % T::THREADS == 0, "whole pieces a thread");
  static_assert(bytes <= 64 * 1024, "more LDS than a launch gets unasked");
  hipLaunchKernelGGL((gemm_q8_kernel<MS, RP, TP, WR, WT, KB, ST, OCC>), dim3((unsigned)(per * 8)), dim3(T::THREADS), bytes, st, p);
  return hipGetLastError();
}

// What a workgroup of each kind of tile takes for 4,096 columns, microseconds, with 1, 2, ... of them on a CU (4,096 rows on 64 to
// 2,304 tokens): a small tile is the shortest chain of steps, a large one reads LDS less a result.  Workgroups past those that fit
// take over the places that come free, all but the largest's, which start and end together.  (4096 x 4096 on 1,000 tokens: 128 x 64 68.9
// us, 64 x 64 84.4; 9728 x 896 on 301 20.2 and 18.7; 4096 x 4096 on 4,096 261, 312, and 230 for 128 x 128.)  Other widths are chosen for by
// the same figures: what grows with the columns and what a launch costs by itself are not apart in them.
struct Q8Kind { int rows, tokens, fit; float us[5]; };
constexpr Q8Kind kQ8Tiles[] = {
  {32, 32, 4, {15.2f, 19.0f, 26.0f, 33.2f}},
  {64, 64, 5, {33.0f, 43.8f, 65.8f, 84.6f, 102.0f}},
  {128, 64, 3, {54.5f, 69.2f, 102.0f}},
  {128, 128, 2, {90.0f, 116.8f}},
};
float q8_time(const Q8Kind& c, const Q8Params& p) {
  long long n = 0;
  for (int i = 0; i < p.nmat; i++) n += (p.mat[i].rows + c.rows - 1) / c.rows;
  n *= (p.ntok + c.tokens - 1) / c.tokens;
  const long long full = 256LL * c.fit, rest = n % full;
  if (n <= full) return c.us[(n + 255) / 256 - 1];
  if (c.rows * c.tokens < 128 * 128) return c.us[c.fit - 1] * (float)n / (float)full;
  return (float)(n / full) * c.us[c.fit - 1] + (rest ? c.us[(rest + 255) / 256 - 1] : 0.0f);
}

}  // namespace

hipError_t ilt_k_gemm_q8(int nmat, const uint8_t* const* ws, const uint16_t* const* wds, const int* rows, float* const* ys, const float* const* biases,
                         int cols, const int8_t* xq, const float* xs, int ntok, int acc, hipStream_t st, long long ldy) {
  if (nmat < 1 || nmat > 4 || ntok < 1 || cols < 64 || cols % 64 || (long long)128 * cols >= 0x7FFFFFFFLL || ((uintptr_t)xq & 15) || ((uintptr_t)xs & 3)) return hipErrorNotSupported;
  Q8Params p = {};
  p.nmat = nmat; p.cols = cols; p.ntok = ntok; p.acc = acc; p.xq = xq; p.xs = xs;
  for (int i = 0; i < nmat; i++) {
    Q8Mat& m = p.mat[i];
    m.w = ws[i]; m.wd = wds[i]; m.y = ys[i]; m.bias = biases ? biases[i] : nullptr; m.rows = rows[i]; m.ldy = ldy ? ldy : rows[i];
    if (rows[i] < 1 || m.ldy < rows[i] || m.ldy * 1024 >= 0x7FFFFFFFLL || ((uintptr_t)ws[i] & 15) || ((uintptr_t)wds[i] & 3)) return hipErrorNotSupported;
  }
  // ILT_Q8_TILE (tests): 1 to 4, that one.
  const char* const f = getenv("ILT_Q8_TILE");
  int v = f ? atoi(f) : 0;
  if (v < 1 || v > 4) {
    float least = 0.0f;
    for (int k = cols % 128 ? 1 : 0; k < 4; k++) {
      const float us = q8_time(kQ8Tiles[k], p);
      if (!v || us < least) { v = k + 1; least = us; }
    }
  }
  if (v == 1 && cols % 128) v = 2;
  switch (v) {
    case 1: return q8_launch<16, 1, 1, 2, 2, 4, 4, 4>(p, st);
    case 2: return q8_launch<16, 2, 2, 2, 2, 2, 3, 5>(p, st);
    case 3: return q8_launch<32, 2, 1, 2, 2, 2, 3, 3>(p, st);
    default: return q8_launch<32, 2, 2, 2, 2, 2, 3, 2>(p, st);
  }
}
