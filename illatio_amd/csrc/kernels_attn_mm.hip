// A prompt chunk's attention with its products made by the matrix cores (heads of 64 and 128 columns), every number the CPU
// path's (attend-head!, model.lisp:298-334; F32-DOT16, tensor.lisp:370-378).
//
// Both halves of it are products rounded to single and then added in a fixed order, so no fused multiply-add and no sum
// inside the matrix cores will do.  But v_mfma_f32_16x16x1_4b_f32 has one product a result, and with zeros to add to, each
// result is that product rounded once (denormals and all: compared with v_mul_f32 over 26 million pairs; a product that
// rounds to -0 stays -0, where 0 + -0 would be +0: no sum here shows it).  A thousand products are one instruction that
// takes the time of sixteen adds, and its operands are sixteen rows and sixteen columns in one register each, straight from
// memory (the query rows of a long chunk's scores by way of LDS, a read an instruction).  The adds are the vector ALU's, a register of sixty-four sums an instruction.  (The
// two do not run at the same time on gfx950: an instruction with 16 results and 16 adds beside it take 33-36 ns a SIMD, 15
// and 17 apart; as mul and add they take 32.  What the matrix cores save is the operands' way: sixteen chains a thread
// read LDS once a chain and four products.)
//
// The query heads of a KV head see the same keys and values, so a KV head's rows -- token t, head g of its group: row
// t * group + g -- go through in tiles of 16 (or 4), whatever heads they are of.
#include "ilt_act_blocks.h"
#include "ilt_device.h"
#include "ilt_kernels.h"
#include "ilt_softmax.h"
#include "ilt_value_sets.h"
#include <type_traits>

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float part(const float4& v, int e) { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; }

constexpr int kShortMost = 448;        // positions of attn_short_mm_kernel

// raw[(t * nh + h) * spitch + p] = F32-DOT16(K[p], q) * scale.  A wave takes 16 rows and, one after another, npt tiles of 16
// positions.  Block m of the instruction has columns 4m + e of every sixteen, so its results are the running sums e, 4 + e,
// 8 + e and 12 + e of 256 scores, and a lane's four 16-byte pieces of a row (or a key) are its operands for e = 0 .. 3.
// Positions are the results' rows: a lane stores four scores of one row.
// QL: the rows' operands in LDS, a read an instruction, and four waves a SIMD instead of three.
// The grid's columns are pairs of row tiles' sets, one from the start and one from the end: a set for a column left as many workgroups without
// a position as with one, and a wave needed sixteen tiles where the pairs are quickest with eight (us: 2,048 tokens at none, 32 heads
// of 128 over 8, 407 -> 369, 1,000 115 -> 104, 1,250 at 1,250 419 -> 403; 14 of 64 over 2, 2,048 at none 118 -> 88).
// The waves, npt position tiles each, that the positions of row tiles 4 set .. 4 set + 3 take
__host__ __device__ __forceinline__ int score_waves(int set, int pos0, int rows, int group, int npt) {
  const int last = 64 * set + 63 < rows ? 64 * set + 63 : rows - 1;
  return (pos0 + last / group + 16 * npt) / (16 * npt);
}
template <int NJ, bool QL>      // hd / 16
__global__ __launch_bounds__(256, QL ? 4 : 3) void attn_scores_mm_kernel(const float* __restrict__ q, const float* __restrict__ kc, float* __restrict__ raw,
                                                                int nh, int group, int kvd, int pos0, int ntok, float scale, int spitch, int npt) {
  constexpr int HD = 16 * NJ;
  const int kvh = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, m = lane >> 4, rows = ntok * group;
  // (the four waves: row tiles on the same positions, whose keys then come from the CU's own cache; a column of the grid's is the
  // positions of a set of row tiles and then those of the set as far from the last, so that every one has as many)
  const int sets = (rows + 63) / 64;
  int set = blockIdx.z, pw = blockIdx.y;
  if (const int nw = score_waves(set, pos0, rows, group, npt); pw >= nw) {
    pw -= nw;
    if (set == sets - 1 - set) return;
    set = sets - 1 - set;
  }
  const int r0 = (set * 4 + wave) * 16, p0 = pw * npt * 16;
  if (r0 >= rows) return;
  const int nposmax = pos0 + (min(r0 + 15, rows - 1)) / group + 1, pend = min(p0 + 16 * npt, nposmax);
  if (p0 >= pend) return;
  const int row = min(r0 + i, rows - 1), t = row / group, h = kvh * group + row - t * group;
  const float* const qr = q + ((long long)t * nh + h) * HD + 4 * m;
  __shared__ float qs[QL ? 4 : 1][QL ? 4 * NJ : 1][64];       // (a wave's own: no barrier)
  float4 qa[NJ], ka[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) qa[j] = *(const float4*)(qr + 16 * j);
  if constexpr (QL) {
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) qs[wave][4 * j + e][lane] = part(qa[j], e);
  }
  auto qpart = [&](int j, int e) { if constexpr (QL) return qs[wave][4 * j + e][lane]; else return part(qa[j], e); };
  float* const dst = raw + ((long long)t * nh + h) * spitch + 4 * m;
  const float* const kbase = kc + (long long)kvh * HD + 4 * m;
  auto load = [&](int p) {
    const float* kr = kbase + (long long)min(p + i, nposmax - 1) * kvd;
#pragma unroll
    for (int j = 0; j < NJ; j++) ka[j] = *(const float4*)(kr + 16 * j);
  };
  for (int p = p0; p < pend; p += 16) {
    load(p);
    v4f y, z;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const v16f zero = {};
      v16f s = __builtin_amdgcn_mfma_f32_16x16x1f32(part(ka[0], e), qpart(0, e), zero, 0, 0, 0);
      v16f d = __builtin_amdgcn_mfma_f32_16x16x1f32(part(ka[1], e), qpart(1, e), zero, 0, 0, 0);
#pragma unroll
      for (int j = 2; j <= NJ; j++) {
        v16f dn = {};
        if (j < NJ) dn = __builtin_amdgcn_mfma_f32_16x16x1f32(part(ka[j], e), qpart(j, e), zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = s[r] + d[r];
        asm volatile("" : "+v"(s));
        d = dn;
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float x = (s[r] + s[4 + r]) + (s[8 + r] + s[12 + r]);
        if (e == 0) y[r] = x;
        if (e == 1) y[r] = y[r] + x;
        if (e == 2) z[r] = x;
        if (e == 3) z[r] = z[r] + x;
      }
    }
    if (r0 + i < rows && p + 4 * m < spitch) {       // (what lies past the row's own positions is never read)
      v4f o;
#pragma unroll
      for (int r = 0; r < 4; r++) o[r] = (y[r] + z[r]) * scale;
      *(v4f*)(dst + p) = o;
    }
  }
}

// A workgroup's NTILE x HD results, rows from rb on, in LDS (HD + 4 floats a row) to the blocks of the output product's activations: a
// launch and the results' way to memory and back less, 2.5 us a layer of 97 at 21 tokens of the Qwen3-4B shape, 4 of 440 at 700.
struct RowsQuant { i8* q; float* d; int* sums; int kind; };      // kind: ILT_ROWS_Q8 or ILT_ROWS_Q8K
template <int HD, int NW>      // (NW: the workgroup's waves)
__device__ __forceinline__ void rows_to_blocks(const float* tile, int ntile, const RowsQuant& o, int rb, int rows, int nh, int group, int kvh, int wave, int lane) {
  __syncthreads();
  for (int c = wave; c < (ntile * HD + 255) / 256; c += NW) {
    const int at = 256 * c + 4 * lane, r = at / HD, row = rb + r, t = row / group;
    const float4 f = *(const float4*)(tile + min(r, ntile - 1) * (HD + 4) + at % HD);
    const float v[4] = {f.x, f.y, f.z, f.w};
    const long long p = ((long long)t * nh + kvh * group + row - t * group) * HD + at % HD;
    const bool live = r < ntile && row < rows;
    int q[4];
    if (o.kind == ILT_ROWS_Q8K) {
      const float d = q8k_block(v, lane, q);
      if (live) q8k_store(q, d, lane, o.q, o.d, o.sums, p >> 8);      // (a block's rows are all there or none is)
    } else {
      const float d = q8_block(v, q);
      if (live) {
        const u32 packed = act_pack(q);
        __builtin_memcpy(o.q + p, &packed, 4);
        if ((lane & 7) == 0) o.d[p >> 5] = __half2float(__float2half_rn(d));
      }
    }
  }
}

// out = the values' rows times the scaled scores (attn_softmax_kernel's), position after position.  A wave takes R rows
// (16, or 4: v_mfma_f32_4x4x1_16b_f32) and 64 columns; an instruction is one position, its operands the position's values in
// the wave's columns and its scores in the wave's rows.
// R 16: the values are the product's rows and four scores a 16-byte load of a row's lane the columns, the same in all four
// blocks.  R 4: a register holds the four rows' scores of sixteen positions, a block each, and the instruction broadcasts one
// block to all (16-byte loads there, sixteen lanes with the same address, were the launch's time: 321 positions 11.2 -> 8 us).
template <int R> struct ValMM;
template <> struct ValMM<16> {
  typedef v16f V;
  static constexpr int P = 8, AHEAD = 2, NS = 8;     // positions a set of registers, sets, registers of scores in one
  template <int K> static __device__ __forceinline__ V mul(const float (&s)[NS], float v) { const V z = {}; return __builtin_amdgcn_mfma_f32_16x16x1f32(v, s[K], z, 0, 0, 0); }
};
template <> struct ValMM<4> {
  typedef v4f V;
  static constexpr int P = 16, AHEAD = 3, NS = 1;
  template <int K> static __device__ __forceinline__ V mul(const float (&s)[NS], float v) { const V z = {}; return __builtin_amdgcn_mfma_f32_4x4x1f32(s[0], v, z, 4, K, 0); }
};

template <int R, int HD, bool QUANT>
__global__ __launch_bounds__(256, R == 16 ? 4 : 2) void attn_values_mm_kernel(const float* __restrict__ prob, const float* __restrict__ vc, float* __restrict__ out,
                                                                int nh, int group, int kvd, int pos0, int ntok, int spitch, RowsQuant quant) {
  using M = ValMM<R>;
  using V = typename M::V;
  constexpr int CG = HD / 64, WR = 4 / CG;           // column groups and row tiles of a workgroup's four waves
  constexpr int P = M::P, AHEAD = M::AHEAD;
  const int kvh = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rows = ntok * group, cg = wave % CG;
  // (the last rows, which see the most positions, first: the launch ends with the short ones)
  const int rb = (int)(gridDim.y - 1 - blockIdx.y) * WR * R;
  int r0 = rb + wave / CG * R;
  if (r0 >= rows) {
    if constexpr (!QUANT) return;
    r0 = rows - 1;                                   // (the last row again, for nobody)
  }
  const int t0 = r0 / group, t1 = min(r0 + R - 1, rows - 1) / group;
  const int npos0 = pos0 + t0 + 1, nposmax = pos0 + t1 + 1;
  // (through buffer loads: a set's values are one vector offset and scalar ones that never change, all of them within the cache
  // -- ilt_value_sets.h --, since how a buffer load's range check counts a scalar offset the public descriptions do not agree on.
  // The scores' whole offset is in the vector part: what lies past the tile's last row is zero, what lies past a row's last
  // position or in the next row is never added.)
  const __amdgpu_buffer_rsrc_t rs = ilt_rsrc(ilt_uniform_ptr(prob + ((long long)t0 * nh + kvh * group) * spitch), (u32)((t1 - t0) * nh + group) * (u32)spitch * 4u);
  const __amdgpu_buffer_rsrc_t rv = ilt_rsrc(ilt_uniform_ptr(vc), (u32)nposmax * (u32)kvd * 4u);
  const int srow = min(r0 + (lane & (R - 1)), rows - 1), st = srow / group;
  const u32 so = ((u32)((st - t0) * nh + srow - st * group) * (u32)spitch + (R == 4 ? (u32)(lane >> 2) : 0u)) * 4u, vo = (u32)(kvh * HD + 64 * cg + lane) * 4u;
  struct Set { float s[M::NS], v[P]; };
  int ko[P];
#pragma unroll
  for (int k = 0; k < P; k++) ko[k] = ilt_set_at(k, nposmax) * kvd * 4;
  auto load = [&](Set& x, int p) {
    const u32 base = (u32)ilt_set_base(p, P, nposmax);
#pragma unroll
    for (int k = 0; k < M::NS; k += 4) {
      if constexpr (R == 4) x.s[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, so + 4u * base, 0, 0));
      else {
        const float4 f = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, so + 4u * base + 4u * k, 0, 0));
        x.s[k] = f.x; x.s[k + 1] = f.y; x.s[k + 2] = f.z; x.s[k + 3] = f.w;
      }
    }
    const u32 pv = vo + base * (u32)kvd * 4u;
#pragma unroll
    for (int k = 0; k < P; k++) x.v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, pv, ko[k], 0));
  };
  V acc = {};
  int npos[R == 4 ? 4 : 1];                          // R 16: a lane's results are one row's; R 4: its column's in four rows
#pragma unroll
  for (int r = 0; r < (R == 4 ? 4 : 1); r++) npos[r] = pos0 + (R == 4 ? min(r0 + r, rows - 1) / group : st) + 1;
  auto set = [&](const Set& x, int p, auto ownc) {   // OWN: rows may end inside these positions, and they may lie further down
    constexpr bool OWN = decltype(ownc)::value;
    const int base = ilt_set_base(p, P, nposmax);
    u32 left[R == 4 ? 4 : 1];
#pragma unroll
    for (int r = 0; r < (R == 4 ? 4 : 1); r++) left[r] = ilt_set_left(p, npos[r]);
    auto mul = [&](auto kc) { constexpr int k = decltype(kc)::value; return M::template mul<k>(x.s, x.v[k]); };
    auto add = [&](const V& d, int k) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float a = acc[r] + d[r];
        acc[r] = !OWN || ilt_set_from(p, base, k) < left[R == 4 ? r : 0] ? a : acc[r];
      }
      asm volatile("" : "+v"(acc));
    };
    using std::integral_constant;
    V d0 = mul(integral_constant<int, 0>{}), d1;
    auto two = [&](auto kc) {                        // a product ahead of the sums
      constexpr int k = decltype(kc)::value;
      d1 = mul(integral_constant<int, k + 1>{});
      add(d0, k);
      if constexpr (k + 2 < P) d0 = mul(integral_constant<int, k + 2>{});
      add(d1, k + 1);
    };
    two(integral_constant<int, 0>{}); two(integral_constant<int, 2>{}); two(integral_constant<int, 4>{}); two(integral_constant<int, 6>{});
    if constexpr (P == 16) { two(integral_constant<int, 8>{}); two(integral_constant<int, 10>{}); two(integral_constant<int, 12>{}); two(integral_constant<int, 14>{}); }
  };
  Set x[AHEAD];
  ilt_value_sets<P, AHEAD>(x, npos0, nposmax, load, [&](const Set& x, int p) { set(x, p, std::false_type{}); },
                           [&](const Set& x, int p) { set(x, p, std::true_type{}); });
  if constexpr (QUANT) {
    __shared__ __align__(16) float tile[WR * R * (HD + 4)];
    float* const mine = tile + wave / CG * R * (HD + 4) + 64 * cg;
    if constexpr (R == 4) {
#pragma unroll
      for (int r = 0; r < 4; r++) mine[r * (HD + 4) + lane] = acc[r];
    } else {
#pragma unroll
      for (int b = 0; b < 4; b++) *(v4f*)(mine + (lane & 15) * (HD + 4) + 16 * b + 4 * (lane >> 4)) = v4f{acc[4 * b], acc[4 * b + 1], acc[4 * b + 2], acc[4 * b + 3]};
    }
    rows_to_blocks<HD, 4>(tile, WR * R, quant, rb, rows, nh, group, kvh, wave, lane);
    return;
  }
  auto row_out = [&](int row) { return out + ((long long)(row / group) * nh + kvh * group + row % group) * HD + 64 * cg; };
  if constexpr (R == 4) {
#pragma unroll
    for (int r = 0; r < 4; r++) if (r0 + r < rows) row_out(r0 + r)[lane] = acc[r];
  } else if (r0 + (lane & 15) < rows) {
    float* const o = row_out(srow) + 4 * (lane >> 4);
#pragma unroll
    for (int b = 0; b < 4; b++) *(v4f*)(o + 16 * b) = v4f{acc[4 * b], acc[4 * b + 1], acc[4 * b + 2], acc[4 * b + 3]};
  }
}

// Four registers of the four groups of 16 lanes, register and group exchanged.
__device__ __forceinline__ void across(float* v) {
  auto swap32 = [](float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(a), __float_as_int(b), false, false);
    const int x = r[0], y = r[1];
    a = __int_as_float(x); b = __int_as_float(y);
  };
  auto swap16 = [](float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(a), __float_as_int(b), false, false);
    const int x = r[0], y = r[1];
    a = __int_as_float(x); b = __int_as_float(y);
  };
  swap32(v[0], v[2]); swap32(v[1], v[3]);
  swap16(v[0], v[1]); swap16(v[2], v[3]);
}

// The same for few rows, by the vector ALU alone: a wave takes one row and 64 columns.  What bounds a launch of few waves is a wave's chain of positions, and
// what a position costs is instructions (a wave alone on its SIMD issues one in 5 cycles): four rows a wave are an instruction of
// the matrix cores, four adds and a load, one row a multiplication by a score broadcast within its row of lanes, an addition
// and, the values as 16-byte loads of four positions a wave, a quarter of a load and an exchange between lanes.
// us for scores, softmax and values: 32 heads of 128 over 8, 8 tokens at 300 positions 16.4 -> 13.4, 21 18.6 -> 17.6, 3 at 2,000
// 50 -> 36; 14 of 64 over 2, 48 at 300 17.4 -> 15.2, 21 at 2,000 52 -> 37.
template <int K> __device__ __forceinline__ float times_score(float s, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x150 + K, 0xF, 0xF, true)) * v;      // row_newbcast:K
}
// columns 64 cg + 4 (lane & 15) + (lane >> 4) of a row that sees npos positions; scores(base): those of positions base + (lane & 15)
template <int HD, int AHEAD, class Scores>
__device__ __forceinline__ float row_values(Scores scores, const float* vc, int kvd, int kvh, int cg, int npos, int lane) {
  constexpr int P = 16;
  const __amdgpu_buffer_rsrc_t rv = ilt_rsrc(ilt_uniform_ptr(vc), (u32)npos * (u32)kvd * 4u);
  const int col = 64 * cg + 4 * (lane & 15);
  u32 vo[P / 4];                                     // the lane's position of each four
#pragma unroll
  for (int k = 0; k < P / 4; k++) vo[k] = (u32)(ilt_set_at(4 * k + (lane >> 4), npos) * kvd + kvh * HD + col) * 4u;
  struct Set { float s, v[P]; };
  auto load = [&](Set& x, int p) {
    const u32 base = (u32)ilt_set_base(p, P, npos), bv = base * (u32)kvd * 4u;
    x.s = scores(base);
#pragma unroll
    for (int k = 0; k < P; k += 4) {
      const float4 f = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rv, vo[k / 4] + bv, 0, 0));
      x.v[k] = f.x; x.v[k + 1] = f.y; x.v[k + 2] = f.z; x.v[k + 3] = f.w;
    }
  };
  float acc = 0.0f;
  auto set = [&](Set& x, int p, auto ownc) {
    constexpr bool OWN = decltype(ownc)::value;
    const int base = ilt_set_base(p, P, npos);
    const u32 left = ilt_set_left(p, npos);
    auto four = [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      across(x.v + k);
      const float d[4] = {times_score<k>(x.s, x.v[k]), times_score<k + 1>(x.s, x.v[k + 1]), times_score<k + 2>(x.s, x.v[k + 2]), times_score<k + 3>(x.s, x.v[k + 3])};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float a = acc + d[i];
        acc = !OWN || ilt_set_from(p, base, k + i) < left ? a : acc;
      }
    };
    using std::integral_constant;
    four(integral_constant<int, 0>{}); four(integral_constant<int, 4>{}); four(integral_constant<int, 8>{}); four(integral_constant<int, 12>{});
  };
  Set x[AHEAD];
  ilt_value_sets<P, AHEAD>(x, npos, npos, load, [&](Set& x, int p) { set(x, p, std::false_type{}); }, [&](Set& x, int p) { set(x, p, std::true_type{}); });
  return acc;                                        // (the exchange leaves column 4 c + g of sixteen c in lane 16 g + c)
}
template <int HD, int AHEAD, bool QUANT>
__global__ __launch_bounds__(256) void attn_values_mm_row_kernel(const float* __restrict__ prob, const float* __restrict__ vc, float* __restrict__ out,
                                                              int nh, int group, int kvd, int pos0, int ntok, int spitch, RowsQuant quant) {
  constexpr int CG = HD / 64;
  const int kvh = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rb = ((int)gridDim.y - 1 - (int)blockIdx.y) * (4 / CG), cg = wave % CG;
  int row = rb + wave / CG;
  if (row >= ntok * group) {
    if constexpr (!QUANT) return;
    row = ntok * group - 1;                          // (again, for nobody)
  }
  const int t = row / group, h = kvh * group + row - t * group, npos = pos0 + t + 1;
  const __amdgpu_buffer_rsrc_t rs = ilt_rsrc(ilt_uniform_ptr(prob + ((long long)t * nh + h) * spitch), (u32)npos * 4u);
  const int col = 64 * cg + 4 * (lane & 15) + (lane >> 4);
  const float acc = row_values<HD, AHEAD>([&](u32 base) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, 4u * (base + (u32)(lane & 15)), 0, 0)); },
                                          vc, kvd, kvh, cg, npos, lane);
  if constexpr (QUANT) {
    __shared__ __align__(16) float tile[4 / CG * (HD + 4)];
    tile[wave / CG * (HD + 4) + col] = acc;
    rows_to_blocks<HD, 4>(tile, 4 / CG, quant, rb, ntok * group, nh, group, kvh, wave, lane);
    return;
  }
  out[((long long)t * nh + h) * HD + col] = acc;
}

// All of it in one launch where a chunk is short: a workgroup a KV head and token, its rows the heads of the group.  Scores with four
// lanes a position (sums 4 m + e of F32-DOT16 in lane m), 16 positions a wave at a time, into LDS; a wave a row's softmax; the values a row
// and 64 columns a wave as above.  Three launches of few workgroups are mostly their own starts and ends, 3 us each; what is left is 10 us
// for scores and values of 300 positions on eight waves, instructions for the most part (keys or values through LDS, the next keys asked
// for first, two rows a wave, two waves a row's softmax: none changed it by 5 %).  us for the three and for this: 21 tokens at none 11.3 and 5.6, at
// 300 19.6 and 15.5, at 900 36.6 and 32.4, 8 at 900 25.4 and 30.4 (32 heads of 128 over 8); 14 of 64 over 2, 48 at none 10.3 and 6.4.
template <int HD, bool QUANT>
__global__ __launch_bounds__(512) void attn_short_mm_kernel(const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc, float* __restrict__ out,
                                                         int nh, int group, int kvd, int pos0, int ntok, float scale, int pitch, RowsQuant quant) {
  constexpr int CG = HD / 64, NJ = HD / 16, NW = 8;
  extern __shared__ __align__(16) float sc[];        // group rows of pitch scores, then of HD + 4 results
  const int kvh = blockIdx.x, t = (int)gridDim.y - 1 - (int)blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int npos = pos0 + t + 1, m = lane & 3, pl = lane >> 2;
  const float* const kb = kc + (long long)kvh * HD + 4 * m;
  for (int rb = 0; rb < group; rb += 4) {
    float4 qa[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float* const qr = q + ((long long)t * nh + kvh * group + min(rb + i, group - 1)) * HD + 4 * m;
#pragma unroll
      for (int j = 0; j < NJ; j++) qa[i][j] = *(const float4*)(qr + 16 * j);
    }
    for (int p0 = 16 * wave; p0 < npos; p0 += 16 * NW) {
      const float* const kr = kb + (long long)min(p0 + pl, npos - 1) * kvd;
      float4 ka[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) ka[j] = *(const float4*)(kr + 16 * j);
      float x[4][4];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float d = part(qa[i][j], e) * part(ka[j], e);
            x[i][e] = j ? x[i][e] + d : d;
          }
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          x[i][e] = x[i][e] + ilt_dppf<ILT_DPP_XOR1>(x[i][e]);
          x[i][e] = x[i][e] + ilt_dppf<ILT_DPP_XOR2>(x[i][e]);
        }
        const float v = ((x[i][0] + x[i][1]) + (x[i][2] + x[i][3])) * scale;
        if (m == 0 && rb + i < group && p0 + pl < npos) sc[(rb + i) * pitch + p0 + pl] = v;
      }
    }
  }
  __syncthreads();
  for (int row = wave; row < group; row += NW) {     // (a wave's own row: nobody else's until the barrier)
    float* const w = sc + row * pitch;
    float mx = -3.402823466e38f;
    for (int p = lane; p < npos; p += 64) mx = fmaxf(mx, w[p]);
    mx = wave_max_float(mx);
    double sum = 0.0;
    for (int p = lane; p < npos; p += 64) { const float e = ilt_expf_via_double(w[p] - mx); w[p] = e; sum += (double)e; }
    sum = wave_sum_double(sum);
    float inv;
    if (!recip_settled<sum_adds(kShortMost / 64, 0)>(sum, npos, &inv)) {      // the same in every lane
      wave_lds_sync();
      sum = 0.0;
      for (int p = 0; p < npos; p++) sum += (double)w[p];
      inv = (float)(1.0 / sum);
    }
    wave_lds_sync();
    for (int p = lane; p < npos; p += 64) w[p] = w[p] * inv;
  }
  __syncthreads();
  float* const tile = sc + group * pitch;
  for (int pr = wave; pr < group * CG; pr += NW) {
    const int row = pr / CG, cg = pr % CG, col = 64 * cg + 4 * (lane & 15) + (lane >> 4);
    const float* const pw = sc + row * pitch + (lane & 15);
    const float acc = row_values<HD, 3>([&](u32 base) { return pw[base]; }, vc, kvd, kvh, cg, npos, lane);
    if constexpr (QUANT) tile[row * (HD + 4) + col] = acc;
    else out[((long long)t * nh + kvh * group + row) * HD + col] = acc;
  }
  if constexpr (QUANT) rows_to_blocks<HD, NW>(tile, group, quant, t * group, ntok * group, nh, group, kvh, wave, lane);
}

}  // namespace

// (The values may lie on any dword: they are read by buffer loads, which want no more, also of 16 bytes.)
bool ilt_k_attn_mm_takes(const float* q, const float* kc, const float* scratch, const float* out, int nh, int nkv, int hd, int ctx) {
  return (hd == 64 || hd == 128) && ((((uintptr_t)q) | ((uintptr_t)kc) | ((uintptr_t)scratch) | ((uintptr_t)out)) & 15) == 0 &&      // 16-byte loads and stores of them
         (long long)ctx * nkv * hd < (1LL << 30) && 17LL * nh * (ctx + 3) < (1LL << 30);                         // 32-bit offsets: the values, a tile's rows
}

// hipErrorNotSupported, and nothing launched, where three launches are better: more workgroups than CUs, positions that a few workgroups are
// long over (whole prompts, one launch's gain: the Qwen3-4B shape, 2 tokens at 16 positions 6.5 %, at 128 2.6, at 300 -0.2; 21 at 300 4.0, at 400 2.1; 40
// at 128, 320 workgroups, -3.5; the Qwen2.5-0.5B one, 8 at 64 6.5, at 200 1.9; 128 at 200 4.0), groups of fewer than three heads (scores are made
// for four at a time).  Five heads of 128 and more are two rounds of the eight waves' values and of the scores, and over after a third of those
// positions (us for one launch and for three, on 8 workgroups: five heads at 96 positions 10.2 and 10.3, at 104 12.2 and 10.4, at 200 16.0 and 11.8; eight at
// 64 10.0 and 10.3, at 72 11.1 and 10.3, at 200 18.4 and 11.8; on 128 eight heads at 94 11.9 and 12.8, at 102 13.8 and 13.3; on 240 at 108 13.7 and 13.8).
hipError_t ilt_k_attn_short_mm(const float* q, const float* kc, const float* vc, float* out, int nh, int nkv, int hd, int pos0, int ntok, float scale,
                               const IltRowsQuant* to, hipStream_t st) {
  const int group = nh / nkv, ctx = pos0 + ntok, pitch = (ctx + 15) & ~15;
  const long long wgs = (long long)ntok * nkv;
  const int most = group * hd > 8 * 64 ? (wgs >= 128 || group <= 6 ? 96 : 64) : wgs >= 128 ? kShortMost : 256;
  if (group < 3 || group > 8 || wgs > 256 || ctx > most) return hipErrorNotSupported;
  const RowsQuant quant = to ? RowsQuant{to->q, to->d, to->sums, to->kind} : RowsQuant{};
  const dim3 grid(nkv, ntok);
  const size_t smem = sizeof(float) * group * (pitch + hd + 4);
#define ILT_SHORT(HD, QUANT) hipLaunchKernelGGL((attn_short_mm_kernel<HD, QUANT>), grid, dim3(512), smem, st, q, kc, vc, out, nh, group, nkv * hd, pos0, ntok, scale, pitch, quant)
  if (hd == 128) { if (to) ILT_SHORT(128, true); else ILT_SHORT(128, false); }
  else { if (to) ILT_SHORT(64, true); else ILT_SHORT(64, false); }
#undef ILT_SHORT
  return hipGetLastError();
}

// Blocks of 32 lie within a row; blocks of 256 are rows of one token and start where a tile's rows do where a group's columns are whole blocks.
bool ilt_k_attn_mm_quantizes(int kind, int nh, int nkv, int hd) { return kind == ILT_ROWS_Q8 || (kind == ILT_ROWS_Q8K && nh / nkv * hd % 256 == 0); }

// A wave's position tiles, its rows' loads and the launch's waves shared among them, by all the launch's tiles (us of the scores for one,
// two, four and eight of them): 2,944 tiles 10.0, 10.5, 11.3, 17.5; 6,912 17.3, 14.5, 16.3, 18.2; 14,336 15.4, 14.8, 15.8, 18.7; 32,768 39.8, 35.5, 36.1,
// 38.8; 45,600 52.6, 45.6, 44.2, 49.0; 75,000 four 107, eight 104, sixteen 119; 205,000 155, 150, 158;
// 393,000 421, 403, 404 (and 2,500 tokens as two halves 68.6, 68.7 and 68.3 ms).  The rows' operands in LDS past 16,384
// tiles (512 tokens at none 40.5 -> 39.1; 256 at none, 8,192, 15.3 against 16.0).
hipError_t ilt_k_attn_scores_mm(const float* q, const float* kc, float* raw, int nh, int nkv, int hd, int pos0, int ntok, float scale, int spitch,
                                hipStream_t st) {
  const int group = nh / nkv, rtiles = (ntok * group + 15) / 16, ptiles = (pos0 + ntok + 15) / 16;
  const long long tiles = (long long)rtiles * nkv * ptiles;
  const int npt = tiles < 6000 ? 1 : tiles <= 16384 ? 2 : tiles < 70000 ? 4 : tiles < 300000 ? 8 : 16;
  const int rows = ntok * group, sets = (rows + 63) / 64;
  // (a column's positions: no pair of sets has more than this)
  const int waves = sets == 1 ? score_waves(0, pos0, rows, group, npt) : (2 * pos0 + (64 * sets + 62) / group + 32 * npt) / (16 * npt);
  const dim3 grid(nkv, waves, (sets + 1) / 2);
#define ILT_SCORES(NJ, QL) hipLaunchKernelGGL((attn_scores_mm_kernel<NJ, QL>), grid, dim3(256), 0, st, q, kc, raw, nh, group, nkv * hd, pos0, ntok, scale, spitch, npt)
  if (tiles > 16384) { if (hd == 128) ILT_SCORES(8, true); else ILT_SCORES(4, true); }
  else { if (hd == 128) ILT_SCORES(8, false); else ILT_SCORES(4, false); }
#undef ILT_SCORES
  return hipGetLastError();
}

// Sixteen rows a wave once that leaves about six waves a CU (32 heads of 128 over 8 on 512 tokens, 2,048 waves: 95.7 us for the
// chunk's attention against 97.6 with four; 1,250 at 1,250 893 against 1,102), else four: a wave's chain of positions, an
// instruction every few cycles, is the launch's time (256 tokens 41 us against 43, 64 tokens 13.9 against 15.5, 14 heads of 64
// over 2 on 1,250 121 against 137).  Further into a conversation than the chunk is long, sixteen as soon as their chain, 53 ns a position, is over
// before the four times as many waves of four rows, 19 ns a position each, are through: by how many waves they are and how much of the longest chain
// their average is (values, us, four and sixteen; 32 heads of 128 over 8: 128
// tokens at 1,900, 502 by this count, 76 and 107; 200 at 1,200, 743, 90 and 78; 300 at 1,700, 1,110, 161 and 139; 380 at 600 87 and 69; 14 of
// 64 over 2, 700 at 3,000, 556, 173 and 192).  So also beside a prompt's other half, where it lies as far in (whole prompts, ms, all its halves with four and
// by this rule: 400 tokens at 600, as 256 and 144, 12.8 and 12.3; 512 at 900 17.3 and 16.2; 400 at 300 11.3 and 11.7); a half no further in than it is long has four
// (512 at none, its second half 256 at 256, 768 by this count: 10.7 ms, with sixteen 11.0), alone the two are within 5 % there (32 heads of 128 over 8,
// the chunk's attention: 300 at 200 67.8 us with four, 66.6 with sixteen; 28 over 4, 400 at 300 99.4 and 95.2).  One row a wave up to 1,400 waves, a little more
// than the SIMDs (32 heads of 128 over 8 at 300
// positions, 1,344 waves 17.6 us against 18.6, 2,112 21.1 against 19.3; 14 of 64 over 2, 1,400 19.8 against 20.9, 2,800 30.5 against
// 29.1); its values three sets ahead up to 512 positions, four past them (3 tokens at 2,000: 35.5 against 39.7).
hipError_t ilt_k_attn_values_mm(const float* prob, const float* vc, float* out, int nh, int nkv, int hd, int pos0, int ntok, int spitch, const IltRowsQuant* to,
                                hipStream_t st) {
  const int group = nh / nkv, rows = ntok * group, cg = hd / 64, wr = 4 / cg;
  const RowsQuant quant = to ? RowsQuant{to->q, to->d, to->sums, to->kind} : RowsQuant{};
  if ((long long)rows * nkv * cg <= 1400) {
    const dim3 grid(nkv, (rows * cg + 3) / 4);
#define ILT_VALUES(HD, AHEAD, QUANT) hipLaunchKernelGGL((attn_values_mm_row_kernel<HD, AHEAD, QUANT>), grid, dim3(256), 0, st, prob, vc, out, nh, group, nkv * hd, pos0, ntok, spitch, quant)
#define ILT_VALUES_OF(AHEAD, QUANT) do { if (hd == 128) ILT_VALUES(128, AHEAD, QUANT); else ILT_VALUES(64, AHEAD, QUANT); } while (0)
    if (pos0 + ntok <= 512) { if (to) ILT_VALUES_OF(3, true); else ILT_VALUES_OF(3, false); }
    else { if (to) ILT_VALUES_OF(4, true); else ILT_VALUES_OF(4, false); }
#undef ILT_VALUES_OF
#undef ILT_VALUES
    return hipGetLastError();
  }
  const long long w16 = (long long)((rows + 15) / 16) * nkv * cg;
  const int r = w16 >= 1600 || (pos0 > ntok && w16 * (2LL * pos0 + ntok) >= 1440LL * (pos0 + ntok)) ? 16 : 4;
  const dim3 grid(nkv, ((rows + r - 1) / r + wr - 1) / wr);
#define ILT_VALUES(R, HD, QUANT) hipLaunchKernelGGL((attn_values_mm_kernel<R, HD, QUANT>), grid, dim3(256), 0, st, prob, vc, out, nh, group, nkv * hd, pos0, ntok, spitch, quant)
#define ILT_VALUES_OF(R, QUANT) do { if (hd == 128) ILT_VALUES(R, 128, QUANT); else ILT_VALUES(R, 64, QUANT); } while (0)
  if (r == 16) { if (to) ILT_VALUES_OF(16, true); else ILT_VALUES_OF(16, false); }
  else { if (to) ILT_VALUES_OF(4, true); else ILT_VALUES_OF(4, false); }
#undef ILT_VALUES_OF
#undef ILT_VALUES
  return hipGetLastError();
}
