// The exact prefill product of many tokens, the weights made in the matrix cores' operand registers: Y[t][r] = W[r].x_t, W in
// GGUF Q4_K / Q6_K / Q2_K / IQ2_XXS blocks, every result with the CPU path's bits (MATMUL!: kquant.lisp:180-236, batch.lisp:128).
//
// What bounds it: the vector ALU and the matrix cores together (gfx950 issues a multiply or an add of two waves in the time a
// third of an MFMA takes, and an MFMA hides permutes and 16-bit arithmetic but only half of the plain float work beside it),
// and the latencies between them.  A super-block of 256 columns leaves one integer a result, however it comes about, and two
// (Q4_K: four) roundings after it; the integer goes through v_mfma_i32_32x32x32_i8 as two planes:
//   Q4_K: a scale is two digits, sc = 8 sh + sl, and q * digit is at most 105: four bytes times a digit is one 16-bit packed
//         multiply with no carry between them.  isum = 8 * (sh q . xq) + (sl q . xq).
//   Q6_K: T = sc (q - 32) = 256 hi + lo with lo signed: 16-bit fields, one packed multiply-add for two weights.
//   Q2_K: sc * q is at most 45, one plane; IQ2_XXS: a group's sums scaled by the lanes (below).
// The minimums (Q4_K) are one f16 product of the tokens' sums of 32, in two parts of seven bits, with the 6-bit minimums:
// whole numbers below 2^21, exact in its single-precision sums.
//
// A wave takes 32 rows and holds a whole super-block of them as operands (64 registers), so a weight is unpacked once for the
// wave's 64 or 128 tokens and nothing of it passes through LDS twice; the rows' blocks come into LDS as they are (direct
// loads of consecutive bytes: the same bytes as 16-byte loads a lane, of 32 rows each, cost the memory pipeline four times
// as much and half the kernel's time), the tokens' quants beside them, 64 tokens' room at a time, so that two workgroups of
// four waves fit a CU and one's start and end run beside the other's middle.  Everything is one step ahead: while patch a's
// products run, patch a-1's integer sums become float terms, and with a block's last patch each group's operands are replaced
// by the next block's as soon as they have been multiplied.  Two barriers a super-block, loads half a super-block ahead.
// A patch's float work beside its MFMAs one result after another left every instruction waiting for the one before it; two
// results go step by step side by side, and what a step wants from LDS is asked for a step before.
//
// Measured against the kernel of 64-column steps with planes through LDS that this one replaced (us; Q4_K 19456 x 2560 on 256,
// 512, 2048 tokens; 2560 x 4096 on 512; Q6_K 2560 x 9728 on 512; 17408 x 5120 on 4096): 88 -> 54, 137 -> 82, 583 -> 278;
// 62 -> 40; 110 -> 79; 1,400 -> 985 (741 TFLOP/s).
#include "ilt_device.h"
#include "ilt_gemm_tile.h"
#include "ilt_iq2xxs_tables.h"
#include "ilt_kernels.h"
#include <stdlib.h>
#include <algorithm>
#include <type_traits>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef unsigned short v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u32 wordr(const int4& v, int i) { return (u32)(i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w); }
__device__ __forceinline__ v2u as2(u32 v) { return __builtin_bit_cast(v2u, v); }
__device__ __forceinline__ u32 asw(v2u v) { return __builtin_bit_cast(u32, v); }
// half H of the two 16-bit fields of V, in both
template <int H> __device__ __forceinline__ v2u splat(u32 v) { const v2u a = as2(v); return v2u{a[H], a[H]}; }

__device__ __forceinline__ float4 lds_f4(const float* p) {
  const int4 v = ilt_lds_ld16(p);
  return make_float4(__builtin_bit_cast(float, v.x), __builtin_bit_cast(float, v.y), __builtin_bit_cast(float, v.z), __builtin_bit_cast(float, v.w));
}

template <int FMT> struct RegW;

// ilt_g2lds16 as the compiler does not see it: behind the one that it does see it waits for every load in flight before it reads
// LDS again, and the kernel waits for its loads itself (6 of 256 experts, 1,000 tokens: IQ2_XXS's gate and up 550 -> 475 us, the
// tables of 4 bytes an entry included).  Not so behind the buffer loads, which want addresses of whole dwords.
__device__ __forceinline__ void g2lds16_untracked(const void* src, void* dst) {
  u32 m0;                                            // (the compiler's, put back)
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(m0) : "v"(src), "s"(__builtin_amdgcn_readfirstlane((u32)(uintptr_t)(ILT_LDS void*)dst)) : "memory");
}

template <> struct RegW<ILT_Q4_K> {
  static constexpr int BLOCK = 144;
  static constexpr bool MINS = true;
  static constexpr int PLANES = 2, SH = 3;  // isum = (hi sums << SH) + (lo sums)
  struct Block { u32 sc[2]; float d, dm; v8h mins; };
  struct Quants { int4 q[2]; };
  // In LDS: the quants of eight rows a kilobyte, piece p of row r at p ^ (r >> 1 & 7); behind them a header a row.
  static constexpr int LOADS = 5, LBYTES = 5120;             // direct loads, bytes of LDS for 32 rows
  struct At { u32 a, b, h; };
  static __device__ __forceinline__ At place(u32 row_bytes, int lane, int, int) {
    const u32 pc = 16 * (u32)((lane & 7) ^ ((lane >> 4) & 3)), rr = (u32)(lane >> 3) * row_bytes + 16;
    return At{rr + pc, rr + (pc ^ 64), (u32)(lane & 31) * row_bytes};
  }
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t rw, const u8*, const At& at, u32 row_bytes, u32 row0, u32 block, u8* dst) {
    if (i < 4) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (ILT_LDS void*)(dst + 1024 * i), 16, (i & 1 ? at.b : at.a) + (row0 + 8 * i) * row_bytes, block, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (ILT_LDS void*)(dst + 4096), 16, at.h + row0 * row_bytes, block, 0, 0);
  }
  static __device__ __forceinline__ void block(Block& o, const u8* src, int l32, int) {
    const int4 h = ilt_lds_ld16(src + 4096 + 16 * l32);
    o.d = ilt_h2f((u16)((u32)h.x & 0xFFFF));
    o.dm = ilt_h2f((u16)((u32)h.x >> 16));
    const u32 a = (u32)h.y, b = (u32)h.z, c = (u32)h.w;                          // get_scale_min_k4, four groups a word
    o.sc[0] = a & 0x3F3F3F3Fu; o.sc[1] = (c & 0x0F0F0F0Fu) | ((a >> 2) & 0x30303030u);
    const u32 mn[2] = { b & 0x3F3F3F3Fu, ((c >> 4) & 0x0F0F0F0Fu) | ((b >> 2) & 0x30303030u) };
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const v2h k = {(_Float16)1024.0f, (_Float16)1024.0f};
      const v2h m01 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0, mn[i], 0x0C010C00u) | 0x64006400u) - k;
      const v2h m23 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0, mn[i], 0x0C030C02u) | 0x64006400u) - k;
      o.mins[4 * i] = m01[0]; o.mins[4 * i + 1] = m01[1]; o.mins[4 * i + 2] = m23[0]; o.mins[4 * i + 3] = m23[1];
    }
  }
  // the quants of groups g and g + 1 (g even)
  static __device__ __forceinline__ void quants(Quants& o, const u8* src, int g, int l32, int lh) {
    if (g % 2 == 0) o.q[(g >> 1) & 1] = ilt_lds_ld16(src + 128 * l32 + 16 * ((g + lh) ^ ((l32 >> 1) & 7)));
  }
  static __device__ __forceinline__ void quants_now(Quants&, const u8*, int, int, int) {}
  static __device__ __forceinline__ void group(Block& b, const Quants& r, int g, int, v4i& hi, v4i& lo) {
    const v2u l = splat<0>((b.sc[g >> 2] >> (8 * (g & 3))) & 7), h = splat<0>((b.sc[g >> 2] >> (8 * (g & 3) + 3)) & 7);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const u32 w = wordr(r.q[(g >> 1) & 1], k);
      const v2u n = as2((g % 2 ? w >> 4 : w) & 0x0F0F0F0Fu);
      lo[k] = (int)asw(n * l);
      hi[k] = (int)asw(n * h);
    }
  }
};

template <> struct RegW<ILT_Q6_K> {
  static constexpr int BLOCK = ILT_Q6K_STRIDE;
  static constexpr bool MINS = false;
  static constexpr int PLANES = 2, SH = 8;
  struct Block { int4 sc; float d, dm; v8h mins; };
  struct Quants { int4 l[2], h; };
  // In LDS: four rows a kilobyte and 64 bytes, piece p of row r at p ^ (r & 3) of its 256; piece 13 the block's last 16 bytes.
  static constexpr int LOADS = 8, LBYTES = 8704;
  struct At { u32 a; };
  static __device__ __forceinline__ At place(u32 row_bytes, int lane, int, int) {
    return At{(u32)(lane >> 4) * row_bytes + min(16u * (u32)((lane & 15) ^ (lane >> 4)), 196u)};
  }
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t rw, const u8*, const At& at, u32 row_bytes, u32 row0, u32 block, u8* dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (ILT_LDS void*)(dst + 1088 * i), 16, at.a + (row0 + 4 * i) * row_bytes, block, 0, 0);
  }
  static __device__ __forceinline__ const u8* row_of(const u8* src, int l32) { return src + (l32 >> 2) * 1088 + (l32 & 3) * 256; }
  static __device__ __forceinline__ void block(Block& o, const u8* src, int l32, int) {
    const u8* row = row_of(src, l32);
    o.sc = ilt_lds_ld16(row + 16 * (12 ^ (l32 & 3)));
    o.d = ilt_h2f(*ILT_LDS_PTR(const u16, row + 16 * (13 ^ (l32 & 3)) + 12));
  }
  // what group g needs that no group before it has brought: groups g and g + 2 of a half share 16 bytes of low bits, a half's
  // four groups 16 bytes of high ones
  static __device__ __forceinline__ void quants(Quants& o, const u8* src, int g, int l32, int lh) {
    const u8* row = row_of(src, l32);
    const int x = l32 & 3, n = g >> 2;
    if (g % 4 < 2) o.l[g % 4] = ilt_lds_ld16(row + 16 * ((4 * n + 2 * (g % 4) + lh) ^ x));
  }
  // (the high ones once the last of the half before has been made)
  static __device__ __forceinline__ void quants_now(Quants& o, const u8* src, int g, int l32, int lh) {
    if (g % 4 == 0) o.h = ilt_lds_ld16(row_of(src, l32) + 16 * ((8 + 2 * (g >> 2) + lh) ^ (l32 & 3)));
  }
  static __device__ __forceinline__ void group(Block& b, const Quants& r, int g, int lh, v4i& hi, v4i& lo) {
    const int j = g & 3;                             // columns 32g + 16lh ..: scale 2g + lh
    const int s = (int)(i8)((wordr(b.sc, g >> 1) >> (8 * lh)) >> (16 * (g & 1)));
    const u32 kk = (u32)(128 - 32 * s);
    const v2u s2 = {(unsigned short)s, (unsigned short)s}, k2 = {(unsigned short)kk, (unsigned short)kk};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const u32 w = wordr(r.l[j & 1], k), qh = wordr(r.h, k);
      const u32 v = ((j >> 1 ? w >> 4 : w) & 0x0F0F0F0Fu) | ((j < 2 ? qh << (4 - 2 * j) : qh >> (2 * j - 4)) & 0x30303030u);
      const u32 te = asw(as2(v & 0x00FF00FFu) * s2 + k2), to = asw((as2(v) >> 8) * s2 + k2);
      hi[k] = (int)__builtin_amdgcn_perm(to, te, 0x07030501u);
      lo[k] = (int)(__builtin_amdgcn_perm(to, te, 0x06020400u) ^ 0x80808080u);
    }
  }
};

// Q2_K: scale * quant is at most 45, one plane.  In LDS: eight rows a kilobyte, piece p of row r at p ^ (r >> 1 & 7); piece 5
// the block's last 16 bytes.
template <> struct RegW<ILT_Q2_K> {
  static constexpr int BLOCK = 84;
  static constexpr bool MINS = true;
  static constexpr int PLANES = 1, SH = 0;
  struct Block { u32 sc[4]; float d, dm; v8h mins; };
  struct Quants { int4 q[2]; };
  static constexpr int LOADS = 4, LBYTES = 4096;
  struct At { u32 a, b; };
  static __device__ __forceinline__ At place(u32 row_bytes, int lane, int, int) {
    const u32 pc = (u32)((lane & 7) ^ ((lane >> 4) & 3)), rr = (u32)(lane >> 3) * row_bytes;
    return At{rr + min(16 * pc, 68u), rr + min(16 * (pc ^ 4), 68u)};
  }
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t rw, const u8*, const At& at, u32 row_bytes, u32 row0, u32 block, u8* dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (ILT_LDS void*)(dst + 1024 * i), 16, (i & 1 ? at.b : at.a) + (row0 + 8 * i) * row_bytes, block, 0, 0);
  }
  static __device__ __forceinline__ void block(Block& o, const u8* src, int l32, int lh) {
    const u8* row = src + 128 * l32;
    const int x = (l32 >> 1) & 7;
    const int4 s = ilt_lds_ld16(row + 16 * x);
    const u32 dd = *ILT_LDS_PTR(const u32, row + 16 * (5 ^ x) + 12);
    o.d = ilt_h2f((u16)(dd & 0xFFFF));
    o.dm = ilt_h2f((u16)(dd >> 16));
#pragma unroll
    for (int i = 0; i < 4; i++) o.sc[i] = wordr(s, i) & 0x0F0F0F0Fu;
#pragma unroll
    for (int i = 0; i < 2; i++) {                    // the minimums of groups 8 lh ..
      const u32 m = ((u32)(lh ? wordr(s, 2 + i) : wordr(s, i)) >> 4) & 0x0F0F0F0Fu;
      const v2h k = {(_Float16)1024.0f, (_Float16)1024.0f};
      const v2h m01 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0, m, 0x0C010C00u) | 0x64006400u) - k;
      const v2h m23 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0, m, 0x0C030C02u) | 0x64006400u) - k;
      o.mins[4 * i] = m01[0]; o.mins[4 * i + 1] = m01[1]; o.mins[4 * i + 2] = m23[0]; o.mins[4 * i + 3] = m23[1];
    }
  }
  // a half's four groups share 16 bytes, two bits each
  static __device__ __forceinline__ void quants(Quants& o, const u8* src, int g, int l32, int lh) {
    if (g % 4 == 0) o.q[g >> 2] = ilt_lds_ld16(src + 128 * l32 + 16 * ((1 + 2 * (g >> 2) + lh) ^ ((l32 >> 1) & 7)));
  }
  static __device__ __forceinline__ void quants_now(Quants&, const u8*, int, int, int) {}
  static __device__ __forceinline__ void group(Block& b, const Quants& r, int g, int lh, v4i&, v4i& lo) {
    const v2u s = splat<0>((b.sc[g >> 1] >> (8 * lh + 16 * (g & 1))) & 15);       // scale 2g + lh
#pragma unroll
    for (int k = 0; k < 4; k++) lo[k] = (int)asw(as2((wordr(r.q[g >> 2], k) >> (2 * (g & 3))) & 0x03030303u) * s);
  }
};

// The same for a matrix on a two-byte boundary (an expert's slot may lie on one; buffer loads of dwords want four): the blocks by
// loads through pointers, as IQ2_XXS's, a row past the matrix's its last one.
struct RegWQ2KHalf : RegW<ILT_Q2_K> {
  struct At { u32 a[4]; };
  static __device__ __forceinline__ At place(u32 row_bytes, int lane, int row0, int rows) {
    At o;
#pragma unroll
    for (int i = 0; i < 4; i++)
      o.a[i] = (u32)min(row0 + 8 * i + (lane >> 3), rows - 1) * row_bytes + min(16 * (u32)((lane & 7) ^ ((lane >> 4) & 3) ^ (i & 1 ? 4 : 0)), 68u);
    return o;
  }
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t, const u8* w, const At& at, u32, u32, u32 block, u8* dst) {
    ilt_g2lds16(w + (size_t)block + at.a[i], dst + 1024 * i);
  }
};

// IQ2_XXS: a block's eight groups of 32 weights add (float(sumi) * (0.5 + scale)) alternately to two sums, and the block's term
// is (d yd) times the two together (iquant.lisp:161-215).  Every partial sum is a multiple of 1/2 whose double stays below 2^24
// (test_oracle.py asserts it from the codebook), so nothing rounds before the two meet, and their sum is float(isum) / 2 for
// isum = sum of (2 scale + 1) * sumi.  The signed codebook entries (at most 43) are the operand and a group is one MFMA, whose
// results are scaled by the lanes (a row's scale is its lane's own): as two planes of scaled weights the entries take three
// times the arithmetic, which is what groups of a few tokens would wait for.
// In LDS: a row's 64 bytes of indices and signs, piece p of row r at p ^ (r >> 2 & 3), and behind them 16 bytes with its d.
__device__ const u64 iq2_grid_reg[256] = { ILT_IQ2XXS_GRID_VALUES };
// Four bytes an entry: a nibble a weight (weight k < 4 in byte k's low one, 4 + k in its high one), of the codebook which of the
// three magnitudes it is, of the 128 sign patterns 4 where it is negative; together the selector of a byte permutation.
__device__ __forceinline__ u32* iq2_tables() {
  __shared__ u32 tab[384];
  return tab;
}
__device__ __forceinline__ void iq2_tables_load(int t, int threads) {       // a barrier follows
  u32* const tab = iq2_tables();
  for (int i = t; i < 384; i += threads) {
    u32 v;
    if (i < 256) {
      const u64 g = iq2_grid_reg[i];
      v = ((u32)(g >> 4) & 0x03030303u) | ((u32)(g >> 32) & 0x30303030u);
    } else {
      const u32 s = (u32)(i - 256) | ((u32)(__popc(i - 256) & 1) << 7);
      v = 0;
#pragma unroll
      for (int j = 0; j < 4; j++) v |= (((s >> j) & 1) << (8 * j + 2)) | (((s >> (4 + j)) & 1) << (8 * j + 6));
    }
    tab[i] = v;
  }
}
template <> struct RegW<ILT_IQ2_XXS> {
  static constexpr int BLOCK = 66;
  static constexpr bool MINS = false;
  static constexpr int PLANES = 0, SH = 0;           // PLANES 0: a group's sums scaled by the lanes
  struct Block { int k[8]; float d, dm; v8h mins; };  // the groups' scales
  struct Quants { int4 q[2]; u32 sel[2]; };
  static constexpr int LOADS = 3, LBYTES = 3072;
  struct At { int lane, row0, rows; };
  static __device__ __forceinline__ At place(u32, int lane, int row0, int rows) { return At{lane, row0, rows}; }
  // (the blocks are two-byte aligned; a row past the matrix's is its last one; the offsets made each time: kept, they are in
  // scratch memory, whose reads wait for the loads before them)
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t, const u8* w, const At& at, u32 row_bytes, u32, u32 block, u8* dst) {
    u32 lane = (u32)at.lane;
    asm volatile("" : "+v"(lane));
    const u32 r = i < 2 ? 16 * i + (lane >> 2) : lane & 31, o = i < 2 ? 2 + 16 * ((lane & 3) ^ ((lane >> 4) & 3)) : 0;
    g2lds16_untracked(w + (size_t)block + (u32)min(at.row0 + (int)r, at.rows - 1) * row_bytes + o, dst + 1024 * i);
  }
  static __device__ __forceinline__ void block(Block& o, const u8* src, int l32, int) {
    o.d = ilt_h2f(*ILT_LDS_PTR(const u16, src + 2048 + 16 * l32));
  }
  static __device__ __forceinline__ void quants(Quants& o, const u8* src, int g, int l32, int) {
    if (g % 2 == 0) o.q[(g >> 1) & 1] = ilt_lds_ld16(src + 64 * l32 + 16 * ((g >> 1) ^ ((l32 >> 2) & 3)));
  }
  static __device__ __forceinline__ u32 index_word(const Quants& r, int g) { return wordr(r.q[(g >> 1) & 1], 2 * (g & 1)); }
  static __device__ __forceinline__ u32 sign_word(const Quants& r, int g) { return wordr(r.q[(g >> 1) & 1], 2 * (g & 1) + 1); }
  // the table entries of the lane's two runs of eight weights
  static __device__ __forceinline__ void quants_now(Quants& o, const u8*, int g, int, int lh) {
    const u32* const tab = iq2_tables();
    const u32 idx = index_word(o, g) >> (16 * lh), sg = sign_word(o, g) >> (14 * lh);
#pragma unroll
    for (int l = 0; l < 2; l++) o.sel[l] = *ILT_LDS_PTR(const u32, tab + ((idx >> (8 * l)) & 0xFF)) | *ILT_LDS_PTR(const u32, tab + 256 + ((sg >> (7 * l)) & 127));
  }
  static __device__ __forceinline__ void group(Block& b, const Quants& r, int g, int, v4i&, v4i& lo) {
    b.k[g] = (int)((sign_word(r, g) >> 27) | 1);
#pragma unroll
    for (int k = 0; k < 4; k++)                      // 8, 25, 43 and what they are negated
      lo[k] = (int)__builtin_amdgcn_perm(0x00D5E7F8u, 0x002B1908u, (k & 1 ? r.sel[k >> 1] >> 4 : r.sel[k >> 1]) & 0x07070707u);
  }
  static __device__ __forceinline__ int scale(const Block& b, int g) { return b.k[g]; }
};

template <int TN, int RAW, bool MINS, int XB = 1> struct RegSmem {
  // the tokens' quants of a super-block: four tokens a kilobyte and 64 bytes, piece p of token t at p ^ (t & 3) of its 256
  __align__(16) u8 xs[XB][TN / 4 * 1088];
  __align__(16) u8 ms[3][MINS ? TN * 32 : 16];          // the sums of 32 as halves: eight times 128 * (sum >> 7), eight times sum & 127 (Q2_K: the sums of 16, exact as they are)
  __align__(16) u8 ws[RAW];                 // the rows' blocks
  float xd[3][TN];
};
template <int FMT, int NP, int WR, int WT> constexpr int raw_bytes() { return (WT == 1 && NP > 1 ? 1 : 2) * WR * RegW<FMT>::LBYTES; }
template <int FMT, int NP, int WR, int WT> using RegSmemOf = RegSmem<32 * NP * WT, raw_bytes<FMT, NP, WR, WT>(), RegW<FMT>::MINS, NP == 1 ? 2 : 1>;

// Rows r0 .. of one matrix (p.rows of them, results to p.y) x tokens tok0 .. tok0 + ntok - 1: WR x WT waves of 32 rows x 32 NP
// tokens.  NP 1: nothing to share out between two halves, so the tokens and the rows' blocks are in two buffers and a block ahead.
template <int FMT, int NP, int WR, int WT, class F = RegW<FMT>>
__device__ __forceinline__ void reg_tile(const BfParams& p, const u8* w, int r0, long tok0, int ntok, unsigned char* smem) {
  constexpr int TN = 32 * NP * WT, THREADS = 64 * WR * WT;
  constexpr bool DEEP = NP == 1;
  constexpr int NI = DEEP ? 8 / WR : TN / (8 * WR * WT);       // direct loads of a wave a super-block's half (NP 1: all) of the tokens (four tokens each)
  constexpr int NW = (F::LOADS + WT - 1) / WT;       // and of the rows' blocks
  constexpr int NC = (2 * TN + THREADS - 1) / THREADS;         // half tokens' sums a thread brings
  static_assert(NP == 1 ? WT == 1 && 8 % WR == 0 : NP == 2 || NP == 4, "patches a wave");
  using Smem = RegSmemOf<FMT, NP, WR, WT>;
  Smem& S = *(Smem*)smem;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nsb = p.cols / 256;
  const int l32 = lane & 31, lh = lane >> 5;
  const int wr0 = 32 * (wave % WR), wt0 = 32 * NP * (wave / WR);
  const __amdgpu_buffer_rsrc_t rw = ilt_rsrc(ilt_uniform_ptr(w), (u32)p.rows * (u32)(nsb * F::BLOCK));
  // (past the matrix's rows: zeros.  What may lie past the end goes into the loads' vector offset, which the descriptor's bound
  // is checked against whatever the scalar one is; the scalar offset is the block's within a row.)
  const u32 row_bytes = (u32)(nsb * F::BLOCK);
  const typename F::At at = F::place(row_bytes, lane, r0 + wr0, p.rows);
  const int wg = wave % WR, wq = wave / WR;          // the wave's group of rows, its place among those that share it
  auto issue_w = [&](int sb, int buf) {
    u8* const dst = S.ws + ((WT == 1 && !DEEP ? 0 : buf) * WR + wg) * F::LBYTES;
    u32 rb = row_bytes;
    asm volatile("" : "+s"(rb));                     // (offsets made here each time: kept, they are registers the products want)
#pragma unroll
    for (int i = 0; i < NW; i++)
      if (F::LOADS % WT == 0 || wq * NW + i < F::LOADS) F::issue(wq * NW + i, rw, w, at, rb, (u32)(r0 + wr0), (u32)sb * F::BLOCK, dst);
  };
  const u8* xbase = (const u8*)ilt_uniform_ptr((const i8*)p.x + tok0 * (long)p.cols);
  // (past the tile's tokens: zeros)
  const __amdgpu_buffer_rsrc_t rx = ilt_rsrc(xbase, (u32)(__builtin_amdgcn_readfirstlane(ntok) * p.cols));
  const u32 xlane = (u32)(lane >> 4) * (u32)p.cols + 16 * (u32)((lane & 15) ^ (lane >> 4));
  // half H of the tokens: the first or the second NP / 2 patches of every wave's (NP 1: all of them, into buffer H)
  auto issue_x = [&](int sb, int h) {
    u32 cols = (u32)p.cols;
    asm volatile("" : "+s"(cols));
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int j = wave * NI + i, q = j / (4 * NP), k4 = DEEP ? j : 8 * NP * q + 4 * NP * h + j % (4 * NP);      // tokens 4 k4 .. + 3
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (ILT_LDS void*)(S.xs[DEEP ? h : 0] + k4 * 1088), 16, xlane + (u32)(k4 * 4) * cols, sb * 256, 0, 0);
    }
  };
  // the tokens' scales and sums of 32 of a super-block, through registers
  const __amdgpu_buffer_rsrc_t rd = ilt_rsrc(ilt_uniform_ptr(p.xd + tok0 * nsb), (u32)(__builtin_amdgcn_readfirstlane(ntok) * nsb) * 4);
  const __amdgpu_buffer_rsrc_t rb = ilt_rsrc(ilt_uniform_ptr(p.bsums + (F::MINS ? tok0 * (p.cols >> 4) : 0)), F::MINS ? (u32)(__builtin_amdgcn_readfirstlane(ntok) * (p.cols >> 4)) * 4 : 0);
  float c_yd[NC]; int4 c_bs[NC][2];                  // (past the tile's tokens: zeros)
  auto load_consts = [&](int sb) {
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int h = t + i * THREADS;
      if (2 * TN < THREADS && h >= 2 * TN) return;
      const u32 ctok = (u32)((h >> 1) * nsb);
      c_yd[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, ctok * 4, sb * 4, 0));
      if constexpr (F::MINS) {
        const u32 o = ctok * 64 + 32 * (h & 1);
        const ilt_v4i a = __builtin_amdgcn_raw_buffer_load_b128(rb, o, sb * 64, 0), b = __builtin_amdgcn_raw_buffer_load_b128(rb, o + 16, sb * 64, 0);
        c_bs[i][0] = make_int4(a.x, a.y, a.z, a.w); c_bs[i][1] = make_int4(b.x, b.y, b.z, b.w);
      }
    }
  };
  auto store_consts = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int h = t + i * THREADS;
      if (2 * TN < THREADS && h >= 2 * TN) return;
      if ((h & 1) == 0) S.xd[buf][h >> 1] = c_yd[i];
      const int4 &b0 = c_bs[i][0], &b1 = c_bs[i][1];
      if constexpr (FMT == ILT_Q2_K) {
        _Float16 hh[8];
#pragma unroll
        for (int k = 0; k < 8; k++) hh[k] = (_Float16)(float)(k < 4 ? (int)wordr(b0, k) : (int)wordr(b1, k - 4));
        __builtin_memcpy(S.ms[buf] + 32 * (h >> 1) + 16 * (h & 1), hh, 16);
      } else if constexpr (F::MINS) {
        const int s[4] = { b0.x + b0.y, b0.z + b0.w, b1.x + b1.y, b1.z + b1.w };
        _Float16 hh[4], ll[4];
#pragma unroll
        for (int k = 0; k < 4; k++) { hh[k] = (_Float16)(float)(s[k] & ~127); ll[k] = (_Float16)(float)(s[k] & 127); }
        _Float16* const dst = (_Float16*)(S.ms[buf] + 32 * (h >> 1)) + 4 * (h & 1);
        __builtin_memcpy(dst, hh, 8);
        __builtin_memcpy(dst + 8, ll, 8);
      }
    }
  };
  v16f sum[NP][1];
#pragma unroll
  for (int a = 0; a < NP; a++)
#pragma unroll
    for (int r = 0; r < 16; r++) sum[a][0][r] = 0.0f;
  const u32 x0 = (u32)((wt0 + l32) >> 2) * 1088 + (u32)(l32 & 3) * 256 + 16 * (u32)(lh ^ (l32 & 3)), x1 = x0 ^ 32;
  const u8* const wsrc = S.ws + wg * F::LBYTES;
  v4i hi[8], lo[8];
  typename F::Block blk;
  issue_w(0, 0);
  if (DEEP) issue_w(min(1, nsb - 1), 1);
  issue_x(0, 0);
  load_consts(0);
  store_consts(0);
  for (int i = t; i < TN; i += THREADS) S.xd[2][i] = 0.0f;       // (the block before the first: nothing)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the direct loads have landed
  ilt_barrier_lds();
  F::block(blk, wsrc, l32, lh);
  {
    typename F::Quants qs;
#pragma unroll
    for (int g = 0; g < 8; g++) { F::quants(qs, wsrc, g, l32, lh); F::quants_now(qs, wsrc, g, l32, lh); F::group(blk, qs, g, lh, hi[g], lo[g]); }
  }
  if (DEEP && WT > 1) ilt_barrier_lds();             // (a shared first buffer is written again)
  // integer sums: of the patch being multiplied, and of the one before as they are, or put together where registers are short
  constexpr bool TIGHT = (NP == 4 && F::PLANES == 2) || DEEP;
  v16i X[TIGHT || F::PLANES < 2 ? 1 : 2], Y[TIGHT ? 1 : 2], P, D[2];      // (D: a group's sums, still without its scale)
#pragma unroll
  for (int r = 0; r < 16; r++) { if (TIGHT) P[r] = 0; else { X[F::PLANES == 2][r] = 0; Y[1][r] = 0; } }
  v16f im = {};                                      // and of the minimums
  float dprev = 0.0f, dmprev = 0.0f;
  int c0 = 0, c1 = 1, c2 = 2;                        // where the tokens' constants of this block, the next and the one before are
  // Patch a of the block: its products, and beside them the terms of the patch before it and, with the last patch, the next
  // block's operands, each group's as soon as this block's have been multiplied.
  auto patch = [&](auto ac, const u8* wnext, const u8* xs) {
    constexpr int a = decltype(ac)::value, par = a & 1, pa = (a + NP - 1) % NP;
    constexpr bool last = a == NP - 1;
    constexpr int XI = TIGHT || F::PLANES < 2 ? 0 : 1, YI = TIGHT ? 0 : 1;
    v16i &XC = X[par * XI], &YC = Y[par * YI], &XP = X[(par ^ 1) * XI], &YP = Y[(par ^ 1) * YI];

    const float dp = a == 0 ? dprev : blk.d, dmp = a == 0 ? dmprev : blk.dm;
    const float* const xp = S.xd[a == 0 ? c2 : c0] + wt0 + 32 * pa + 4 * lh;
    auto frag = [&](int g) { return __builtin_bit_cast(v4i, ilt_lds_ld16((DEEP ? xs : S.xs[0]) + (g & 1 ? x1 : x0) + 8704 * a + 64 * (g >> 1))); };
    const v16i zi = {};
    typename F::Block nb = {};
    typename F::Quants qs;
    v4i f0 = frag(0), f1 = frag(1);
    float4 yp = lds_f4(xp), yn;
    v8h sums;
    if constexpr (last) { F::block(nb, wnext, l32, lh); F::quants(qs, wnext, 0, l32, lh); }
#pragma unroll
    for (int g = 0; g < 8; g++) {
      const v4i f = f0;
      f0 = f1;
      // (what the next step wants from LDS is asked for before this one's products)
      if (g < 6) f1 = frag(g + 2);
      if (last) F::quants_now(qs, wnext, g, l32, lh);
      if (last && g < 7) F::quants(qs, wnext, g + 1, l32, lh);
      if (g % 2 == 0 && g < 6) yn = lds_f4(xp + 4 * g + 8);
      if (F::MINS && g == 6) sums = __builtin_bit_cast(v8h, ilt_lds_ld16(S.ms[c0] + 32 * (wt0 + 32 * a + l32) + 16 * lh));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (F::PLANES == 2) XC = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, hi[g], g ? XC : zi, 0, 0, 0);
      if constexpr (F::PLANES > 0) YC = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, lo[g], g ? YC : zi, 0, 0, 0);
      else {                                         // the group before's sums by its scale while this one's are made
        D[g & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, lo[g], zi, 0, 0, 0);
        if (g > 0) {
          const int sc = F::scale(blk, g - 1);
#pragma unroll
          for (int r = 0; r < 16; r++) YC[r] = g > 1 ? ilt_mad24(D[(g & 1) ^ 1][r], sc, YC[r]) : ilt_mul24(D[(g & 1) ^ 1][r], sc);
          asm volatile("" : "+v"(YC));
        }
      }
      // two results' terms, step by step side by side (one after the other every instruction waits for the one before it)
      {
        const int r = 2 * g;
        const float y0 = r & 2 ? yp.z : yp.x, y1 = r & 2 ? yp.w : yp.y;
        const int i0 = TIGHT ? P[r] : F::PLANES == 2 ? (XP[r] << F::SH) + YP[r] : YP[r], i1 = TIGHT ? P[r + 1] : F::PLANES == 2 ? (XP[r + 1] << F::SH) + YP[r + 1] : YP[r + 1];
        float b0 = y0 * dp, b1 = y1 * dp, f0_ = (float)i0, f1_ = (float)i1, s0 = sum[pa][0][r], s1 = sum[pa][0][r + 1];
        if constexpr (F::MINS) {
          float a0 = y0 * dmp, a1 = y1 * dmp;
          asm volatile("" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1), "+v"(f0_), "+v"(f1_));
          a0 = a0 * im[r]; a1 = a1 * im[r + 1]; b0 = b0 * f0_; b1 = b1 * f1_;
          asm volatile("" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
          s0 = s0 - a0; s1 = s1 - a1;
          asm volatile("" : "+v"(s0), "+v"(s1));
        } else {
          asm volatile("" : "+v"(b0), "+v"(b1), "+v"(f0_), "+v"(f1_));
          if constexpr (F::PLANES == 0) { f0_ = f0_ * 0.5f; f1_ = f1_ * 0.5f; }
          b0 = b0 * f0_; b1 = b1 * f1_;
          asm volatile("" : "+v"(b0), "+v"(b1));
        }
        sum[pa][0][r] = s0 + b0; sum[pa][0][r + 1] = s1 + b1;
      }
      if (g % 2 == 1) yp = yn;
      // (pinned here: the compiler would put all of it off to the block's end, where nothing runs beside it)
      asm volatile("" : "+v"(sum[pa][0]));
      if constexpr (last) {
        F::group(nb, qs, g, lh, hi[g], lo[g]);
        if constexpr (F::PLANES == 2) asm volatile("" : "+v"(hi[g]), "+v"(lo[g]));
        else asm volatile("" : "+v"(lo[g]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (F::PLANES == 0) {
      const int sc = F::scale(blk, 7);
#pragma unroll
      for (int r = 0; r < 16; r++) YC[r] = ilt_mad24(D[1][r], sc, YC[r]);
      asm volatile("" : "+v"(YC));
    }
    if constexpr (F::MINS) {
      const v16f zf = {};
      im = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, blk.mins, zf, 0, 0, 0);
    }
    if constexpr (TIGHT) {
#pragma unroll
      for (int r = 0; r < 16; r++) P[r] = F::PLANES == 2 ? (XC[r] << F::SH) + YC[r] : YC[r];
      asm volatile("" : "+v"(P));
    }
    if constexpr (last) { dprev = blk.d; dmprev = blk.dm; blk = nb; }
  };
#pragma unroll 1
  for (int sb = 0; sb < nsb; sb++) {

    const int nx = min(sb + 1, nsb - 1), nbuf = (sb + 1) & 1;       // (the last block's again, for nobody)
    using std::integral_constant;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (DEEP) {
      issue_x(nx, nbuf);
      issue_w(min(sb + 2, nsb - 1), sb & 1);         // (this block's operands are made)
    } else {
      issue_x(sb, 1);                                // (the block before's second half has been multiplied)
      issue_w(nx, nbuf);                             // (and this block's operands are made)
    }
    load_consts(nx);
    __builtin_amdgcn_sched_barrier(0);
    const u8* const wnext = wsrc + (WT == 1 && !DEEP ? 0 : nbuf) * WR * F::LBYTES;
    const u8* const xs = S.xs[DEEP ? sb & 1 : 0];
    patch(integral_constant<int, 0>{}, wnext, xs);
    if constexpr (NP == 4) patch(integral_constant<int, 1>{}, wnext, xs);
    store_consts(c1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    ilt_barrier_lds();
    if constexpr (!DEEP) {
      __builtin_amdgcn_sched_barrier(0);
      issue_x(nx, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NP == 4) {
        patch(integral_constant<int, 2>{}, wnext, xs);
        patch(integral_constant<int, 3>{}, wnext, xs);
      } else {
        patch(integral_constant<int, 1>{}, wnext, xs);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      ilt_barrier_lds();
    }
    const int c = c2; c2 = c0; c0 = c1; c1 = c;
  }
  {
    const float* const xp = S.xd[c2] + wt0 + 32 * (NP - 1) + 4 * lh;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      if constexpr (F::MINS) sum[NP - 1][0][r] = sum[NP - 1][0][r] - (xp[8 * (r >> 2) + (r & 3)] * dmprev) * im[r];
      const int is = TIGHT ? P[r] : F::PLANES == 2 ? (X[F::PLANES == 2 && !TIGHT][r] << F::SH) + Y[!TIGHT][r] : Y[!TIGHT][r];
      sum[NP - 1][0][r] = sum[NP - 1][0][r] + (xp[8 * (r >> 2) + (r & 3)] * dprev) * (F::PLANES == 0 ? (float)is * 0.5f : (float)is);
    }
  }
  if constexpr (F::PLANES == 0) {
#pragma unroll
    for (int a = 0; a < NP; a++)
#pragma unroll
      for (int r = 0; r < 16; r++) sum[a][0][r] = 0.25f * sum[a][0][r];
  }
  store_tile<NP, 1>(sum, p, tok0, ntok, r0, wt0, wr0, l32, lh);
}

// A quarter of a tile's results to y: tokens t0 .. t0 + 3 of the row
__device__ __forceinline__ void split_store(const BfParams& p, const v4f& sum, long tok0, int ntok, int row, int t0) {
  const bool ok = row < p.rows;
  const __amdgpu_buffer_rsrc_t ry = ilt_rsrc(ilt_uniform_ptr(p.y + tok0 * p.ldy), ((u32)(ntok - 1) * (u32)p.ldy + (u32)p.rows) * 4);
  const u32 rows4 = (u32)p.ldy * 4, base = ok ? (u32)(t0 * (int)p.ldy + row) * 4 : 0x80000000u;
  const float bv = p.bias && ok ? p.bias[row] : 0.0f;
  float old[4];
  if (p.acc) {
#pragma unroll
    for (int r = 0; r < 4; r++) old[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ry, base + (u32)r * rows4, 0, 0));
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    float v = sum[r];
    if (p.bias) v = v + bv;
    if (p.acc) v = old[r] + v;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(u32, v), ry, base + (u32)r * rows4, 0, 0);
  }
}

// Rows r0 .. x tokens tok0 .. tok0 + ntok - 1 where the launch has few tiles: a tile of 32 rows x 32 tokens is a workgroup's, its
// super-block u wave u mod 4's.  What bounds such a launch is the chain of a row's blocks: a wave alone on its SIMD issues an
// instruction in 5 cycles, 1.4 us a block, whatever the rest of the chip could do meanwhile.  A block's integers and float terms
// depend on nothing before them, only the sums' order does, so every wave makes its blocks' terms as reg_tile does (its own loads,
// operands and products, a block ahead: nothing shared), leaves them in LDS, and once a round -- four blocks -- each adds the terms of
// its own quarter of the tile in the CPU's order.  A round takes 1.95 us (four waves of a CU share its LDS and the loads' way: 1.6
// without the loads).  us before and now, matrices from memory: Q6_K 2560 x 9728 on 33 to 96 tokens 41-43 -> 26-27; 4096 x 4096 on 64
// 28 -> 15; Q4_K 2560 x 4096 on 40 16.7 -> 12.8.  (Two waves a tile and two tiles of rows a workgroup: on 160 tokens 43.)
constexpr int KS = 4;                  // waves of a workgroup, and super-blocks of a round
template <int FMT> struct SplitSmem {
  RegSmem<32, 2 * RegW<FMT>::LBYTES, RegW<FMT>::MINS, 2> w[KS];
  __align__(16) float ex[KS][KS][RegW<FMT>::MINS ? 2 : 1][256];       // terms [quarter][wave][a term][lane's four]
};
template <int FMT>
__device__ __forceinline__ void reg_split(const BfParams& p, const u8* w, int r0, long tok0, int ntok, unsigned char* smem) {
  using F = RegW<FMT>;
  constexpr int TERMS = F::MINS ? 2 : 1;
  static_assert(F::PLANES == 2, "a result's integer is two planes");
  SplitSmem<FMT>& W = *(SplitSmem<FMT>*)smem;
  const int lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto& S = W.w[ks];
  const int nsb = p.cols / 256, rounds = (nsb + KS - 1) / KS;
  const int l32 = lane & 31, lh = lane >> 5;
  const u32 row_bytes = (u32)(nsb * F::BLOCK);
  const __amdgpu_buffer_rsrc_t rw = ilt_rsrc(ilt_uniform_ptr(w), (u32)p.rows * row_bytes);      // (past the matrix's rows: zeros)
  const typename F::At at = F::place(row_bytes, lane, r0, p.rows);
  auto issue_w = [&](int sb, int buf) {
#pragma unroll
    for (int i = 0; i < F::LOADS; i++) F::issue(i, rw, w, at, row_bytes, (u32)r0, (u32)sb * F::BLOCK, S.ws + buf * F::LBYTES);
  };
  ntok = __builtin_amdgcn_readfirstlane(ntok);
  const __amdgpu_buffer_rsrc_t rx = ilt_rsrc(ilt_uniform_ptr((const i8*)p.x + tok0 * (long)p.cols), (u32)(ntok * p.cols));      // (past the tile's tokens: zeros)
  const u32 xlane = (u32)(lane >> 4) * (u32)p.cols + 16 * (u32)((lane & 15) ^ (lane >> 4));
  auto issue_x = [&](int sb, int buf) {
#pragma unroll
    for (int i = 0; i < 8; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (ILT_LDS void*)(S.xs[buf] + i * 1088), 16, xlane + (u32)(i * 4) * (u32)p.cols, sb * 256, 0, 0);
  };
  const __amdgpu_buffer_rsrc_t rd = ilt_rsrc(ilt_uniform_ptr(p.xd + tok0 * nsb), (u32)(ntok * nsb) * 4);
  const __amdgpu_buffer_rsrc_t rb = ilt_rsrc(ilt_uniform_ptr(p.bsums + (F::MINS ? tok0 * (p.cols >> 4) : 0)), F::MINS ? (u32)(ntok * (p.cols >> 4)) * 4 : 0);
  float c_yd; int4 c_bs[2];
  auto load_consts = [&](int sb) {                   // half a token's sums of 16 a lane
    const u32 ctok = (u32)((lane >> 1) * nsb);
    c_yd = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, ctok * 4, sb * 4, 0));
    if constexpr (F::MINS) {
      const u32 o = ctok * 64 + 32 * (lane & 1);
      const ilt_v4i a = __builtin_amdgcn_raw_buffer_load_b128(rb, o, sb * 64, 0), b = __builtin_amdgcn_raw_buffer_load_b128(rb, o + 16, sb * 64, 0);
      c_bs[0] = make_int4(a.x, a.y, a.z, a.w); c_bs[1] = make_int4(b.x, b.y, b.z, b.w);
    }
  };
  auto store_consts = [&](int buf) {
    if ((lane & 1) == 0) S.xd[buf][lane >> 1] = c_yd;
    if constexpr (F::MINS) {
      const int4 &b0 = c_bs[0], &b1 = c_bs[1];
      const int s[4] = { b0.x + b0.y, b0.z + b0.w, b1.x + b1.y, b1.z + b1.w };
      _Float16 hh[4], ll[4];
#pragma unroll
      for (int k = 0; k < 4; k++) { hh[k] = (_Float16)(float)(s[k] & ~127); ll[k] = (_Float16)(float)(s[k] & 127); }
      _Float16* const dst = (_Float16*)(S.ms[buf] + 32 * (lane >> 1)) + 4 * (lane & 1);
      __builtin_memcpy(dst, hh, 8);
      __builtin_memcpy(dst + 8, ll, 8);
    }
  };
  const u32 x0 = (u32)(l32 >> 2) * 1088 + (u32)(l32 & 3) * 256 + 16 * (u32)(lh ^ (l32 & 3)), x1 = x0 ^ 32;
  v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
  v4i hi[8], lo[8];
  typename F::Block blk;
  auto mine = [&](int i) { return min(i * KS + ks, nsb - 1); };      // the wave's block of round i (past the last: the last again, for nobody)
  issue_w(mine(0), 0);
  issue_x(mine(0), 0);
  load_consts(mine(0));
  issue_w(mine(1), 1);
  store_consts(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  F::block(blk, S.ws, l32, lh);
  {
    typename F::Quants qs;
#pragma unroll
    for (int g = 0; g < 8; g++) { F::quants(qs, S.ws, g, l32, lh); F::quants_now(qs, S.ws, g, l32, lh); F::group(blk, qs, g, lh, hi[g], lo[g]); }
  }
  v16i X, Y, P;
  v16f im = {};
  float dprev = 0.0f, dmprev = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; r++) P[r] = 0;
  float* const ex = (float*)W.ex;
  // four results' terms, of the round before, to their quarter's place
  auto term = [&](int j, const float4& y) {
    float a[4], b[4], f[4];
    const float yv[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
    for (int i = 0; i < 4; i++) { b[i] = yv[i] * dprev; f[i] = (float)P[4 * j + i]; if constexpr (F::MINS) a[i] = yv[i] * dmprev; }
#pragma unroll
    for (int i = 0; i < 4; i++) { b[i] = b[i] * f[i]; if constexpr (F::MINS) a[i] = a[i] * im[4 * j + i]; }
    float* const o = ex + ((j * KS + ks) * TERMS) * 256 + 4 * lane;
    if constexpr (F::MINS) *ILT_LDS_PTR(v4f, o) = v4f{a[0], a[1], a[2], a[3]};
    *ILT_LDS_PTR(v4f, o + (TERMS - 1) * 256) = v4f{b[0], b[1], b[2], b[3]};
  };
  // the wave's quarter: the terms of round i's blocks in order
  auto add = [&](int i) {
    v4f t[KS][TERMS];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
      for (int k = 0; k < TERMS; k++) t[s][k] = *ILT_LDS_PTR(const v4f, ex + ((ks * KS + s) * TERMS + k) * 256 + 4 * lane);
#pragma unroll
    for (int s = 0; s < KS; s++)
      if (i * KS + s < nsb) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if constexpr (F::MINS) sum[r] = sum[r] - t[s][0][r];
          sum[r] = sum[r] + t[s][TERMS - 1][r];
        }
      }
    asm volatile("" : "+v"(sum));                    // (the reads have come back before the wave meets the next barrier)
  };
  int c0 = 0, c1 = 1, c2 = 2;
#pragma unroll 1
  for (int i = 0; i < rounds; i++) {
    const int nbuf = (i + 1) & 1;
    __builtin_amdgcn_sched_barrier(0);
    issue_x(mine(i + 1), nbuf);
    load_consts(mine(i + 1));
    issue_w(mine(i + 2), i & 1);                     // (this block's operands are made)
    __builtin_amdgcn_sched_barrier(0);
    const u8 *const wnext = S.ws + nbuf * F::LBYTES, *const xs = S.xs[i & 1];
    const float* const xp = S.xd[c2] + 4 * lh;
    auto frag = [&](int g) { return __builtin_bit_cast(v4i, ilt_lds_ld16(xs + (g & 1 ? x1 : x0) + 64 * (g >> 1))); };
    const v16i zi = {};
    typename F::Block nb = {};
    typename F::Quants qs;
    v4i f0 = frag(0), f1 = frag(1);
    float4 y = lds_f4(xp);
    v8h sums;
    F::block(nb, wnext, l32, lh); F::quants(qs, wnext, 0, l32, lh);
#pragma unroll
    for (int g = 0; g < 8; g++) {
      const v4i f = f0;
      f0 = f1;
      if (g < 6) f1 = frag(g + 2);
      F::quants_now(qs, wnext, g, l32, lh);
      if (g < 7) F::quants(qs, wnext, g + 1, l32, lh);
      if (F::MINS && g == 6) sums = __builtin_bit_cast(v8h, ilt_lds_ld16(S.ms[c0] + 32 * l32 + 16 * lh));
      __builtin_amdgcn_sched_barrier(0);
      X = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, hi[g], g ? X : zi, 0, 0, 0);
      Y = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, lo[g], g ? Y : zi, 0, 0, 0);
      if (g == 0) asm volatile("s_barrier" ::: "memory");      // (the round before's terms have been added)
      if (g % 2 == 1) {
        term(g >> 1, y);
        if (g < 7) y = lds_f4(xp + 8 * (g >> 1) + 8);
      }
      F::group(nb, qs, g, lh, hi[g], lo[g]);
      asm volatile("" : "+v"(hi[g]), "+v"(lo[g]));
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (F::MINS) {
      const v16f zf = {};
      im = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, blk.mins, zf, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) P[r] = (X[r] << F::SH) + Y[r];
    dprev = blk.d; dmprev = blk.dm; blk = nb;
    store_consts(c1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    ilt_barrier_lds();
    if (i > 0) add(i - 1);
    const int c = c2; c2 = c0; c0 = c1; c1 = c;
  }
  ilt_barrier_lds();
  {
    const float* const xp = S.xd[c2] + 4 * lh;
#pragma unroll
    for (int j = 0; j < 4; j++) term(j, lds_f4(xp + 8 * j));
  }
  ilt_barrier_lds();
  add(rounds - 1);
  split_store(p, sum, tok0, ntok, r0 + l32, 8 * ks + 4 * lh);
}

// The same with two workgroups a CU, where there are more tiles than CUs: one buffer for the tokens and one for the rows' blocks, asked
// for anew as soon as a block is through, so that a wave waits for them while the other workgroup's waves work; the tokens' sums in
// registers; and of a block's terms only those in LDS that another wave adds: 77 to 79 KB.  Alone on a CU it takes 2.25 us
// a round for reg_split's 1.95, two of them 3.25.  us with whole tiles and now, matrices from memory: Q6_K 2560 x 9728 on 160 tokens
// 62 -> 37, on 256 62 -> 54; 4096 x 4096 on 128 28 -> 20; Q4_K 2560 x 4096 on 128 24 -> 18.
template <int FMT> struct SplitSmem2 {
  struct { __align__(16) u8 xs[8192]; __align__(16) u8 ws[RegW<FMT>::LBYTES]; float xd[2][32]; } w[KS];
  __align__(16) float ex[KS][KS - 1][RegW<FMT>::MINS ? 2 : 1][256];       // terms [quarter][the other waves in turn][a term][lane's four]
};
template <int FMT>
__device__ __forceinline__ void reg_split2(const BfParams& p, const u8* w, int r0, long tok0, int ntok, unsigned char* smem) {
  using F = RegW<FMT>;
  constexpr int TERMS = F::MINS ? 2 : 1;
  static_assert(F::PLANES == 2, "a result's integer is two planes");
  SplitSmem2<FMT>& W = *(SplitSmem2<FMT>*)smem;
  const int lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto& S = W.w[ks];
  const int nsb = p.cols / 256, rounds = (nsb + KS - 1) / KS;
  const int l32 = lane & 31, lh = lane >> 5;
  const u32 row_bytes = (u32)(nsb * F::BLOCK);
  const __amdgpu_buffer_rsrc_t rw = ilt_rsrc(ilt_uniform_ptr(w), (u32)p.rows * row_bytes);      // (past the matrix's rows: zeros)
  const typename F::At at = F::place(row_bytes, lane, r0, p.rows);
  ntok = __builtin_amdgcn_readfirstlane(ntok);
  const __amdgpu_buffer_rsrc_t rx = ilt_rsrc(ilt_uniform_ptr((const i8*)p.x + tok0 * (long)p.cols), (u32)(ntok * p.cols));      // (past the tile's tokens: zeros)
  // the tokens' quants: a kilobyte the half of a super-block of eight tokens, piece q of token t at q ^ (t >> 1 & 7) of its eight
  const u32 xpc = 16 * (u32)((lane & 7) ^ ((lane >> 4) & 3)), xrow = (u32)(lane >> 3) * (u32)p.cols;
  const __amdgpu_buffer_rsrc_t rd = ilt_rsrc(ilt_uniform_ptr(p.xd + tok0 * nsb), (u32)(ntok * nsb) * 4);
  const __amdgpu_buffer_rsrc_t rb = ilt_rsrc(ilt_uniform_ptr(p.bsums + (F::MINS ? tok0 * (p.cols >> 4) : 0)), F::MINS ? (u32)(ntok * (p.cols >> 4)) * 4 : 0);
  float c_yd; int4 c_bs[4];
  auto mine = [&](int i) { return min(i * KS + ks, nsb - 1); };      // the wave's block of round i (past the last: the last again, for nobody)
  auto issue_w = [&](int sb) {
#pragma unroll
    for (int i = 0; i < F::LOADS; i++) F::issue(i, rw, w, at, row_bytes, (u32)r0, (u32)sb * F::BLOCK, S.ws);
  };
  auto issue_x = [&](int sb) {                       // and the token's scale and sums of 16, a token two lanes
#pragma unroll
    for (int i = 0; i < 8; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (ILT_LDS void*)(S.xs + i * 1024), 16, xrow + (i & 1 ? xpc ^ 64 : xpc) + (u32)(8 * (i & 3)) * (u32)p.cols + 128 * (i >> 2), sb * 256, 0, 0);
    const u32 ctok = (u32)(l32 * nsb);
    c_yd = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, ctok * 4, sb * 4, 0));
    if constexpr (F::MINS) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const ilt_v4i a = __builtin_amdgcn_raw_buffer_load_b128(rb, ctok * 64 + 16 * k, sb * 64, 0);
        c_bs[k] = make_int4(a.x, a.y, a.z, a.w);
      }
    }
  };
  const u8* const xb = S.xs + 128 * l32;
  const int xsw = (l32 >> 1) & 7;
  auto frag = [&](int g) { return __builtin_bit_cast(v4i, ilt_lds_ld16(xb + 4096 * (g >> 2) + 16 * ((2 * (g & 3) + lh) ^ xsw))); };
  v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
  v4i hi[8], lo[8];
  typename F::Block blk;
  issue_w(mine(0));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  F::block(blk, S.ws, l32, lh);
  {
    typename F::Quants qs;
#pragma unroll
    for (int g = 0; g < 8; g++) { F::quants(qs, S.ws, g, l32, lh); F::quants_now(qs, S.ws, g, l32, lh); F::group(blk, qs, g, lh, hi[g], lo[g]); }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the blocks' place is written again)
  issue_x(mine(0));
  issue_w(mine(1));
  v16i X, Y, P;
  v16f im = {};
  float dprev = 0.0f, dmprev = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; r++) P[r] = 0;
  float* const ex = (float*)W.ex;
  auto place = [&](int j, int s) { return ex + ((j * (KS - 1) + s) * TERMS) * 256 + 4 * lane; };      // (s: the source's number without the owner's)
  v4f own[TERMS];
  // four results' terms, of the round before
  auto term = [&](int j, const float4& y) {
    v4f a = {}, b;
    const float yv[4] = {y.x, y.y, y.z, y.w};
    float f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) { b[i] = yv[i] * dprev; f[i] = (float)P[4 * j + i]; if constexpr (F::MINS) a[i] = yv[i] * dmprev; }
#pragma unroll
    for (int i = 0; i < 4; i++) { b[i] = b[i] * f[i]; if constexpr (F::MINS) a[i] = a[i] * im[4 * j + i]; }
    if (j == ks) {
      if constexpr (F::MINS) own[0] = a;
      own[TERMS - 1] = b;
    } else {
      float* const o = place(j, ks - (ks > j ? 1 : 0));
      if constexpr (F::MINS) *ILT_LDS_PTR(v4f, o) = a;
      *ILT_LDS_PTR(v4f, o + (TERMS - 1) * 256) = b;
    }
  };
  // the wave's quarter: the terms of round i's blocks in order, its own among the others'
  auto add = [&](int i) {
    v4f t[KS][TERMS];
#pragma unroll
    for (int s = 0; s < KS - 1; s++)
#pragma unroll
      for (int k = 0; k < TERMS; k++) t[s][k] = *ILT_LDS_PTR(const v4f, place(ks, s) + k * 256);
#pragma unroll
    for (int s = KS - 1; s >= 0; s--)                // (moved up from the wave's place on)
#pragma unroll
      for (int k = 0; k < TERMS; k++) t[s][k] = s == ks ? own[k] : s > ks ? t[s - (s > 0)][k] : t[s][k];
#pragma unroll
    for (int s = 0; s < KS; s++)
      if (i * KS + s < nsb) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if constexpr (F::MINS) sum[r] = sum[r] - t[s][0][r];
          sum[r] = sum[r] + t[s][TERMS - 1][r];
        }
      }
    asm volatile("" : "+v"(sum));                    // (the reads have come back before the wave meets the next barrier)
  };
#pragma unroll 1
  for (int i = 0; i < rounds; i++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const float* const xp = S.xd[(i & 1) ^ 1] + 4 * lh;
    const v16i zi = {};
    typename F::Block nb = {};
    typename F::Quants qs;
    v4i f0 = frag(0), f1 = frag(1);
    float4 y = lds_f4(xp);
    F::block(nb, S.ws, l32, lh); F::quants(qs, S.ws, 0, l32, lh);
    if (lh == 0) S.xd[i & 1][l32] = c_yd;
    v8h sums;
    if constexpr (F::MINS) {                         // the sums of 32, eight times 128 * (sum >> 7) or eight times sum & 127
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int v = k & 1 ? wordr(c_bs[k >> 1], 2) + wordr(c_bs[k >> 1], 3) : wordr(c_bs[k >> 1], 0) + wordr(c_bs[k >> 1], 1);
        sums[k] = (_Float16)(float)(v & (lh ? 127 : ~127));
      }
    }
#pragma unroll
    for (int g = 0; g < 8; g++) {
      const v4i f = f0;
      f0 = f1;
      if (g < 6) f1 = frag(g + 2);
      F::quants_now(qs, S.ws, g, l32, lh);
      if (g < 7) F::quants(qs, S.ws, g + 1, l32, lh);
      __builtin_amdgcn_sched_barrier(0);
      X = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, hi[g], g ? X : zi, 0, 0, 0);
      Y = __builtin_amdgcn_mfma_i32_32x32x32_i8(f, lo[g], g ? Y : zi, 0, 0, 0);
      if (g == 0) asm volatile("s_barrier" ::: "memory");      // (the round before's terms have been added)
      if (g % 2 == 1) {
        term(g >> 1, y);
        if (g < 7) y = lds_f4(xp + 8 * (g >> 1) + 8);
      }
      F::group(nb, qs, g, lh, hi[g], lo[g]);
      asm volatile("" : "+v"(hi[g]), "+v"(lo[g]));
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (F::MINS) {
      const v16f zf = {};
      im = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, blk.mins, zf, 0, 0, 0);
    }
    dprev = blk.d; dmprev = blk.dm; blk = nb;
    asm volatile("" : "+v"(blk.d));
    ilt_barrier_lds();                               // the terms are in, and this wave has read its tokens and blocks
    issue_x(mine(i + 1));
    issue_w(mine(i + 2));
    if (i > 0) add(i - 1);
#pragma unroll
    for (int r = 0; r < 16; r++) P[r] = (X[r] << F::SH) + Y[r];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last round's loads, for nobody: nothing may land in LDS after the workgroup ends)
  ilt_barrier_lds();
  {
    const float* const xp = S.xd[(rounds & 1) ^ 1] + 4 * lh;
#pragma unroll
    for (int j = 0; j < 4; j++) term(j, lds_f4(xp + 8 * j));
  }
  ilt_barrier_lds();
  add(rounds - 1);
  split_store(p, sum, tok0, ntok, r0 + l32, 8 * ks + 4 * lh);
}

// Rows r0 .. + 15 x tokens tok0 .. tok0 + ntok - 1 (16 NT at most): a super-block in eight a wave's, two waves a SIMD.  A launch of some
// twenty tokens has 80 tiles of 32 x 32 and a chain of 38 blocks (2560 x 9728), on 4 waves each: most of the chip idle.  Tiles of half the
// rows are twice as many CUs', eight waves' chains are five blocks, and a block of 16 rows is half the operands and terms: a round takes 1.5 us
// (NT 1) or 2 (NT 2), a fifth of it the wait for the next blocks, which are asked for as soon as a block is in registers.  The terms go through LDS a
// float a lane: the wave that adds a result of the lanes reads the eight blocks' in the CPU's order.  NT 2: two places for a round's terms, one
// barrier a round; NT 1: one, so that two workgroups are a CU's (480 tiles 22 -> 18 us).  us before (four or eight waves with 16-byte loads straight
// into the operands, or reg_split) and now, matrices from memory: Q6_K 2560 x 9728 on 8 tokens 13.6 -> 11.6, 16 14.9 -> 12.4, 21 23.6 -> 14.7, 32 25.4 ->
// 15.5, 48 26.2 -> 18.2; 1024 x 2560 on 32 10.5 -> 6.4; Q4_K 2560 x 4096 on 8 7.8 -> 6.4, 21 11.0 -> 8.3, 48 12.6 -> 11.1.
constexpr int HS = 8;                  // waves of a workgroup, and super-blocks of a round
template <int FMT> struct HalfW;
template <> struct HalfW<ILT_Q4_K> {
  using F = RegW<ILT_Q4_K>;
  static constexpr int LOADS = 3, LBYTES = 3072;     // RegW's places for 16 rows, the headers behind them
  struct At { u32 a, b, h; };
  static __device__ __forceinline__ At place(u32 row_bytes, int lane) {
    const F::At at = F::place(row_bytes, lane, 0, 0);
    return At{at.a, at.b, (u32)(lane & 15) * row_bytes};
  }
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t rw, const At& at, u32 row_bytes, u32 row0, u32 block, u8* dst) {
    if (i < 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (ILT_LDS void*)(dst + 1024 * i), 16, (i ? at.b : at.a) + (row0 + 8 * i) * row_bytes, block, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (ILT_LDS void*)(dst + 2048), 16, at.h + row0 * row_bytes, block, 0, 0);
  }
  // a lane's half of the columns (HQ): what its four groups need
  static __device__ __forceinline__ void read(F::Block& b, F::Quants& q, const u8* ws, int l16, int lh, int hq) {
    F::quants(q, ws, 0, l16, lh + 4 * hq); F::quants(q, ws, 2, l16, lh + 4 * hq);
    F::block(b, ws - 2048, l16, lh);
    b.sc[0] = hq ? b.sc[1] : b.sc[0];
  }
};
template <> struct HalfW<ILT_Q6_K> {
  using F = RegW<ILT_Q6_K>;
  static constexpr int LOADS = 4, LBYTES = 4352;
  using At = F::At;
  static __device__ __forceinline__ At place(u32 row_bytes, int lane) { return F::place(row_bytes, lane, 0, 0); }
  static __device__ __forceinline__ void issue(int i, __amdgpu_buffer_rsrc_t rw, const At& at, u32 row_bytes, u32 row0, u32 block, u8* dst) {
    F::issue(i, rw, nullptr, at, row_bytes, row0, block, dst);
  }
  static __device__ __forceinline__ void read(F::Block& b, F::Quants& q, const u8* ws, int l16, int lh, int hq) {
    F::quants(q, ws, 0, l16, lh + 4 * hq); F::quants(q, ws, 1, l16, lh + 4 * hq);
    F::quants_now(q, ws, 0, l16, lh + 2 * hq);
    F::block(b, ws, l16, lh);
    b.sc.x = hq ? b.sc.z : b.sc.x; b.sc.y = hq ? b.sc.w : b.sc.y;
  }
};
template <int FMT, int NT> struct HalfSmem {
  struct { __align__(16) u8 xs[4096 * NT]; __align__(16) u8 ws[HalfW<FMT>::LBYTES]; __align__(16) float xd[16 * NT]; } w[HS];
  float ex[NT][4 * NT][HS][RegW<FMT>::MINS ? 2 : 1][64];       // a round's terms [result of a lane][wave][a term][lane]
};
template <int FMT, int NT>
__device__ __forceinline__ void reg_half(const BfParams& p, const u8* w, int r0, long tok0, int ntok, unsigned char* smem) {
  using F = RegW<FMT>;
  using H = HalfW<FMT>;
  constexpr int TERMS = F::MINS ? 2 : 1;
  static_assert(NT == 1 || NT == 2, "a wave adds one of a lane's results");
  HalfSmem<FMT, NT>& W = *(HalfSmem<FMT, NT>*)smem;
  const int lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto& S = W.w[ks];
  const int nsb = p.cols / 256, rounds = (nsb + HS - 1) / HS;
  // lane (l16, lh, hq): row (and token) l16, columns 128 hq + 32 s + 16 lh .. of step s
  const int l16 = lane & 15, lq = lane >> 4, lh = lq & 1, hq = lq >> 1;
  const u32 row_bytes = (u32)(nsb * F::BLOCK);
  const __amdgpu_buffer_rsrc_t rw = ilt_rsrc(ilt_uniform_ptr(w), (u32)p.rows * row_bytes);      // (past the matrix's rows: zeros)
  const typename H::At at = H::place(row_bytes, lane);
  ntok = __builtin_amdgcn_readfirstlane(ntok);
  const __amdgpu_buffer_rsrc_t rx = ilt_rsrc(ilt_uniform_ptr((const i8*)p.x + tok0 * (long)p.cols), (u32)(ntok * p.cols));      // (past the tile's tokens: zeros)
  // the tokens' quants: a kilobyte the half of a super-block of eight tokens, piece q of token t at q ^ (t >> 1 & 7) of its eight
  const u32 xpc = 16 * (u32)((lane & 7) ^ ((lane >> 4) & 3)), xrow = (u32)(lane >> 3) * (u32)p.cols;
  const __amdgpu_buffer_rsrc_t rd = ilt_rsrc(ilt_uniform_ptr(p.xd + tok0 * nsb), (u32)(ntok * nsb) * 4);
  const __amdgpu_buffer_rsrc_t rb = ilt_rsrc(ilt_uniform_ptr(p.bsums + (F::MINS ? tok0 * (p.cols >> 4) : 0)), F::MINS ? (u32)(ntok * (p.cols >> 4)) * 4 : 0);
  float c_yd; int4 c_bs[NT][2];
  auto issue = [&](int i) {
    const int sb = min(i * HS + ks, nsb - 1);        // the wave's block of round i (past the last: the last again, for nobody)
#pragma unroll
    for (int k = 0; k < H::LOADS; k++) H::issue(k, rw, at, row_bytes, (u32)r0, (u32)sb * F::BLOCK, S.ws);
#pragma unroll
    for (int k = 0; k < 4 * NT; k++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (ILT_LDS void*)(S.xs + k * 1024), 16, xrow + (k & 1 ? xpc ^ 64 : xpc) + (u32)(8 * (k % (2 * NT))) * (u32)p.cols + 128 * (k / (2 * NT)), sb * 256, 0, 0);
    c_yd = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, (u32)((lane & (16 * NT - 1)) * nsb) * 4, sb * 4, 0));
    if constexpr (F::MINS) {
#pragma unroll
      for (int h = 0; h < NT; h++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const ilt_v4i a = __builtin_amdgcn_raw_buffer_load_b128(rb, (u32)((l16 + 16 * h) * nsb) * 64 + 32 * lh + 16 * k, sb * 64, 0);
          c_bs[h][k] = make_int4(a.x, a.y, a.z, a.w);
        }
    }
  };
  const int xsw = (l16 >> 1) & 7;
  float sum = 0.0f;
  issue(0);
#pragma unroll 1
  for (int i = 0; i < rounds; i++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane < 16 * NT) S.xd[lane] = c_yd;
    typename F::Block blk = {};
    typename F::Quants qs;
    H::read(blk, qs, S.ws, l16, lh, hq);
    v4i x[NT][4]; float4 y[NT]; v4h sums[NT];
#pragma unroll
    for (int h = 0; h < NT; h++) {
#pragma unroll
      for (int s = 0; s < 4; s++) x[h][s] = __builtin_bit_cast(v4i, ilt_lds_ld16(S.xs + 2048 * NT * hq + 128 * (l16 + 16 * h) + 16 * ((2 * s + lh) ^ xsw)));
      y[h] = lds_f4(S.xd + 16 * h + 4 * lq);
      if constexpr (F::MINS) {                       // sums of 32: eight times 128 * (sum >> 7) (the lower half's lanes) or eight times sum & 127
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int4& b = c_bs[h][k >> 1];
          const int v = k & 1 ? b.z + b.w : b.x + b.y;
          sums[h][k] = (_Float16)(float)(v & (hq ? 127 : ~127));
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (their places are written again)
    __builtin_amdgcn_sched_barrier(0);
    issue(i + 1);
    __builtin_amdgcn_sched_barrier(0);
    v4i X[NT], Y[NT];
    const v4i zi = {};
#pragma unroll
    for (int s = 0; s < 4; s++) {
      v4i hi, lo;
      F::group(blk, qs, s, lh, hi, lo);
#pragma unroll
      for (int h = 0; h < NT; h++) {
        X[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[h][s], hi, s ? X[h] : zi, 0, 0, 0);
        Y[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[h][s], lo, s ? Y[h] : zi, 0, 0, 0);
      }
    }
    if (NT == 1 && i > 0) asm volatile("s_barrier" ::: "memory");      // (the round before's terms have been added)
    float* const ex = &W.ex[i & (NT - 1)][0][ks][0][lane];
#pragma unroll
    for (int h = 0; h < NT; h++) {
      v4f im = {};
      if constexpr (F::MINS) {
        v4h m;
#pragma unroll
        for (int k = 0; k < 4; k++) m[k] = lh ? blk.mins[4 + k] : blk.mins[k];
        im = __builtin_amdgcn_mfma_f32_16x16x16f16(sums[h], m, im, 0, 0, 0);
      }
      const float yv[4] = {y[h].x, y[h].y, y[h].z, y[h].w};
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float* const o = ex + (4 * h + r) * (HS * TERMS * 64);
        if constexpr (F::MINS) *ILT_LDS_PTR(float, o) = (yv[r] * blk.dm) * im[r];
        *ILT_LDS_PTR(float, o + (TERMS - 1) * 64) = (yv[r] * blk.d) * (float)((X[h][r] << F::SH) + Y[h][r]);
      }
    }
    ilt_barrier_lds();                               // (and the reads of the round before have come back)
    if (ks < 4 * NT) {
      const float* const o = &W.ex[i & (NT - 1)][ks][0][0][lane];
      float t[HS][TERMS];
#pragma unroll
      for (int s = 0; s < HS; s++)
#pragma unroll
        for (int k = 0; k < TERMS; k++) t[s][k] = *ILT_LDS_PTR(const float, o + (s * TERMS + k) * 64);
#pragma unroll
      for (int s = 0; s < HS; s++)
        if (i * HS + s < nsb) {
          if constexpr (F::MINS) sum = sum - t[s][0];
          sum = sum + t[s][TERMS - 1];
        }
      asm volatile("" : "+v"(sum));                  // (the reads have come back before the wave meets the next barrier)
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last round's loads, for nobody: nothing may land in LDS after the workgroup ends)
  const int tok = 16 * (ks >> 2) + 4 * lq + (ks & 3), row = r0 + l16;
  if (ks < 4 * NT && tok < ntok && row < p.rows) {
    float* const o = p.y + (tok0 + tok) * p.ldy + row;
    float v = sum;
    if (p.bias) v = v + p.bias[row];
    if (p.acc) v = *o + v;
    *o = v;
  }
}

// Rows r0 .. + 63 x tokens tok0 .. tok0 + ntok - 1 (16 NT at most): four waves of 16 rows, each through all the blocks, on the same tokens in LDS;
// a barrier a block.  For matrices of many rows on few tokens, where a tile of 32 rows is one wave's, of which there are not enough for the
// SIMDs, and its block twice the instructions: 0.55, 0.75 and 1.15 us a block for NT 1, 2 and 4 a workgroup a CU, what their 190 to 380
// instructions take at a wave a SIMD; two workgroups 1.0, 1.25 and 1.75.  (The loads a block further ahead, six or eight waves a workgroup: within 5 %.)
// us with the tiles before and now, matrices from memory: Q4_K 19456 x 2560 on 21 tokens 17.4 -> 16.6, 48 24.4 -> 22, 64 25.2 -> 23; 6144 x 2560 on 64
// 14.4 -> 11.9, 128 17.0 -> 15.6, 256 23.4 -> 21.5; 24576 x 4096 on 16 26.7 -> 21.1, 64 39.9 -> 33; Q6_K 12288 x 4096 on 16 20.5 -> 16.3, 21 20.9 -> 18.0,
// 64 30.7 -> 24.1, 128 41 -> 33.4.
template <int FMT, int NT> struct RowsSmem {
  static constexpr int XB = NT > 2 ? 2 : 3;          // buffers of a block's tokens and rows
  __align__(16) u8 xs[XB][4096 * NT];
  __align__(16) u8 ws[4][XB][HalfW<FMT>::LBYTES];
  __align__(16) u8 ms[2][RegW<FMT>::MINS ? 512 * NT : 16];       // the tokens' sums of 32 as halves (RegSmem's)
  __align__(16) float xd[2][16 * NT];
};
template <int FMT, int NT>
__device__ __forceinline__ void reg_rows(const BfParams& p, const u8* w, int r0, long tok0, int ntok, unsigned char* smem) {
  using F = RegW<FMT>;
  using H = HalfW<FMT>;
  using Smem = RowsSmem<FMT, NT>;
  constexpr int XB = Smem::XB, AHEAD = XB - 1;
  static_assert(NT <= 8, "half a token a thread");
  Smem& S = *(Smem*)smem;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nsb = p.cols / 256;
  const int l16 = lane & 15, lq = lane >> 4, lh = lq & 1, hq = lq >> 1;      // (reg_half's)
  const u32 row_bytes = (u32)(nsb * F::BLOCK);
  const __amdgpu_buffer_rsrc_t rw = ilt_rsrc(ilt_uniform_ptr(w), (u32)p.rows * row_bytes);      // (past the matrix's rows: zeros)
  const typename H::At at = H::place(row_bytes, lane);
  ntok = __builtin_amdgcn_readfirstlane(ntok);
  const __amdgpu_buffer_rsrc_t rx = ilt_rsrc(ilt_uniform_ptr((const i8*)p.x + tok0 * (long)p.cols), (u32)(ntok * p.cols));      // (past the tile's tokens: zeros)
  const u32 xpc = 16 * (u32)((lane & 7) ^ ((lane >> 4) & 3)), xrow = (u32)(lane >> 3) * (u32)p.cols;
  const __amdgpu_buffer_rsrc_t rd = ilt_rsrc(ilt_uniform_ptr(p.xd + tok0 * nsb), (u32)(ntok * nsb) * 4);
  const __amdgpu_buffer_rsrc_t rb = ilt_rsrc(ilt_uniform_ptr(p.bsums + (F::MINS ? tok0 * (p.cols >> 4) : 0)), F::MINS ? (u32)(ntok * (p.cols >> 4)) * 4 : 0);
  auto issue = [&](int sb) {
    const int b = sb % XB, at_sb = min(sb, nsb - 1);      // (past the last: the last again, for nobody)
#pragma unroll
    for (int k = 0; k < H::LOADS; k++) H::issue(k, rw, at, row_bytes, (u32)(r0 + 16 * wave), (u32)at_sb * F::BLOCK, S.ws[wave][b]);
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const int k = wave * NT + j;                   // a kilobyte: half k / 2 NT of the block, eight tokens
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (ILT_LDS void*)(S.xs[b] + k * 1024), 16, xrow + (k & 1 ? xpc ^ 64 : xpc) + (u32)(8 * (k % (2 * NT))) * (u32)p.cols + 128 * (k / (2 * NT)),
                                               at_sb * 256, 0, 0);
    }
  };
  // the tokens' scales and sums of 32, half a token a thread
  float c_yd; int4 c_bs[2];
  auto load_consts = [&](int sb) {
    if (t >= 32 * NT) return;
    const u32 ctok = (u32)((t >> 1) * nsb);
    c_yd = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, ctok * 4, min(sb, nsb - 1) * 4, 0));
    if constexpr (F::MINS) {
      const u32 o = ctok * 64 + 32 * (t & 1);
      const ilt_v4i a = __builtin_amdgcn_raw_buffer_load_b128(rb, o, min(sb, nsb - 1) * 64, 0), b = __builtin_amdgcn_raw_buffer_load_b128(rb, o + 16, min(sb, nsb - 1) * 64, 0);
      c_bs[0] = make_int4(a.x, a.y, a.z, a.w); c_bs[1] = make_int4(b.x, b.y, b.z, b.w);
    }
  };
  auto store_consts = [&](int buf) {
    if (t >= 32 * NT) return;
    if ((t & 1) == 0) S.xd[buf][t >> 1] = c_yd;
    if constexpr (F::MINS) {
      const int4 &b0 = c_bs[0], &b1 = c_bs[1];
      const int s[4] = { b0.x + b0.y, b0.z + b0.w, b1.x + b1.y, b1.z + b1.w };
      _Float16 hh[4], ll[4];
#pragma unroll
      for (int k = 0; k < 4; k++) { hh[k] = (_Float16)(float)(s[k] & ~127); ll[k] = (_Float16)(float)(s[k] & 127); }
      _Float16* const dst = (_Float16*)(S.ms[buf] + 32 * (t >> 1)) + 4 * (t & 1);
      __builtin_memcpy(dst, hh, 8);
      __builtin_memcpy(dst + 8, ll, 8);
    }
  };
  const int xsw = (l16 >> 1) & 7;
  v4f sum[NT];
#pragma unroll
  for (int h = 0; h < NT; h++) sum[h] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  if (AHEAD == 2) { issue(0); __builtin_amdgcn_sched_barrier(0); }
  load_consts(0);
  __builtin_amdgcn_sched_barrier(0);
  issue(AHEAD - 1);
#pragma unroll 1
  for (int sb = 0; sb < nsb; sb++) {
    // this block's loads and its constants' have landed; with three buffers the next block's are still on their way
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"((AHEAD - 1) * (H::LOADS + NT)) : "memory");
    store_consts(sb & 1);
    ilt_barrier_lds();
    __builtin_amdgcn_sched_barrier(0);
    const int b = sb % XB;
    typename F::Block blk = {};
    typename F::Quants qs;
    v4i x[NT][4]; float4 y[NT]; v4h sums[NT];
    H::read(blk, qs, S.ws[wave][b], l16, lh, hq);
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int h = 0; h < NT; h++) x[h][s] = __builtin_bit_cast(v4i, ilt_lds_ld16(S.xs[b] + 2048 * NT * hq + 128 * (l16 + 16 * h) + 16 * ((2 * s + lh) ^ xsw)));
#pragma unroll
    for (int h = 0; h < NT; h++) {
      if constexpr (F::MINS) __builtin_memcpy(&sums[h], S.ms[sb & 1] + 32 * (l16 + 16 * h) + 8 * lq, 8);
      y[h] = lds_f4(S.xd[sb & 1] + 16 * h + 4 * lq);
    }
    __builtin_amdgcn_sched_barrier(6);               // (the reads first; what is made of them may wait)
    load_consts(sb + 1);
    __builtin_amdgcn_sched_barrier(6);
    issue(sb + AHEAD);
    __builtin_amdgcn_sched_barrier(6);
    v4i X[NT], Y[NT];
    const v4i zi = {};
#pragma unroll
    for (int s = 0; s < 4; s++) {
      v4i hi, lo;
      F::group(blk, qs, s, lh, hi, lo);
#pragma unroll
      for (int h = 0; h < NT; h++) {
        X[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[h][s], hi, s ? X[h] : zi, 0, 0, 0);
        Y[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[h][s], lo, s ? Y[h] : zi, 0, 0, 0);
      }
    }
    v4h m = {};
    if constexpr (F::MINS) {
#pragma unroll
      for (int k = 0; k < 4; k++) m[k] = lh ? blk.mins[4 + k] : blk.mins[k];
    }
#pragma unroll
    for (int h = 0; h < NT; h++) {
      v4f im = {};
      if constexpr (F::MINS) im = __builtin_amdgcn_mfma_f32_16x16x16f16(sums[h], m, im, 0, 0, 0);
      const float yv[4] = {y[h].x, y[h].y, y[h].z, y[h].w};
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if constexpr (F::MINS) sum[h][r] = sum[h][r] - (yv[r] * blk.dm) * im[r];
        sum[h][r] = sum[h][r] + (yv[r] * blk.d) * (float)((X[h][r] << F::SH) + Y[h][r]);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last loads, for nobody: nothing may land in LDS after the workgroup ends)
#pragma unroll
  for (int h = 0; h < NT; h++) split_store(p, sum[h], tok0, ntok, r0 + 16 * wave + l16, 16 * h + 4 * lq);
}

// FSET: the matrices' format, or 0 where Q4_K and Q6_K meet in a launch
template <int FSET, int NP, int WR, int WT>
__global__ __launch_bounds__(64 * WR * WT, WR * WT == 1 ? 1 : 2) void gemm_i8r_kernel(BfParams p) {
  constexpr int TM = 32 * WR, TN = 32 * NP * WT;
  extern __shared__ __align__(16) unsigned char smem[];
  long tok0; int ntok, rt; const u8* w = p.w;
  if (!pick_tile<TM, TN>(p, tok0, ntok, rt, w)) return;
  // which of the launch's matrices the row tile belongs to
  const int n0 = (p.mrows[0] + TM - 1) / TM, n1 = n0 + (p.mrows[1] + TM - 1) / TM;
  const int m = rt < n0 ? 0 : rt < n1 ? 1 : 2;
  rt -= m == 0 ? 0 : m == 1 ? n0 : n1;
  w = m == 0 ? p.mw[0] : m == 1 ? p.mw[1] : p.mw[2];
  p.rows = m == 0 ? p.mrows[0] : m == 1 ? p.mrows[1] : p.mrows[2];
  p.y = m == 0 ? p.my[0] : m == 1 ? p.my[1] : p.my[2];
  p.bias = m == 0 ? p.mbias[0] : m == 1 ? p.mbias[1] : p.mbias[2];
  if (p.nmulti > 1) p.ldy = p.rows;
  const int fmt = m == 0 ? p.mfmt[0] : m == 1 ? p.mfmt[1] : p.mfmt[2];
  if constexpr (FSET == ILT_IQ2_XXS) { iq2_tables_load(threadIdx.x, 64 * WR * WT); __syncthreads(); }
  if constexpr (FSET != 0) reg_tile<FSET, NP, WR, WT>(p, w, rt * TM, tok0, ntok, smem);
  else if (fmt == ILT_Q4_K) reg_tile<ILT_Q4_K, NP, WR, WT>(p, w, rt * TM, tok0, ntok, smem);
  else reg_tile<ILT_Q6_K, NP, WR, WT>(p, w, rt * TM, tok0, ntok, smem);
}

// TWO: reg_split2, two workgroups a CU
template <int FSET, bool TWO>
__global__ __launch_bounds__(256, TWO ? 2 : 1) void gemm_i8s_kernel(BfParams p) {
  constexpr int TM = 32;
  extern __shared__ __align__(16) unsigned char smem[];
  long tok0; int ntok, rt; const u8* w = p.w;
  if (!pick_tile<TM, 32>(p, tok0, ntok, rt, w)) return;
  // which of the launch's matrices the row tile belongs to
  const int n0 = (p.mrows[0] + TM - 1) / TM, n1 = n0 + (p.mrows[1] + TM - 1) / TM;
  const int m = rt < n0 ? 0 : rt < n1 ? 1 : 2;
  rt -= m == 0 ? 0 : m == 1 ? n0 : n1;
  w = m == 0 ? p.mw[0] : m == 1 ? p.mw[1] : p.mw[2];
  p.rows = m == 0 ? p.mrows[0] : m == 1 ? p.mrows[1] : p.mrows[2];
  p.y = m == 0 ? p.my[0] : m == 1 ? p.my[1] : p.my[2];
  p.bias = m == 0 ? p.mbias[0] : m == 1 ? p.mbias[1] : p.mbias[2];
  if (p.nmulti > 1) p.ldy = p.rows;
  const int fmt = m == 0 ? p.mfmt[0] : m == 1 ? p.mfmt[1] : p.mfmt[2];
  if constexpr (TWO) {
    if constexpr (FSET != 0) reg_split2<FSET>(p, w, rt * TM, tok0, ntok, smem);
    else if (fmt == ILT_Q4_K) reg_split2<ILT_Q4_K>(p, w, rt * TM, tok0, ntok, smem);
    else reg_split2<ILT_Q6_K>(p, w, rt * TM, tok0, ntok, smem);
  } else {
    if constexpr (FSET != 0) reg_split<FSET>(p, w, rt * TM, tok0, ntok, smem);
    else if (fmt == ILT_Q4_K) reg_split<ILT_Q4_K>(p, w, rt * TM, tok0, ntok, smem);
    else reg_split<ILT_Q6_K>(p, w, rt * TM, tok0, ntok, smem);
  }
}

template <int FSET, int NT>
__global__ __launch_bounds__(64 * HS, NT == 1 ? 2 : 1) void gemm_i8h_kernel(BfParams p) {
  constexpr int TM = 16;
  extern __shared__ __align__(16) unsigned char smem[];
  long tok0; int ntok, rt; const u8* w = p.w;
  if (!pick_tile<TM, 16 * NT>(p, tok0, ntok, rt, w)) return;
  // which of the launch's matrices the row tile belongs to
  const int n0 = (p.mrows[0] + TM - 1) / TM, n1 = n0 + (p.mrows[1] + TM - 1) / TM;
  const int m = rt < n0 ? 0 : rt < n1 ? 1 : 2;
  rt -= m == 0 ? 0 : m == 1 ? n0 : n1;
  w = m == 0 ? p.mw[0] : m == 1 ? p.mw[1] : p.mw[2];
  p.rows = m == 0 ? p.mrows[0] : m == 1 ? p.mrows[1] : p.mrows[2];
  p.y = m == 0 ? p.my[0] : m == 1 ? p.my[1] : p.my[2];
  p.bias = m == 0 ? p.mbias[0] : m == 1 ? p.mbias[1] : p.mbias[2];
  if (p.nmulti > 1) p.ldy = p.rows;
  const int fmt = m == 0 ? p.mfmt[0] : m == 1 ? p.mfmt[1] : p.mfmt[2];
  if constexpr (FSET != 0) reg_half<FSET, NT>(p, w, rt * TM, tok0, ntok, smem);
  else if (fmt == ILT_Q4_K) reg_half<ILT_Q4_K, NT>(p, w, rt * TM, tok0, ntok, smem);
  else reg_half<ILT_Q6_K, NT>(p, w, rt * TM, tok0, ntok, smem);
}

template <int FSET, int NT>
__global__ __launch_bounds__(256, 2) void gemm_i8w_kernel(BfParams p) {
  constexpr int TM = 64;
  extern __shared__ __align__(16) unsigned char smem[];
  long tok0; int ntok, rt; const u8* w = p.w;
  if (!pick_tile<TM, 16 * NT>(p, tok0, ntok, rt, w)) return;
  // which of the launch's matrices the row tile belongs to
  const int n0 = (p.mrows[0] + TM - 1) / TM, n1 = n0 + (p.mrows[1] + TM - 1) / TM;
  const int m = rt < n0 ? 0 : rt < n1 ? 1 : 2;
  rt -= m == 0 ? 0 : m == 1 ? n0 : n1;
  w = m == 0 ? p.mw[0] : m == 1 ? p.mw[1] : p.mw[2];
  p.rows = m == 0 ? p.mrows[0] : m == 1 ? p.mrows[1] : p.mrows[2];
  p.y = m == 0 ? p.my[0] : m == 1 ? p.my[1] : p.my[2];
  p.bias = m == 0 ? p.mbias[0] : m == 1 ? p.mbias[1] : p.mbias[2];
  if (p.nmulti > 1) p.ldy = p.rows;
  const int fmt = m == 0 ? p.mfmt[0] : m == 1 ? p.mfmt[1] : p.mfmt[2];
  if constexpr (FSET != 0) reg_rows<FSET, NT>(p, w, rt * TM, tok0, ntok, smem);
  else if (fmt == ILT_Q4_K) reg_rows<ILT_Q4_K, NT>(p, w, rt * TM, tok0, ntok, smem);
  else reg_rows<ILT_Q6_K, NT>(p, w, rt * TM, tok0, ntok, smem);
}

template <int FMT, int NP, int WR, int WT> constexpr size_t reg_smem() {
  if constexpr (FMT != 0) return sizeof(RegSmemOf<FMT, NP, WR, WT>);
  else return reg_smem<ILT_Q4_K, NP, WR, WT>() > reg_smem<ILT_Q6_K, NP, WR, WT>() ? reg_smem<ILT_Q4_K, NP, WR, WT>() : reg_smem<ILT_Q6_K, NP, WR, WT>();
}

template <int FSET, int NP, int WR, int WT>
hipError_t launch_i8r(BfParams& p, hipStream_t st) {
  constexpr int TM = 32 * WR, TN = 32 * NP * WT;
  constexpr size_t smem = reg_smem<FSET, NP, WR, WT>();
  static_assert(2 * smem <= 160 * 1024, "two workgroups a CU");
  static bool attr_set[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!attr_set[dev]) {            // more dynamic LDS than the default 64 KB: asked for once per device
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_i8r_kernel<FSET, NP, WR, WT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    attr_set[dev] = true;
  }
  long long tiles = 0;
  for (int m = 0; m < p.nmulti; m++) tiles += (p.mrows[m] + TM - 1) / TM;
  p.rows = (int)(tiles * TM);
  const long long total = (long long)((p.ntok + TN - 1) / TN) * tiles, per = (total + 7) / 8;
  if (per * 8 > 0x7FFFFFFFLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_i8r_kernel<FSET, NP, WR, WT>), dim3((unsigned)(per * 8)), dim3(64 * WR * WT), smem, st, p);
  return hipGetLastError();
}

template <int FSET, bool TWO>
hipError_t launch_i8s(BfParams& p, hipStream_t st) {
  constexpr size_t s4 = TWO ? sizeof(SplitSmem2<ILT_Q4_K>) : sizeof(SplitSmem<ILT_Q4_K>), s6 = TWO ? sizeof(SplitSmem2<ILT_Q6_K>) : sizeof(SplitSmem<ILT_Q6_K>);
  constexpr size_t smem = FSET == ILT_Q4_K ? s4 : FSET == ILT_Q6_K ? s6 : s4 > s6 ? s4 : s6;
  static_assert((TWO ? 2 : 1) * smem <= 160 * 1024, "one workgroup's LDS, or two's");
  static bool attr_set[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_i8s_kernel<FSET, TWO>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    attr_set[dev] = true;
  }
  long long tiles = 0;
  for (int m = 0; m < p.nmulti; m++) tiles += (p.mrows[m] + 31) / 32;
  p.rows = (int)(tiles * 32);
  const long long total = (long long)((p.ntok + 31) / 32) * tiles, per = (total + 7) / 8;
  if (per * 8 > 0x7FFFFFFFLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_i8s_kernel<FSET, TWO>), dim3((unsigned)(per * 8)), dim3(256), smem, st, p);
  return hipGetLastError();
}
template <int FSET, int NT>
hipError_t launch_i8h(BfParams& p, hipStream_t st) {
  constexpr size_t s4 = sizeof(HalfSmem<ILT_Q4_K, NT>), s6 = sizeof(HalfSmem<ILT_Q6_K, NT>);
  constexpr size_t smem = FSET == ILT_Q4_K ? s4 : FSET == ILT_Q6_K ? s6 : s4 > s6 ? s4 : s6;
  static_assert((NT == 1 ? 2 : 1) * smem <= 160 * 1024, "two workgroups' LDS, or one's");
  static bool attr_set[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_i8h_kernel<FSET, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    attr_set[dev] = true;
  }
  long long tiles = 0;
  for (int m = 0; m < p.nmulti; m++) tiles += (p.mrows[m] + 15) / 16;
  p.rows = (int)(tiles * 16);
  const long long total = (long long)((p.ntok + 16 * NT - 1) / (16 * NT)) * tiles, per = (total + 7) / 8;
  if (per * 8 > 0x7FFFFFFFLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_i8h_kernel<FSET, NT>), dim3((unsigned)(per * 8)), dim3(64 * HS), smem, st, p);
  return hipGetLastError();
}

template <int FSET, int NT>
hipError_t launch_i8w(BfParams& p, hipStream_t st) {
  constexpr size_t s4 = sizeof(RowsSmem<ILT_Q4_K, NT>), s6 = sizeof(RowsSmem<ILT_Q6_K, NT>);
  constexpr size_t smem = FSET == ILT_Q4_K ? s4 : FSET == ILT_Q6_K ? s6 : s4 > s6 ? s4 : s6;
  static_assert(2 * smem <= 160 * 1024, "two workgroups' LDS");
  static bool attr_set[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_i8w_kernel<FSET, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    attr_set[dev] = true;
  }
  long long tiles = 0;
  for (int m = 0; m < p.nmulti; m++) tiles += (p.mrows[m] + 63) / 64;
  p.rows = (int)(tiles * 64);
  const long long total = (long long)((p.ntok + 16 * NT - 1) / (16 * NT)) * tiles, per = (total + 7) / 8;
  if (per * 8 > 0x7FFFFFFFLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_i8w_kernel<FSET, NT>), dim3((unsigned)(per * 8)), dim3(256), smem, st, p);
  return hipGetLastError();
}

// The experts' products: token tiles of every expert's rows in turn, 128 rows of the expert's matrix (of two, one behind the
// other in the output: gate and up) a workgroup.  A group of up to 32 (64) rows goes as one (two) patches of 32.
template <int FMT>
__global__ __launch_bounds__(256, 2) void gemm_i8r_group_kernel(BfParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  long tok0; int ntok, rt; const u8* w;
  const int rows = p.rows, nr = (rows + 127) / 128;
  if (p.nmulti > 1) p.rows = 2 * nr * 128;
  if (!pick_tile<128, 128>(p, tok0, ntok, rt, w)) return;
  if constexpr (FMT == ILT_IQ2_XXS) { iq2_tables_load(threadIdx.x, 256); __syncthreads(); }
  p.rows = rows;
  if (rt >= nr) { rt -= nr; w += p.up_delta; p.y = p.my[1]; }
  ntok = __builtin_amdgcn_readfirstlane(ntok);
  if constexpr (FMT == ILT_Q2_K) {
    if ((u32)(uintptr_t)ilt_uniform_ptr(w) & 3) { reg_tile<FMT, 4, 4, 1, RegWQ2KHalf>(p, w, rt * 128, tok0, ntok, smem); return; }
  }
  if (ntok <= 32) reg_tile<FMT, 1, 4, 1>(p, w, rt * 128, tok0, ntok, smem);
  else if (ntok <= 64) reg_tile<FMT, 2, 4, 1>(p, w, rt * 128, tok0, ntok, smem);
  else reg_tile<FMT, 4, 4, 1>(p, w, rt * 128, tok0, ntok, smem);
}

template <int FMT>
hipError_t launch_i8r_group(const BfParams& p, long long total_rows, hipStream_t st) {
  constexpr size_t a = reg_smem<FMT, 1, 4, 1>(), b = reg_smem<FMT, 2, 4, 1>(), c = reg_smem<FMT, 4, 4, 1>();
  constexpr size_t smem = a > b ? (a > c ? a : c) : (b > c ? b : c);
  static_assert(2 * (smem + 5120) <= 160 * 1024, "two workgroups a CU");
  static bool attr_set[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (!attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_i8r_group_kernel<FMT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    attr_set[dev] = true;
  }
  // sum over experts of ceil(count / 128) <= total / 128 + those with a row
  const long long total = (total_rows / 128 + std::min<long long>(p.ne, total_rows)) * ((p.rows + 127) / 128) * p.nmulti, per = (total + 7) / 8;
  if (per * 8 > 0x7FFFFFFFLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(gemm_i8r_group_kernel<FMT>, dim3((unsigned)(per * 8)), dim3(256), smem, st, p);
  return hipGetLastError();
}

// The tiles a launch may be cut into.  What a workgroup of each takes for a super-block, microseconds, with 1, 2, ... of them on
// a CU, as many as fit (Q4_K; Q6_K), measured on 1,024 to 19,456 rows and 17 to 1,280 tokens, the matrices from memory: a wave alone on its SIMD issues an
// instruction in 2.1 ns, two in 1.05 each, so tiles of one wave are the fastest way through the columns while there are fewer
// of them than SIMDs, and large tiles, which unpack a weight for more tokens, once there are more.  (Workgroups of two waves come
// to lie on the same two SIMDs of a CU: 1.4, then 2.35.)  The chip is taken to be empty: where another stream's launches run beside
// (the halves of a prompt) a launch takes longer than this says -- down at the Qwen3-4B shape on 256 tokens 49 us here and alone, 60-70 beside the
// other half -- and the choice is the one for a launch alone, but for the largest tiles, which do the most for an instruction: two on a CU take
// 5.45 and 5.0 alone, and with those figures here 512 tokens as halves take 11.2 ms instead of 10.7, 1,024 21.0 instead of 20.2 (2,048 50.3 instead of 50.5).
// A product alone pays for that: of 260 random ones of each format (512 to 17,408 rows, 1,024 to 9,728 columns, 96 to 4,096 tokens) the tile taken is 1.3 %
// (Q6_K 0.8) slower on average than the quickest of them, more than 5 % for 29 (20), at most 10; with 5.0 for both 0.9 (0.7), with 5.45 1.1 (1.3).
// Of such products from 8 tokens on, 32 x 32 and 32 x 64 are the choice for one in 400 (Q6_K 600), where larger tiles leave most of a round empty (Q4_K 798 x
// 2304 on 1,257 tokens 17.4 us, with four waves of 16 rows 19.9; 1685 x 8960 on 1,198 75, with 64 x 64 87), 64 x 128 for one in 600 and within 4 % of
// 64 x 64 there (Q4_K 1085 x 1792 on 3,673 28.9 and 27.7, Q6_K 1284 x 1280 on 3,020 23.7 and 24.0), reg_split2 for one in 1,200 (Q6_K 130).
struct RegTile { int rows, tokens, fit; float us[2][5]; };
constexpr RegTile kRegTiles[] = {
  {32, 32, 5, {{1.1f, 1.18f, 1.3f, 1.35f, 2.0f}, {1.4f, 1.5f, 1.65f, 1.8f, 4.0f}}},       // (Q6_K: four fit, a fifth is a second round)
  {32, 64, 4, {{1.75f, 1.95f, 2.1f, 2.55f}, {1.95f, 2.05f, 2.15f, 2.35f}}},
  {64, 64, 4, {{1.55f, 2.5f, 2.8f, 3.3f}, {2.0f, 2.7f, 2.9f, 3.3f}}},
  {64, 128, 2, {{2.0f, 3.1f}, {2.25f, 3.1f}}},
  {128, 128, 2, {{3.0f, 4.4f}, {2.85f, 4.4f}}},
  {64, 16, 2, {{0.57f, 1.04f}, {0.77f, 1.16f}}},     // reg_rows from here on
  {64, 32, 2, {{0.8f, 1.23f}, {0.86f, 1.38f}}},
  {64, 64, 2, {{1.2f, 1.88f}, {1.2f, 1.8f}}},
};
constexpr int kTileOf[] = {0, 1, 2, 3, 4, 9, 10, 11};      // their numbers in dispatch_i8r
// The same for tiles whose super-blocks are shared out, where a round is KS of them, whatever the format: a workgroup a CU (reg_split)
// 1.95 us a round, one of two (reg_split2) 2.25, two 3.25; besides, microseconds, a tile's start and end, and the launch's, which tiles
// of the other kinds have once.  Workgroups past those that fit start as the first ones end: 0.7 of what they take alone.
constexpr float kRegStart = 4.0f, kSplitStart = 2.8f, kSplitTile = 2.2f, kSplitRound = 1.95f, kSplitRound2[2] = {2.25f, 3.25f};
// And for tiles of 16 rows (reg_half), a round eight super-blocks: of 32 tokens 2.1 us, 256 tiles at a time; of 16 tokens 1.75 a workgroup a CU, 2.6 two.
constexpr float kHalfStart2 = 3.8f, kHalfStart1 = 3.2f, kHalfTile = 1.6f, kHalfRound2 = 2.1f, kHalfRound1[2] = {1.75f, 2.6f};
// Which of them, by the rounds that the chip takes the launch's workgroups in.  (Shapes, us for the tiles taken and for 64 or 128
// rows x 128 tokens: Q6_K 2560 x 9728 on 256 tokens 48 and 89, on 512 71 and 90; Q4_K 2560 x 4096 on 256 22 and 33; 19456 x 2560 on 32
// 16.8 and 31, on 192 37 and 48.)
template <int FSET>
int reg_tile_of(const BfParams& p) {
  const int f = FSET == ILT_Q4_K ? 0 : 1, nsb = p.cols / 256;
  auto workgroups = [&](int rows, int tokens) {
    long long n = 0;
    for (int m = 0; m < p.nmulti; m++) n += (p.mrows[m] + rows - 1) / rows;
    return n * ((p.ntok + tokens - 1) / tokens);
  };
  int best = 0;
  float least = 0.0f;
  for (int v = 0; v < 8; v++) {
    const RegTile& c = kRegTiles[v];
    const int fit = v == 0 && f ? 4 : c.fit;
    const long long n = workgroups(c.rows, c.tokens), round = 256LL * fit, rest = n % round;
    const float us = kRegStart + (float)nsb * ((float)(n / round) * c.us[f][fit - 1] + (rest ? c.us[f][(rest + 255) / 256 - 1] : 0.0f));
    if (v == 0 || us < least) { best = kTileOf[v]; least = us; }
  }
  const long long n = workgroups(32, 32), rest = n % 512;
  const float rounds = (float)((nsb + KS - 1) / KS);
  auto take = [&](int v, float us) { if (us < least) { best = v; least = us; } };
  if (n <= 256) take(5, kSplitStart + kSplitTile + kSplitRound * rounds);
  else {
    const float part = rest ? kSplitTile + kSplitRound2[(rest - 1) / 256] * rounds : 0.0f;
    take(6, kSplitStart + (float)(n / 512) * (kSplitTile + kSplitRound2[1] * rounds) + (n > 512 ? 0.7f : 1.0f) * part);
  }
  const float rounds8 = (float)((nsb + HS - 1) / HS);
  const long long n2 = workgroups(16, 32), n1 = workgroups(16, 16), rest1 = n1 % 512;
  take(7, kHalfStart2 + (float)((n2 + 255) / 256) * (kHalfRound2 * rounds8 + kHalfTile) - kHalfTile);
  const float part1 = rest1 == 0 ? 0.0f : rest1 <= 256 ? kHalfRound1[0] * rounds8 : kHalfTile + kHalfRound1[1] * rounds8;
  take(8, kHalfStart1 + (float)(n1 / 512) * (kHalfTile + kHalfRound1[1] * rounds8) + part1);
  return best;
}

template <int FSET>
hipError_t dispatch_i8r(BfParams& p, int forced, hipStream_t st) {
  if constexpr (FSET == ILT_Q2_K || FSET == ILT_IQ2_XXS) {
    // 128 rows x 128 tokens from 150 such tiles on; fewer leave CUs idle, and 64 x 128 fills twice as many
    const bool big = forced ? forced == 128 : (long long)((p.mrows[0] + 127) / 128) * ((p.ntok + 127) / 128) >= 150;
    return big ? launch_i8r<FSET, 4, 4, 1>(p, st) : launch_i8r<FSET, 2, 2, 2>(p, st);
  } else {
    switch (forced == 128 ? 4 : forced == 64 ? 3 : forced >= 1 && forced <= 12 ? forced - 1 : reg_tile_of<FSET>(p)) {
      case 0: return launch_i8r<FSET, 1, 1, 1>(p, st);
      case 1: return launch_i8r<FSET, 2, 1, 1>(p, st);
      case 2: return launch_i8r<FSET, 2, 2, 1>(p, st);
      case 3: return launch_i8r<FSET, 2, 2, 2>(p, st);
      case 5: return launch_i8s<FSET, false>(p, st);
      case 6: return launch_i8s<FSET, true>(p, st);
      case 7: return launch_i8h<FSET, 2>(p, st);
      case 8: return launch_i8h<FSET, 1>(p, st);
      case 9: return launch_i8w<FSET, 1>(p, st);
      case 10: return launch_i8w<FSET, 2>(p, st);
      case 11: return launch_i8w<FSET, 4>(p, st);
      default: return launch_i8r<FSET, 4, 4, 1>(p, st);
    }
  }
}

constexpr int block_bytes_of(int fmt) {
  return fmt == ILT_Q4_K ? RegW<ILT_Q4_K>::BLOCK : fmt == ILT_Q6_K ? RegW<ILT_Q6_K>::BLOCK : fmt == ILT_Q2_K ? RegW<ILT_Q2_K>::BLOCK : RegW<ILT_IQ2_XXS>::BLOCK;
}

}  // namespace

// Up to three matrices (Q4_K, Q6_K in any mix, or all Q2_K, or all IQ2_XXS) on the same tokens in one launch, their row tiles one after another.
// hipErrorNotSupported, and nothing launched, where the shapes are not this kernel's.  ILT_I8_TM (tests): 64 or 128 rows by 128 tokens
// whatever the shape, 1 to 5 the tiles in kRegTiles' order, 6 and 7 the two kernels for few tiles, 8 and 9 the tiles of 16 rows, 32 and 16
// tokens, 10 to 12 those of four waves of 16 rows.
hipError_t ilt_k_gemm_i8_reg(int nmat, const int* fmts, const uint8_t* const* ws, const int* rows, float* const* ys, const float* const* biases,
                             int cols, const int8_t* xq, const float* xd, const int* bsums, int ntok, int acc, hipStream_t st, long long ldy) {
  if (nmat < 1 || nmat > 3 || ntok < 1 || cols < 256 || cols % 256 != 0 || cols >= ILT_REG_COLS) return hipErrorNotSupported;
  BfParams p = {};
  long long tiles128 = 0;
  int fset = fmts[0];
  for (int m = 0; m < nmat; m++) {
    const bool two = fmts[m] == ILT_Q2_K || fmts[m] == ILT_IQ2_XXS;
    if (fmts[m] != ILT_Q4_K && fmts[m] != ILT_Q6_K && !two) return hipErrorNotSupported;
    if (fmts[m] != fset) { if (two || fset == ILT_Q2_K || fset == ILT_IQ2_XXS) return hipErrorNotSupported; fset = 0; }
    const long long bytes = (long long)rows[m] * (cols / 256) * block_bytes_of(fmts[m]);
    if (rows[m] < 1 || bytes >= 0x7FFFFFFFLL || (((uintptr_t)ws[m]) & (fmts[m] == ILT_IQ2_XXS ? 1 : 3)) || rows[m] >= ILT_REG_ROWS) return hipErrorNotSupported;
    p.mw[m] = ws[m]; p.mrows[m] = rows[m]; p.my[m] = ys[m]; p.mbias[m] = biases ? biases[m] : nullptr; p.mfmt[m] = fmts[m];
    tiles128 += (rows[m] + 127) / 128;
  }
  p.ldy = nmat > 1 || ldy == 0 ? rows[0] : ldy;
  if (p.ldy < rows[0] || p.ldy >= ILT_REG_ROWS || tiles128 * 128 >= (1 << 30)) return hipErrorNotSupported;
  p.nmulti = nmat; p.cols = cols; p.x = (const u16*)xq; p.xd = xd; p.bsums = bsums; p.acc = acc; p.ntok = ntok;
  const char* force = getenv("ILT_I8_TM");
  const int forced = force ? atoi(force) : 0;
  switch (fset) {
    case ILT_Q4_K: return dispatch_i8r<ILT_Q4_K>(p, forced, st);
    case ILT_Q6_K: return dispatch_i8r<ILT_Q6_K>(p, forced, st);
    case ILT_Q2_K: return dispatch_i8r<ILT_Q2_K>(p, forced, st);
    case ILT_IQ2_XXS: return dispatch_i8r<ILT_IQ2_XXS>(p, forced, st);
    default: return dispatch_i8r<0>(p, forced, st);
  }
}

// The grouped product of the experts' IQ2_XXS and Q2_K matrices: expert z's rows counts[z] from bases[z] on; y2 set: a second
// matrix at add2 as well, its results there.  Slots on two-byte boundaries.  hipErrorNotSupported, and nothing launched, where the shapes are not this kernel's.
hipError_t ilt_k_gemm_i8_reg_id(int fmt, const uint64_t* ptrs, long long add, long long add2, const uint32_t* counts, const uint32_t* bases, int ne,
                                int rows, int cols, const int8_t* xq, const float* xd, const int* bsums, long long total_rows, float* y, float* y2,
                                hipStream_t st) {
  const long long row_bytes = (long long)(cols / 256) * block_bytes_of(fmt), delta = y2 ? add2 - add : 0;
  if ((fmt != ILT_IQ2_XXS && fmt != ILT_Q2_K) || ne < 1 || ne > 256 || rows < 1 || rows >= (1 << 21) || cols < 256 || cols % 256 || rows * row_bytes >= 0x7FFFFFFFLL ||
      cols >= (1 << 22) || total_rows < 1 || total_rows >= 0x7FFFFFFFLL || delta < 0 || delta > 0x7FFFFFFFLL)
    return hipErrorNotSupported;
  BfParams p = {};
  p.ptrs = ptrs; p.add = add; p.up_delta = (unsigned)delta; p.counts = counts; p.bases = bases; p.ne = ne;
  p.rows = rows; p.cols = cols; p.row_bytes = row_bytes; p.x = (const u16*)xq; p.xd = xd; p.bsums = bsums;
  p.y = y; p.my[1] = y2; p.nmulti = y2 ? 2 : 1; p.ntok = (int)total_rows; p.ldy = rows;
  return fmt == ILT_IQ2_XXS ? launch_i8r_group<ILT_IQ2_XXS>(p, total_rows, st) : launch_i8r_group<ILT_Q2_K>(p, total_rows, st);
}
