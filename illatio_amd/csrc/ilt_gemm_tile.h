// What the pipelined prefill kernels share: their parameters, which tile a workgroup takes, and a wave's results to memory.
#ifndef ILT_GEMM_TILE_H
#define ILT_GEMM_TILE_H

#include "ilt_device.h"
#include "ilt_kernels.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int GR = 8;                  // row tiles per block of tiles sharing an L2

struct BfParams {
  const u8* w;                               // dense
  const u64* ptrs; long long add;            // grouped: expert z's matrix at ptrs[z] + add
  const u32* counts; const u32* bases; int ne;
  int rows, cols; long long row_bytes;
  const u16* x;                              // bf16 activations, cols per token (the gathered rows when grouped)
  const u32* rmap;                           // grouped: row i of the groups is x's row rmap[i] (null: row i)
  float* y; const float* bias; int acc; int ntok;
  long long ldy;                             // floats from a token's results to the next token's in y (rows, unless p covers a part of the rows)
  // several matrices of one format on the same tokens in one launch (gemm_i8r_kernel): matrix m's row tiles follow
  // matrix m-1's; rows = the tiles of all of them together times 128 until the workgroup has found its matrix
  int nmulti; const u8* mw[3]; int mrows[3]; float* my[3]; const float* mbias[3]; int mfmt[3];
  // the grouped gate and up products with the gated activation (gemm_bf16_regb_kernel<FMT, true>): rows = the width of
  // each; up's matrix at ptrs[z] + add + up_delta; mid[i][r] = bf16((silu(gate) * up) * wrow[i]), clamped as d4_swiglu_w does
  unsigned up_delta; const float* wrow; float clamp; u16* mid;
  // the exact products (gemm_i8r_kernel): x = the tokens' Q8_K quants (a byte a column), with their block scales and sums of 16
  const float* xd; const int* bsums;
  // the planes made beforehand (gemm_i8pp_kernel): w = the hi plane, wlo the lo plane (a byte a weight, rows of cols bytes), wdf = d per row and super-block
  const u8* wlo; const float* wdf;
  // the columns split over workgroups (gemm_bf16_kernel, dense): workgroups from split_from on take the tiles from
  // split_from on, ksplit of them a tile, each a run of the super-blocks, and leave their sums in part (a tile of TM x TN
  // floats each, token after token); bf16_split_sum_kernel adds a tile's parts in order and writes y.  ksplit 0: none
  int ksplit, split_from; float* part;
};

// ---- a wave's results to y ----
// Patch (a, b), register r of a lane: token wt0 + 32a + 8*(r/4) + 4*lh + r%4, row wr0 + 32b + l32
// of the tile, so a store instruction writes 32 consecutive rows of two tokens.  With one
// workgroup on a CU nothing else runs while it stores, so the loop is kept to an address add
// and a store per value and has no branches: the stores go through a buffer descriptor that
// ends with the tile's last token, which drops what lies past it, and a lane whose row the
// matrix does not have starts 2 GiB out.  (ldy * 1024 < 2^31, checked by the host.)
template <int NA, int NB, bool BIAS, bool ACC>
__device__ __forceinline__ void store_patches(const v16f (&acc)[NA][NB], const BfParams& p, __amdgpu_buffer_rsrc_t ry, int r0,
                                              int wt0, int wr0, int l32, int lh) {
  const u32 rows4 = (u32)p.ldy * 4;
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int row = r0 + wr0 + 32 * b + l32;
    const bool ok = row < p.rows;
    const u32 base = ok ? (u32)((wt0 + 4 * lh) * (int)p.ldy + row) * 4 : 0x80000000u;
    float bv = 0.0f;
    if (BIAS) bv = ok ? p.bias[row] : 0.0f;
#pragma unroll
    for (int a = 0; a < NA; a++) {
      float old[16];
      if (ACC) {
#pragma unroll
        for (int r = 0; r < 16; r++)
          old[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ry, base + (u32)(32 * a + 8 * (r >> 2) + (r & 3)) * rows4, 0, 0));
      }
#pragma unroll
      for (int r = 0; r < 16; r++) {
        float v = acc[a][b][r];
        if (BIAS) v = v + bv;
        if (ACC) v = old[r] + v;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(u32, v), ry, base + (u32)(32 * a + 8 * (r >> 2) + (r & 3)) * rows4, 0, 0);
      }
    }
  }
}

template <int NA, int NB>
__device__ __forceinline__ void store_tile(const v16f (&acc)[NA][NB], const BfParams& p, long tok0, int ntok, int r0,
                                           int wt0, int wr0, int l32, int lh) {
  // (ntok may come out of LDS: the same in every lane, said so to the compiler)
  const u32 ybytes = ((u32)(__builtin_amdgcn_readfirstlane(ntok) - 1) * (u32)p.ldy + (u32)p.rows) * 4;
  const __amdgpu_buffer_rsrc_t ry = ilt_rsrc(ilt_uniform_ptr(p.y + tok0 * p.ldy), ybytes);
  if (p.bias) {
    if (p.acc) store_patches<NA, NB, true, true>(acc, p, ry, r0, wt0, wr0, l32, lh);
    else store_patches<NA, NB, true, false>(acc, p, ry, r0, wt0, wr0, l32, lh);
  } else {
    if (p.acc) store_patches<NA, NB, false, true>(acc, p, ry, r0, wt0, wr0, l32, lh);
    else store_patches<NA, NB, false, false>(acc, p, ry, r0, wt0, wr0, l32, lh);
  }
}

// Which tile a workgroup takes: row tile rt, tokens tok0 .. tok0+ntok-1 (of expert z's group,
// with w its matrix, when grouped).  Tiles are numbered so that the eight XCDs' workgroups (the
// hardware deals them round-robin) each walk a contiguous run, GR row tiles of one token tile
// after another.  False: none (the grid is rounded up).
// (dense) tile number s of the NT x NR: its row tile and its first token
__device__ __forceinline__ void tile_place(int s, int NT, int NR, int& rt, int& tt) {
  const int rg = s / (GR * NT), rem = s - rg * GR * NT, nr = min(GR, NR - rg * GR);
  tt = rem / nr;
  rt = rg * GR + (rem - tt * nr);
}

// LIMIT >= 0: only the tiles before it are dealt out (a multiple of 8; the workgroups from it on take parts of the rest).
// Grouped: every wave adds up the groups' tiles by itself, four groups a lane (up to 256), without LDS or a barrier: the scan
// through LDS took 17 barriers, some 2 us of every workgroup's time, those with no tile (two of three) included (24 tokens, 6 of
// 256 experts, 4,096 x 2,048: Q2_K's down product 44.5 -> 31.3 us, IQ2_XXS's gate and up 87 -> 78).
template <int TM, int TN>
__device__ __forceinline__ bool pick_tile(const BfParams& p, long& tok0, int& ntok, int& rt, const u8*& w, int limit = -1) {
  const int NR = (p.rows + TM - 1) / TM, lane = threadIdx.x & 63;
  int NT;
  u32 n[4], upto = 0;                                  // grouped: the lane's four counts; the tiles of its groups and those before
  if (p.ptrs) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int z = 4 * lane + k;
      n[k] = z < p.ne ? p.counts[z] : 0;
      upto += (n[k] + TN - 1) / TN;
    }
    upto = wave_sums_upto(upto);
    NT = (int)__builtin_amdgcn_readlane(upto, 63);
  } else {
    NT = (p.ntok + TN - 1) / TN;
  }
  const int total = limit >= 0 ? limit : NT * NR, per = (total + 7) / 8;
  const int L = blockIdx.x, j = L >> 3;
  const int s = (L & 7) * per + j;
  if (j >= per || s >= total) return false;
  int tt;
  tile_place(s, NT, NR, rt, tt);
  if (p.ptrs) {
    // the lane whose groups the tile is among, then which of the four
    const int l = __builtin_ctzll(__ballot(upto > (u32)tt));
    u32 z = 4 * l, c = 0, first = l ? (u32)__builtin_amdgcn_readlane(upto, l - 1) : 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const u32 ck = (u32)__builtin_amdgcn_readlane(n[k], l), tiles = (ck + TN - 1) / TN;
      if (c == 0) {                                    // (not found yet)
        if ((u32)tt < first + tiles) { z = 4 * l + k; c = ck; }
        else first += tiles;
      }
    }
    const u32 skip = ((u32)tt - first) * TN;
    tok0 = (long)(p.bases[z] + skip);
    ntok = (int)min((u32)TN, c - skip);
    w = (const u8*)(p.ptrs[z] + p.add);
  } else {
    tok0 = (long)tt * TN;
    ntok = min(TN, p.ntok - (int)tok0);
  }
  return true;
}

}  // namespace

#endif  // ILT_GEMM_TILE_H
