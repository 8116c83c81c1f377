// A block of activations to int8, as quantize-q8! and quantize-q8k! do (tensor.lisp:245-262, kquant.lisp:130-167), four
// consecutive values a lane.
#ifndef ILT_ACT_BLOCKS_H
#define ILT_ACT_BLOCKS_H
#include "ilt_device.h"

namespace {

__device__ __forceinline__ u32 act_pack(const int (&q)[4]) { return (u32)(q[0] & 0xFF) | ((u32)(q[1] & 0xFF) << 8) | ((u32)(q[2] & 0xFF) << 16) | ((u32)(q[3] & 0xFF) << 24); }
// Q8_0: 32 values, eight lanes'; d before it is rounded to a half.
__device__ __forceinline__ float q8_block(const float (&v)[4], int (&q)[4]) {
  float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  amax = fmaxf(amax, ilt_dppf<ILT_DPP_XOR1>(amax));
  amax = fmaxf(amax, ilt_dppf<ILT_DPP_XOR2>(amax));
  amax = fmaxf(amax, ilt_dppf<ILT_DPP_HALF_MIRROR>(amax));
  const float d = amax / 127.0f;
  const float id = d == 0.0f ? 0.0f : 1.0f / d;
#pragma unroll
  for (int k = 0; k < 4; k++) q[k] = (int)rintf(v[k] * id);
  return d;
}
// Q8_K: 256, a wave's.
__device__ __forceinline__ float q8k_block(const float (&v)[4], int lane, int (&q)[4]) {
  // |v|'s bits order as |v| does; the low word prefers the earlier index
  u64 key = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const u64 kk = ((u64)__float_as_uint(fabsf(v[k])) << 32) | (u32)(255 - (4 * lane + k));
    key = kk > key ? kk : key;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const u32 hi = __shfl_xor((u32)(key >> 32), off), lo = __shfl_xor((u32)key, off);
    const u64 o = ((u64)hi << 32) | lo;
    key = o > key ? o : key;
  }
  const int idx = 255 - (int)(key & 0xFFFFFFFFu);             // the same in every lane
  const int ik = idx & 3;
  const float mine = ik == 0 ? v[0] : ik == 1 ? v[1] : ik == 2 ? v[2] : v[3];
  const float mx = __shfl(mine, idx >> 2);
  const bool any = (key >> 32) != 0;
  const float iscale = any ? -127.0f / mx : 0.0f;
#pragma unroll
  for (int k = 0; k < 4; k++) q[k] = any ? min(127, (int)rintf(iscale * v[k])) : 0;
  return any ? 1.0f / iscale : 0.0f;
}
// and they to block b's place, with the sums of each 16
__device__ __forceinline__ void q8k_store(const int (&q)[4], float d, int lane, i8* __restrict__ xq, float* __restrict__ xd, int* __restrict__ bsums, long long b) {
  ((u32*)(xq + b * 256))[lane] = act_pack(q);
  int s = (q[0] + q[1]) + (q[2] + q[3]);
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  if ((lane & 3) == 0) bsums[b * 16 + (lane >> 2)] = s;
  if (lane == 0) xd[b] = d;
}

}  // namespace

#endif  // ILT_ACT_BLOCKS_H
