// The arithmetic of QK-norm and RoPE on 16-bit rows, for the kernels that do it behind a load (producer.hip) or behind the projection
// that makes the rows (qkv.hip).  Both give the same bits: order and contraction of every sum are written out here.
#pragma once

#include "dt_common.h"

namespace dt {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// kHalf: the 16-bit type is IEEE half, else bfloat16
template <bool kHalf>
__device__ __forceinline__ float round16(float v) {
  if constexpr (kHalf) return (float)(_Float16)v;
  else return (float)(__bf16)v;
}

template <bool kHalf>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  f32x2 f;
  f.x = lo;
  f.y = hi;
  // round to nearest even
  if constexpr (kHalf) return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

template <bool kHalf>
__device__ __forceinline__ void unpack8(const u32x4 r, float (&v)[8]) {
  const uint32_t u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (kHalf) {
      const f32x2 f = __builtin_convertvector(__builtin_bit_cast(f16x2, u[i]), f32x2);
      v[2 * i] = f.x;
      v[2 * i + 1] = f.y;
    } else {
      v[2 * i] = __builtin_bit_cast(float, u[i] << 16);
      v[2 * i + 1] = __builtin_bit_cast(float, u[i] & 0xffff0000u);
    }
  }
}

// DPP: lane i of every row of 16 reads another lane of that row inside the vector instruction itself, where __shfl is an LDS
// access.  Only whole groups of 8 or 16 neighbouring lanes leave the kernel early, so the lanes read are active.
constexpr int kDppXor1 = 0xb1, kDppXor2 = 0x4e;                 // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kDppHalfMirror = 0x141, kDppMirror = 0x140;       // i -> 7 - i within 8 lanes, i -> 15 - i within 16
template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kCtrl, 0xf, 0xf, true));
}

// Sum over the lane group, the same in all of its lanes: neighbours, pairs, quads (all lanes of a quad agree by then, so the
// mirrored lane is as good as lane ^ 4) and halves, the order and the bits of a butterfly with __shfl_xor.
template <int G>
__device__ __forceinline__ float group_sum(float v) {
  static_assert(G == 8 || G == 16, "a lane group is 8 or 16 lanes");
  v += dpp<kDppXor1>(v);
  v += dpp<kDppXor2>(v);
  v += dpp<kDppHalfMirror>(v);
  if constexpr (G == 16) v += dpp<kDppMirror>(v);
  return v;
}

// Sums over a row of 8 G values, a lane's eight one after the other, and of their squares.
template <int G>
__device__ __forceinline__ float row_sum(const float (&v)[8]) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) t += v[i];
  return group_sum<G>(t);
}
template <int G>
__device__ __forceinline__ float row_squares(const float (&v)[8]) {
  float t = __builtin_fmaf(v[0], v[0], v[1] * v[1]);
#pragma unroll
  for (int i = 2; i < 8; ++i) t = __builtin_fmaf(v[i], v[i], t);
  return group_sum<G>(t);
}
__device__ __forceinline__ float layer_norm(float v, float mean, float rs, float w, float b) { return __builtin_fmaf((v - mean) * rs, w, b); }
// ... rounded to the row's type.  (Half: the multiply-add and its rounding are one instruction, v_fma_mixlo_f16, and one rounding.)
template <bool kHalf>
__device__ __forceinline__ float layer_norm16(float v, float mean, float rs, float w, float b) { return round16<kHalf>(layer_norm(v, mean, rs, w, b)); }
__device__ __forceinline__ float rotated(float v, float rot, float cos, float sin) { return __builtin_fmaf(rot, sin, v * cos); }

// 1 / sqrt(ss / D + eps) of four rows.  The square root and the division are some 25 instructions at full precision, and all
// lanes of a group would do the same ones: lane i of a quad takes row i and the quad exchanges the results.
// With the LDS butterfly and a root per row the kernel took as long for its arithmetic as for its bytes; us per launch before, with
// the sums by DPP, and with the shared roots too: 14882 tokens x 24 heads of 128 35.2 / 34.5 / 34.1, 119056 x 24 256 / 245 / 240
// (6.6 TB/s), 9000 x 20 20.3 / 19.6 / 19.3, 12444 x 48 of 64 with LayerNorm 30.0 / 28.9 / 28.7; 14882 x 24 without a norm 32.8.
// Short launches, replayed from a graph, before and with both: 512 x 4 of 64 5.7 / 4.8, 2250 x 48 of 64 with LayerNorm 8.8 / 8.0, 8000 x
// 3 of 128 5.7 / 5.5, 5000 x 10 9.1 / 8.1 (called one by one from Python the host is the limit there, 13 to 16 us).
// (The sums come as values: from an array the compiler makes the choice one of addresses and the array a piece of LDS, which
// costs every launch 8 us.)
template <int D>
__device__ __forceinline__ void inverse_rms4(float s0, float s1, float s2, float s3, float eps, float (&rs)[4]) {
  const int i = threadIdx.x & 3;
  const float lo = i & 1 ? s1 : s0, hi = i & 1 ? s3 : s2;
  const float mine = 1.0f / sqrtf((i & 2 ? hi : lo) * (1.0f / D) + eps);
  rs[0] = dpp<0x00>(mine);   // quad_perm [0,0,0,0] ... [3,3,3,3]
  rs[1] = dpp<0x55>(mine);
  rs[2] = dpp<0xaa>(mine);
  rs[3] = dpp<0xff>(mine);
}

}  // namespace
}  // namespace dt
