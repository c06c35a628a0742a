// What the decode kernels (attention.hip) and the prefill kernels
// (attention_prefill.hip) of the attention share.
#pragma once
#include "common.h"

namespace htn {

constexpr int D = HTN_HEAD_DIM;
constexpr int kSplit = 64;  // cache slots per tile

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Max / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (the four quads'
// copies of one query row): gfx950's row-swap permutes, no LDS round trip.
// permlane16_swap pairs row r with row r ^ 1 and permlane32_swap the wave's
// halves; both results of each swap hold the two partners.
__device__ __forceinline__ float quad_max(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float quad_sum(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Causal attention over many queries per sequence, without a split.
struct PrefillArgs {
  const bf16_t* q; long q_sb, q_sh, q_st;
  const bf16_t* keys; const bf16_t* values; long cap;
  const int64_t* pos;
  bf16_t* out;  // row (b, h, t) at b*o_sb + h*o_sh + t*o_st (dims contiguous)
  long o_sb, o_sh, o_st;
  int B, Hq, Hkv, G, Q;
  int turn;     // attention_prefill_long: the query rank from which ranks run in reverse
  float scale;
};

// Needs 16-byte query fragments and 8-byte output stores; one launch, no scratch.
int prefill_attention(PrefillArgs& a, hipStream_t st);

}  // namespace htn
