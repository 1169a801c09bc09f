// RMSNorm of one token row with the residual add, shared by the standalone norm launch
// (small_ops.hip) and the W8A16 split-K epilogue that feeds it (w8a16.hip), so that both compute
// the same values with the same instructions (ops/triton_rmsnorm.py:10-46, twin
// ops/reference.py:13-22): the residual add is an fp32 add rounded to fp16; RMS is taken in fp32
// over the rounded sum and the normalised row is rounded to fp16 before the weight multiply.
#pragma once

#include "common.h"

namespace ts {

constexpr int kRowThreads = 256;
constexpr int kRowVec = 8;                 // halves per 16-byte access
constexpr int kRmsMaxIter = 4;             // N <= 4 * 256 * 8 = 8192

template <int C>                           // an integer as a type, for the arguments of generic lambdas
struct IntC { static constexpr int value = C; };

// Sum over a wavefront, the same in every lane: the butterfly of lane xors 32, 16, 8, 4, 2, 1 on the
// VALU (row and half-wave swaps, then DPP; a rotation by 4 of rows already equal 8 apart is the xor).
__device__ __forceinline__ float wave_sum(float v) {
  auto dpp = [](float x, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf,
                                                      0xf, true));
  };
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  v += dpp(v, IntC<0x128>{});                 // row_ror:8
  v += dpp(v, IntC<0x124>{});                 // row_ror:4
  v += dpp(v, IntC<0x4e>{});                  // quad_perm [2, 3, 0, 1]
  return v + dpp(v, IntC<0xb1>{});            // quad_perm [1, 0, 3, 2]
}

__device__ __forceinline__ float block_sum_256(float v, float* s_red) {
  v = wave_sum(v);
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (lane == 0) s_red[w] = v;
  __syncthreads();
  return (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
}

// One row of N features by a workgroup of kRowThreads threads. load_x(i) returns features
// i .. i+7 of the row's input; with kRes, res is added and the sum written to res_out.
//
// A row is a chain of load latencies (one workgroup per row, a few KB), so the residual and the
// weight are requested together with the input, not after the reduction of a split product and
// after the sum of squares (a row of the M = 1 projections with the norm behind it: 1536 x 8960 8.0 ->
// 7.9 us, 3584 x 18944 20.0 -> 19.7 us; 2048 rows of 8192 alone 25.7 -> 24.4 us).
template <bool kRes, class LoadX>
__device__ __forceinline__ void rmsnorm_row(LoadX load_x, const half_t* __restrict__ res,
                                            const half_t* __restrict__ w, half_t* __restrict__ out,
                                            half_t* __restrict__ res_out, int N, float eps) {
  __shared__ float s_red[kRowThreads / kWave];
  const int tid = threadIdx.x;
  half8_t v[kRmsMaxIter], wv[kRmsMaxIter], rv[kRmsMaxIter];
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < kRmsMaxIter; ++it) {
    const int i = (it * kRowThreads + tid) * kRowVec;
    if (i < N) {
      if constexpr (kRes) rv[it] = ld<half8_t>(res + i);
      wv[it] = ld<half8_t>(w + i);
    }
  }
#pragma unroll
  for (int it = 0; it < kRmsMaxIter; ++it) {
    const int i = (it * kRowThreads + tid) * kRowVec;
    if (i < N) {
      half8_t a = load_x(i);
      if constexpr (kRes) {
#pragma unroll
        for (int e = 0; e < kRowVec; ++e) a[e] = (half_t)((float)a[e] + (float)rv[it][e]);
        st<half8_t>(res_out + i, a);
      }
      v[it] = a;
#pragma unroll
      for (int e = 0; e < kRowVec; ++e) ss += (float)a[e] * (float)a[e];
    }
  }
  const float inv = rsqrtf(block_sum_256(ss, s_red) / (float)N + eps);
#pragma unroll
  for (int it = 0; it < kRmsMaxIter; ++it) {
    const int i = (it * kRowThreads + tid) * kRowVec;
    if (i < N) {
      half8_t o;
#pragma unroll
      for (int e = 0; e < kRowVec; ++e) {
        const half_t y = (half_t)((float)v[it][e] * inv);          // cast before the weight
        o[e] = (half_t)((float)wv[it][e] * (float)y);
      }
      st<half8_t>(out + i, o);
    }
  }
}

// One workgroup per token row of N = hidden features.
template <bool kRes>
__global__ void __launch_bounds__(kRowThreads) rmsnorm_kernel(
    const half_t* __restrict__ x, int64_t x_st, const half_t* __restrict__ res, int64_t res_st,
    const half_t* __restrict__ w, half_t* __restrict__ out, int64_t out_st,
    half_t* __restrict__ res_out, int64_t res_out_st, int N, float eps) {
  const int64_t t = blockIdx.x;
  const half_t* xr = x + t * x_st;
  rmsnorm_row<kRes>([&](int i) { return ld<half8_t>(xr + i); }, kRes ? res + t * res_st : nullptr,
                    w, out + t * out_st, kRes ? res_out + t * res_out_st : nullptr, N, eps);
}

}  // namespace ts
