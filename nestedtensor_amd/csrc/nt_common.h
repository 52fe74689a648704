// Shared helpers of the nestedtensor_amd HIP library (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <atomic>

#include "../../include/nestedtensor_amd.h"

namespace nt {

constexpr int kWave = 64;

// Error text of the calling thread, returned by nt_last_error().
char* error_buffer();

inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(error_buffer(), 512, fmt, ap);
  va_end(ap);
  return code;
}

inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    return fail(NT_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  }
  return NT_OK;
}

// Dynamic LDS beyond 48 KiB has to be allowed on every device that a kernel runs on: once per
// kernel and device (the first 64 of them; on any other every time).
template <auto KERNEL>
inline int allow_lds(int bytes, const char* what) {
  static std::atomic<uint64_t> allowed{0};
  if (bytes <= 48 * 1024) return NT_OK;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t(1) << dev : 0;
  if (e == hipSuccess && (allowed.load(std::memory_order_relaxed) & bit) == 0) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) allowed.fetch_or(bit, std::memory_order_relaxed);
  }
  if (e == hipSuccess) return NT_OK;
  (void)hipGetLastError();
  return fail(NT_ERR_HIP, "%s: cannot raise the dynamic LDS limit: %s", what, hipGetErrorString(e));
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 16-byte load from an address of any alignment (gfx950 runs with unaligned
// access mode; the compiler emits one global_load_dwordx4).
__device__ __forceinline__ u32x4 load16_unaligned(const char* p) {
  u32x4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

__device__ __forceinline__ void store16(char* p, u32x4 v) {
  *reinterpret_cast<u32x4*>(p) = v;
}

__device__ __forceinline__ void store16_stream(char* p, u32x4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}

// fp32 operands of products on the bf16 matrix instruction are taken times 2^16 and split into
// three bf16 parts, each the rounded rest of the one before.  Of any fp32 number below 2^111 the
// parts are exact: it is a multiple of 2^-149, 2^16 times it one of 2^-133, the smallest bf16
// number, so no rest falls below what a part can hold.  From 2^111 on (and of what is no
// finite number) a part is infinite or NaN, and so is every sum that it enters.
constexpr float kSplitScale = 0x1p16f;
constexpr float kSplitUnscale = 0x1p-32f;      // of a product of two

// The parts of two scaled numbers, a packed pair each.
__device__ __forceinline__ void split_bf16_pair(float x, float y, uint32_t& first, uint32_t& second, uint32_t& third) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  auto round_pair = [&] { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, bf16x2)); };
  auto take_rest = [&](uint32_t pair) {
    x -= __builtin_bit_cast(float, pair << 16);
    y -= __builtin_bit_cast(float, pair & 0xffff0000u);
  };
  first = round_pair();
  take_rest(first);
  second = round_pair();
  take_rest(second);
  third = round_pair();
}

// gelu(x) = x Phi(x), Phi the normal distribution function, from its tail: Phi(-|x|) is
// 2^Q(|x|) with Q a polynomial of degree 8 fitted to log2 Phi(-u) on [0, 5] (least
// squares reweighted towards the smallest largest error of Phi).  Q falls without end past 5, so the tail
// goes to 0 by itself.  In a projection's epilogue nothing hides these instructions: eight
// multiply-adds and one 2^x, against a reciprocal, a 2^x and fourteen others of the erf of
// Abramowitz & Stegun 7.1.26 that was here.  Against 64 bits the largest error over
// [-12, 12] is 3.8e-7 (4.7e-7 before), its root mean square 4.0e-8 (6.3e-8), and between
// -5.5 and -2, where 1 + erf cancels, 1.6e-3 of the result (0.57).
__device__ __forceinline__ float gelu_erf(float x) {
  const float u = fabsf(x);
  float q = -1.1560465309e-06f;
  q = fmaf(q, u, 1.9096820324e-05f);
  q = fmaf(q, u, -9.0532266768e-05f);
  q = fmaf(q, u, -3.6171370631e-04f);
  q = fmaf(q, u, 7.3426929303e-03f);
  q = fmaf(q, u, -5.2675705403e-02f);
  q = fmaf(q, u, -4.5915418863e-01f);
  q = fmaf(q, u, -1.1511111259f);
  q = fmaf(q, u, -9.9999988079e-01f);
  const float tail = __builtin_amdgcn_exp2f(q);
  return x * (x >= 0.0f ? 1.0f - tail : tail);
}

// b with offsets[b] <= i < offsets[b + 1] (offsets non-decreasing, offsets[B] > i)
__device__ __forceinline__ int64_t find_segment(const int64_t* offsets, int64_t B, int64_t i) {
  int64_t lo = 0, hi = B;   // answer in [lo, hi)
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) >> 1;
    if (offsets[mid] <= i) {
      lo = mid;
    } else {
      hi = mid;
    }
  }
  return lo;
}

// find_segment for an i that a whole wavefront shares: its lanes look at 64 entries at a
// time, one round trip to memory for up to 64 segments and two for up to 4096.
__device__ __forceinline__ int64_t find_segment_uniform(const int64_t* offsets, int64_t B, int64_t i) {
  const int64_t lane = threadIdx.x & (kWave - 1);
  int64_t lo = 0, n = B;      // answer in [lo, lo + n)
  for (;;) {
    const int64_t step = (n + kWave - 1) / kWave;
    const int64_t at = lane * step;
    const int64_t below = __popcll(__ballot(at < n && offsets[lo + (at < n ? at : 0)] <= i)) - 1;
    lo += below * step;
    if (step == 1) return lo;
    n = n - below * step < step ? n - below * step : step;
  }
}

// Reductions over the 64 lanes of a wavefront on the vector ALU's data-parallel
// primitives: four shifted adds within each row of 16 lanes, then the row totals
// are passed on to rows 1 and 3 and to rows 2 and 3 (row_bcast:15, row_bcast:31);
// lane 63 holds the total and is read back as a scalar, so the result is uniform.
// Seven vector instructions, against six LDS-crossbar permutes and their address
// arithmetic for the same reduction written with __shfl_xor.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_move(float old, float src) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, src),
                                                               CTRL, ROW_MASK, 0xf, false));
}
__device__ __forceinline__ float wave_reduce_sum(float v) {
  v += dpp_move<0x111, 0xf>(0.0f, v);   // row_shr:1
  v += dpp_move<0x112, 0xf>(0.0f, v);   // row_shr:2
  v += dpp_move<0x114, 0xf>(0.0f, v);   // row_shr:4
  v += dpp_move<0x118, 0xf>(0.0f, v);   // row_shr:8
  v += dpp_move<0x142, 0xa>(0.0f, v);   // row_bcast:15 into rows 1 and 3
  v += dpp_move<0x143, 0xc>(0.0f, v);   // row_bcast:31 into rows 2 and 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ int wave_reduce_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ float wave_reduce_max(float v) {
  const float lowest = -__builtin_inff();
  v = fmaxf(v, dpp_move<0x111, 0xf>(lowest, v));
  v = fmaxf(v, dpp_move<0x112, 0xf>(lowest, v));
  v = fmaxf(v, dpp_move<0x114, 0xf>(lowest, v));
  v = fmaxf(v, dpp_move<0x118, 0xf>(lowest, v));
  v = fmaxf(v, dpp_move<0x142, 0xa>(lowest, v));
  v = fmaxf(v, dpp_move<0x143, 0xc>(lowest, v));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

}  // namespace nt
