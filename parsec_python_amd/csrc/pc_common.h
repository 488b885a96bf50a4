// Shared helpers for the PARSEC hot-path HIP library (gfx950 / CDNA4).
#pragma once
#include <type_traits>
#include <utility>
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>

namespace pc {

// Thread-local text of the last failure; the C-ABI returns an int status and
// pc_last_error() hands this string to the caller.
void set_error(const std::string& msg);
const char* last_error();

enum Status : int {
  PC_OK = 0,
  PC_ERR_ARG = 1,      // invalid argument (shape, pointer, size)
  PC_ERR_HIP = 2,      // HIP runtime error
  PC_ERR_SOLVER = 3,   // dense solver failure (not SPD, no convergence)
  PC_ERR_LIMIT = 4,    // size above a documented maximum
};

constexpr int kWave = 64;

// Workgroups per launch, at most: a grid dimension holds fewer than 2^32
// work-items, and a launch of more wraps round without an error.  Entry points
// whose workgroups may be more launch in parts.
constexpr long long kMaxGrid = 1LL << 21;

}  // namespace pc

#define PC_CHECK_ARG(cond, msg)                                   \
  do {                                                            \
    if (!(cond)) {                                                \
      pc::set_error(std::string(__func__) + ": " + (msg));        \
      return pc::PC_ERR_ARG;                                      \
    }                                                             \
  } while (0)

#define PC_HIP(call)                                                                   \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess) {                                                            \
      pc::set_error(std::string(__func__) + ": " #call " -> " + hipGetErrorString(e_)); \
      return pc::PC_ERR_HIP;                                                           \
    }                                                                                  \
  } while (0)

#define PC_LAUNCH_CHECK() PC_HIP(hipGetLastError())

// Sum over the 64 lanes of a wavefront, in every lane: lane l and l ^ 32, then
// ^ 16, 8, 4, 2, 1 (the order of a shuffle-down tree, whose lane 0 has the same
// bits).  Lane swaps and row rotations instead of six LDS permutes, which a
// short kernel's reduction waits for one after the other.
__device__ __forceinline__ double pc_wave_sum(double v) {
  auto bits = [](double x) { return __builtin_bit_cast(unsigned long long, x); };
  auto make = [](unsigned lo, unsigned hi) {
    return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
  };
  {
    const unsigned lo = (unsigned)bits(v), hi = (unsigned)(bits(v) >> 32);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    v = make(l[0], h[0]) + make(l[1], h[1]);
  }
  {
    const unsigned lo = (unsigned)bits(v), hi = (unsigned)(bits(v) >> 32);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    v = make(l[0], h[0]) + make(l[1], h[1]);
  }
#define PC_ROW_ROR(N)                                                                                       \
  v += make((unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)bits(v), 0x120 + N, 0xf, 0xf, true),          \
            (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(bits(v) >> 32), 0x120 + N, 0xf, 0xf, true));
  PC_ROW_ROR(8) PC_ROW_ROR(4) PC_ROW_ROR(2) PC_ROW_ROR(1)
#undef PC_ROW_ROR
  return v;
}

// f(integral_constant I) for I = 0, 1, ...
template <int... I, class F>
__device__ __forceinline__ void pc_unroll_seq(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// Block-wide FP64 sum of one value per thread (blockDim.x multiple of 64,
// <= 1024).  Result valid in thread 0.
__device__ inline double pc_block_sum(double v, double* sh) {
  v = pc_wave_sum(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
    const int nw = (blockDim.x + 63) >> 6;
    for (int w = 0; w < nw; ++w) r += sh[w];
  }
  return r;
}

// Sum of part[0 .. nb), nb <= 8 NT, in every thread: thread t < NT adds
// part[t], part[t + NT], ... in order, then the wavefronts' sums are added in
// order.  All loads are in flight together.  sh: blockDim.x / 64 doubles, not
// used since the last barrier by anything else.
template <int NT>
__device__ __forceinline__ double pc_parts_load(const double* part, int nb) {
  double v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    v[k] = 0.0;
    if (NT * k < nb) {   // the same in every thread
      const int b = (int)threadIdx.x + NT * k;
      const double t = part[b < nb ? b : 0];
      v[k] = b < nb && threadIdx.x < NT ? t : 0.0;
    }
  }
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 8; ++k) s += v[k];
  return s;
}
__device__ __forceinline__ void pc_parts_post(double s, double* sh) {
  s = pc_wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
}
template <int NT>   // after a barrier
__device__ __forceinline__ double pc_parts_get(const double* sh) {
  double r = 0.0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) r += sh[w];
  return r;
}
