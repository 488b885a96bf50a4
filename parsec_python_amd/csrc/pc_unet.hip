// Learned density initialiser: the kernels of a small 3D U-Net (forward,
// backward, Adam), BF16 storage with FP32 accumulation on the bf16 MFMA.
//
// Layout: one volume, channel-last: element (voxel v, channel c) at v*ld + c,
// v = (z*H + y)*W + x.  A channel stride ld larger than the channel count lets
// a layer read or write a slice of a concatenated tensor in place.
// Weights: W[co][t][ci] (tap t = (dz+1)*9 + (dy+1)*3 + (dx+1), ci fastest),
// 3x3x3 taps, zero padding 1.
//
// conv3d (implicit GEMM, M = output channels, N = voxels, K = 27 * C_in): a
// workgroup owns a box of voxels, stages it with its halo in LDS and issues
// v_mfma_f32_16x16x16_bf16 tap by tap.  The input gradient is the same kernel on the tap-flipped, channel-transposed
// weights; the weight gradient is a GEMM over voxels, one wavefront per dz.
#include "pc_common.h"
#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// round to nearest even (finite inputs)
__device__ __forceinline__ unsigned short f2bf(float f) {
  const unsigned u = __float_as_uint(f);
  return (unsigned short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

struct Vol {
  int D, H, W;
  long long V;
};

__device__ __forceinline__ void tap_offsets(int t, int& dz, int& dy, int& dx) {
  dz = t / 9 - 1;
  dy = (t / 3) % 3 - 1;
  dx = t % 3 - 1;
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

// Boxes of a TX x TY x TZ tiling and the box of this workgroup (consecutive
// boxes on one XCD, whose L2 then serves the halos).
struct Boxes {
  int nx, ny, nz;     // boxes per axis
  int nblocks, nb8;   // boxes x channel blocks
};

// One result of lane (n, lk): channels co0 .. co0 + 3 of a voxel.
// mode: 0 = FP32 output with bias, 1 = leaky ReLU -> BF16 output (with bias),
//       2 = FP32 output, no bias
__device__ __forceinline__ void conv_store(f32x4 acc, long long v, int co0, int cout, const float* __restrict__ bias,
                                           int mode, float slope, void* Y, int ldy, bool vec) {
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    o[r] = acc[r];
    if (mode != 2) o[r] += bias[min(co0 + r, cout - 1)];
    if (mode == 1) o[r] = o[r] > 0.f ? o[r] : slope * o[r];
  }
  if (mode == 1) {
    unsigned short* y = static_cast<unsigned short*>(Y) + v * ldy + co0;
    if (vec && co0 + 3 < cout) {
      const u32x2 t = {f2bf(o[0]) | (unsigned)f2bf(o[1]) << 16, f2bf(o[2]) | (unsigned)f2bf(o[3]) << 16};
      *reinterpret_cast<u32x2*>(y) = t;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (co0 + r < cout) y[r] = f2bf(o[r]);
    }
  } else {
    float* y = static_cast<float*>(Y) + v * ldy + co0;
    if (vec && co0 + 3 < cout) {
      *reinterpret_cast<f32x4*>(y) = f32x4{o[0], o[1], o[2], o[3]};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (co0 + r < cout) y[r] = o[r];
    }
  }
}

constexpr int kNT = 2;   // 16-voxel tiles per wavefront
constexpr int kWaves = 4;

// Any number of input channels (a multiple of 16, or 1): each wavefront owns 16*MT
// output channels x 32 voxels in flat order, its operands gathered straight from
// the channel-last tensors.
template <int MT, bool CIN1>
__global__ __launch_bounds__(256) void conv_fwd(Vol vol, const unsigned short* __restrict__ X, int ldx, int cin,
                                                const unsigned short* __restrict__ Wt, const float* __restrict__ bias,
                                                int cout, int mode, float slope, void* Y, int ldy) {
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int co_base = blockIdx.y * 64;
  const long long vbase = ((long long)blockIdx.x * kWaves + wv) * (16 * kNT);
  const int ln = lane & 15, lk = lane >> 4;

  // the voxels of this lane's B columns
  int vz[kNT], vy[kNT], vx[kNT];
  bool vin[kNT];
#pragma unroll
  for (int n = 0; n < kNT; ++n) {
    const long long v = vbase + 16 * n + ln;
    vin[n] = v < vol.V;
    const long long vv = vin[n] ? v : 0;
    vx[n] = (int)(vv % vol.W);
    vy[n] = (int)((vv / vol.W) % vol.H);
    vz[n] = (int)(vv / ((long long)vol.W * vol.H));
  }
  f32x4 acc[MT][kNT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < kNT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  if constexpr (!CIN1) {
    const int ncb = cin >> 4;
    for (int t = 0; t < 27; ++t) {
      int dz, dy, dx;
      tap_offsets(t, dz, dy, dx);
      long long src[kNT];
      bool ok[kNT];
#pragma unroll
      for (int n = 0; n < kNT; ++n) {
        const int z = vz[n] + dz, y = vy[n] + dy, x = vx[n] + dx;
        ok[n] = vin[n] && z >= 0 && z < vol.D && y >= 0 && y < vol.H && x >= 0 && x < vol.W;
        src[n] = ok[n] ? ((long long)(z * vol.H + y) * vol.W + x) * ldx : 0;
      }
      for (int cb = 0; cb < ncb; ++cb) {
        const int ci = cb * 16 + 4 * lk;
        bf16x4 b[kNT];
#pragma unroll
        for (int n = 0; n < kNT; ++n) {
          b[n] = ok[n] ? *reinterpret_cast<const bf16x4*>(X + src[n] + ci) : bf16x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int co = co_base + 16 * m + ln;
          const bf16x4 a = co < cout ? *reinterpret_cast<const bf16x4*>(Wt + ((long long)co * 27 + t) * cin + ci)
                                     : bf16x4{0, 0, 0, 0};
#pragma unroll
          for (int n = 0; n < kNT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[n], acc[m][n], 0, 0, 0);
        }
      }
    }
  } else {
    // one input channel: K = the 27 taps (two k-steps of 16, taps 27..31 zero)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x4 b[kNT];
      short av[MT][4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = ks * 16 + 4 * lk + j;
        int dz = 0, dy = 0, dx = 0;
        if (t < 27) tap_offsets(t, dz, dy, dx);
#pragma unroll
        for (int n = 0; n < kNT; ++n) {
          const int z = vz[n] + dz, y = vy[n] + dy, x = vx[n] + dx;
          const bool ok = t < 27 && vin[n] && z >= 0 && z < vol.D && y >= 0 && y < vol.H && x >= 0 && x < vol.W;
          b[n][j] = ok ? (short)X[((long long)(z * vol.H + y) * vol.W + x) * ldx] : (short)0;
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int co = co_base + 16 * m + ln;
          av[m][j] = (t < 27 && co < cout) ? (short)Wt[(long long)co * 27 + t] : (short)0;
        }
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const bf16x4 a = {av[m][0], av[m][1], av[m][2], av[m][3]};
#pragma unroll
        for (int n = 0; n < kNT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[n], acc[m][n], 0, 0, 0);
      }
    }
  }

  // epilogue: lane holds D[co = 16m + 4*lk + r][voxel = 16n + ln]
#pragma unroll
  for (int n = 0; n < kNT; ++n) {
    if (!vin[n]) continue;
    const long long v = vbase + 16 * n + ln;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int co0 = co_base + 16 * m + 4 * lk;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int co = co0 + r;
        if (co >= cout) continue;
        float o = acc[m][n][r];
        if (mode != 2) o += bias[co];
        if (mode == 1) {
          o = o > 0.f ? o : slope * o;
          static_cast<unsigned short*>(Y)[v * ldy + co] = f2bf(o);
        } else {
          static_cast<float*>(Y)[v * ldy + co] = o;
        }
      }
    }
  }
}

// Workgroup: 4 wavefronts, a box of TX x TY x TZ voxels (NT tiles of 16 per
// wavefront, in the box's flat order) x 16 output channels.  The box with its
// halo goes to LDS once, all 16 NCB channels of a voxel together, 8 loads per
// thread in flight; the products then run tap by tap and, inside a tap, 16
// channels by 16 channels (the order of conv_fwd, so the same bits), each tile's
// operand one 8-byte LDS read per lane, the next tap's weights loaded meanwhile.
// Bound by the LDS reads (2 bytes per voxel, tap and channel) and the staging;
// 64^3 volume: 48 -> 16 channels 39 us, 16 -> 48 31 us (115
// and 91 us with every operand gathered from global memory per tap).
template <int NCB, int TX, int TY, int TZ>
__global__ __launch_bounds__(256, NCB == 1 ? 4 : 2) void conv_tile(Vol vol, Boxes bx,
                                                                   const unsigned short* __restrict__ X, int ldx,
                                                                   const unsigned short* __restrict__ Wt,
                                                                   const float* __restrict__ bias, int cout, int mode,
                                                                   float slope, void* Y, int ldy, bool yvec) {
  constexpr int CIN = 16 * NCB;
  constexpr int VS = CIN + 8;   // LDS voxel stride: an odd number of 16-byte pieces, so 16 voxels meet different banks
  constexpr int NT = TX * TY * TZ / 64;
  constexpr int HX = TX + 2, HY = TY + 2, HZ = TZ + 2, HV = HX * HY * HZ;
  __shared__ __align__(16) unsigned short xs[HV * VS];
  const int L = (blockIdx.x & 7) * bx.nb8 + (blockIdx.x >> 3);
  if (L >= bx.nblocks) return;
  const int nbox = bx.nx * bx.ny * bx.nz;
  const int cb = L / nbox, box = L - cb * nbox;
  const int x0 = box % bx.nx * TX, y0 = box / bx.nx % bx.ny * TY, z0 = box / (bx.nx * bx.ny) * TZ;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ln = lane & 15, lk = lane >> 4;
  // the box and its halo, zero outside the volume, 8 channels per step
  constexpr int PV = 2 * NCB, UNITS = HV * PV, U = 8;
  for (int e0 = threadIdx.x; e0 < UNITS; e0 += 256 * U) {
    u32x4 t[U];
    unsigned inside = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + 256 * u, q = e / PV, h = e % PV * 8;
      const int x = x0 + q % HX - 1, y = y0 + q / HX % HY - 1, z = z0 + q / (HX * HY) - 1;
      const bool in = e < UNITS && x >= 0 && x < vol.W && y >= 0 && y < vol.H && z >= 0 && z < vol.D;
      inside |= (unsigned)in << u;
      t[u] = *reinterpret_cast<const u32x4*>(X + (in ? ((long long)(z * vol.H + y) * vol.W + x) * ldx + h : 0));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + 256 * u;
      if (e < UNITS) *reinterpret_cast<u32x4*>(&xs[e / PV * VS + e % PV * 8]) = inside >> u & 1 ? t[u] : u32x4{0, 0, 0, 0};
    }
  }
  int base[NT];          // LDS position of this lane's voxel of each tile (its tap (0, 0, 0))
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int q = (wv * NT + n) * 16 + ln;
    base[n] = ((q / (TX * TY) * HY + q / TX % TY) * HX + q % TX) * VS + 4 * lk;
  }
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool win = cb * 16 + ln < cout;
  const unsigned short* wp = Wt + (long long)min(cb * 16 + ln, cout - 1) * 27 * CIN + 4 * lk;
  // the three taps of a row at a time; the next row's weights are in flight meanwhile
  bf16x4 a[3][NCB], an[3][NCB];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int c = 0; c < NCB; ++c) a[k][c] = *reinterpret_cast<const bf16x4*>(wp + k * CIN + 16 * c);
  __syncthreads();
  for (int r = 0; r < 9; ++r) {
    const int rn = min(r + 1, 8);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < NCB; ++c) an[k][c] = *reinterpret_cast<const bf16x4*>(wp + (3 * rn + k) * CIN + 16 * c);
    __builtin_amdgcn_sched_barrier(0);   // or the loads are sunk to their uses
    const int off = (r / 3 * HY + r % 3) * HX * VS;
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < NCB; ++c) {
        const bf16x4 av = win ? a[k][c] : bf16x4{0, 0, 0, 0};
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const bf16x4 b = *reinterpret_cast<const bf16x4*>(&xs[base[n] + off + k * VS + 16 * c]);
          acc[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b, acc[n], 0, 0, 0);
        }
      }
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int c = 0; c < NCB; ++c) a[k][c] = an[k][c];
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int q = (wv * NT + n) * 16 + ln;
    const int x = x0 + q % TX, y = y0 + q / TX % TY, z = z0 + q / (TX * TY);
    if (x < vol.W && y < vol.H && z < vol.D && cb * 16 + 4 * lk < cout)
      conv_store(acc[n], (long long)(z * vol.H + y) * vol.W + x, cb * 16 + 4 * lk, cout, bias, mode, slope, Y, ldy,
                 yvec);
  }
}

// One input channel: K = the 27 taps in two products of 16 (lane group lk holds
// taps 16 ks + 4 lk .. + 3, those past 26 zero), the box with its halo in LDS.
template <int TX, int TY, int TZ>
__global__ __launch_bounds__(256) void conv_tile1(Vol vol, Boxes bx, const unsigned short* __restrict__ X, int ldx,
                                                  const unsigned short* __restrict__ Wt,
                                                  const float* __restrict__ bias, int cout, int mode, float slope,
                                                  void* Y, int ldy, bool yvec) {
  constexpr int NT = TX * TY * TZ / 64;
  constexpr int HX = TX + 2, HY = TY + 2, HZ = TZ + 2, HV = HX * HY * HZ;
  __shared__ unsigned short xs[HV];
  const int L = (blockIdx.x & 7) * bx.nb8 + (blockIdx.x >> 3);
  if (L >= bx.nblocks) return;
  const int nbox = bx.nx * bx.ny * bx.nz;
  const int cb = L / nbox, box = L - cb * nbox;
  const int x0 = box % bx.nx * TX, y0 = box / bx.nx % bx.ny * TY, z0 = box / (bx.nx * bx.ny) * TZ;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ln = lane & 15, lk = lane >> 4;
  for (int q = threadIdx.x; q < HV; q += 256) {
    const int x = x0 + q % HX - 1, y = y0 + q / HX % HY - 1, z = z0 + q / (HX * HY) - 1;
    const bool in = x >= 0 && x < vol.W && y >= 0 && y < vol.H && z >= 0 && z < vol.D;
    xs[q] = in ? X[((long long)(z * vol.H + y) * vol.W + x) * ldx] : (unsigned short)0;
  }
  const int co = cb * 16 + ln;
  int off[8];
  unsigned av[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int t = 16 * (e >> 2) + 4 * lk + (e & 3), tt = t < 27 ? t : 0;
    off[e] = (tt / 9 * HY + tt / 3 % 3) * HX + tt % 3;
    av[e] = (t < 27 && co < cout) ? Wt[(long long)co * 27 + t] : 0;
  }
  // of the second product's taps 16 + 4 lk .. + 3, those below 27
  const unsigned tm[2] = {lk < 3 ? ~0u : 0u, lk < 2 ? ~0u : (lk == 2 ? 0xffffu : 0u)};
  const u32x2 a0 = {av[0] | av[1] << 16, av[2] | av[3] << 16}, a1 = {av[4] | av[5] << 16, av[6] | av[7] << 16};
  __syncthreads();
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int q = (wv * NT + n) * 16 + ln;
    const int p = (q / (TX * TY) * HY + q / TX % TY) * HX + q % TX;
    u32x4 b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = xs[p + off[2 * e]] | (unsigned)xs[p + off[2 * e + 1]] << 16;
    b[2] &= tm[0];   // (a tap past 26 repeats tap 0, and 0 times an infinite value would be a NaN)
    b[3] &= tm[1];
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4, a0),
                                                    __builtin_bit_cast(bf16x4, u32x2{b[0], b[1]}), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4, a1),
                                                    __builtin_bit_cast(bf16x4, u32x2{b[2], b[3]}), acc, 0, 0, 0);
    const int x = x0 + q % TX, y = y0 + q / TX % TY, z = z0 + q / (TX * TY);
    if (x < vol.W && y < vol.H && z < vol.D && cb * 16 + 4 * lk < cout)
      conv_store(acc, (long long)(z * vol.H + y) * vol.W + x, cb * 16 + 4 * lk, cout, bias, mode, slope, Y, ldy, yvec);
  }
}

// Wt[ci][t][co] = W[co][26 - t][ci]: the weights of the input-gradient conv
__global__ void conv_wflip(const unsigned short* __restrict__ W, int cout, int cin, unsigned short* __restrict__ Wt) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long n = (long long)cout * cin * 27;
  if (i >= n) return;
  const int ci = (int)(i % cin);
  const int t = (int)((i / cin) % 27);
  const int co = (int)(i / ((long long)cin * 27));
  Wt[((long long)ci * 27 + (26 - t)) * cout + co] = W[i];
}

// Weight gradient: workgroup (16 output channels, 16 input channels, voxel split
// s); it stages boxes of TX x TY x TZ voxels of dZ and, with the halo, of X into
// LDS transposed (channel by channel, x fastest), so that a lane's 8 voxels of
// one channel are two 8-byte reads.  Wavefronts (dz, k): the 9 taps of one dz on
// every second group of 32 voxels; the x-shifted operands of a row's three taps
// share their reads (funnel shifts).  dW_part[s][co][t][ci].  Bound by LDS reads
// and the transposing staging; 64^3 volume, 48 x 16 channels: 47 us (611 us
// with 2-byte gathers from global memory per tap).
// RAGGED: boxes may reach beyond the volume.
template <int TX, int TY, int TZ, bool ZVEC, bool XVEC, bool RAGGED>   // VEC: 16-byte aligned channels, a multiple of 16
__global__ __launch_bounds__(384) void conv_wgrad(Vol vol, Boxes bx, const unsigned short* __restrict__ dZ, int ldz,
                                                  int cout, const unsigned short* __restrict__ X, int ldx, int cin,
                                                  int nsplit, float* __restrict__ part) {
  constexpr int HY = TY + 2, HZ = TZ + 2;
  constexpr int RS = TX + 8;                      // row stride: x = -4 .. TX + 3
  // channel strides of 40 bytes beyond a multiple of 256, so that 16 channels' reads meet different banks
  constexpr int CX = (HZ * HY * RS + 107) / 128 * 128 + 20;
  constexpr int CZ = (TZ * TY * TX + 107) / 128 * 128 + 20;
  constexpr int RPK = 32 / TX;                    // rows per group of 32 voxels
  constexpr int NG = TX * TY * TZ / 32;           // groups per box
  constexpr int ZERO = HZ * HY * RS + 4;          // zeros in the first channel's padding
  static_assert(ZERO + 12 <= CX && ZERO % 4 == 0, "no room for the zeros");
  __shared__ __align__(16) unsigned short xs[16 * CX], zs[16 * CZ];
  const int co0 = blockIdx.x * 16, ci0 = blockIdx.y * 16;
  const int s = blockIdx.z;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ln = lane & 15, lk = lane >> 4;
  const int dz = wv % 3, kh = wv / 3;
  f32x4 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // staging unit: 4 voxels x 8 channels of a row, transposed in registers on
  // the way to LDS
  constexpr int XG = RS / 4, ZG = TX / 4;         // 4-voxel groups per row
  constexpr int XU = HZ * HY * XG * 2, ZU = TZ * TY * ZG * 2;
  constexpr int NX = (XU + 383) / 384, NZ = (ZU + 383) / 384;
  u32x4 tx[NX][4], tz[NZ][4];
  unsigned mx[NX], mz[NZ];                        // which of a unit's voxels lie in the volume
  auto fetch = [&](auto vec, const unsigned short* __restrict__ src, int ld, int nch, int c0, int e, int units,
                   int groups, int ny, int xo, int bx0, int by0, int bz0, u32x4 (&t)[4], unsigned& m) {
    const int h = (e & 1) * 8, g = (e >> 1) % groups, row = (e >> 1) / groups;
    const int y = by0 + row % ny, z = bz0 + row / ny;
    const bool rin = e < units && y >= 0 && y < vol.H && z >= 0 && z < vol.D;
    m = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int x = bx0 + 4 * g + xo + k;
      const bool in = rin && x >= 0 && x < vol.W;
      m |= (unsigned)in << k;
      const unsigned short* p = src + (in ? ((long long)(z * vol.H + y) * vol.W + x) * ld + c0 : 0);
      if constexpr (decltype(vec)::value) {
        t[k] = *reinterpret_cast<const u32x4*>(p + (in ? h : 0));
      } else {
        t[k] = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (in && c0 + h + c < nch) t[k][c >> 1] |= (unsigned)p[h + c] << (16 * (c & 1));
      }
    }
  };
  auto put = [&](u32x4 (&t)[4], unsigned m, unsigned short* dst, int cstride, int rs, int groups, int e) {
    const int h = (e & 1) * 8, g = (e >> 1) % groups, row = (e >> 1) / groups;
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] = m >> k & 1 ? t[k] : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const unsigned sel = c & 1 ? 0x07060302u : 0x05040100u;   // the high or the low halves of two words
      const u32x2 w = {__builtin_amdgcn_perm(t[1][c >> 1], t[0][c >> 1], sel),
                       __builtin_amdgcn_perm(t[3][c >> 1], t[2][c >> 1], sel)};
      *reinterpret_cast<u32x2*>(&dst[(h + c) * cstride + row * rs + 4 * g]) = w;
    }
  };
  const int nbox = bx.nx * bx.ny * bx.nz;
  auto fetch_box = [&](int box) {
    const int x0 = box % bx.nx * TX, y0 = box / bx.nx % bx.ny * TY, z0 = box / (bx.nx * bx.ny) * TZ;
#pragma unroll
    for (int u = 0; u < NX; ++u)
      fetch(std::integral_constant<bool, XVEC>{}, X, ldx, cin, ci0, threadIdx.x + 384 * u, XU, XG, HY, -4, x0, y0 - 1,
            z0 - 1, tx[u], mx[u]);
#pragma unroll
    for (int u = 0; u < NZ; ++u)
      fetch(std::integral_constant<bool, ZVEC>{}, dZ, ldz, cout, co0, threadIdx.x + 384 * u, ZU, ZG, TY, 0, x0, y0, z0,
            tz[u], mz[u]);
  };
  if (RAGGED && threadIdx.x < 16) xs[ZERO - 4 + threadIdx.x] = 0;
  fetch_box(s);
  for (int box = s; box < nbox; box += nsplit) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NX; ++u)
      if ((int)threadIdx.x + 384 * u < XU) put(tx[u], mx[u], xs, CX, RS, XG, threadIdx.x + 384 * u);
#pragma unroll
    for (int u = 0; u < NZ; ++u)
      if ((int)threadIdx.x + 384 * u < ZU) put(tz[u], mz[u], zs, CZ, TX, ZG, threadIdx.x + 384 * u);
    __syncthreads();
    if (box + nsplit < nbox) fetch_box(box + nsplit);   // in flight during the products
    // A voxel just beyond the volume has gradient zero, but its tap towards the
    // volume reads an activation, and 0 times an infinite one would be a NaN: planes
    // beyond the volume are left out, rows beyond it read zeros in the first y-tap,
    // and such a voxel of a row is zeroed in the first x-tap.
    const int x0 = box % bx.nx * TX, y0 = box / bx.nx % bx.ny * TY, z0 = box / (bx.nx * bx.ny) * TZ;
    const int ng = RAGGED ? min(NG, (vol.D - z0) * (TY / RPK)) : NG;
    u32x4 first = {~0u, ~0u, ~0u, ~0u};
    if constexpr (RAGGED) {
      const int j = vol.W - x0 - (TX == 16 ? 8 * (lk & 1) : 0);   // that voxel among this lane's 8
#pragma unroll
      for (int w = 0; w < 4; ++w) first[w] = j == 2 * w ? 0xffff0000u : j == 2 * w + 1 ? 0xffffu : ~0u;
    }
#pragma unroll 2
    for (int g = kh; g < ng; g += 2) {
      const int row = g * RPK + (TX == 16 ? lk >> 1 : lk);        // this lane's row of the box
      const int xh = TX == 16 ? 8 * (lk & 1) : 0;
      const int y = row % TY, z = row / TY;
      const u32x2* za = reinterpret_cast<const u32x2*>(&zs[ln * CZ + row * TX + xh]);
      const u32x2 z0v = za[0], z1v = za[1];
      const u32x4 a = {z0v[0], z0v[1], z1v[0], z1v[1]};
#pragma unroll
      for (int dy = 0; dy < 3; ++dy) {
        const unsigned short* xr = &xs[ln * CX + ((z + dz) * HY + y + dy) * RS + 4 + xh];
        if (RAGGED && dy == 0) xr = y0 + y >= vol.H ? &xs[ZERO] : xr;
        const unsigned wm = *reinterpret_cast<const unsigned*>(xr - 2), wp = *reinterpret_cast<const unsigned*>(xr + 8);
        const u32x2 wa = *reinterpret_cast<const u32x2*>(xr), wb = *reinterpret_cast<const u32x2*>(xr + 4);
        const unsigned s0 = __builtin_amdgcn_alignbit(wa[0], wm, 16), s1 = __builtin_amdgcn_alignbit(wa[1], wa[0], 16);
        const unsigned s2 = __builtin_amdgcn_alignbit(wb[0], wa[1], 16), s3 = __builtin_amdgcn_alignbit(wb[1], wb[0], 16);
        const unsigned s4 = __builtin_amdgcn_alignbit(wp, wb[1], 16);
        acc[3 * dy] = mfma32(a, u32x4{s0, s1, s2, s3} & first, acc[3 * dy]);
        acc[3 * dy + 1] = mfma32(a, u32x4{wa[0], wa[1], wb[0], wb[1]}, acc[3 * dy + 1]);
        acc[3 * dy + 2] = mfma32(a, u32x4{s1, s2, s3, s4}, acc[3 * dy + 2]);
      }
    }
  }
  // add the two k-halves (lane (ln, lk) register r: channel 4 lk + r of dZ, channel ln of X)
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(xs);     // 3 * 9 * 64 of them
  static_assert(sizeof(f32x4) * 3 * 9 * 64 <= sizeof(xs), "partial sums do not fit");
  if (kh == 1) {
#pragma unroll
    for (int t = 0; t < 9; ++t) red[(dz * 9 + t) * 64 + lane] = acc[t];
  }
  __syncthreads();
  if (kh == 0 && ci0 + ln < cin) {
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const f32x4 o = red[(dz * 9 + t) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int co = co0 + 4 * lk + r;
        if (co < cout) part[(((long long)s * cout + co) * 27 + dz * 9 + t) * cin + ci0 + ln] = acc[t][r] + o[r];
      }
    }
  }
}

// The same over voxels in flat order, for volumes that boxes cover badly: workgroup
// (tap t, 16 output channels, 16 NTC input channels, voxel split s), its operands
// gathered from global memory.
template <int NTC>
__global__ __launch_bounds__(256) void conv_wgrad_flat(Vol vol, const unsigned short* __restrict__ dZ, int ldz,
                                                       int cout, const unsigned short* __restrict__ X, int ldx, int cin,
                                                       long long vchunk, float* __restrict__ part) {
  __shared__ float red[kWaves][16 * 16 * NTC];
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int ln = lane & 15, lk = lane >> 4;
  const int t = blockIdx.x % 27;
  const int cob = blockIdx.x / 27;
  const int cib = blockIdx.y;
  const int s = blockIdx.z;
  int dz, dy, dx;
  tap_offsets(t, dz, dy, dx);
  const int co = cob * 16 + ln;
  const long long v0 = (long long)s * vchunk;
  const long long v1 = min(v0 + vchunk, vol.V);
  f32x4 acc[NTC];
#pragma unroll
  for (int n = 0; n < NTC; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  // each wavefront takes every 4th group of 16 voxels
  for (long long vb = v0 + 16 * wv; vb < v1; vb += 16 * kWaves) {
    bf16x4 a;
    bf16x4 b[NTC];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const long long v = vb + 4 * lk + j;
      const bool vok = v < v1;
      a[j] = (vok && co < cout) ? (short)dZ[v * ldz + co] : (short)0;
      long long src = -1;
      if (vok) {
        const int x = (int)(v % vol.W) + dx;
        const int y = (int)((v / vol.W) % vol.H) + dy;
        const int z = (int)(v / ((long long)vol.W * vol.H)) + dz;
        if (z >= 0 && z < vol.D && y >= 0 && y < vol.H && x >= 0 && x < vol.W)
          src = ((long long)(z * vol.H + y) * vol.W + x) * ldx;
      }
#pragma unroll
      for (int n = 0; n < NTC; ++n) {
        const int ci = cib * 16 * NTC + 16 * n + ln;
        b[n][j] = (src >= 0 && ci < cin) ? (short)X[src + ci] : (short)0;
      }
    }
#pragma unroll
    for (int n = 0; n < NTC; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[n], acc[n], 0, 0, 0);
  }
  // D[m = co row 4*lk + r][n = ci col ln]
#pragma unroll
  for (int n = 0; n < NTC; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][(4 * lk + r) * (16 * NTC) + 16 * n + ln] = acc[n][r];
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * 16 * NTC; e += 256) {
    const float sum = red[0][e] + red[1][e] + red[2][e] + red[3][e];
    const int m = e / (16 * NTC), c = e % (16 * NTC);
    const int com = cob * 16 + m, cim = cib * 16 * NTC + c;
    if (com < cout && cim < cin) part[(((long long)s * cout + com) * 27 + t) * cin + cim] = sum;
  }
}

// dW[i] = sum_s part[s][i]: 32 elements per workgroup, 8 threads each taking
// every 8th split in order, their sums added in order
__global__ __launch_bounds__(256) void reduce_splits(const float* __restrict__ part, int nsplit, long long n,
                                                     float* __restrict__ out) {
  __shared__ float red[8][32];
  const int el = threadIdx.x & 31, g = threadIdx.x >> 5;
  const long long i = (long long)blockIdx.x * 32 + el;
  float s = 0.f;
  if (i < n) {
#pragma unroll 8
    for (int k = g; k < nsplit; k += 8) s += part[(long long)k * n + i];
  }
  red[g][el] = s;
  __syncthreads();
  if (g == 0 && i < n) {
    float t = red[0][el];
#pragma unroll
    for (int q = 1; q < 8; ++q) t += red[q][el];
    out[i] = t;
  }
}

// dZ = dA * (a > 0 ? 1 : slope) (a == nullptr: identity), rounded to BF16;
// per-block partial bias gradients sum(dZ) per channel (FP32 before rounding).
__global__ __launch_bounds__(256) void act_bwd(const float* __restrict__ dA, int lda,
                                               const unsigned short* __restrict__ a, int lda_a, int C, long long V,
                                               float slope, unsigned short* __restrict__ dZ, int ldz,
                                               long long vchunk, float* __restrict__ dbpart) {
  __shared__ float red[256];
  const int c = threadIdx.x % C;             // C divides 256 or C <= 256 handled by the grid-stride below
  const int lanes = (256 / C) * C;
  const int slot = threadIdx.x / C;
  const int nslot = 256 / C;
  float s = 0.f;
  if (threadIdx.x < lanes) {
    const long long v0 = (long long)blockIdx.x * vchunk;
    const long long v1 = min(v0 + vchunk, V);
    for (long long v = v0 + slot; v < v1; v += nslot) {
      float g = dA[v * lda + c];
      if (a) g = bf2f(a[v * lda_a + c]) > 0.f ? g : slope * g;
      dZ[v * ldz + c] = f2bf(g);
      s += g;
    }
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < C) {
    float tot = 0.f;
    for (int k = 0; k < nslot; ++k) tot += red[k * C + threadIdx.x];
    dbpart[(long long)blockIdx.x * C + threadIdx.x] = tot;
  }
}

// The same for C = 4 C4 channels in 16- and 8-byte pieces: a thread takes 4
// channels of every (256 / C4)-th voxel.
__global__ __launch_bounds__(256) void act_bwd4(const float* __restrict__ dA, int lda,
                                                const unsigned short* __restrict__ a, int lda_a, int C4, long long V,
                                                float slope, unsigned short* __restrict__ dZ, int ldz,
                                                long long vchunk, float* __restrict__ dbpart) {
  __shared__ f32x4 red[256];
  const int c = threadIdx.x % C4 * 4, slot = threadIdx.x / C4, nslot = 256 / C4;
  const long long v0 = (long long)blockIdx.x * vchunk;
  const long long v1 = slot < nslot ? min(v0 + vchunk, V) : v0;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (long long v = v0 + slot; v < v1; v += nslot) {
    f32x4 g = *reinterpret_cast<const f32x4*>(dA + v * lda + c);
    if (a) {
      const u32x2 t = *reinterpret_cast<const u32x2*>(a + v * lda_a + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float av = __uint_as_float(r & 1 ? t[r >> 1] & 0xffff0000u : t[r >> 1] << 16);
        g[r] = av > 0.f ? g[r] : slope * g[r];
      }
    }
    const u32x2 o = {f2bf(g[0]) | (unsigned)f2bf(g[1]) << 16, f2bf(g[2]) | (unsigned)f2bf(g[3]) << 16};
    *reinterpret_cast<u32x2*>(dZ + v * ldz + c) = o;
    s += g;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int n = nslot; n > 1;) {
    const int h = (n + 1) / 2;
    if (slot + h < n) red[threadIdx.x] += red[threadIdx.x + h * C4];
    __syncthreads();
    n = h;
  }
  if (slot == 0) *reinterpret_cast<f32x4*>(dbpart + (long long)blockIdx.x * 4 * C4 + c) = red[threadIdx.x];
}

__global__ void pool2_fwd(Vol out, const unsigned short* __restrict__ X, int ldx, int C,
                          unsigned short* __restrict__ Y, int ldy) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= out.V * C) return;
  const int c = (int)(i % C);
  const long long v = i / C;
  const int x = (int)(v % out.W), y = (int)((v / out.W) % out.H), z = (int)(v / ((long long)out.W * out.H));
  const int W2 = 2 * out.W, H2 = 2 * out.H;
  float s = 0.f;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
    s += bf2f(X[((long long)(zz * H2 + yy) * W2 + xx) * ldx + c]);
  }
  Y[v * ldy + c] = f2bf(s * 0.125f);
}

// dX (fine) = dY(coarse)/8 + dSkip (fine, optional)
__global__ void pool2_bwd(Vol fine, const float* __restrict__ dY, int ldy, const float* __restrict__ dS, int lds,
                          int C, float* __restrict__ dX, int ldx) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= fine.V * C) return;
  const int c = (int)(i % C);
  const long long v = i / C;
  const int x = (int)(v % fine.W), y = (int)((v / fine.W) % fine.H), z = (int)(v / ((long long)fine.W * fine.H));
  const int Wc = fine.W / 2, Hc = fine.H / 2;
  float g = dY[((long long)((z / 2) * Hc + y / 2) * Wc + x / 2) * ldy + c] * 0.125f;
  if (dS) g += dS[v * lds + c];
  dX[v * ldx + c] = g;
}

__global__ void up2_fwd(Vol fine, const unsigned short* __restrict__ X, int ldx, int C,
                        unsigned short* __restrict__ Y, int ldy) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= fine.V * C) return;
  const int c = (int)(i % C);
  const long long v = i / C;
  const int x = (int)(v % fine.W), y = (int)((v / fine.W) % fine.H), z = (int)(v / ((long long)fine.W * fine.H));
  const int Wc = fine.W / 2, Hc = fine.H / 2;
  Y[v * ldy + c] = X[((long long)((z / 2) * Hc + y / 2) * Wc + x / 2) * ldx + c];
}

// dX (coarse) = sum of the 8 fine children of dY
__global__ void up2_bwd(Vol coarse, const float* __restrict__ dY, int ldy, int C, float* __restrict__ dX, int ldx) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= coarse.V * C) return;
  const int c = (int)(i % C);
  const long long v = i / C;
  const int x = (int)(v % coarse.W), y = (int)((v / coarse.W) % coarse.H);
  const int z = (int)(v / ((long long)coarse.W * coarse.H));
  const int W2 = 2 * coarse.W, H2 = 2 * coarse.H;
  float s = 0.f;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
    s += dY[((long long)(zz * H2 + yy) * W2 + xx) * ldy + c];
  }
  dX[v * ldx + c] = s;
}

__global__ void cast_bf16(const float* __restrict__ src, long long n, unsigned short* __restrict__ dst) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = f2bf(src[i]);
}

// Adam with bias correction; writes the BF16 copy of the updated weights.
__global__ void adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                     long long n, float lr, float b1, float b2, float eps, float wd, float bc1, float bc2,
                     unsigned short* __restrict__ wbf) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i] + wd * w[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wn = w[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  w[i] = wn;
  if (wbf) wbf[i] = f2bf(wn);
}

// dy = 2 (y - t) / n; per-block partial sums of (y - t)^2 (FP64)
__global__ __launch_bounds__(256) void mse(const float* __restrict__ y, const float* __restrict__ t, long long n,
                                           float* __restrict__ dy, double* __restrict__ part) {
  __shared__ double red[4];
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float d = y[i] - t[i];
    dy[i] = 2.f * d / (float)n;
    s += (double)d * d;
  }
  const double tot = pc_block_sum(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// out[c] = sum over the blocks, one workgroup per channel
__global__ __launch_bounds__(256) void sum_parts_f32(const float* __restrict__ part, int nblk, int C,
                                                     float* __restrict__ out) {
  __shared__ float red[256];
  const int c = blockIdx.x;
  float s = 0.f;
  for (int b = threadIdx.x; b < nblk; b += 256) s += part[(long long)b * C + c];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = red[0];
}

__global__ void sum_parts_f64(const double* __restrict__ part, int nblk, double* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double s = 0.0;
  for (int b = 0; b < nblk; ++b) s += part[b];
  out[0] = s;
}

Vol make_vol(int D, int H, int W) { return Vol{D, H, W, (long long)D * H * W}; }

inline int nblk(long long n, int b = 256) { return (int)((n + b - 1) / b); }

constexpr int kWgradSplit = 128;     // voxel splits of the weight gradient, at most
constexpr int kWgradSplitMin = 64;   // splits whose workspace every caller has to bring
constexpr int kActChunk = 512;       // voxels per workgroup of the activation backward, at least
constexpr int kActChunkMax = 2048;   // (chunk whose workspace every caller has to bring)
constexpr int kMseBlocks = 512;

Boxes make_boxes(const Vol& v, int tx, int ty, int tz, int cblocks) {
  Boxes b;
  b.nx = (v.W + tx - 1) / tx;
  b.ny = (v.H + ty - 1) / ty;
  b.nz = (v.D + tz - 1) / tz;
  b.nblocks = b.nx * b.ny * b.nz * cblocks;
  b.nb8 = (b.nblocks + 7) / 8;
  return b;
}
inline long long box_count(const Vol& v, int tx, int ty, int tz) {
  return (long long)((v.W + tx - 1) / tx) * ((v.H + ty - 1) / ty) * ((v.D + tz - 1) / tz);
}
inline bool aligned(const void* p, size_t n) { return reinterpret_cast<uintptr_t>(p) % n == 0; }

}  // namespace

extern "C" {

int pc_unet_conv3d_fwd(const void* X, int ldx, int cin, const void* W, const float* bias, int cout, int D, int H,
                       int Wd, int mode, float slope, void* Y, int ldy, void* stream) {
  PC_CHECK_ARG(X && W && Y, "null pointer");
  PC_CHECK_ARG(D > 0 && H > 0 && Wd > 0, "bad volume");
  PC_CHECK_ARG(cin == 1 || (cin % 16 == 0), "cin must be 1 or a multiple of 16");
  PC_CHECK_ARG(cout >= 1, "cout < 1");
  PC_CHECK_ARG(ldx >= cin && ldy >= cout, "channel stride smaller than the channel count");
  PC_CHECK_ARG(cin == 1 || (ldx % 4 == 0), "ldx must be a multiple of 4");
  PC_CHECK_ARG(mode >= 0 && mode <= 2, "bad mode");
  PC_CHECK_ARG(mode == 2 || bias, "bias required");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Vol vol = make_vol(D, H, Wd);
  PC_CHECK_ARG(vol.V < (1LL << 31), "volume too large");
  auto X16 = static_cast<const unsigned short*>(X);
  auto W16 = static_cast<const unsigned short*>(W);
  const int ct = (cout + 15) / 16;
  const bool yvec = ldy % 4 == 0 && aligned(Y, mode == 1 ? 8 : 16);
  const bool xvec = ldx % 8 == 0 && aligned(X, 16);
  // Boxes of 512 voxels for one group of 16 input channels, 256 for two or
  // three and 128 for up to seven (LDS: two workgroups per CU, one for seven groups
  // and for six in 16-wide boxes), 16 or 8 wide
  // (whichever pads the volume less); 128 also where larger ones would not give
  // every CU a workgroup.
  const int ncb = cin / 16;
  auto padded = [&](int tx, int ty, int tz) { return box_count(vol, tx, ty, tz) * tx * ty * tz; };
  const bool fill512 = padded(16, 8, 4) / 512 * ct >= 256, fill256 = padded(16, 4, 4) / 256 * ct >= 256;
  const int size = cin == 1 || ncb == 1 ? (fill512 ? 512 : 128) : ncb <= 3 ? (fill256 ? 256 : 128) : 128;
  const bool w8 = size == 512   ? padded(8, 8, 8) < padded(16, 8, 4)
                  : size == 256 ? padded(8, 8, 4) < padded(16, 4, 4)
                                : padded(8, 4, 4) < padded(16, 4, 2);
  // conv_fwd: more input channels, columns without 16-byte alignment, and volumes
  // that the boxes pad by so much that gathering every operand is the shorter
  // (once the chip is full, at 2^18 padded voxels x channel blocks; a 300,000 x 1 x 1
  // volume, 64 -> 64 channels: 14.5 ms in boxes, 0.53 gathered; 300 x 2 x 300, padded
  // twice: 112 -> 48 channels 0.75 and 0.38, 48 -> 64 0.18 and 0.27).
  const long long pad = size == 512   ? std::min(padded(8, 8, 8), padded(16, 8, 4))
                        : size == 256 ? std::min(padded(8, 8, 4), padded(16, 4, 4))
                                      : std::min(padded(8, 4, 4), padded(16, 4, 2));
  const double most = cin == 1 ? 12.0 : ncb == 1 ? 4.2 : ncb <= 3 ? 2.2 : ncb <= 5 ? 1.8 : 1.3;
  const bool gather = pad * ct >= (1 << 18) && (double)pad > most * (double)vol.V;
  // the channel blocks that one launch holds at a time
#define PC_CONV_PARTS(KERNEL, TX, TY, TZ)                                                                            \
  do {                                                                                                               \
    const int step = (int)std::max(1LL, std::min<long long>(ct, pc::kMaxGrid / box_count(vol, TX, TY, TZ)));         \
    for (int c = 0; c < ct; c += step) {                                                                             \
      const Boxes bx = make_boxes(vol, TX, TY, TZ, std::min(step, ct - c));                                          \
      void* y = mode == 1 ? (void*)(static_cast<unsigned short*>(Y) + 16 * c) : (void*)(static_cast<float*>(Y) + 16 * c); \
      hipLaunchKernelGGL((KERNEL), dim3(8 * bx.nb8), dim3(256), 0, st, vol, bx, X16, ldx, W16 + 16LL * c * 27 * cin, \
                         bias ? bias + 16 * c : nullptr, cout - 16 * c, mode, slope, y, ldy, yvec);                  \
      PC_LAUNCH_CHECK();                                                                                             \
    }                                                                                                                \
  } while (0)
#define PC_CONV(NCB, TX, TY, TZ) PC_CONV_PARTS((conv_tile<NCB, TX, TY, TZ>), TX, TY, TZ)
#define PC_CONV1(TX, TY, TZ) PC_CONV_PARTS((conv_tile1<TX, TY, TZ>), TX, TY, TZ)
#define PC_CONV128(NCB)                \
  do {                                 \
    if (w8) PC_CONV(NCB, 8, 4, 4);     \
    else PC_CONV(NCB, 16, 4, 2);       \
  } while (0)
#define PC_CONV256(NCB)                \
  do {                                 \
    if (w8) PC_CONV(NCB, 8, 8, 4);     \
    else PC_CONV(NCB, 16, 4, 4);       \
  } while (0)
  if (gather || (cin > 1 && (ncb > 7 || !xvec))) {
    const long long vox_per_block = 16LL * kNT * kWaves;
    dim3 grid((unsigned)((vol.V + vox_per_block - 1) / vox_per_block), (unsigned)((cout + 63) / 64));
    auto general = ct == 1 ? conv_fwd<1, false> : ct == 2 ? conv_fwd<2, false> : ct == 3 ? conv_fwd<3, false> : conv_fwd<4, false>;
    if (cin == 1) general = ct == 1 ? conv_fwd<1, true> : ct == 2 ? conv_fwd<2, true> : ct == 3 ? conv_fwd<3, true> : conv_fwd<4, true>;
    hipLaunchKernelGGL(general, grid, dim3(256), 0, st, vol, X16, ldx, cin, W16, bias, cout, mode, slope, Y, ldy);
  } else if (cin == 1) {
    if (size == 512) {
      if (w8) PC_CONV1(8, 8, 8);
      else PC_CONV1(16, 8, 4);
    } else {
      if (w8) PC_CONV1(8, 4, 4);
      else PC_CONV1(16, 4, 2);
    }
  } else {
    switch (ncb) {
      case 1:
        if (size == 512) {
          if (w8) PC_CONV(1, 8, 8, 8);
          else PC_CONV(1, 16, 8, 4);
        } else {
          PC_CONV128(1);
        }
        break;
      case 2:
        if (size == 256) PC_CONV256(2);
        else PC_CONV128(2);
        break;
      case 3:
        if (size == 256) PC_CONV256(3);
        else PC_CONV128(3);
        break;
      case 4: PC_CONV128(4); break;
      case 5: PC_CONV128(5); break;
      case 6: PC_CONV128(6); break;
      default: PC_CONV128(7); break;
    }
  }
#undef PC_CONV
#undef PC_CONV1
#undef PC_CONV_PARTS
#undef PC_CONV128
#undef PC_CONV256
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

int pc_unet_conv3d_wflip(const void* W, int cout, int cin, void* Wt, void* stream) {
  PC_CHECK_ARG(W && Wt, "null pointer");
  PC_CHECK_ARG(cout >= 1 && cin >= 1, "bad channels");
  const long long n = (long long)cout * cin * 27;
  hipLaunchKernelGGL(conv_wflip, dim3(nblk(n)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const unsigned short*>(W), cout, cin, static_cast<unsigned short*>(Wt));
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

int pc_unet_wgrad_workspace(int cout, int cin, size_t* out_bytes) {
  PC_CHECK_ARG(out_bytes, "null pointer");
  *out_bytes = (size_t)kWgradSplit * cout * 27 * cin * sizeof(float);
  return pc::PC_OK;
}

// dW[co][t][ci] = sum_v dZ[v][co] X[v + off_t][ci]  (FP32 result)
int pc_unet_conv3d_wgrad(const void* dZ, int ldz, int cout, const void* X, int ldx, int cin, int D, int H, int Wd,
                         float* dW, void* work, size_t work_bytes, void* stream) {
  PC_CHECK_ARG(dZ && X && dW && work, "null pointer");
  PC_CHECK_ARG(D > 0 && H > 0 && Wd > 0, "bad volume");
  PC_CHECK_ARG(ldz >= cout && ldx >= cin, "channel stride smaller than the channel count");
  const long long n = (long long)cout * 27 * cin;
  PC_CHECK_ARG(work_bytes >= kWgradSplitMin * n * sizeof(float), "workspace too small");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Vol vol = make_vol(D, H, Wd);
  auto dZ16 = static_cast<const unsigned short*>(dZ);
  auto X16 = static_cast<const unsigned short*>(X);
  float* part = static_cast<float*>(work);
  const bool zvec = ldz % 8 == 0 && cout % 16 == 0 && aligned(dZ, 16);
  const bool xvec = ldx % 8 == 0 && cin % 16 == 0 && aligned(X, 16);
  const bool w8 = box_count(vol, 8, 8, 4) * 8 < box_count(vol, 16, 8, 4) * 16;   // padded rows
  const int room = (int)std::min<long long>(kWgradSplit, (long long)(work_bytes / sizeof(float)) / n);
  // Volumes that the boxes pad twelvefold and more (lines of voxels): over the
  // voxels in flat order.  1 x 1 x 300,000, 48 -> 16 channels: 1.9 ms in boxes,
  // 0.6 flat; 2 x 2 x 40,000, padded eightfold: 0.27 and 0.36.
  if ((w8 ? box_count(vol, 8, 8, 4) * 256 : box_count(vol, 16, 8, 4) * 512) >= 12 * vol.V && vol.V >= 512) {
    const int splits = (int)std::min<long long>(std::min(room, kWgradSplitMin), (vol.V + 255) / 256);
    const long long vchunk = (vol.V + splits - 1) / splits;
    const int ntc = cin >= 32 ? 2 : 1;
    hipLaunchKernelGGL((ntc == 2 ? conv_wgrad_flat<2> : conv_wgrad_flat<1>),
                       dim3(27 * ((cout + 15) / 16), (cin + 16 * ntc - 1) / (16 * ntc), splits), dim3(256), 0, st, vol,
                       dZ16, ldz, cout, X16, ldx, cin, vchunk, part);
    PC_LAUNCH_CHECK();
    hipLaunchKernelGGL(reduce_splits, dim3(nblk(n, 32)), dim3(256), 0, st, part, splits, n, dW);
    PC_LAUNCH_CHECK();
    return pc::PC_OK;
  }
  const Boxes bx = w8 ? make_boxes(vol, 8, 8, 4, 1) : make_boxes(vol, 16, 8, 4, 1);
  const int nsplit = std::min(room, bx.nblocks);
  dim3 grid((cout + 15) / 16, (cin + 15) / 16, nsplit);
  const bool ragged = Wd % (w8 ? 8 : 16) != 0 || H % 8 != 0 || D % 4 != 0;
#define PC_WGRAD(TX, ZV, XV, RG)                                                                                     \
  hipLaunchKernelGGL((conv_wgrad<TX, 8, 4, ZV, XV, RG>), grid, dim3(384), 0, st, vol, bx, dZ16, ldz, cout, X16, ldx, \
                     cin, nsplit, part)
#define PC_WGRAD_V(TX, RG)                             \
  do {                                                 \
    if (zvec && xvec) PC_WGRAD(TX, true, true, RG);    \
    else if (zvec) PC_WGRAD(TX, true, false, RG);      \
    else if (xvec) PC_WGRAD(TX, false, true, RG);      \
    else PC_WGRAD(TX, false, false, RG);               \
  } while (0)
  if (w8) {
    if (ragged) PC_WGRAD_V(8, true);
    else PC_WGRAD_V(8, false);
  } else {
    if (ragged) PC_WGRAD_V(16, true);
    else PC_WGRAD_V(16, false);
  }
#undef PC_WGRAD
#undef PC_WGRAD_V
  PC_LAUNCH_CHECK();
  hipLaunchKernelGGL(reduce_splits, dim3(nblk(n, 32)), dim3(256), 0, st, part, nsplit, n, dW);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

int pc_unet_act_bwd_workspace(int C, long long V, size_t* out_bytes) {
  PC_CHECK_ARG(out_bytes && C >= 1 && V >= 1, "bad argument");
  *out_bytes = (size_t)((V + kActChunk - 1) / kActChunk) * C * sizeof(float);
  return pc::PC_OK;
}

// dZ (BF16) = dA * leaky'(a) (a == NULL: identity); db[c] = sum_v dZ (FP32)
int pc_unet_act_bwd(const float* dA, int lda, const void* a, int lda_a, int C, int D, int H, int Wd, float slope,
                    void* dZ, int ldz, float* db, void* work, size_t work_bytes, void* stream) {
  PC_CHECK_ARG(dA && dZ && db && work, "null pointer");
  PC_CHECK_ARG(C >= 1 && C <= 256, "C must be in [1, 256]");
  const long long V = (long long)D * H * Wd;
  PC_CHECK_ARG(work_bytes >= (size_t)((V + kActChunkMax - 1) / kActChunkMax) * C * sizeof(float), "workspace too small");
  hipStream_t st = static_cast<hipStream_t>(stream);
  // the smallest chunk of at least kActChunk voxels whose partial sums fit and whose workgroups one launch holds
  long long chunk = kActChunk;
  while ((size_t)((V + chunk - 1) / chunk) * C * sizeof(float) > work_bytes || (V + chunk - 1) / chunk > pc::kMaxGrid)
    chunk *= 2;
  const int nb = (int)((V + chunk - 1) / chunk);
  float* part = static_cast<float*>(work);
  auto a16 = static_cast<const unsigned short*>(a);
  auto z16 = static_cast<unsigned short*>(dZ);
  const int c4 = C / 4;
  const bool vec = C % 4 == 0 && lda % 4 == 0 && aligned(dA, 16) && ldz % 4 == 0 &&
                   aligned(dZ, 8) && (!a || (lda_a % 4 == 0 && aligned(a, 8))) && aligned(part, 16);
  if (vec)
    hipLaunchKernelGGL(act_bwd4, dim3(nb), dim3(256), 0, st, dA, lda, a16, lda_a, c4, V, slope, z16, ldz, chunk, part);
  else
    hipLaunchKernelGGL(act_bwd, dim3(nb), dim3(256), 0, st, dA, lda, a16, lda_a, C, V, slope, z16, ldz, chunk, part);
  PC_LAUNCH_CHECK();
  hipLaunchKernelGGL(sum_parts_f32, dim3(C), dim3(256), 0, st, part, nb, C, db);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

// pooled (D/2, H/2, W/2) from X (D, H, W)
int pc_unet_pool2_fwd(const void* X, int ldx, int C, int D, int H, int Wd, void* Y, int ldy, void* stream) {
  PC_CHECK_ARG(X && Y, "null pointer");
  PC_CHECK_ARG(D % 2 == 0 && H % 2 == 0 && Wd % 2 == 0, "even volume required");
  const Vol out = make_vol(D / 2, H / 2, Wd / 2);
  hipLaunchKernelGGL(pool2_fwd, dim3(nblk(out.V * C)), dim3(256), 0, static_cast<hipStream_t>(stream), out,
                     static_cast<const unsigned short*>(X), ldx, C, static_cast<unsigned short*>(Y), ldy);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

int pc_unet_pool2_bwd(const float* dY, int ldy, const float* dS, int lds, int C, int D, int H, int Wd, float* dX,
                      int ldx, void* stream) {
  PC_CHECK_ARG(dY && dX, "null pointer");
  PC_CHECK_ARG(D % 2 == 0 && H % 2 == 0 && Wd % 2 == 0, "even volume required");
  const Vol fine = make_vol(D, H, Wd);
  hipLaunchKernelGGL(pool2_bwd, dim3(nblk(fine.V * C)), dim3(256), 0, static_cast<hipStream_t>(stream), fine, dY, ldy,
                     dS, lds, C, dX, ldx);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

// fine (D, H, W) from coarse X (D/2, H/2, W/2)
int pc_unet_up2_fwd(const void* X, int ldx, int C, int D, int H, int Wd, void* Y, int ldy, void* stream) {
  PC_CHECK_ARG(X && Y, "null pointer");
  PC_CHECK_ARG(D % 2 == 0 && H % 2 == 0 && Wd % 2 == 0, "even volume required");
  const Vol fine = make_vol(D, H, Wd);
  hipLaunchKernelGGL(up2_fwd, dim3(nblk(fine.V * C)), dim3(256), 0, static_cast<hipStream_t>(stream), fine,
                     static_cast<const unsigned short*>(X), ldx, C, static_cast<unsigned short*>(Y), ldy);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

// coarse gradient (D/2, H/2, W/2) from the fine gradient dY (D, H, W)
int pc_unet_up2_bwd(const float* dY, int ldy, int C, int D, int H, int Wd, float* dX, int ldx, void* stream) {
  PC_CHECK_ARG(dY && dX, "null pointer");
  PC_CHECK_ARG(D % 2 == 0 && H % 2 == 0 && Wd % 2 == 0, "even volume required");
  const Vol coarse = make_vol(D / 2, H / 2, Wd / 2);
  hipLaunchKernelGGL(up2_bwd, dim3(nblk(coarse.V * C)), dim3(256), 0, static_cast<hipStream_t>(stream), coarse, dY,
                     ldy, C, dX, ldx);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

int pc_unet_cast_bf16(const float* src, long long n, void* dst, void* stream) {
  PC_CHECK_ARG(src && dst && n >= 0, "bad argument");
  if (n == 0) return pc::PC_OK;
  hipLaunchKernelGGL(cast_bf16, dim3(nblk(n)), dim3(256), 0, static_cast<hipStream_t>(stream), src, n,
                     static_cast<unsigned short*>(dst));
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

// step >= 1; wbf (optional) receives the BF16 rounding of the updated weights
int pc_unet_adam(float* w, const float* g, float* m, float* v, long long n, double lr, double b1, double b2,
                 double eps, double wd, int step, void* wbf, void* stream) {
  PC_CHECK_ARG(w && g && m && v && n >= 0 && step >= 1, "bad argument");
  if (n == 0) return pc::PC_OK;
  const float bc1 = (float)(1.0 - std::pow(b1, step));
  const float bc2 = (float)(1.0 - std::pow(b2, step));
  hipLaunchKernelGGL(adam, dim3(nblk(n)), dim3(256), 0, static_cast<hipStream_t>(stream), w, g, m, v, n, (float)lr,
                     (float)b1, (float)b2, (float)eps, (float)wd, bc1, bc2, static_cast<unsigned short*>(wbf));
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

int pc_unet_mse_workspace(size_t* out_bytes) {
  PC_CHECK_ARG(out_bytes, "null pointer");
  *out_bytes = (size_t)kMseBlocks * sizeof(double);
  return pc::PC_OK;
}

// dy = 2 (y - t)/n; loss_dev[0] (FP64, device) = sum (y - t)^2
int pc_unet_mse(const float* y, const float* t, long long n, float* dy, double* loss_dev, void* work,
                size_t work_bytes, void* stream) {
  PC_CHECK_ARG(y && t && dy && loss_dev && work && n > 0, "bad argument");
  PC_CHECK_ARG(work_bytes >= (size_t)kMseBlocks * sizeof(double), "workspace too small");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nb = (int)std::min<long long>(kMseBlocks, (n + 255) / 256);
  double* part = static_cast<double*>(work);
  hipLaunchKernelGGL(mse, dim3(nb), dim3(256), 0, st, y, t, n, dy, part);
  PC_LAUNCH_CHECK();
  hipLaunchKernelGGL(sum_parts_f64, dim3(1), dim3(64), 0, st, part, nb, loss_dev);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

}  // extern "C"
