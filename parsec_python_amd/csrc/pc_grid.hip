// Grid index map and the fused multi-vector finite-difference stencil.
//
// Storage ("compact, vector-major"): the domain is a set of x-rows (j,k) of an
// nx*ny*nz cube, each row holding the contiguous points lo[j,k] <= i < hi[j,k]
// (cube: the whole row; sphere: the chord).  Points are numbered k-major, then
// j, then i, so row (j,k) starts at off[j,k].  Vector v of a block lives at
// [v*ld, v*ld + npts).  Outside the domain values are zero (Dirichlet), which
// is the reference's truncated-diagonal Laplacian (src/Laplacian/fd3d.py:79-100)
// when the domain is the full cube.
//
// One launch computes, for every vector v and domain point p,
//     out = sum_d w_d * (6 neighbours at distance d) + w_0 * y  (the -lap weights,
//           pre-multiplied by the caller's scale)
//         + (a*V[p] + b) * y[p] + c * x[p]
// which is H*y (a=1,b=0,c=0) and every step of the reference's scaled and slim
// Chebyshev filters (src/Eigensolvers/ch_filter.py:66-80, first_filt.py:94-101).
// x may alias out (each point reads x before writing out at the same place).
//
// Kernel shape (CDNA4; stencil_win, and stencil_zmarch where partial sums are asked
// for): a workgroup owns one vector, a slab of y-rows and a window of up to 64 or 128
// columns (its whole rows), and marches along z.  Each thread keeps its point's 2R+1
// z-values in registers; the current plane of the slab plus R halo rows
// above/below sits in LDS for the x/y differences.  Workgroup ids are remapped so
// the windows of one vector run on the same XCD (its L2 then serves the halos).
#include "pc_common.h"
#include "pc_zmarch.h"
#include <type_traits>
#include <utility>
#include <vector>
#include <algorithm>
#include <cstring>

namespace {

// One way to cut the windows into z-chunks: planes per chunk, chunks of the longest
// window; over all windows the chunks that have planes and their planes in whole
// blocks; the longest chunk.
struct WinSplit {
  int zc, nzc, wgs;
  long long planes;
  int longest;
};

struct GridDev {
  int nx, ny, nz;
  long long npts;
  void* tables;  // the one allocation that the tables below lie in
  int* lo;       // [ny*nz]
  int* hi;       // [ny*nz]
  int* off;      // [ny*nz]
  int* zrange;   // [2*ny]: min z, max z+1 of non-empty rows per y
  int2* meta;    // [ny*nz]: {off - lo, lo | hi << 16}
  int* prow;     // [npts]: row (j + ny*k) of each domain point
  int radius;
  double w[8];   // 1D -d2/dx2 weights, centre first (unscaled)
  int4* win;     // stencil_win: windows {first row, first column | columns << 16 | left halo lanes << 28, zb, ze}
  int nwin;        // their number
  std::vector<WinSplit> splits;   // ways to cut them, the longest chunks first
  int winsx;       // wavefronts of 64 columns per row of a window
  int2* pmeta;   // its padded row table {offset, lo | length << 16}, nyp x nzp
  int nyp, nzp;
};

struct StArgs {
  int nx, ny, nz;
  long long npts;
  const int* lo;
  const int* hi;
  const int* off;
  const int* zrange;
  const int2* meta;
  long long ld;
  int nslab;
  int nvec;
  int nblocks;   // real (unpadded) number of workgroups
  int nb8;       // ceil(nblocks/8)
  double w[8];   // scaled weights; w[0] already includes the factor 3
};

template <typename T>
__device__ __forceinline__ T row_val(const T* __restrict__ y, int lo, int hi, int off, int i) {
  return (i >= lo && i < hi) ? y[off + (i - lo)] : T(0);
}

// LDS-only workgroup barrier: waits for this wave's LDS traffic, not for
// outstanding global loads (the prefetch of the next plane stays in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt/expcnt left at max
  __builtin_amdgcn_s_barrier();
}

template <typename T>
__device__ __forceinline__ T meta_val(const T* __restrict__ y, int2 m, int i) {
  const int lo = m.y & 0xffff, hi = m.y >> 16;
  return (i >= lo && i < hi) ? y[m.x + i] : T(0);
}

// The step with per-workgroup sums of out * y: a workgroup owns one vector and 4
// y-rows, one wavefront of SX 64-column parts per row, and marches z.  While plane
// z is computed from LDS and the register queues, the loads for the next plane
// (queue entry z+R+1, halo rows, V and x) are in flight.  Two LDS tiles alternate,
// so one barrier per plane suffices.
template <typename T, int R, int SX, bool HASX>
__global__ __launch_bounds__(256) void stencil_zmarch(StArgs g, const T* __restrict__ Y, const T* X, T* Out,
                                                      const T* __restrict__ V, T ca, T cb, T cc,
                                                      double* __restrict__ dot_part) {
  constexpr int TY = 4;
  constexpr int LW = 64 * SX + 2 * R;          // LDS row stride (R zero columns each side)
  constexpr int LR = TY + 2 * R;               // LDS rows
  constexpr int HT = (2 * R + TY - 1) / TY;    // halo rows per wave
  __shared__ T tile[2][LR * LW];
  __shared__ double red[TY];

  const int bid = blockIdx.x;
  const int L = (bid & 7) * g.nb8 + (bid >> 3);
  if (L >= g.nblocks) return;
  const int v = L / g.nslab;
  const int j0 = (L - v * g.nslab) * TY;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ny = g.ny, nz = g.nz;
  const int2* __restrict__ meta = g.meta;
  const long long base = (long long)v * g.ld;
  const T* yv = Y + base;
  const T* xv = HASX ? X + base : nullptr;
  T* ov = Out + base;

  int zb = nz, ze = 0;
  for (int t = 0; t < TY; ++t) {
    const int j = j0 + t;
    if (j < ny) {
      zb = min(zb, g.zrange[2 * j]);
      ze = max(ze, g.zrange[2 * j + 1]);
    }
  }
  if (zb >= ze) {
    if (threadIdx.x == 0) dot_part[L] = 0.0;
    return;
  }
  for (int t = threadIdx.x; t < 2 * LR * LW; t += 256) (&tile[0][0])[t] = T(0);
  __syncthreads();

  auto rowmeta = [&](int j, int z) -> int2 {
    return (j >= 0 && j < ny && z >= 0 && z < nz) ? meta[j + ny * z] : make_int2(0, 0);
  };
  // Row metadata windows: lane l of a window holds meta(j, wb + l), so the
  // per-plane lookups are register reads (readlane) and the addresses of a
  // plane's loads never wait for a metadata load; a window is reloaded once
  // every 64 planes.  Own row: planes z (output) and z + R (queue front).
  struct Win {
    int2 v;
    int wb;
  };
  auto win_load = [&](Win& w, int j, int wb) {
    w.wb = wb;
    w.v = rowmeta(j, wb + lane);
  };
  auto win_at = [&](const Win& w, int z) -> int2 {
    const int l = z - w.wb;
    return make_int2(__builtin_amdgcn_readlane(w.v.x, l), __builtin_amdgcn_readlane(w.v.y, l));
  };
  // tile row of this wavefront's t-th halo row (LR and more: none)
  auto halo = [&](int t) { return wv + TY * t < R ? wv + TY * t : wv + TY * t + TY; };
  Win wown, whalo[HT];
  win_load(wown, j0 + wv, zb - R);
#pragma unroll
  for (int t = 0; t < HT; ++t) win_load(whalo[t], j0 - R + halo(t), zb);

  T q[SX][2 * R + 1], xq[SX], vq[SX], hc[HT][SX] = {};
  T nq[SX], nxv[SX], nv[SX], hn[HT][SX] = {};   // the next plane's
  int2 mcur, mnext;
  // planes zb-R .. zb+R-1
#pragma unroll
  for (int s = 0; s < SX; ++s) q[s][0] = T(0);
#pragma unroll
  for (int dz = 1; dz <= 2 * R; ++dz) {
    const int2 m = win_at(wown, zb - R - 1 + dz);
#pragma unroll
    for (int s = 0; s < SX; ++s) q[s][dz] = meta_val(yv, m, lane + 64 * s);
  }
  auto prefetch = [&](int z) {
    if (z + R >= wown.wb + 64) win_load(wown, j0 + wv, z);
    const int2 mq = win_at(wown, z + R);
    mnext = win_at(wown, z);
    const int lo = mnext.y & 0xffff, hi = mnext.y >> 16;
#pragma unroll
    for (int s = 0; s < SX; ++s) {
      const int i = lane + 64 * s;
      const bool in = i >= lo && i < hi;
      nv[s] = in ? V[mnext.x + i] : T(0);
      nq[s] = meta_val(yv, mq, i);
      nxv[s] = (HASX && in) ? xv[mnext.x + i] : T(0);
    }
#pragma unroll
    for (int t = 0; t < HT; ++t) {
      if (halo(t) >= LR) continue;
      if (z >= whalo[t].wb + 64) win_load(whalo[t], j0 - R + halo(t), z);
      const int2 mh = win_at(whalo[t], z);
#pragma unroll
      for (int s = 0; s < SX; ++s) hn[t][s] = meta_val(yv, mh, lane + 64 * s);
    }
  };
  double dot = 0.0;
  prefetch(zb);
  for (int z = zb; z < ze; ++z) {
    T* tb = tile[(z - zb) & 1];
    mcur = mnext;
#pragma unroll
    for (int s = 0; s < SX; ++s) {
      vq[s] = nv[s];
#pragma unroll
      for (int d = 0; d < 2 * R; ++d) q[s][d] = q[s][d + 1];
      q[s][2 * R] = nq[s];
      xq[s] = nxv[s];
#pragma unroll
      for (int t = 0; t < HT; ++t) hc[t][s] = hn[t][s];
    }
    if (z + 1 < ze) prefetch(z + 1);
#pragma unroll
    for (int s = 0; s < SX; ++s) tb[(wv + R) * LW + R + lane + 64 * s] = q[s][R];
#pragma unroll
    for (int t = 0; t < HT; ++t) {
      if (halo(t) >= LR) continue;
#pragma unroll
      for (int s = 0; s < SX; ++s) tb[halo(t) * LW + R + lane + 64 * s] = hc[t][s];
    }
    lds_barrier();
    const int lo = mcur.y & 0xffff, hi = mcur.y >> 16;
#pragma unroll
    for (int s = 0; s < SX; ++s) {
      const int i = lane + 64 * s;
      // computed on every lane (values outside the domain are zeros), stored inside it
      const T va = ca * vq[s] + cb;
      const T yc = q[s][R];
      T acc = T(g.w[0]) * yc;
      const T* trow = tb + (wv + R) * LW + R + i;
#pragma unroll
      for (int d = 1; d <= R; ++d) {
        const T nb = trow[-d] + trow[d] + trow[-d * LW] + trow[d * LW] + q[s][R - d] + q[s][R + d];
        acc += T(g.w[d]) * nb;
      }
      T o = acc + va * yc;
      if constexpr (HASX) o += cc * xq[s];
      if (i >= lo && i < hi) {
        ov[mcur.x + i] = o;
        dot += (double)o * (double)yc;
      }
    }
  }
  const double s = pc_block_sum(dot, red);
  if (threadIdx.x == 0) dot_part[L] = s;
}

// ---- the windowed z-march (one vector per workgroup, no partial sums) ---------
// A workgroup owns one vector and one window of a slab of win_ty(R, SX) y-rows, one
// wavefront of 64 columns (SX = 1) or two (SX = 2) per row.  A window is all the
// columns that the slab's rows touch, where these are at most 64 SX (the columns
// beyond are zero); else a part of them, with R columns of each neighbouring window
// among its lanes.
// The host lists the windows with the planes they touch.  The march along z:
//   * the z-queue is a ring of QL registers per lane, indexed by the plane's
//     phase; the plane loop is unrolled QL times so the ring turns by renaming
//     instead of register moves (slot (z - zb + R) mod QL holds plane z);
//   * every global access is a raw buffer access on the row's own chord (its begin
//     as the scalar offset, its end as num_records: a lane is in range if its
//     offset is less than their difference): a lane outside the chord, before or
//     after it, has an out-of-range offset, so its load returns 0 and its store is
//     dropped; one vector subtraction per access, no masks and no branches;
//   * a row's begin, end and first column of 64 planes, in bytes, sit in a lane
//     each and are read with v_readlane; the table is padded with empty rows, so
//     nothing is clamped;
//   * X, V and the halo rows of plane z+1 go out before plane z is computed, the
//     queue front of plane z-R+QL right after plane z's last use of slot z-R.
// What bounds it: per row and plane 40 vector, 11 scalar and 10 LDS instructions
// at radius 4 against 5 loads and stores, with one barrier; no unit is busy more
// than half of the time.  Large blocks on a sphere are bound by the fabric: 3.7 GB
// per step for 2.0 GB of Y, X and Out at 605,808 x 275 FP32 (V per vector, and halo
// rows of slabs that march out of phase).  Occupancy is the
// registers': two vectors per workgroup, three register sets or forced occupancy
// were slower, and so were 4, 6 and 16 rows at radius 4 (the halo is 2R rows per
// slab, the barrier is over all its wavefronts) and non-temporal X or stores.
// Row ranges by readlane and buffer ranges instead of scalar arithmetic on a base
// per row (38 scalar instructions): FP32 98 -> 85 us on C10H8.
// One recurrence step; before: one slab and two 64-column chunks of a row in one
// workgroup, masks and tables in vector registers, the windows full or half empty:
//   605,808 points, radius 4 (Si87H76 sphere), 275 vectors:
//                                   FP32 721 -> 680 us, FP64 1508 -> 1250 us
//   C10H8 sphere, radius 4, 49:     FP32 111 -> 80 us,  FP64 260 -> 175 us
//   52^3 cube, radius 4, 23:        FP32 17.2 -> 15.0,  FP64 30.2 -> 22.0 us
//   128^3 sphere r = 60, radius 6:  256 vectors FP32 1310 -> 1165 us,
//                                   64 vectors FP64 640 -> 551 us
//   70^3 cube, 40 vectors:          radius 3 FP32 49 -> 48, radius 2 FP64 87.5 -> 80.5 us
//   52^3 cube, 150 vectors:         radius 1 FP32 52 -> 48, radius 2 FP64 138 -> 126 us
//                                   (55 and 147 us with 8 rows per workgroup)
//   128^3 cube, 23 vectors (SX 2):  radius 4 FP32 147 -> 141, FP64 292 -> 274 us (174
//                                   and 341 us as three windows), radius 6 FP64 338 -> 298
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pc_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T pc_bload(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
  }
}
template <typename T>
__device__ __forceinline__ void pc_bstore(__amdgpu_buffer_rsrc_t r, int off, int soff, T v) {
  if constexpr (sizeof(T) == 4) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, soff, 0);
  } else {
    using V2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, v), r, off, soff, 0);
  }
}

// rows (wavefronts) per workgroup: one halo row per wavefront from radius 4 on
// (radius 1 and 2: half of that, their plane is short against its barrier); two
// wavefronts per row (SX = 2): 16 wavefronts at most
constexpr int win_ty(int R, int SX) { return SX == 2 ? (R == 1 ? 4 : 8) : R <= 2 ? 4 : R <= 4 ? 8 : 2 * R; }
constexpr int win_ns(int R) { return R == 1 ? 3 : 2; }    // register sets of X, V and halo values in flight
// queue length: 2R+1 planes plus 3 fronts in flight, rounded up to a multiple of
// 2 win_ns (tile parity and register sets repeat within the block)
constexpr int win_ql(int R) { return (2 * R + 1 + 3 + 2 * win_ns(R) - 1) / (2 * win_ns(R)) * (2 * win_ns(R)); }
constexpr int kWinPadY = 24;  // empty rows around the padded row table (>= win_ty(R, SX) + R) ...
constexpr int kWinPadZ = 64;  // ... and planes above (>= 2 win_ql(R)); R planes below

struct WinArgs {
  const int4* win;     // {first row, first column | columns << 16 | halo lanes << 28, zb, ze}
  const int2* meta;    // padded row table {offset, lo | length << 16}
  int nyp, nzp;        // its rows and planes
  long long ld;
  int nwin, nzc, zc;   // windows, z-chunks per window and planes per chunk
  int nblocks, nb8;
  double w[8];         // scaled weights; w[0] already includes the factor 3
};

// (two workgroups of 16 wavefronts per CU in FP32: 64 registers at radius 4, which has 65 otherwise)
constexpr int win_occ(int bytes, int R, int SX) { return SX == 2 && bytes == 4 && R <= 4 ? 8 : 1; }

template <typename T, int R, bool HASX, int SX>
__global__ __launch_bounds__(64 * SX * win_ty(R, SX), win_occ(sizeof(T), R, SX))
void stencil_win(WinArgs g, const T* Y, const T* X, T* Out, const T* V, T ca, T cb, T cc) {
  constexpr int TY = win_ty(R, SX), NS = win_ns(R), QL = win_ql(R);
  constexpr int LR = TY + 2 * R;
  constexpr int HT = (2 * R + TY - 1) / TY;   // halo rows per wavefront
  constexpr int ES = (int)sizeof(T);
  constexpr int LW = 64 * SX + 2 * R;    // R zero columns either side
  // row LR takes what wavefronts without a halo row write
  __shared__ T tile[2][(LR + 1) * LW];
  const int L = (blockIdx.x & 7) * g.nb8 + (blockIdx.x >> 3);
  if (L >= g.nblocks) return;
  // workgroup L: vector v, z-chunk zci, window wi (fastest)
  const int per = g.nwin * g.nzc;
  const int v = L / per, zci = (L - v * per) / g.nwin, wi = L - v * per - zci * g.nwin;
  const int4 win = g.win[wi];
  const int zb = win.z + zci * g.zc, ze = min(win.w, zb + g.zc);
  if (zb >= ze) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wv = SX == 2 ? wave >> 1 : wave;                      // row of the slab
  const int col = SX == 2 ? lane + 64 * (wave & 1) : lane;        // column of the window
  const long long base = (long long)v * g.ld;
  const T* __restrict__ yv = Y + base;
  const T* xv = HASX ? X + base : Y + base;
  T* ov = Out + base;
  // win.y: first column | columns << 16 | halo lanes << 28
  const int halo = win.y >> 28, width = win.y >> 16 & 0xfff;
  const int lx = ((win.y & 0xffff) - halo + col) * ES;                         // loads of Y
  const int lo_ = col >= halo && col < halo + width ? lx : 0x40000000;          // X, V and the store: the window's columns
  for (int e = threadIdx.x; e < 2 * (LR + 1) * 2 * R; e += 64 * SX * TY) {
    const int row = e / (2 * R), c = e % (2 * R);
    (&tile[0][0])[row * LW + (c < R ? c : 64 * SX + c)] = T(0);
  }

  // row metadata: lane l holds plane wb + l
  const int jo = win.x + wv + kWinPadY;
  int jh[HT], th[HT];
#pragma unroll
  for (int u = 0; u < HT; ++u) {
    const int k = wv + TY * u;
    th[u] = k < 2 * R ? (k < R ? k : k + TY) : LR;
    jh[u] = k < 2 * R ? win.x - R + th[u] + kWinPadY : 0;                  // (row 0 of the table is empty)
  }
  struct Row { int off, end, lo; };   // in bytes
  auto row_load = [&](int i) -> Row {
    const int2 m = g.meta[i];
    return {m.x * ES, (m.x + (m.y >> 16)) * ES, (m.y & 0xffff) * ES};
  };
  int wb;
  Row wo, wh[HT];
  auto windows = [&](int z) {
    wb = z;
    const int row = min(z + R + lane, g.nzp - 1) * g.nyp;
    wo = row_load(row + jo);
#pragma unroll
    for (int u = 0; u < HT; ++u) wh[u] = row_load(row + jh[u]);
  };
  auto row_of = [&](Row w, int z) -> Row {
    return {__builtin_amdgcn_readlane(w.off, z - wb), __builtin_amdgcn_readlane(w.end, z - wb),
            __builtin_amdgcn_readlane(w.lo, z - wb)};
  };
  auto yload = [&](Row r) -> T { return pc_bload<T>(pc_rsrc(yv, r.end), lx - r.lo, r.off); };

  T q[QL];
  T xq[NS], vq[NS], hq[NS][HT];
  Row ro[NS];
  windows(zb - R);
#pragma unroll
  for (int d = 0; d < QL; ++d) q[d] = yload(row_of(wo, zb - R + d));
  // X, V, halo rows of plane z into set S
  auto issue_plane = [&](auto set, int z) {
    constexpr int S = decltype(set)::value;
    const Row r = row_of(wo, z);
    ro[S] = r;
    const int off = lo_ - r.lo;
    vq[S] = pc_bload<T>(pc_rsrc(V, r.end), off, r.off);
    if constexpr (HASX) xq[S] = pc_bload<T>(pc_rsrc(xv, r.end), off, r.off);
#pragma unroll
    for (int u = 0; u < HT; ++u) hq[S][u] = yload(row_of(wh[u], z));
  };
  pc_unroll_seq(std::make_integer_sequence<int, NS - 1>{}, [&](auto k) {
    constexpr int K = decltype(k)::value;
    issue_plane(std::integral_constant<int, K>{}, zb + K);
  });
  const T w0 = T(g.w[0]);
  T wd[R + 1];
#pragma unroll
  for (int d = 1; d <= R; ++d) wd[d] = T(g.w[d]);

  // Planes run in whole blocks of QL, past ze up to the next multiple of QL:
  // those planes are not stored (their store size is 0; the next z-chunk's
  // workgroup stores them) and what they load is empty or not used.
  auto plane = [&](auto phase, int z) {
    constexpr int P = decltype(phase)::value;
    constexpr int S = P % NS;      // (z - zb) mod NS: the register set of plane z
    constexpr int B = P & 1;       // LDS tile of this plane
    issue_plane(std::integral_constant<int, (P + NS - 1) % NS>{}, z + NS - 1);
    __builtin_amdgcn_sched_barrier(0);
    T* tb = &tile[B][R];
    tb[(wv + R) * LW + col] = q[(P + R) % QL];
#pragma unroll
    for (int u = 0; u < HT; ++u) tb[th[u] * LW + col] = hq[S][u];
    lds_barrier();
    const T* trow = tb + (wv + R) * LW + col;
    const T yc = q[(P + R) % QL];
    T acc = w0 * yc;
#pragma unroll
    for (int d = 1; d <= R; ++d) {
      const T nb = trow[-d] + trow[d] + trow[-d * LW] + trow[d * LW] + q[(P + R - d) % QL] + q[(P + R + d) % QL];
      acc += wd[d] * nb;
      // one distance's LDS reads at a time: all 24 at once cost radius 6 its
      // second workgroup per CU (FP32 1598 -> 1209 us), radius 4 nothing
      if (R > 4 && d < R) __builtin_amdgcn_sched_barrier(0);
    }
    T o = acc + (ca * vq[S] + cb) * yc;
    if constexpr (HASX) o += cc * xq[S];
    const Row r = ro[S];
    pc_bstore<T>(pc_rsrc(ov, z < ze ? r.end : r.off), lo_ - r.lo, r.off, o);
    // slot P (plane z-R) is free: plane z-R+QL, the queue front of plane z-2R+QL
    q[P] = yload(row_of(wo, z - R + QL));
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int z0 = zb; z0 < ze; z0 += QL) {
    if (z0 + 2 * QL > wb + 64) windows(z0);
    pc_unroll_seq(std::make_integer_sequence<int, QL>{}, [&](auto ph) {
      constexpr int P = decltype(ph)::value;
      plane(ph, z0 + P);
    });
  }
}

// z-chunks: a window's z-range is split where that fills the chip better.  The march
// runs whole blocks of win_ql planes, so chunks are multiples of that.  A CU holds
// kSlots workgroups (32 wavefronts in FP32, 16 in FP64 where the registers or the
// bandwidth allow no more; the 12 wavefronts of radius 6 count as 16).  A round of r
// workgroups per CU costs r + kSlots / 4 for each plane, and 2 planes for its start;
// its planes are the mean chunk's, nearer to the longest's the fewer rounds there
// are.  The cheapest cut is taken: 0.8 % slower in the mean than the fastest one over
// 1,417 cubes and spheres of 18 to 128 points, 1 to 200 vectors, both types.  Against
// rounds of the whole chip, counted by planes without the blocks: 64^3, 23 vectors,
// radius 4 FP32 27.4 -> 21 us; 41^3 sphere, 49 vectors, radius 3 FP32 22.5 -> 17,
// FP64 37 -> 27; 5 % in the mean.
template <typename T, int R, int SX>
void win_zchunks(WinArgs& a, const std::vector<WinSplit>& splits, int nvec) {
  constexpr int kSlots = (sizeof(T) == 4 ? 32 : 16) / (SX * (R > 4 ? 16 / SX : win_ty(R, SX)));
  double least = 0.0;
  a.nzc = 0;
  for (const WinSplit& s : splits) {
    const long long per_cu = ((long long)s.wgs * nvec + 255) / 256, rest = per_cu % kSlots;
    const double mean = (double)s.planes / s.wgs, rounds = (double)((per_cu + kSlots - 1) / kSlots);
    const double len = 2.0 + mean + ((double)s.longest - mean) / rounds;
    const double cost = len * (1.25 * (double)(per_cu - rest) + (rest ? (double)rest + 0.25 * kSlots : 0.0));
    if (a.nzc == 0 || cost < least) {
      least = cost;
      a.zc = s.zc;
      a.nzc = s.nzc;
    }
  }
}

template <typename T, int R, int SX>
int launch_win(const GridDev* gd, const T* Y, const T* X, T* Out, const T* V, int nvec, long long ld, double scale,
               double ca, double cb, double cc, hipStream_t st) {
  WinArgs a;
  a.win = gd->win;
  a.nwin = gd->nwin;
  if (a.nwin == 0) return pc::PC_OK;   // no points
  a.meta = gd->pmeta; a.nyp = gd->nyp; a.nzp = gd->nzp;
  a.ld = ld;
  win_zchunks<T, R, SX>(a, gd->splits, nvec);
  for (int d = 0; d < 8; ++d) a.w[d] = 0.0;
  a.w[0] = 3.0 * gd->w[0] * scale;
  for (int d = 1; d <= R; ++d) a.w[d] = gd->w[d] * scale;
  const int per = a.nwin * a.nzc, step = (int)std::max<long long>(1, pc::kMaxGrid / per);   // vectors per launch
  for (int v0 = 0; v0 < nvec; v0 += step) {
    const long long at = (long long)v0 * ld;
    a.nblocks = per * std::min(step, nvec - v0);
    a.nb8 = (a.nblocks + 7) / 8;
    const dim3 grid(8 * a.nb8), block(64 * SX * win_ty(R, SX));
    if (X)
      hipLaunchKernelGGL((stencil_win<T, R, true, SX>), grid, block, 0, st, a, Y + at, X + at, Out + at, V, T(ca), T(cb),
                         T(cc));
    else
      hipLaunchKernelGGL((stencil_win<T, R, false, SX>), grid, block, 0, st, a, Y + at, X, Out + at, V, T(ca), T(cb),
                         T(cc));
    PC_LAUNCH_CHECK();
  }
  return pc::PC_OK;
}

// With per-vector partial sums: one vector and 4 rows (wavefronts) per workgroup.
template <typename T, int R, int SX>
int launch_dot(const GridDev* gd, const T* Y, const T* X, T* Out, const T* V, int nvec, long long ld, double scale,
               double ca, double cb, double cc, double* dot_part, hipStream_t st) {
  StArgs a;
  a.nx = gd->nx; a.ny = gd->ny; a.nz = gd->nz; a.npts = gd->npts;
  a.lo = gd->lo; a.hi = gd->hi; a.off = gd->off; a.zrange = gd->zrange; a.meta = gd->meta;
  a.ld = ld;
  a.nslab = (gd->ny + 3) / 4;
  a.nvec = nvec;
  a.nblocks = a.nslab * nvec;
  a.nb8 = (a.nblocks + 7) / 8;
  for (int d = 0; d < 8; ++d) a.w[d] = 0.0;
  a.w[0] = 3.0 * gd->w[0] * scale;
  for (int d = 1; d <= R; ++d) a.w[d] = gd->w[d] * scale;
  const dim3 grid(8 * a.nb8), block(256);
  if (X)
    hipLaunchKernelGGL((stencil_zmarch<T, R, SX, true>), grid, block, 0, st, a, Y, X, Out, V,
                       T(ca), T(cb), T(cc), dot_part);
  else
    hipLaunchKernelGGL((stencil_zmarch<T, R, SX, false>), grid, block, 0, st, a, Y, X, Out, V,
                       T(ca), T(cb), T(cc), dot_part);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

template <typename T, int R>
int launch_r(const GridDev* gd, const T* Y, const T* X, T* Out, const T* V, int nvec, long long ld, double scale,
             double ca, double cb, double cc, double* dot_part, hipStream_t st) {
  if (!dot_part && gd->winsx == 2) return launch_win<T, R, 2>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, st);
  if (!dot_part) return launch_win<T, R, 1>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, st);
  if (gd->nx <= 64) return launch_dot<T, R, 1>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
  if (gd->nx <= 128) return launch_dot<T, R, 2>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
  return launch_dot<T, R, 4>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
}

template <typename T>
int stencil_dispatch(void* grid, const T* Y, const T* X, T* Out, const T* V, int nvec, long long ld, double scale,
                     double ca, double cb, double cc, double* dot_part, void* stream) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  PC_CHECK_ARG(gd != nullptr, "null grid");
  PC_CHECK_ARG(Y && Out && V, "null operand");
  PC_CHECK_ARG(Y != Out, "output must not alias the stencil input");
  PC_CHECK_ARG(nvec >= 1, "nvec < 1");
  PC_CHECK_ARG(ld >= gd->npts, "ld < npts");
  PC_CHECK_ARG(gd->npts * (long long)sizeof(T) < 0x7ffffff0LL, "vector larger than 2 GiB");
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (gd->radius) {
    case 1: return launch_r<T, 1>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 2: return launch_r<T, 2>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 3: return launch_r<T, 3>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 4: return launch_r<T, 4>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 6: return launch_r<T, 6>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    default:
      pc::set_error("stencil: unsupported radius");
      return pc::PC_ERR_ARG;
  }
}

// Direct form for few vectors (Lanczos, CG): one wave per x-row, neighbours
// read through the caches.  Used where the z-march has too few workgroups.
template <typename T, int R>
__global__ __launch_bounds__(256) void stencil_direct(StArgs g, const T* __restrict__ Y, const T* X, T* Out,
                                                      const T* __restrict__ V, T ca, T cb, T cc,
                                                      double* __restrict__ dot_part) {
  __shared__ double red[4];
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int v = blockIdx.y;
  const int nrow = g.ny * g.nz;
  const T* __restrict__ yv = Y + (long long)v * g.ld;
  const T* xv = X ? X + (long long)v * g.ld : nullptr;
  T* ov = Out + (long long)v * g.ld;
  double dot = 0.0;
  if (row < nrow) {
    const int j = row % g.ny, k = row / g.ny;
    const int lo = g.lo[row], hi = g.hi[row], off = g.off[row];
    for (int i = lo + lane; i < hi; i += 64) {
      const long long p = off + (i - lo);
      const T yc = yv[p];
      T acc = T(g.w[0]) * yc;
#pragma unroll
      for (int d = 1; d <= R; ++d) {
        T nb = row_val(yv, lo, hi, off, i - d) + row_val(yv, lo, hi, off, i + d);
        if (j - d >= 0) {
          const int r2 = row - d;
          nb += row_val(yv, g.lo[r2], g.hi[r2], g.off[r2], i);
        }
        if (j + d < g.ny) {
          const int r2 = row + d;
          nb += row_val(yv, g.lo[r2], g.hi[r2], g.off[r2], i);
        }
        if (k - d >= 0) {
          const int r2 = row - d * g.ny;
          nb += row_val(yv, g.lo[r2], g.hi[r2], g.off[r2], i);
        }
        if (k + d < g.nz) {
          const int r2 = row + d * g.ny;
          nb += row_val(yv, g.lo[r2], g.hi[r2], g.off[r2], i);
        }
        acc += T(g.w[d]) * nb;
      }
      T o = acc + (ca * V[p] + cb) * yc;
      if (xv) o += cc * xv[p];
      ov[p] = o;
      dot += (double)o * (double)yc;
    }
  }
  if (dot_part) {
    const double s = pc_block_sum(dot, red);
    if (threadIdx.x == 0) dot_part[(long long)v * gridDim.x + blockIdx.x] = s;
  }
}

template <typename T, int R>
int launch_direct_r(const GridDev* gd, const T* Y, const T* X, T* Out, const T* V, int nvec, long long ld,
                    double scale, double ca, double cb, double cc, double* dot_part, hipStream_t st) {
  StArgs a;
  a.nx = gd->nx; a.ny = gd->ny; a.nz = gd->nz; a.npts = gd->npts;
  a.lo = gd->lo; a.hi = gd->hi; a.off = gd->off; a.zrange = gd->zrange; a.meta = gd->meta;
  a.ld = ld; a.nslab = 0; a.nvec = nvec; a.nblocks = 0; a.nb8 = 0;
  for (int d = 0; d < 8; ++d) a.w[d] = 0.0;
  a.w[0] = 3.0 * gd->w[0] * scale;
  for (int d = 1; d <= R; ++d) a.w[d] = gd->w[d] * scale;
  const int nrow = gd->ny * gd->nz;
  dim3 grid((nrow + 3) / 4, nvec);
  hipLaunchKernelGGL((stencil_direct<T, R>), grid, dim3(256), 0, st, a, Y, X, Out, V, T(ca), T(cb), T(cc), dot_part);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

// One FP64 vector (the Lanczos bounds): the pass of the CG step (pc_zmarch.h),
// so each point's neighbours come from registers and LDS instead of dependent
// row-table loads.  Out may alias X.
struct SinglePass {
  struct Raw { double y; };
  struct Ext { double v, x; };
  static constexpr bool DOT = false, POST = false;
  const double* __restrict__ Y;
  const double* X;
  double* Out;
  const double* __restrict__ V;
  double ca, cb, cc;
  __device__ __forceinline__ Raw load(long long idx, bool, int, int, int) const { return {Y[idx]}; }
  __device__ __forceinline__ Ext ext(long long idx) const { return {V[idx], X ? X[idx] : 0.0}; }
  __device__ __forceinline__ bool pre() const { return true; }
  __device__ __forceinline__ double comb(Raw r) const { return r.y; }
  __device__ __forceinline__ void out(bool in, long long idx, Raw, Ext e, double qc, double acc, double&,
                                      double&) const {
    double o = acc + (ca * e.v + cb) * qc;
    if (X) o += cc * e.x;
    if (in) Out[idx] = o;
  }
};

template <int R, int SX>
__global__ __launch_bounds__(pcz::threads(SX), SX == 2 && R <= 4 ? 4 : 2) void stencil_single(pcz::ZMap zm, SinglePass p) {
  __shared__ double tile[pcz::Tile<R, SX>::SIZE];
  const int L = pcz::block_of(zm);
  if (L >= zm.nwg) return;
  double s;
  pcz::zpass<R, SX, pcz::kZW, false, false, false>(zm, L, tile, p, s);
}

template <int R>
int launch_single_r(const pcz::ZMap& zm, const double* Y, const double* X, double* Out, const double* V, double ca,
                    double cb, double cc, hipStream_t st) {
  const dim3 grid(8 * zm.nwg8), block(pcz::threads(zm.sx));
  const SinglePass p{Y, X, Out, V, ca, cb, cc};
  switch (zm.sx) {
    case 1: hipLaunchKernelGGL((stencil_single<R, 1>), grid, block, 0, st, zm, p); break;
    case 2: hipLaunchKernelGGL((stencil_single<R, 2>), grid, block, 0, st, zm, p); break;
    default: hipLaunchKernelGGL((stencil_single<R, 4>), grid, block, 0, st, zm, p); break;
  }
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

// Measured on the C10H8 sphere (394,264 points, radius 4): one FP64 vector 12.2
// us (17.0 us marching with one plane of loads in flight; on Si87H76's 605,808
// points that was 17 us, stencil_direct 46 us; the same bits).
int single_dispatch(void* grid, const double* Y, const double* X, double* Out, const double* V, double scale,
                    double ca, double cb, double cc, hipStream_t st, bool* done) {
  *done = false;
  const GridDev* gd = static_cast<const GridDev*>(grid);
  double w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  w[0] = 3.0 * gd->w[0] * scale;
  for (int d = 1; d <= gd->radius && d < 8; ++d) w[d] = gd->w[d] * scale;
  pcz::ZMap zm;
  int radius = 0;
  if (pcz::zmap_init(grid, w, zm, &radius) != 0) return pc::PC_OK;   // nx > 256: direct form
  int rc = pc::PC_OK;
  switch (radius) {
    case 1: rc = launch_single_r<1>(zm, Y, X, Out, V, ca, cb, cc, st); break;
    case 2: rc = launch_single_r<2>(zm, Y, X, Out, V, ca, cb, cc, st); break;
    case 3: rc = launch_single_r<3>(zm, Y, X, Out, V, ca, cb, cc, st); break;
    case 4: rc = launch_single_r<4>(zm, Y, X, Out, V, ca, cb, cc, st); break;
    case 6: rc = launch_single_r<6>(zm, Y, X, Out, V, ca, cb, cc, st); break;
    default: return pc::PC_OK;
  }
  *done = rc == pc::PC_OK;
  return rc;
}

template <typename T>
int direct_dispatch(void* grid, const T* Y, const T* X, T* Out, const T* V, int nvec, long long ld, double scale,
                    double ca, double cb, double cc, double* dot_part, void* stream) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  PC_CHECK_ARG(gd != nullptr, "null grid");
  PC_CHECK_ARG(Y && Out && V, "null operand");
  PC_CHECK_ARG(Y != Out, "output must not alias the stencil input");
  PC_CHECK_ARG(nvec >= 1 && nvec <= 65535, "nvec out of range");
  PC_CHECK_ARG(ld >= gd->npts, "ld < npts");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if constexpr (std::is_same<T, double>::value) {
    if (nvec == 1 && dot_part == nullptr) {
      bool done = false;
      const int rc = single_dispatch(grid, Y, X, Out, V, scale, ca, cb, cc, st, &done);
      if (rc != pc::PC_OK || done) return rc;
    }
  }
  switch (gd->radius) {
    case 1: return launch_direct_r<T, 1>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 2: return launch_direct_r<T, 2>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 3: return launch_direct_r<T, 3>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 4: return launch_direct_r<T, 4>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    case 6: return launch_direct_r<T, 6>(gd, Y, X, Out, V, nvec, ld, scale, ca, cb, cc, dot_part, st);
    default:
      pc::set_error("stencil: unsupported radius");
      return pc::PC_ERR_ARG;
  }
}

}  // namespace

// Used by the CG solver in pc_pcg.hip.
int pc_internal_stencil_direct_f64(void* grid, const double* Y, const double* X, double* Out, const double* V,
                                   double scale, double ca, double cb, double cc, double* dot_part, void* stream,
                                   int* out_nblocks) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  if (out_nblocks) *out_nblocks = (gd->ny * gd->nz + 3) / 4;
  return direct_dispatch<double>(grid, Y, X, Out, V, 1, gd->npts, scale, ca, cb, cc, dot_part, stream);
}

long long pc_internal_grid_npts(void* grid) { return static_cast<const GridDev*>(grid)->npts; }
int pc_internal_grid_view(void* grid, int* nx, int* ny, int* nz, const int** lo, const int** hi, const int** off) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  *nx = gd->nx; *ny = gd->ny; *nz = gd->nz;
  *lo = gd->lo; *hi = gd->hi; *off = gd->off;
  return 0;
}
// Point map for single-vector kernels (the Hartree CG): row metadata
// {off-lo, lo|hi<<16}, the row of every point, and the unscaled weights.
int pc_internal_grid_points(void* grid, int* ny, int* nz, int* radius, const int2** meta, const int** prow,
                            double* w8) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  *ny = gd->ny; *nz = gd->nz; *radius = gd->radius;
  *meta = gd->meta; *prow = gd->prow;
  for (int d = 0; d < 8; ++d) w8[d] = gd->w[d];
  return 0;
}
// z-extent per y (min z, max z + 1 of the non-empty rows) and nx, for z-marching kernels
int pc_internal_grid_zmap(void* grid, int* nx, const int** zrange) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  *nx = gd->nx;
  *zrange = gd->zrange;
  return 0;
}
long long pc_internal_grid_nrow(void* grid) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  return (long long)gd->ny * gd->nz;
}

extern "C" {

int pc_stencil_direct_f64(void* grid, const double* Y, const double* X, double* Out, const double* V, int nvec,
                          long long ld, double scale, double a, double b, double c, double* dot_part, void* stream) {
  return direct_dispatch<double>(grid, Y, X, Out, V, nvec, ld, scale, a, b, c, dot_part, stream);
}

int pc_stencil_direct_f32(void* grid, const float* Y, const float* X, float* Out, const float* V, int nvec,
                          long long ld, double scale, double a, double b, double c, double* dot_part, void* stream) {
  return direct_dispatch<float>(grid, Y, X, Out, V, nvec, ld, scale, a, b, c, dot_part, stream);
}

int pc_grid_create(int nx, int ny, int nz, const int* row_lo, const int* row_hi, int radius, const double* weights,
                   void** out_grid, long long* out_npts) {
  PC_CHECK_ARG(out_grid && row_lo && row_hi && weights, "null pointer");
  PC_CHECK_ARG(nx >= 1 && ny >= 1 && nz >= 1, "bad dims");
  PC_CHECK_ARG(nx <= 256, "nx > 256 not supported (x rows are held by one workgroup)");
  PC_CHECK_ARG(radius == 1 || radius == 2 || radius == 3 || radius == 4 || radius == 6,
               "radius must be 1,2,3,4 or 6");
  const int nrow = ny * nz;
  std::vector<int> off(nrow), zr(2 * ny);
  for (int j = 0; j < ny; ++j) { zr[2 * j] = nz; zr[2 * j + 1] = 0; }
  long long cnt = 0;
  for (int k = 0; k < nz; ++k)
    for (int j = 0; j < ny; ++j) {
      const int r = j + ny * k;
      PC_CHECK_ARG(row_lo[r] >= 0 && row_hi[r] <= nx, "row extent outside [0,nx]");
      off[r] = (int)cnt;
      const int len = std::max(0, row_hi[r] - row_lo[r]);
      if (len > 0) {
        zr[2 * j] = std::min(zr[2 * j], k);
        zr[2 * j + 1] = std::max(zr[2 * j + 1], k + 1);
      }
      cnt += len;
    }
  PC_CHECK_ARG(cnt < (1LL << 31), "too many points");
  // normalise empty rows to lo=hi=0
  std::vector<int> lo(row_lo, row_lo + nrow), hi(row_hi, row_hi + nrow);
  for (int r = 0; r < nrow; ++r)
    if (hi[r] <= lo[r]) { lo[r] = 0; hi[r] = 0; }
  std::vector<int2> meta(nrow);
  for (int r = 0; r < nrow; ++r) meta[r] = make_int2(off[r] - lo[r], lo[r] | (hi[r] << 16));
  GridDev* g = new GridDev();
  g->nx = nx; g->ny = ny; g->nz = nz; g->npts = cnt; g->radius = radius;
  // stencil_win: per slab of rows the columns they touch, as one window of up to
  // 64 sx or as windows of equal lane counts (an inner edge has radius halo lanes,
  // an outer one none), with the planes they touch; lanes: those of all planes
  int most = 0;   // windows of one slab
  auto windows = [&](int sx, std::vector<int4>& win) {
    long long lanes_all = 0;
    const int ty = win_ty(radius, sx), lw = 64 * sx;
    for (int j0 = 0; j0 < ny; j0 += ty) {
      int xl = nx, xh = 0;
      const int j1 = std::min(ny, j0 + ty);
      for (int j = j0; j < j1; ++j)
        for (int k = zr[2 * j]; k < zr[2 * j + 1]; ++k)
          if (hi[j + ny * k] > lo[j + ny * k]) {
            xl = std::min(xl, lo[j + ny * k]);
            xh = std::max(xh, hi[j + ny * k]);
          }
      if (xl >= xh) continue;
      int n = 1;
      while (xh - xl + 2 * radius * (n - 1) > lw * n) ++n;
      most = std::max(most, n);
      const int lanes = xh - xl + 2 * radius * (n - 1);
      auto cut = [&](int i) { return i == 0 ? xl : i == n ? xh : xl + lanes * i / n - radius * (2 * i - 1); };
      for (int i = 0; i < n; ++i) {
        const int x0 = cut(i), x1 = cut(i + 1);
        int zb = nz, ze = 0;
        for (int j = j0; j < j1; ++j)
          for (int k = zr[2 * j]; k < zr[2 * j + 1]; ++k)
            if (std::max(lo[j + ny * k], x0) < std::min(hi[j + ny * k], x1)) {
              zb = std::min(zb, k);
              ze = std::max(ze, k + 1);
            }
        if (zb >= ze) continue;
        win.push_back(make_int4(j0, x0 | ((x1 - x0) << 16) | ((i ? radius : 0) << 28), zb, ze));
        lanes_all += (long long)(ze - zb) * lw * ty;
      }
    }
    return lanes_all;
  };
  std::vector<int4> win, win2;
  g->winsx = 1;
  const long long lanes1 = windows(1, win);
  // Two wavefronts per row share one tile, so a row of up to 128 columns has no
  // inner edges: taken where that saves a fifth of the lanes (121 to 128 full
  // columns at radius 4, which are three windows otherwise: 128^3, 23 vectors,
  // FP64 341 -> 280 us, radius 6 361 -> 298), and where it costs none at radius 1
  // (126^3, 49 vectors FP32 289 -> 263) and up to radius 4 on rows that are full to
  // seven eighths (120^3, 23 vectors FP32 radius 2 130 -> 107, 3 130 -> 114, 4 129 ->
  // 117 us; 112 columns gain nothing at radius 3 and 4).  Elsewhere, with two windows
  // either way, one wavefront per row is the faster (100^3 radius 4 3 to 15 %,
  // spheres 5 to 40 %).
  const bool full = radius <= 4 && 8 * cnt > 7 * 128LL * ny * nz;
  if (nx > 64 && nx <= 128 && most >= (radius == 1 || full ? 2 : 3)) {
    const long long lanes2 = windows(2, win2);
    if (radius == 1 || full ? lanes2 <= lanes1 : 5 * lanes2 <= 4 * lanes1) {
      g->winsx = 2;
      win.swap(win2);
    }
  }
  // the longest first: what runs last is short
  std::stable_sort(win.begin(), win.end(), [](const int4& x, const int4& y) { return x.w - x.z > y.w - y.z; });
  g->nwin = (int)win.size();
  const int ql = win_ql(radius), blocks = win.empty() ? 0 : (win[0].w - win[0].z + ql - 1) / ql;
  for (int n = 1, last = 0; n <= std::min(blocks, 256); ++n) {   // n chunks of about equal numbers b of blocks
    const int b = (blocks + n - 1) / n;
    if (b == last) continue;
    last = b;
    WinSplit s{b * ql, (blocks + b - 1) / b, 0, 0, b * ql};
    for (const int4& w : win) {
      const int n = (w.w - w.z + ql - 1) / ql;
      s.wgs += (n + b - 1) / b;
      s.planes += (long long)n * ql;
    }
    g->splits.push_back(s);
  }
  g->nyp = ny + 2 * kWinPadY;
  g->nzp = nz + radius + kWinPadZ;
  std::vector<int2> pmeta((size_t)g->nyp * g->nzp, make_int2(0, 0));
  for (int k = 0; k < nz; ++k)
    for (int j = 0; j < ny; ++j) {
      const int r = j + ny * k;
      pmeta[(size_t)(k + radius) * g->nyp + j + kWinPadY] = make_int2(off[r], lo[r] | ((hi[r] - lo[r]) << 16));
    }
  for (int d = 0; d < 8; ++d) g->w[d] = d <= radius ? weights[d] : 0.0;
  std::vector<int> prow((size_t)std::max(cnt, 1LL));
  for (int r = 0; r < nrow; ++r)
    for (int t = 0; t < hi[r] - lo[r]; ++t) prow[(size_t)off[r] + t] = r;
  // all tables in one allocation, filled by one copy (each costs some 0.1 ms)
  struct Part { void** dst; const void* src; size_t bytes, at; };
  Part parts[] = {{(void**)&g->lo, lo.data(), nrow * sizeof(int), 0},
                  {(void**)&g->hi, hi.data(), nrow * sizeof(int), 0},
                  {(void**)&g->off, off.data(), nrow * sizeof(int), 0},
                  {(void**)&g->zrange, zr.data(), 2 * ny * sizeof(int), 0},
                  {(void**)&g->meta, meta.data(), nrow * sizeof(int2), 0},
                  {(void**)&g->prow, prow.data(), prow.size() * sizeof(int), 0},
                  {(void**)&g->win, win.data(), win.size() * sizeof(int4), 0},
                  {(void**)&g->pmeta, pmeta.data(), pmeta.size() * sizeof(int2), 0}};
  size_t total = 0;
  for (Part& t : parts) {
    t.at = total;
    total += (t.bytes + 255) / 256 * 256 + 256;
  }
  std::vector<char> host(total);
  for (const Part& t : parts)
    if (t.bytes) std::memcpy(host.data() + t.at, t.src, t.bytes);
  hipError_t e = hipMalloc(&g->tables, total);
  if (e == hipSuccess) {
    for (const Part& t : parts) *t.dst = static_cast<char*>(g->tables) + t.at;
    e = hipMemcpy(g->tables, host.data(), total, hipMemcpyHostToDevice);
    if (e != hipSuccess) (void)hipFree(g->tables);
  }
  if (e != hipSuccess) {
    delete g;
    pc::set_error(std::string("pc_grid_create: ") + hipGetErrorString(e));
    return pc::PC_ERR_HIP;
  }
  *out_grid = g;
  if (out_npts) *out_npts = cnt;
  return pc::PC_OK;
}

int pc_grid_destroy(void* grid) {
  GridDev* g = static_cast<GridDev*>(grid);
  if (!g) return pc::PC_OK;
  (void)hipFree(g->tables);
  delete g;
  return pc::PC_OK;
}

// Kept for its callers: one kernel serves every block now, so the value has no effect.
int pc_stencil_set_variant(int variant) {
  PC_CHECK_ARG(variant >= 0 && variant <= 2, "variant must be 0, 1 or 2");
  (void)variant;
  return pc::PC_OK;
}

int pc_stencil_f64(void* grid, const double* Y, const double* X, double* Out, const double* V, int nvec,
                   long long ld, double scale, double a, double b, double c, double* dot_part, void* stream) {
  return stencil_dispatch<double>(grid, Y, X, Out, V, nvec, ld, scale, a, b, c, dot_part, stream);
}

int pc_stencil_f32(void* grid, const float* Y, const float* X, float* Out, const float* V, int nvec,
                   long long ld, double scale, double a, double b, double c, double* dot_part, void* stream) {
  return stencil_dispatch<float>(grid, Y, X, Out, V, nvec, ld, scale, a, b, c, dot_part, stream);
}

// Number of per-workgroup partial sums pc_stencil_* writes when dot_part is
// given (padded layout: entry L of the logical workgroup order, vector-major).
int pc_stencil_num_partials(void* grid, int dtype_bytes, int nvec, int* out_count, int* out_per_vector) {
  const GridDev* gd = static_cast<const GridDev*>(grid);
  PC_CHECK_ARG(gd && out_count && out_per_vector, "null pointer");
  PC_CHECK_ARG(dtype_bytes == 4 || dtype_bytes == 8, "dtype_bytes must be 4 or 8");
  // with partial sums: one vector and one y-row per wavefront, 4 rows per workgroup
  const int nslab = (gd->ny + 3) / 4;
  *out_per_vector = nslab;
  *out_count = nslab * nvec;
  return pc::PC_OK;
}

}  // extern "C"
