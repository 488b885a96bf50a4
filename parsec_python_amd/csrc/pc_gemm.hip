// Rayleigh-Ritz block GEMMs on MFMA (gfx950).
//
//   gram  : S = X^T Y        X: n x kx, Y: n x ky (vector-major, ld), S FP64 kx x ky
//   rotate: Z = X Q          X: n x kx, Q: FP64 kx x ky (column-major), Z: n x ky
//
// The reference forms G = W^T (H W) with a Python double loop of vdot
// (src/Eigensolvers/chefsi1.py:51-53) or cuBLAS (chefsi1_gpu.py:61) and
// rotates with W @ Q (chefsi1.py:67, chefsi1_gpu.py:66).
//
// MFMA 16x16x4 (f64: v_mfma_f64_16x16x4f64, f32: v_mfma_f32_16x16x4f32) lane
// layout on gfx950 (measured with one-hot operands): A[m][k] from lane m + 16k,
// B[k][n] from lane n + 16k; D[m][n] in lane n + 16*(m/4), register m%4 for
// f32, and in lane n + 16*(m%4), register m/4 for f64.  The K index of an operand is only a label
// that A and B must share, so each lane loads 4 consecutive points (one
// 16-byte/32-byte load) and step s of 4 uses point 4*(lane/16)+s.
//
// gram splits the n points into chunks; each workgroup accumulates one output
// tile over one chunk (FP64 MFMA, or FP32 MFMA per 16 points flushed into FP64
// registers) and writes an FP64 partial; a second kernel sums the partials in a
// fixed order (deterministic).
#include "pc_common.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename T> struct Acc;
template <> struct Acc<double> {
  typedef v4d type;
  static __device__ __forceinline__ v4d mfma(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // output row of register r in lane group lk (= lane/16)
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * r + lk; }
};
template <> struct Acc<float> {
  typedef v4f type;
  static __device__ __forceinline__ v4f mfma(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

// Load 4 consecutive points [p, p+4) of column col; zero beyond n.
template <typename T>
__device__ __forceinline__ void load4(const T* __restrict__ base, long long ld, int col, int ncol, long long p,
                                      long long n, T out[4]) {
  if (col < ncol) {
    const T* src = base + (long long)col * ld + p;
#pragma unroll
    for (int s = 0; s < 4; ++s) out[s] = (p + s < n) ? src[s] : T(0);
    return;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) out[s] = T(0);
}

// ---------------------------------------------------------------- gram
// Tile t -> (ti, tj): row-major over ti_n x tj_n, or the upper triangle
// (ti <= tj) row by row when sym.
__device__ __forceinline__ void tile_coords(int t, int ti_n, int tj_n, int sym, int& ti, int& tj) {
  if (!sym) {
    ti = t / tj_n;
    tj = t - ti * tj_n;
    return;
  }
  int i = 0;
  while (t >= ti_n - i) {
    t -= ti_n - i;
    ++i;
  }
  ti = i;
  tj = i + t;
}

// Any alignment: workgroup = 4 waves, output tile 64x64 (each wave 32x32 = 2x2 MFMA tiles).
template <typename T>
__global__ __launch_bounds__(256) void gram_kernel(const T* __restrict__ X, long long ldx, const T* __restrict__ Y,
                                                   long long ldy, long long n, int kx, int ky, int ti_n, int tj_n,
                                                   int ntile, int sym, int nchunk, long long chunk,
                                                   double* __restrict__ part) {
  typedef typename Acc<T>::type AT;
  const int b = blockIdx.x;
  const int tile = b % ntile;
  const int ch = b / ntile;
  int ti, tj;
  tile_coords(tile, ti_n, tj_n, sym, ti, tj);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wi = w >> 1, wj = w & 1;
  const int i0 = ti * 64 + wi * 32, j0 = tj * 64 + wj * 32;
  const int lm = lane & 15, lk = lane >> 4;
  // FP32 inputs: the MFMA accumulates 16 points in FP32, then the block is
  // added into FP64 accumulators (products of FP32 values are exact in FP64,
  // so the only FP32 rounding is within one 16-term block).
  AT acc[2][2];
  double acc64[2][2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      acc[a][c] = AT{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) acc64[a][c][r] = 0.0;
    }
  const long long pbeg = (long long)ch * chunk;
  const long long pend = min(n, pbeg + chunk);
  for (long long p = pbeg; p < pend; p += 16) {
    T a[2][4], bb[2][4];
    const long long pl = p + 4 * lk;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      load4<T>(X, ldx, i0 + 16 * t + lm, kx, pl, pend, a[t]);
      load4<T>(Y, ldy, j0 + 16 * t + lm, ky, pl, pend, bb[t]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int ta = 0; ta < 2; ++ta)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) acc[ta][tb] = Acc<T>::mfma(a[ta][s], bb[tb][s], acc[ta][tb]);
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int ta = 0; ta < 2; ++ta)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc64[ta][tb][r] += (double)acc[ta][tb][r];
          acc[ta][tb] = AT{0, 0, 0, 0};
        }
    }
  }
  // partial layout: part[(ch*ntile + tile)*4096 + jj*64 + ii], tile-local 64x64 col-major
  double* out = part + ((long long)ch * ntile + tile) * 4096;
#pragma unroll
  for (int ta = 0; ta < 2; ++ta)
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ii = wi * 32 + 16 * ta + Acc<T>::row(lk, r);
        const int jj = wj * 32 + 16 * tb + lm;
        out[jj * 64 + ii] = (sizeof(T) == 4) ? acc64[ta][tb][r] : (double)acc[ta][tb][r];
      }
}

// Aligned operands: output tile 32 NT x 32 NT per workgroup (2 x 2 waves of
// NT x NT MFMA tiles).  Per stage of 128 bytes of points (32 FP32, 16 FP64)
// the workgroup loads its X and Y columns once, 16 bytes per lane and 128
// contiguous bytes per column, into one of two LDS buffers; the next stage's
// loads are in flight while the MFMAs run, one barrier per stage.  Columns past
// the edge are loaded from the last column (their products only reach outputs
// that gram_reduce skips), so the stage loop has no branches; only the last
// chunk's last stage checks its points.  FP32: 16 points accumulate in the MFMA
// from zero and are added to the FP64 accumulators while the next 16 run.
// Bound by the MFMA rate once the operand strips stay on chip: consecutive
// workgroups of one XCD take the tiles of one chunk, so its L2 serves the
// columns to all of them (with the tiles dealt over the XCDs every L2 fetched
// every column), and 96-wide tiles read each column a third less often than
// 64-wide ones and pad 275 columns to 288, not 320.  FP32 MFMA and VALU do not
// overlap on this chip (measured: 9 MFMAs and 16 FP64 additions take the sum of
// their times), so the FP64 flush costs a fifth.  605,808 x 275, symmetric and
// full: FP32 668 and 1027 us (803 and 1338 us with 64-wide tiles, every column
// staged once per tile), FP64 1134 and 1701 us = 64 TF/s on the padded product
// (2081 and 3987 us with operands loaded by each wave).
constexpr int kGramStage = 128;   // bytes of one column per stage

template <typename T, int NT>
__global__ __launch_bounds__(256, 2) void gram_tile(const T* __restrict__ X, long long ldx, const T* __restrict__ Y,
                                                    long long ldy, long long n, int kx, int ky, int ti_n, int tj_n,
                                                    int ntile, int sym, int nblocks, int nb8, long long chunk,
                                                    double* __restrict__ part) {
  typedef typename Acc<T>::type AT;
  constexpr int W = 32 * NT;
  constexpr int SP = kGramStage / (int)sizeof(T);   // points per stage
  constexpr int E = 16 / (int)sizeof(T);            // values per 16-byte load
  constexpr int LS = SP + E;                        // LDS row stride (16 bytes of skew)
  constexpr int G = SP / 16;                        // 16-point groups per stage
  typedef T VT __attribute__((ext_vector_type(E)));
  __shared__ __align__(16) T xs[2][W * LS], ys[2][W * LS];
  const int L = (blockIdx.x & 7) * nb8 + (blockIdx.x >> 3);
  if (L >= nblocks) return;
  const int ch = L / ntile;
  int ti, tj;
  tile_coords(L - ch * ntile, ti_n, tj_n, sym, ti, tj);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wi = w >> 1, wj = w & 1;
  const int lm = lane & 15, lk = lane >> 4;
  const int seg = E * (threadIdx.x & 7);
  double* out = part + (long long)L * (W * W);
  // points [pbeg, pend): whole stages, or (EDGE) one stage with some points missing
  auto body = [&](auto edge, long long pbeg, long long pend) {
    constexpr bool EDGE = decltype(edge)::value;
    const T *xp[NT], *yp[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = (threadIdx.x >> 3) + 32 * t;
      xp[t] = X + (long long)min(ti * W + c, kx - 1) * ldx + seg;
      yp[t] = Y + (long long)min(tj * W + c, ky - 1) * ldy + seg;
    }
    VT gx[NT], gy[NT];
    auto gload = [&](long long p) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if constexpr (EDGE) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const bool in = p + seg + e < pend;
            gx[t][e] = in ? xp[t][p + e] : T(0);
            gy[t][e] = in ? yp[t][p + e] : T(0);
          }
        } else {
          gx[t] = *reinterpret_cast<const VT*>(xp[t] + p);
          gy[t] = *reinterpret_cast<const VT*>(yp[t] + p);
        }
      }
    };
    auto sstore = [&](int bf) {
      const int o = (threadIdx.x >> 3) * LS + seg;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        *reinterpret_cast<VT*>(&xs[bf][o + 32 * t * LS]) = gx[t];
        *reinterpret_cast<VT*>(&ys[bf][o + 32 * t * LS]) = gy[t];
      }
    };
    AT acc[NT][NT];
    double acc64[NT][NT][4];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        acc[a][c] = AT{0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < 4; ++r) acc64[a][c][r] = 0.0;
      }
    auto flush = [&]() {
      if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
          for (int c = 0; c < NT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc64[a][c][r] += (double)acc[a][c][r];
      }
    };
    gload(pbeg);
    sstore(0);
    __syncthreads();
    int bf = 0;
    for (long long p = pbeg; p < pend; p += SP) {
      if constexpr (!EDGE) gload(min(p + SP, pend - SP));   // (the last stage re-reads itself)
      __builtin_amdgcn_sched_barrier(0);   // or the loads are sunk to their uses
      const T* xb = &xs[bf][(wi * 16 * NT + lm) * LS + 4 * lk];
      const T* yb = &ys[bf][(wj * 16 * NT + lm) * LS + 4 * lk];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        T a[NT][4], b[NT][4];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int h = 0; h < 4 / E; ++h) {
            const VT av = *reinterpret_cast<const VT*>(xb + 16 * t * LS + 16 * g + E * h);
            const VT bv = *reinterpret_cast<const VT*>(yb + 16 * t * LS + 16 * g + E * h);
#pragma unroll
            for (int e = 0; e < E; ++e) {
              a[t][E * h + e] = av[e];
              b[t][E * h + e] = bv[e];
            }
          }
        flush();   // the previous 16 points
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int ta = 0; ta < NT; ++ta)
#pragma unroll
            for (int tb = 0; tb < NT; ++tb) {
              const AT c0 = (sizeof(T) == 4 && s == 0) ? AT{0, 0, 0, 0} : acc[ta][tb];
              acc[ta][tb] = Acc<T>::mfma(a[ta][s], b[tb][s], c0);
            }
      }
      bf ^= 1;
      if constexpr (!EDGE) sstore(bf);
      __syncthreads();
    }
    flush();
#pragma unroll
    for (int ta = 0; ta < NT; ++ta)
#pragma unroll
      for (int tb = 0; tb < NT; ++tb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int ii = (wi * NT + ta) * 16 + Acc<T>::row(lk, r);
          const int jj = (wj * NT + tb) * 16 + lm;
          out[jj * W + ii] = (sizeof(T) == 4) ? acc64[ta][tb][r] : (double)acc[ta][tb][r];
        }
  };
  // chunk 0 is the last n % SP points when there are any, the others are whole stages
  const long long nw = n / SP * SP;
  if (nw < n && ch == 0) {
    body(std::true_type{}, nw, n);
  } else {
    const long long pbeg = (long long)(ch - (nw < n ? 1 : 0)) * chunk;
    body(std::false_type{}, pbeg, min(nw, pbeg + chunk));
  }
}

// Sum of the chunk partials of a W x W tile (W a multiple of 32): a workgroup
// takes 32 consecutive elements, 8 threads each; thread g of an element adds
// the chunks g, g + 8, ... in order and the 8 sums are added in order
// (deterministic).  With one thread per element the chunks of a single-tile
// Gram matrix were one serial chain (23 us at 385 chunks).
// With at most 8 chunks (ONE) one thread per element adds them in order: the same
// sums from an eighth of the threads.
template <bool ONE>
__global__ __launch_bounds__(256) void gram_reduce(const double* __restrict__ part, int W, int ntile, int nchunk,
                                                   int ti_n, int tj_n, int kx, int ky, double* __restrict__ S,
                                                   long long lds, int sym) {
  __shared__ double red[8][32];
  constexpr int E = ONE ? 256 : 32;   // elements per workgroup
  const int per = W * W / E;
  const int tile = blockIdx.x / per;
  int ti, tj;
  tile_coords(tile, ti_n, tj_n, sym, ti, tj);
  const int el = threadIdx.x & (E - 1), g = threadIdx.x / E;
  const int e = (blockIdx.x - tile * per) * E + el;
  const int jj = e / W, ii = e - jj * W;
  const int i = ti * W + ii, j = tj * W + jj;
  const bool in = i < kx && j < ky;
  double s = 0.0;
  if (in) {
    const double* p = part + (long long)tile * W * W + e;
    const long long st = (long long)ntile * W * W;
#pragma unroll 8
    for (int c = g; c < nchunk; c += ONE ? 1 : 8) s += p[c * st];
  }
  if constexpr (!ONE) {
    red[g][el] = s;
    __syncthreads();
  }
  if (g == 0 && in) {
    double t = s;
    if constexpr (!ONE) {
#pragma unroll
      for (int q = 1; q < 8; ++q) t += red[q][el];
    }
    S[(long long)j * lds + i] = t;
    if (sym && ti != tj) S[(long long)i * lds + j] = t;
  }
}

// ---------------------------------------------------------------- rotate
// Z^T (ky x n) = Q^T (ky x kx) * X^T (kx x n).  Workgroup = 4 waves; wave tile
// = 64 output columns x 32 points (4x2 MFMA tiles); workgroup = 64 cols x 128 pts.
template <typename T>
__global__ __launch_bounds__(256) void rotate_kernel(const T* __restrict__ X, long long ldx,
                                                     const T* __restrict__ Q, int ldq, T* __restrict__ Z,
                                                     long long ldz, long long n, int kx, int ky, int npt_tiles,
                                                     int ncol_tiles, int nblocks, int nb8) {
  typedef typename Acc<T>::type AT;
  const int L = (blockIdx.x & 7) * nb8 + (blockIdx.x >> 3);
  if (L >= nblocks) return;
  const int ct = L % ncol_tiles;
  const int pt = L / ncol_tiles;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lm = lane & 15, lk = lane >> 4;
  const int c0 = ct * 64;
  const long long p0 = (long long)pt * 128 + w * 32;
  AT acc[4][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[a][c] = AT{0, 0, 0, 0};
  for (int k = 0; k < kx; k += 4) {
    const int kk = k + lk;
    T qa[4], xb[2];
#pragma unroll
    for (int ta = 0; ta < 4; ++ta) {
      const int col = c0 + 16 * ta + lm;
      qa[ta] = (kk < kx && col < ky) ? Q[(long long)kk * ldq + col] : T(0);
    }
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const long long p = p0 + 16 * tb + lm;
      xb[tb] = (kk < kx && p < n) ? X[(long long)kk * ldx + p] : T(0);
    }
#pragma unroll
    for (int ta = 0; ta < 4; ++ta)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) acc[ta][tb] = Acc<T>::mfma(qa[ta], xb[tb], acc[ta][tb]);
  }
#pragma unroll
  for (int ta = 0; ta < 4; ++ta)
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = c0 + 16 * ta + Acc<T>::row(lk, r);
        const long long p = p0 + 16 * tb + lm;
        if (col < ky && p < n) Z[(long long)col * ldz + p] = acc[ta][tb][r];
      }
}

// Aligned operands: up to 288 output columns in one workgroup, so X is read
// from memory once.  Waves (pw, cw) = (point half, column half) of 32 E points x
// 32 NCH columns, E = 16 / sizeof(T) points per lane: a wave's points form E
// interleaved tiles (tile j = points E n + j), so each lane loads the E
// consecutive points it feeds to the E tiles with one 16-byte load per vector
// and stores them back with one per output row.  Q^T comes through LDS in slabs
// of KS vectors (two buffers; the next slab's Q and X are in flight while the
// MFMAs run).  Only the last slab and the last workgroup check their edges, so
// the slab loop has no branches.  The k order is that of rotate_kernel, so the
// results are the same bits.  Bound by the MFMA rate and the stores at a
// workgroup's end (without them 80 us less); 605,808 x 275: FP32 818 us = 112
// TF/s (1067 us with Q guarded per value, 115 instead of 31 vector instructions
// beside a slab's 144 MFMAs), FP64 1669 us (2987 us with 64 columns per
// workgroup and Q from memory).
// LONG: 64-bit addresses per lane, for columns whose slab of X exceeds 32-bit
// byte offsets (they take 4 to 8 registers more, which costs FP64 a wavefront
// per SIMD at 96 columns).
template <typename T, int NCH, bool LONG>
__global__ __launch_bounds__(256, 2) void rotate_wide(const T* __restrict__ X, long long ldx,
                                                      const T* __restrict__ Qt, T* __restrict__ Z, long long ldz,
                                                      long long n, int kx, int ky, int ncb, int nblocks, int nb8) {
  typedef typename Acc<T>::type AT;
  constexpr int E = 16 / (int)sizeof(T);
  constexpr int KS = 16;                         // vectors per slab
  constexpr int ST = KS / 4;                     // MFMA steps per slab
  constexpr int NC = 32 * NCH;                   // columns per workgroup
  constexpr int LQ = NC + 64 / (int)sizeof(T);   // LDS row stride
  constexpr int TR = 256 / KS;                   // threads per Q row
  constexpr int QPT = NC / TR;                   // Q values per thread
  typedef T VT __attribute__((ext_vector_type(E)));
  __shared__ T qs[2][KS * LQ];
  const int L = (blockIdx.x & 7) * nb8 + (blockIdx.x >> 3);
  if (L >= nblocks) return;
  const int cb = L % ncb;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int pw = w >> 1, cw = w & 1;
  const int lm = lane & 15, lk = lane >> 4;
  const long long p0 = (long long)(L / ncb) * (32 * E);
  const long long pl = p0 + pw * 16 * E + E * lm;   // this lane's E points
  // blocks of NC columns, the last one moved back to end at ky (the columns it
  // shares with its neighbour are the same bits)
  const int c0 = min(cb * NC, max(ky - NC, 0));
  const int qk = threadIdx.x / TR, qc = threadIdx.x % TR;
  // the whole product for one kind of workgroup (EDGE: some points past n)
  auto body = [&](auto edge) {
    constexpr bool EDGE = decltype(edge)::value;
    AT acc[NCH][E];
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int j = 0; j < E; ++j) acc[c][j] = AT{0, 0, 0, 0};
    // vectors past kx (last slab) are read from the last one and replaced by
    // zero before use; only the last 32 columns of a block can lie past ky:
    // they are read from column ky - 1 and their products are not stored
    T qr[QPT], x[ST][E];
    auto qfetch = [&](int kb) {
      const T* src = Qt + (long long)kb * ky + c0 + (unsigned)(min(qk, kx - 1 - kb) * ky);
#pragma unroll
      for (int t = 0; t < QPT; ++t) {
        const int col = qc + TR * t;
        qr[t] = src[t < QPT - 32 / TR ? col : min(col, ky - 1 - c0)];
      }
    };
    auto qstore = [&](int bf) {
#pragma unroll
      for (int t = 0; t < QPT; ++t) qs[bf][qk * LQ + qc + TR * t] = qr[t];
    };
    // X of step st of the slab at kb
    const T* const xlane = X + (long long)lk * ldx + pl;
    const T* const xlast = X + (long long)(kx - 1) * ldx + pl;
    auto xfetch = [&](int kb, int st) {
      const char* src;
      if constexpr (LONG) {
        const T* s = xlane + (long long)(kb + 4 * st) * ldx;
        src = reinterpret_cast<const char*>(kb + 4 * st + lk < kx ? s : xlast);
      } else {   // 32-bit offsets from the slab's first vector
        const unsigned row = min(4 * st + lk, kx - 1 - kb);
        src = reinterpret_cast<const char*>(X + (long long)kb * ldx) + (row * (unsigned)ldx + (unsigned)pl) * (unsigned)sizeof(T);
      }
      if constexpr (EDGE) {
#pragma unroll
        for (int j = 0; j < E; ++j) x[st][j] = pl + j < n ? *reinterpret_cast<const T*>(src + sizeof(T) * j) : T(0);
      } else {
        const VT t = *reinterpret_cast<const VT*>(src);
#pragma unroll
        for (int j = 0; j < E; ++j) x[st][j] = t[j];
      }
    };
    auto step = [&](int bf, int st) {
      const T* qrow = &qs[bf][(4 * st + lk) * LQ + cw * 16 * NCH + lm];
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const T qa = qrow[16 * c];
#pragma unroll
        for (int j = 0; j < E; ++j) acc[c][j] = Acc<T>::mfma(qa, x[st][j], acc[c][j]);
      }
    };
    const int klast = (kx - 1) / KS * KS;   // the last slab, whole or not
    qfetch(0);
#pragma unroll
    for (int st = 0; st < ST; ++st) xfetch(0, st);
    qstore(0);
    __syncthreads();
    int bf = 0;
    for (int kb = 0; kb < klast; kb += KS) {
      qfetch(kb + KS);
      __builtin_amdgcn_sched_barrier(0);   // or the loads are sunk to their uses
#pragma unroll
      for (int st = 0; st < ST; ++st) {
        step(bf, st);
        xfetch(kb + KS, st);   // into the registers the step has read
        __builtin_amdgcn_sched_barrier(0);
      }
      bf ^= 1;
      qstore(bf);
      __syncthreads();
    }
    if (klast + KS > kx) {
      if (klast + qk >= kx) {
#pragma unroll
        for (int t = 0; t < QPT; ++t) qs[bf][qk * LQ + qc + TR * t] = T(0);
      }
      __syncthreads();
    }
#pragma unroll
    for (int st = 0; st < ST; ++st) {
#pragma unroll
      for (int j = 0; j < E; ++j) x[st][j] = klast + 4 * st + lk < kx ? x[st][j] : T(0);
      if (klast + 4 * st < kx) step(bf, st);
    }
    // register r of tile (c, j): column c0 + 16 c + row(lk, r), point pl + j
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = c0 + (cw * NCH + c) * 16 + Acc<T>::row(lk, r);
        if (col >= ky) continue;
        T* zr = Z + (long long)col * ldz + pl;
        if constexpr (EDGE) {
#pragma unroll
          for (int j = 0; j < E; ++j)
            if (pl + j < n) zr[j] = acc[c][j][r];
        } else {
          VT t;
#pragma unroll
          for (int j = 0; j < E; ++j) t[j] = acc[c][j][r];
          *reinterpret_cast<VT*>(zr) = t;
        }
      }
  };
  if (p0 + 32 * E <= n) body(std::false_type{});
  else body(std::true_type{});
}

// FP32 rotation on bf16 MFMA with three-way splits: every FP32 operand value
// x is split exactly into bf16 parts x = h + m + l (truncation: each part keeps
// the next 8 significant bits), and Z = X Q takes the six products whose parts
// carry at least 2^-16 of the value (lo*hi, mid*mid, hi*lo, mid*hi, hi*mid,
// hi*hi, small terms first) on v_mfma_f32_16x16x32_bf16 with FP32
// accumulation: on random operands the same accuracy as the FP32 MFMA path
// (the dropped products are below 2^-24 relative) at 6 / 16 of its MFMA cost
// (Si87H76 block, 605,808 x 275 x 275: 784 us against 1086 us).  Q (FP64) is rounded
// to FP32 and split once by split_q_bf3 into slabs of 32 k's:
// Qp[slab][column][part][32] (bf16 bits, columns padded to 32 NCH, zero
// beyond kx / ky).  The 16x16x32 operand layouts are only relied on through
// their shared K order: A (Q^T) lane m + 16 g element e and B (X^T) lane
// n + 16 g element e both carry k = 8 g + e; D[m][n] in lane n + 16 (m / 4),
// register m % 4, as for the other 16 x 16 FP32-output MFMAs.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr int kBf3K = 32;   // k's per slab

__device__ __forceinline__ void split3(float x, unsigned& h, unsigned& m, unsigned& l) {
  h = __builtin_bit_cast(unsigned, x) & 0xffff0000u;
  const float r1 = x - __builtin_bit_cast(float, h);
  m = __builtin_bit_cast(unsigned, r1) & 0xffff0000u;
  l = __builtin_bit_cast(unsigned, r1 - __builtin_bit_cast(float, m));   // at most 8 significant bits
}

__global__ void split_q_bf3(const double* __restrict__ Q, int ldq, int kx, int ky, int nc, int nks,
                            unsigned short* __restrict__ Qp) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nks * nc * kBf3K) return;
  const int kk = (int)(t % kBf3K), col = (int)((t / kBf3K) % nc), sl = (int)(t / ((long long)kBf3K * nc));
  const int k = kBf3K * sl + kk;
  const float x = (k < kx && col < ky) ? (float)Q[(long long)col * ldq + k] : 0.0f;
  unsigned h, m, l;
  split3(x, h, m, l);
  unsigned short* o = Qp + ((long long)sl * nc + col) * 3 * kBf3K + kk;
  o[0] = (unsigned short)(h >> 16);
  o[kBf3K] = (unsigned short)(m >> 16);
  o[2 * kBf3K] = (unsigned short)(l >> 16);
}

// Workgroup: 8 waves (pw = point quarter, cw = column half) over 256 points
// and all 32 NCH columns; a wave accumulates 64 points (4 interleaved tiles,
// tile j = points 4 n + j, one float4 of X per vector and lane) x 16 NCH
// columns.  Per slab of 32 k's: the Q parts through LDS (double-buffered),
// X of the next slab loaded into registers while the MFMAs run.  Requires
// 16-byte aligned X/Z columns (ld % 4 == 0).
template <int NCH>
__global__ __launch_bounds__(512) void rotate_bf3(const float* __restrict__ X, long long ldx,
                                                  const unsigned short* __restrict__ Qp, float* __restrict__ Z,
                                                  long long ldz, long long n, int kx, int ky, int nblocks, int nb8) {
  constexpr int NC = 32 * NCH;
  constexpr int SLAB = NC * 3 * kBf3K;   // bf16 values per slab
  __shared__ __attribute__((aligned(16))) unsigned short qs[2][SLAB];
  const int L = (blockIdx.x & 7) * nb8 + (blockIdx.x >> 3);
  if (L >= nblocks) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int pw = w >> 1, cw = w & 1;
  const int lm = lane & 15, g = lane >> 4;
  const long long pl = (long long)L * 256 + pw * 64 + 4 * lm;
  const int c0 = cw * 16 * NCH;
  const int nks = (kx + kBf3K - 1) / kBf3K;
  const bool full = pl + 3 < n;
  v4f acc[NCH][4];
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[c][j] = v4f{0, 0, 0, 0};
  auto qload = [&](int sl, int bf) {
    const u32x4* src = reinterpret_cast<const u32x4*>(Qp + (long long)sl * SLAB);
    u32x4* dst = reinterpret_cast<u32x4*>(qs[bf]);
    for (int t = threadIdx.x; t < SLAB / 8; t += 512) dst[t] = src[t];
  };
  float xr[8][4];
  auto xload = [&](int sl) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int kk = kBf3K * sl + 8 * g + e;
#pragma unroll
      for (int j = 0; j < 4; ++j) xr[e][j] = 0.0f;
      if (kk < kx) {
        const float* xp = X + (long long)kk * ldx + pl;
        if (full) {
          const float4 t = *reinterpret_cast<const float4*>(xp);
          xr[e][0] = t.x; xr[e][1] = t.y; xr[e][2] = t.z; xr[e][3] = t.w;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) xr[e][j] = pl + j < n ? xp[j] : 0.0f;
        }
      }
    }
  };
  qload(0, 0);
  xload(0);
  __syncthreads();
  for (int sl = 0; sl < nks; ++sl) {
    const int bf = sl & 1;
    bf16x8 bh[4], bm[4], bl[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned ph[4], pm[4], pq[4];
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        unsigned h0, m0, l0, h1, m1, l1;
        split3(xr[2 * e2][j], h0, m0, l0);
        split3(xr[2 * e2 + 1][j], h1, m1, l1);
        // the high halves of two floats -> one bf16 pair (element 2 e2 in the low half)
        ph[e2] = __builtin_amdgcn_perm(h1, h0, 0x07060302u);
        pm[e2] = __builtin_amdgcn_perm(m1, m0, 0x07060302u);
        pq[e2] = __builtin_amdgcn_perm(l1, l0, 0x07060302u);
      }
      bh[j] = __builtin_bit_cast(bf16x8, u32x4{ph[0], ph[1], ph[2], ph[3]});
      bm[j] = __builtin_bit_cast(bf16x8, u32x4{pm[0], pm[1], pm[2], pm[3]});
      bl[j] = __builtin_bit_cast(bf16x8, u32x4{pq[0], pq[1], pq[2], pq[3]});
    }
    const bool more = sl + 1 < nks;
    if (more) {
      xload(sl + 1);
      qload(sl + 1, bf ^ 1);
    }
    const unsigned short* qb = qs[bf];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const unsigned short* qa = qb + (c0 + 16 * c + lm) * 3 * kBf3K + 8 * g;
      const bf16x8 ah = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qa));
      const bf16x8 am = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qa + kBf3K));
      const bf16x8 al = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(qa + 2 * kBf3K));
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[j], acc[c][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm[j], acc[c][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[j], acc[c][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bh[j], acc[c][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bm[j], acc[c][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[j], acc[c][j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = c0 + 16 * c + Acc<float>::row(g, r);
      if (col >= ky) continue;
      float* zr = Z + (long long)col * ldz + pl;
      if (full) {
        *reinterpret_cast<float4*>(zr) = make_float4(acc[c][0][r], acc[c][1][r], acc[c][2][r], acc[c][3][r]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (pl + j < n) zr[j] = acc[c][j][r];
      }
    }
}

size_t bf3_work_bytes(int kx, int ky) {
  const size_t nks = (size_t)((kx + kBf3K - 1) / kBf3K), nc = 32 * (size_t)((ky + 31) / 32);
  return nks * nc * 3 * kBf3K * sizeof(unsigned short);
}
// Off by default: on random operands it matches the FP32 MFMA rotation, but
// in the Si87H76 SCF, where the rotation matrix R^-1 Q has large entries that
// cancel, the mixed-precision run took 19 SCF iterations instead of 15 with it
// (same energy to 3.6e-7 Ha/atom), so the 32-product sums inside the bf16 MFMA
// lose more than the FP32 path's sequential accumulation there.
bool g_rotate_bf3 = false;   // pc_rotate_set_split_bf16

__global__ void convert_q_f32(const double* __restrict__ Q, int ldq, int kx, int ky, float* __restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= kx * ky) return;
  const int i = e % kx, j = e / kx;
  out[(long long)i * ky + j] = (float)Q[(long long)j * ldq + i];  // row-major kx x ky -> ldq' = ky
}
__global__ void convert_q_f64(const double* __restrict__ Q, int ldq, int kx, int ky, double* __restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= kx * ky) return;
  const int i = e % kx, j = e / kx;
  out[(long long)i * ky + j] = Q[(long long)j * ldq + i];
}

struct GramPlan {
  int nt;                    // MFMA tiles per wave and side (tile of 32 nt columns)
  int ti_n, tj_n, ntile, nchunk;
  long long chunk;
  long long tile_size() const { return 1024LL * nt * nt; }
};

// Tile width: the one whose padded tiles cost least, a 64-wide tile's product
// counted at 1.1 and a 32-wide one's at 1.4 of a 96-wide one's (they read each
// column 1.5 and 3 times as often); so 275 columns take 96-wide
// tiles, 256 take 64-wide ones and a symmetric product of up to 96 32-wide ones.  Chunks: about as many workgroups as the
// chip holds at once, all with the same work (one round, no short last one),
// at least 256 points each and no more than the workspace holds; sp = points
// per stage.  nchunk = 0: not even one per tile fits.
GramPlan plan_gram(long long n, int kx, int ky, int sym, int sp, size_t bytes) {
  GramPlan p{};
  double best = 0.0;
  for (int nt = 3; nt >= 1; --nt) {
    const int w = 32 * nt, ti = (kx + w - 1) / w, tj = (ky + w - 1) / w;
    const int ntile = sym ? ti * (ti + 1) / 2 : ti * tj;
    const double cost = (double)ntile * w * w * (nt == 3 ? 1.0 : nt == 2 ? 1.1 : 1.4);
    if (p.nt == 0 || cost < best) {
      best = cost;
      p.nt = nt; p.ti_n = ti; p.tj_n = tj; p.ntile = ntile;
    }
  }
  // short columns: narrower tiles until a quarter of the CUs have a workgroup (128
  // points, 275 columns, FP32: 15.1 -> 7.5 us with the reduction's ONE form, 10.4
  // with 64-wide tiles and neither; with every CU 10,000 points, 96 columns lose 10 %)
  const long long maxch = std::max<long long>(1, (n + 255) / 256);
  while (p.nt > 1 && p.ntile * maxch < 64) {
    const int w = 32 * --p.nt;
    p.ti_n = (kx + w - 1) / w;
    p.tj_n = (ky + w - 1) / w;
    p.ntile = sym ? p.ti_n * (p.ti_n + 1) / 2 : p.ti_n * p.tj_n;
  }
  const int resident = p.nt == 3 ? 512 : p.nt == 2 ? 1024 : 2048;
  const int rest = n % sp != 0;   // the points past the last whole stage are a chunk of their own
  const long long nw = n - n % sp;
  const long long room = (long long)(bytes / sizeof(double)) / (p.ntile * p.tile_size()) - rest;
  if (room < (nw > 0 ? 1 : 0)) return p;
  const long long target = std::max<long long>(1, resident / p.ntile - rest);
  p.nchunk = (int)std::min({target, maxch, std::max<long long>(1, room)});
  p.chunk = std::max<long long>(32, ((nw + p.nchunk - 1) / p.nchunk + 31) / 32 * 32);
  p.nchunk = (int)((nw + p.chunk - 1) / p.chunk) + rest;
  return p;
}

// The form for any alignment keeps 64-wide tiles; its workspace is the smallest
// that either form takes.
GramPlan plan_gram_unaligned(long long n, int kx, int ky, int sym) {
  GramPlan p{};
  p.nt = 2;
  p.ti_n = (kx + 63) / 64;
  p.tj_n = (ky + 63) / 64;
  p.ntile = sym ? p.ti_n * (p.ti_n + 1) / 2 : p.ti_n * p.tj_n;
  p.nchunk = (int)std::min(std::max<long long>(1, 2048 / p.ntile), std::max<long long>(1, (n + 1023) / 1024));
  p.chunk = ((n + p.nchunk - 1) / p.nchunk + 31) / 32 * 32;
  p.nchunk = (int)((n + p.chunk - 1) / p.chunk);
  return p;
}

size_t gram_work_bytes(const GramPlan& p) { return (size_t)p.nchunk * p.ntile * p.tile_size() * sizeof(double); }

template <typename T>
int gram_impl(const T* X, long long ldx, const T* Y, long long ldy, long long n, int kx, int ky, double* S,
              long long lds, int sym, void* work, size_t work_bytes, void* stream) {
  PC_CHECK_ARG(X && Y && S && work, "null pointer");
  PC_CHECK_ARG(n >= 1 && kx >= 1 && ky >= 1, "empty operand");
  PC_CHECK_ARG(ldx >= n && ldy >= n && lds >= kx, "leading dimension too small");
  PC_CHECK_ARG(!sym || (kx == ky), "sym requires kx == ky");
  constexpr int E = 16 / (int)sizeof(T);
  const bool vec = (ldx % E == 0) && (ldy % E == 0) && (reinterpret_cast<uintptr_t>(X) % 16 == 0) &&
                   (reinterpret_cast<uintptr_t>(Y) % 16 == 0);
  const GramPlan any = plan_gram_unaligned(n, kx, ky, sym);
  PC_CHECK_ARG(work_bytes >= gram_work_bytes(any), "workspace too small");
  GramPlan p{};
  if (vec) p = plan_gram(n, kx, ky, sym, kGramStage / (int)sizeof(T), work_bytes);
  const bool tiled = p.nchunk > 0;
  if (!tiled) p = any;
  hipStream_t st = static_cast<hipStream_t>(stream);
  double* part = static_cast<double*>(work);
  const int nb = p.ntile * p.nchunk, nb8 = (nb + 7) / 8;
  if (tiled) {
#define PC_GRAM(NT)                                                                                              \
  hipLaunchKernelGGL((gram_tile<T, NT>), dim3(8 * nb8), dim3(256), 0, st, X, ldx, Y, ldy, n, kx, ky, p.ti_n, p.tj_n, \
                     p.ntile, sym, nb, nb8, p.chunk, part)
    if (p.nt == 1) PC_GRAM(1);
    else if (p.nt == 2) PC_GRAM(2);
    else PC_GRAM(3);
#undef PC_GRAM
  } else {
    hipLaunchKernelGGL((gram_kernel<T>), dim3(nb), dim3(256), 0, st, X, ldx, Y, ldy, n, kx, ky, p.ti_n, p.tj_n,
                       p.ntile, sym, p.nchunk, p.chunk, part);
  }
  PC_LAUNCH_CHECK();
  const int w = 32 * p.nt;
  if (p.nchunk <= 8)
    hipLaunchKernelGGL(gram_reduce<true>, dim3(p.ntile * (w * w / 256)), dim3(256), 0, st, part, w, p.ntile, p.nchunk,
                       p.ti_n, p.tj_n, kx, ky, S, lds, sym);
  else
    hipLaunchKernelGGL(gram_reduce<false>, dim3(p.ntile * (w * w / 32)), dim3(256), 0, st, part, w, p.ntile, p.nchunk,
                       p.ti_n, p.tj_n, kx, ky, S, lds, sym);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

template <typename T>
int rotate_impl(const T* X, long long ldx, const double* Q, int ldq, T* Z, long long ldz, long long n, int kx,
                int ky, void* work, size_t work_bytes, void* stream) {
  PC_CHECK_ARG(X && Q && Z && work, "null pointer");
  PC_CHECK_ARG(X != Z, "output must not alias input");
  PC_CHECK_ARG(n >= 1 && kx >= 1 && ky >= 1, "empty operand");
  PC_CHECK_ARG(ldx >= n && ldz >= n && ldq >= kx, "leading dimension too small");
  PC_CHECK_ARG(work_bytes >= (size_t)kx * ky * sizeof(T), "workspace too small");
  hipStream_t st = static_cast<hipStream_t>(stream);
  T* qt = static_cast<T*>(work);
  const int ne = kx * ky;
  auto convert_q = [&]() -> int {
    if constexpr (sizeof(T) == 4)
      hipLaunchKernelGGL(convert_q_f32, dim3((ne + 255) / 256), dim3(256), 0, st, Q, ldq, kx, ky, qt);
    else
      hipLaunchKernelGGL(convert_q_f64, dim3((ne + 255) / 256), dim3(256), 0, st, Q, ldq, kx, ky, qt);
    PC_LAUNCH_CHECK();
    return pc::PC_OK;
  };
  constexpr int E = 16 / (int)sizeof(T);
  const bool vec = (ldx % E == 0) && (ldz % E == 0) && (reinterpret_cast<uintptr_t>(X) % 16 == 0) &&
                   (reinterpret_cast<uintptr_t>(Z) % 16 == 0);
  if constexpr (sizeof(T) == 4) {
    const int nch = (ky + 31) / 32;
    if (vec && nch <= 9 && g_rotate_bf3 && work_bytes >= bf3_work_bytes(kx, ky)) {
      unsigned short* qp = static_cast<unsigned short*>(work);
      const int nks = (kx + kBf3K - 1) / kBf3K;
      const long long nq = (long long)nks * 32 * nch * kBf3K;
      hipLaunchKernelGGL(split_q_bf3, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, st, Q, ldq, kx, ky, 32 * nch,
                         nks, qp);
      PC_LAUNCH_CHECK();
      const int nb = (int)((n + 255) / 256);
      const int nb8 = (nb + 7) / 8;
      switch (nch) {
#define PC_ROTB(N)                                                                                                \
  case N:                                                                                                         \
    hipLaunchKernelGGL(rotate_bf3<N>, dim3(8 * nb8), dim3(512), 0, st, X, ldx, qp, Z, ldz, n, kx, ky, nb, nb8);    \
    break;
        PC_ROTB(1) PC_ROTB(2) PC_ROTB(3) PC_ROTB(4) PC_ROTB(5) PC_ROTB(6) PC_ROTB(7) PC_ROTB(8) PC_ROTB(9)
#undef PC_ROTB
      }
      PC_LAUNCH_CHECK();
      return pc::PC_OK;
    }
  }
  if (vec) {
    if (convert_q() != pc::PC_OK) return pc::PC_ERR_HIP;
    // column blocks of at most 288, of equal width; for short columns narrower ones,
    // until 96 CUs have a workgroup (520 columns, FP32, 1,000 points: 105 -> 48 us,
    // 67 with 64 columns per workgroup in the general form; with every CU 10,000
    // points, 275 columns, FP64 61 -> 87)
    const long long tiles = (n + 32 * E - 1) / (32 * E);
    const int nblk = (ky + 287) / 288;
    int nch = ((ky + nblk - 1) / nblk + 31) / 32;
    while (nch > 2 && tiles * ((ky + 32 * nch - 1) / (32 * nch)) < 96) --nch;
    const int ncb = (ky + 32 * nch - 1) / (32 * nch);
    // a slab's X in 32-bit byte offsets: to 2^26 points per column and more in FP32, 2^25 in FP64
    const bool wide_offsets = ((std::min(kx, 16) - 1) * ldx + n) * (long long)sizeof(T) >= (1LL << 32);
    const long long step = pc::kMaxGrid / ncb * (32 * E);   // points per launch
    for (long long p0 = 0; p0 < n; p0 += step) {
      const long long np = std::min(step, n - p0);
      const int nb = (int)((np + 32 * E - 1) / (32 * E) * ncb);
      const int nb8 = (nb + 7) / 8;
      switch (nch) {
#define PC_ROT(N)                                                                                               \
  case N:                                                                                                       \
    hipLaunchKernelGGL((wide_offsets ? rotate_wide<T, N, true> : rotate_wide<T, N, false>), dim3(8 * nb8),      \
                       dim3(256), 0, st, X + p0, ldx, qt, Z + p0, ldz, np, kx, ky, ncb, nb, nb8);               \
    break;
        PC_ROT(1) PC_ROT(2) PC_ROT(3) PC_ROT(4) PC_ROT(5) PC_ROT(6) PC_ROT(7) PC_ROT(8) PC_ROT(9)
#undef PC_ROT
      }
      PC_LAUNCH_CHECK();
    }
    return pc::PC_OK;
  }
  if (convert_q() != pc::PC_OK) return pc::PC_ERR_HIP;
  const int npt = (int)((n + 127) / 128);
  const int nct = (ky + 63) / 64;
  const int nb = npt * nct;
  const int nb8 = (nb + 7) / 8;
  hipLaunchKernelGGL((rotate_kernel<T>), dim3(8 * nb8), dim3(256), 0, st, X, ldx, qt, ky, Z, ldz, n, kx, ky, npt,
                     nct, nb, nb8);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

}  // namespace

extern "C" {

int pc_gram_workspace(long long n, int kx, int ky, int sym, size_t* out_bytes) {
  PC_CHECK_ARG(out_bytes, "null pointer");
  *out_bytes = std::max({gram_work_bytes(plan_gram(n, kx, ky, sym, 16, SIZE_MAX)),
                         gram_work_bytes(plan_gram(n, kx, ky, sym, 32, SIZE_MAX)),
                         gram_work_bytes(plan_gram_unaligned(n, kx, ky, sym))});
  return pc::PC_OK;
}

int pc_gram_f64(const double* X, long long ldx, const double* Y, long long ldy, long long n, int kx, int ky,
                double* S, long long lds, int sym, void* work, size_t work_bytes, void* stream) {
  return gram_impl<double>(X, ldx, Y, ldy, n, kx, ky, S, lds, sym, work, work_bytes, stream);
}

int pc_gram_f32(const float* X, long long ldx, const float* Y, long long ldy, long long n, int kx, int ky,
                double* S, long long lds, int sym, void* work, size_t work_bytes, void* stream) {
  return gram_impl<float>(X, ldx, Y, ldy, n, kx, ky, S, lds, sym, work, work_bytes, stream);
}

int pc_rotate_workspace(int kx, int ky, int fp32, size_t* out_bytes) {
  PC_CHECK_ARG(out_bytes && kx >= 1 && ky >= 1, "bad argument");
  const size_t base = (size_t)kx * ky * (fp32 ? sizeof(float) : sizeof(double));
  *out_bytes = fp32 ? std::max(base, bf3_work_bytes(kx, ky)) : base;
  return pc::PC_OK;
}

int pc_rotate_set_split_bf16(int on) {
  g_rotate_bf3 = on != 0;
  return pc::PC_OK;
}

int pc_rotate_f64(const double* X, long long ldx, const double* Q, int ldq, double* Z, long long ldz, long long n,
                  int kx, int ky, void* work, size_t work_bytes, void* stream) {
  return rotate_impl<double>(X, ldx, Q, ldq, Z, ldz, n, kx, ky, work, work_bytes, stream);
}

int pc_rotate_f32(const float* X, long long ldx, const double* Q, int ldq, float* Z, long long ldz, long long n,
                  int kx, int ky, void* work, size_t work_bytes, void* stream) {
  return rotate_impl<float>(X, ldx, Q, ldq, Z, ldz, n, kx, ky, work, work_bytes, stream);
}

}  // extern "C"
