// Multigrid-preconditioned CG for the Hartree solve (FP64).
//
// Same system and stop rule as pc_pcg_solve (A = -lap/h^2 with the domain's
// finite-difference stencil, Dirichlet zero outside the domain; stop when
// r.r <= tol^2 r0.r0 or after maxit iterations), preconditioned by one
// symmetric multigrid V-cycle per iteration -- the GPU counterpart of the
// reference's optional preconditioned CG (cg_prec, src/Eigensolvers/pcg.py:7-85,
// whose ILU preconditioner does not map to a GPU).  The preconditioner changes
// the iteration count, not the tolerance the solution meets.
//
// V-cycle, cell-centred: level 0 is the domain with its own stencil; level
// l >= 1 is a full cube of ceil(n_{l-1}/2) cells per axis, a cell active when
// any of its 8 children is, with the 7-point Laplacian at spacing 2^l h.
// Restriction = average of the active children, prolongation = injection
// (R = P^T / 8), one damped-Jacobi step before and after the coarse
// correction on every level, and a fixed-degree Chebyshev iteration on the
// coarsest cube (a polynomial in A, so the cycle is a fixed symmetric linear
// operator and CG theory applies).  From a zero start the pre-smoothed value
// is omega b / D, so the pre-smooth, residual and restriction of a cube level
// are one kernel, and the prolongation with the post-smooth is another.
//
// Launches per iteration:
//   fine level   mg_res0 (b_1 = R (r - c0 A r); rows of more than 128 points:
//                t0 = r - c0 A r and mg_restrict0),
//                mg_up0 (z = post-smooth(c0 r + P e_1), partials of r.z),
//                mg_apply (p = z + beta p, A p, partials of p.Ap), mg_update;
//   cube levels  mg_down / mg_up per level above the tail;
//   tail         mg_tail: the smallest levels and the coarsest Chebyshev in
//                one workgroup with every level in LDS.
// Every launch moves a few MB and is bound by latency.  Si87H76 sphere (605,808
// points), per iteration: 81 us in 9 launches (120 us in 12, before the fine
// passes had all their loads in flight and the small levels were merged):
// res0 10.2, down 4.6 + 4.6, tail 9.2, up 5.0 + 5.3, up0 14.0, apply 15.4,
// update 6.5.
// Arrays of a cube level hold zero on inactive cells, so a neighbour read
// needs no mask.  Every kernel returns at once when the iteration has
// converged, so the host reads the state back only every check_every
// iterations.
#include "pc_common.h"
#include "pc_zmarch.h"
#include <algorithm>
#include <cmath>
#include <vector>

long long pc_internal_grid_npts(void* grid);
int pc_internal_grid_view(void* grid, int* nx, int* ny, int* nz, const int** lo, const int** hi, const int** off);

namespace {

using pcz::ZMap;

constexpr int kB = 256;
constexpr int kNB = 512;          // workgroups of the point-wise launches (= r.r partials)
constexpr int kMaxLev = 8;
constexpr int kCheb = 8;          // Chebyshev steps on the coarsest cube
constexpr int kCoarsest = 512;    // cells of the coarsest cube, at most
constexpr int kTailCells = 4608;  // cells of the levels held in LDS by mg_tail, at most (16^3 + 8^3)
constexpr int kTailThreads = 1024;
// Damped Jacobi: the cycle stays SPD while omega < 2 / lambda_max(D^-1 A)
// (lambda_max(D^-1 A) of the radius-R stencil: 2.28 at R = 4, 2.37 at R = 6,
// so omega < 0.843 for every supported radius; 7-point: < 2, omega < 1).
// A V-cycle emulation on the Si87H76 sphere (smooth charge, tolerance 1e-5):
// 34 CG iterations at (0.6, 0.8), 29 at (0.8, 0.8), 28 at (0.8, 6/7).
constexpr double kOmega0 = 0.8;         // on the domain's own stencil
constexpr double kOmegaC = 6.0 / 7.0;   // on the 7-point cubes
enum { S_RR0 = 0, S_RZ0, S_RZ1, S_TOL1, S_DONE, S_ITS, S_RES, S_COUNT = 8 };

struct Fine {
  const int2* meta;
  const int* prow;
  long long n;
  int nx, ny, nz;
  double w[8];        // weights of A (w[0] = centre)
  double c0;          // omega0 / w[0]
  long long chunk;
  int nb, nb8;
};

struct Cube {
  int nx, ny, nz;
  long long cells;
  double inv_h2;      // 1 / (2^l h)^2
  const unsigned char* mask;
  double* b;
  double* e;
};

__device__ __forceinline__ int chunk_of(int nb8) { return (blockIdx.x & 7) * nb8 + (blockIdx.x >> 3); }

// value of a compact-domain array at cube coordinates (0 outside the domain)
__device__ __forceinline__ double dom_at(const Fine& g, const double* __restrict__ a, int i, int j, int k) {
  if (i < 0 || j < 0 || k < 0 || i >= g.nx || j >= g.ny || k >= g.nz) return 0.0;
  const int2 m = g.meta[j + g.ny * k];
  const int lo = m.y & 0xffff, hi = m.y >> 16;
  return (i >= lo && i < hi) ? a[(long long)m.x + i] : 0.0;
}

// ---------------------------------------------------------------- fine level
// Rows of at most 128 points: slabs of 8 rows, which read 3.3 values per output
// and fill the chip once on a 106^3 box (4 rows: 4.3 values and two rounds; 32.6
// instead of 15.4 us for mg_apply, whose registers then spilled); 4 rows for rows of one
// x-chunk, where twice as many workgroups fill more of the chip.  Chunks of planes from
// multiples of zc, so that every 2 x 2 x 2 cell lies in one workgroup and the
// restriction needs no launch of its own.  Wider rows: the march.
constexpr int mg_rows(int sx, int R) { return sx == 2 && R <= 4 ? 8 : pcz::kZW; }
template <int R, int SX, int VALUES, class P>   // VALUES loaded per point
__device__ __forceinline__ bool mg_pass(const ZMap& zm, int L, double* tile, P& p, double& s) {
  // 128 registers per thread: two values per point of radius 4 do not fit beside the formed field
  constexpr bool early = SX == 2 && R <= 4 && VALUES * (2 * R + pcz::kZP) > 20;
  return pcz::zpass<R, SX, mg_rows(SX, R), false, SX <= 2, early>(zm, L, tile, p, s);
}

// r = rhs - A x; partials of r.r (once per solve)
template <int R>
__global__ __launch_bounds__(kB) void mg_init(Fine g, const double* __restrict__ x, const double* __restrict__ rhs,
                                              double* __restrict__ r, double* __restrict__ prr) {
  __shared__ double red[kB / 64];
  const int c = chunk_of(g.nb8);
  if (c >= g.nb) return;
  const long long p0 = (long long)c * g.chunk, p1 = min(p0 + g.chunk, g.n);
  double s = 0.0;
  for (long long p = p0 + threadIdx.x; p < p1; p += kB) {
    const int row = g.prow[p];
    const int2 m = g.meta[row];
    const int i = (int)(p - m.x), k = row / g.ny, j = row - k * g.ny;
    double acc = g.w[0] * x[p];
#pragma unroll
    for (int d = 1; d <= R; ++d)
      acc += g.w[d] * (dom_at(g, x, i - d, j, k) + dom_at(g, x, i + d, j, k) + dom_at(g, x, i, j - d, k) +
                       dom_at(g, x, i, j + d, k) + dom_at(g, x, i, j, k - d) + dom_at(g, x, i, j, k + d));
    const double rv = rhs[p] - acc;
    r[p] = rv;
    s += rv * rv;
  }
  const double t = pc_block_sum(s, red);
  if (threadIdx.x == 0) prr[c] = t;
}

// t0 = r - c0 A r: the residual after one damped-Jacobi step from zero
// (rows of more than 128 points), or restricted at once: b_1 = the average of
// each cell's children.
template <int R, int SX>
struct Res0Pass {
  struct Raw { double r; };
  typedef pcz::NoExt Ext;
  static constexpr bool DOT = false, POST = SX <= 2;
  double c0;
  const double* __restrict__ r;
  double* __restrict__ t0;
  double* __restrict__ b1;
  int cx, cy, cz;   // cells of level 1
  const double* sc;
  double* buf;      // [kZP / 2][rows / 2][32 SX]
  __device__ __forceinline__ Raw load(long long idx, bool, int, int, int) const { return {r[idx]}; }
  __device__ __forceinline__ Ext ext(long long) const { return {}; }
  __device__ __forceinline__ bool pre() const { return sc[S_DONE] == 0.0; }
  __device__ __forceinline__ double comb(Raw v) const { return v.r; }
  __device__ __forceinline__ void out(bool in, long long idx, Raw, Ext, double qc, double acc, double& a,
                                      double&) const {
    if (POST) a = in ? qc - c0 * acc : 0.0;
    else if (in) t0[idx] = qc - c0 * acc;
  }
  // the plane, x and y pairs of each cell: registers, neighbouring lanes, LDS
  __device__ __forceinline__ void post(const double* t, int i, int j, int z, int zend, int row) const {
    constexpr int W = 32 * SX, H = mg_rows(SX, R) / 2;
    double c[pcz::kZP / 2];
#pragma unroll
    for (int q = 0; q < pcz::kZP / 2; ++q) {
      c[q] = t[2 * q] + t[2 * q + 1];
      c[q] += __shfl_xor(c[q], 1, 64);
      if ((row & 1) && !(i & 1)) buf[(q * H + (row >> 1)) * W + (i >> 1)] = c[q];
    }
    __syncthreads();
    const int I = i >> 1, J = j >> 1;
    if ((row & 1) || (i & 1) || I >= cx || J >= cy) return;
#pragma unroll
    for (int q = 0; q < pcz::kZP / 2; ++q) {
      const int K = (z >> 1) + q;
      if (K < cz && 2 * K < zend) b1[((long long)K * cy + J) * cx + I] = 0.125 * (c[q] + buf[(q * H + (row >> 1)) * W + I]);
    }
  }
};
template <int R, int SX>
__global__ __launch_bounds__(pcz::threads(SX, mg_rows(SX, R)), mg_rows(SX, R) == 8 ? 4 : 2) void mg_res0(ZMap zm, Res0Pass<R, SX> p) {
  __shared__ double tile[pcz::Tile<R, SX, mg_rows(SX, R)>::SIZE];
  __shared__ double buf[SX <= 2 ? pcz::kZP / 2 * (mg_rows(SX, R) / 2) * 32 * SX : 1];
  const int L = pcz::block_of(zm);
  if (L >= zm.nwg) return;
  p.buf = buf;
  double s;
  mg_pass<R, SX, 1>(zm, L, tile, p, s);
}

// level-1 right-hand side: average of the domain children of each cell
__global__ __launch_bounds__(kB) void mg_restrict0(Fine g, const double* __restrict__ t0, Cube c1, const double* sc) {
  if (sc[S_DONE] != 0.0) return;
  const long long q = (long long)blockIdx.x * kB + threadIdx.x;
  if (q >= c1.cells) return;
  const int I = (int)(q % c1.nx), J = (int)((q / c1.nx) % c1.ny), K = (int)(q / ((long long)c1.nx * c1.ny));
  double s = 0.0;
#pragma unroll
  for (int d = 0; d < 8; ++d) s += dom_at(g, t0, 2 * I + (d & 1), 2 * J + ((d >> 1) & 1), 2 * K + (d >> 2));
  c1.b[q] = 0.125 * s;   // zero on inactive cells: none of their children is in the domain
}

// z = post-smooth(c0 r + P e_1) with the domain's stencil; partials of r.z
struct Up0Pass {
  struct Raw { double r, e; };
  typedef pcz::NoExt Ext;
  static constexpr bool DOT = true, POST = false;
  double c0;
  const double* __restrict__ r;
  const double* __restrict__ e1;
  int enx, eny;
  double* __restrict__ z;
  const double* sc;
  __device__ __forceinline__ Raw load(long long idx, bool in, int i, int j, int k) const {
    const int e = in ? ((k >> 1) * eny + (j >> 1)) * enx + (i >> 1) : 0;
    return {r[idx], e1[e]};
  }
  __device__ __forceinline__ Ext ext(long long) const { return {}; }
  __device__ __forceinline__ bool pre() const { return sc[S_DONE] == 0.0; }
  __device__ __forceinline__ double comb(Raw v) const { return c0 * v.r + v.e; }
  __device__ __forceinline__ void out(bool in, long long idx, Raw v, Ext, double qc, double acc, double& a,
                                      double& b) const {
    if (in) {
      const double zn = qc + c0 * (v.r - acc);
      z[idx] = zn;
      a = v.r;
      b = zn;
    }
  }
};
template <int R, int SX>
__global__ __launch_bounds__(pcz::threads(SX, mg_rows(SX, R)), mg_rows(SX, R) == 8 ? 4 : 2) void mg_up0(ZMap zm, Up0Pass p, double* __restrict__ prz) {
  __shared__ double tile[pcz::Tile<R, SX, mg_rows(SX, R)>::SIZE];
  __shared__ double red[16];
  const int L = pcz::block_of(zm);
  if (L >= zm.nwg) return;
  double s;
  if (!mg_pass<R, SX, 2>(zm, L, tile, p, s)) return;
  const double t = pc_block_sum(s, red);
  if (threadIdx.x == 0) prz[L] = t;
}

// PCG step t: convergence from r_t.r_t, beta = rz_t / rz_{t-1}, p = z + beta p_old
// (at t = 0 the caller passes p_old = z and beta is 0), A p, partials of p.Ap.
// Workgroup 0 records the scalars.
struct ApplyPass {
  struct Raw { double z, p; };
  typedef pcz::NoExt Ext;
  static constexpr bool DOT = true, POST = false;
  int t, maxit, nb_rr, nb_rz;
  double tol;
  const double* __restrict__ z;
  const double* __restrict__ p_old;
  double* __restrict__ p_new;
  double* __restrict__ ap;
  const double* __restrict__ prr;
  const double* __restrict__ prz;
  double* sc;
  bool first;
  double *red, *red2;
  double beta;
  __device__ __forceinline__ Raw load(long long idx, bool, int, int, int) const { return {z[idx], p_old[idx]}; }
  __device__ __forceinline__ Ext ext(long long) const { return {}; }
  __device__ __forceinline__ bool pre() {
    const double done0 = t > 0 ? sc[S_DONE] : 0.0, tol0 = t > 0 ? sc[S_TOL1] : 0.0;
    const double rz0 = t > 0 ? sc[S_RZ0 + ((t - 1) & 1)] : 1.0;
    const double s1 = pc_parts_load<256>(prr, nb_rr), s2 = pc_parts_load<256>(prz, nb_rz);
    pc_parts_post(s1, red);
    pc_parts_post(s2, red2);
    __syncthreads();
    if (done0 != 0.0) return false;
    const double rr = pc_parts_get<256>(red), rz = pc_parts_get<256>(red2);
    const double tol1 = t == 0 ? tol * tol * rr : tol0;
    const bool done = t >= maxit || !(rr > tol1);
    beta = t > 0 ? rz / rz0 : 0.0;
    if (first && threadIdx.x == 0) {
      sc[S_RZ0 + (t & 1)] = rz;
      if (t == 0) {
        sc[S_TOL1] = tol1;
        sc[S_RR0] = rr;
      }
      sc[S_ITS] = (double)t;
      sc[S_RES] = rr;
      sc[S_DONE] = done ? 1.0 : 0.0;
    }
    return !done;
  }
  __device__ __forceinline__ double comb(Raw v) const { return v.z + beta * v.p; }
  __device__ __forceinline__ void out(bool in, long long idx, Raw, Ext, double qc, double acc, double& a,
                                      double& b) const {
    if (in) {
      p_new[idx] = qc;
      ap[idx] = acc;
      a = qc;
      b = acc;
    }
  }
};
template <int R, int SX>
__global__ __launch_bounds__(pcz::threads(SX, mg_rows(SX, R)), mg_rows(SX, R) == 8 ? 4 : 2) void mg_apply(ZMap zm, ApplyPass p, double* __restrict__ ppq) {
  __shared__ double tile[pcz::Tile<R, SX, mg_rows(SX, R)>::SIZE];
  __shared__ double red[16], red2[16], red3[16];
  const int L = pcz::block_of(zm);
  if (L >= zm.nwg) return;
  p.first = L == 0;
  p.red = red;
  p.red2 = red2;
  double s;
  if (!mg_pass<R, SX, 2>(zm, L, tile, p, s)) return;
  const double tt = pc_block_sum(s, red3);
  if (threadIdx.x == 0) ppq[L] = tt;
}

// alpha = rz_t / p.Ap; x += alpha p; r -= alpha Ap; partials of
// r_{t+1}.r_{t+1}.  The first points' values are loaded while the p.Ap partials
// are summed.
__global__ __launch_bounds__(kB) void mg_update(Fine g, int npq, int t, const double* sc, double* __restrict__ x,
                                                double* __restrict__ r, const double* __restrict__ p,
                                                const double* __restrict__ ap, const double* __restrict__ ppq,
                                                double* __restrict__ prr) {
  constexpr int U = 5;   // points per thread in flight
  __shared__ double red[kB / 64], red2[kB / 64];
  const int c = chunk_of(g.nb8);
  if (c >= g.nb) return;
  const double done = sc[S_DONE], rz = sc[S_RZ0 + (t & 1)];
  const long long p0 = (long long)c * g.chunk, p1 = min(p0 + g.chunk, g.n);
  double xv[U], rv[U], pv[U], av[U];
  auto load = [&](long long i0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long long i = min(i0 + (long long)u * kB, p1 - 1);
      xv[u] = x[i]; rv[u] = r[i]; pv[u] = p[i]; av[u] = ap[i];
    }
  };
  load(p0 + threadIdx.x);
  pc_parts_post(pc_parts_load<kB>(ppq, npq), red);
  __syncthreads();
  if (done != 0.0) return;
  const double alpha = rz / pc_parts_get<kB>(red);
  double s = 0.0;
  for (long long i0 = p0 + threadIdx.x; i0 < p1; i0 += U * kB) {
    if (i0 != p0 + threadIdx.x) load(i0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long long i = i0 + (long long)u * kB;
      if (i < p1) {
        x[i] = xv[u] + alpha * pv[u];
        const double v = rv[u] - alpha * av[u];
        r[i] = v;
        s += v * v;
      }
    }
  }
  const double tt = pc_block_sum(s, red2);
  if (threadIdx.x == 0) prr[c] = tt;
}

// ---------------------------------------------------------------- cube levels
__device__ __forceinline__ double cube_at(const Cube& c, const double* __restrict__ a, int i, int j, int k) {
  const bool in = i >= 0 && j >= 0 && k >= 0 && i < c.nx && j < c.ny && k < c.nz;
  return in ? a[((long long)k * c.ny + j) * c.nx + i] : 0.0;
}

// b_{l+1} = R (b_l - A_l (omega b_l / D_l)) on the active cells.  One thread
// per child (8 per coarse cell, adjacent lanes), summed across the 8 lanes.
__global__ __launch_bounds__(kB) void mg_down(Cube f, Cube c, const double* sc) {
  if (sc[S_DONE] != 0.0) return;
  const long long gid = (long long)blockIdx.x * kB + threadIdx.x;
  const long long q = gid >> 3;
  const int d = (int)(gid & 7);
  double v = 0.0;
  if (q < c.cells) {
    const int I = (int)(q % c.nx), J = (int)((q / c.nx) % c.ny), K = (int)(q / ((long long)c.nx * c.ny));
    const int i = 2 * I + (d & 1), j = 2 * J + ((d >> 1) & 1), k = 2 * K + (d >> 2);
    if (i < f.nx && j < f.ny && k < f.nz) {
      const long long fq = ((long long)k * f.ny + j) * f.nx + i;
      const double act = f.mask[fq] ? 1.0 : 0.0;
      const double bc = f.b[fq];
      const double nb = cube_at(f, f.b, i - 1, j, k) + cube_at(f, f.b, i + 1, j, k) + cube_at(f, f.b, i, j - 1, k) +
                        cube_at(f, f.b, i, j + 1, k) + cube_at(f, f.b, i, j, k - 1) + cube_at(f, f.b, i, j, k + 1);
      // t = b - (omega/6) (6 b - sum nb)
      v = act * ((1.0 - kOmegaC) * bc + (kOmegaC / 6.0) * nb);
    }
  }
  v += __shfl_xor(v, 1, 64);
  v += __shfl_xor(v, 2, 64);
  v += __shfl_xor(v, 4, 64);
  if (d == 0 && q < c.cells) c.b[q] = 0.125 * v;
}

// e_l = post-smooth(omega b_l / D_l + P e_{l+1}) on the active cells
__global__ __launch_bounds__(kB) void mg_up(Cube f, Cube c, const double* sc) {
  if (sc[S_DONE] != 0.0) return;
  const long long q = (long long)blockIdx.x * kB + threadIdx.x;
  if (q >= f.cells) return;
  const int i = (int)(q % f.nx), j = (int)((q / f.nx) % f.ny), k = (int)(q / ((long long)f.nx * f.ny));
  const double s0 = kOmegaC / (6.0 * f.inv_h2);   // omega / D_l
  auto ev = [&](int a, int b, int cc) -> double {
    const bool in = a >= 0 && b >= 0 && cc >= 0 && a < f.nx && b < f.ny && cc < f.nz;
    if (!in) return 0.0;
    const long long fq = ((long long)cc * f.ny + b) * f.nx + a;
    const long long cq = ((long long)(cc >> 1) * c.ny + (b >> 1)) * c.nx + (a >> 1);
    const double act = f.mask[fq] ? 1.0 : 0.0;
    return act * (s0 * f.b[fq] + c.e[cq]);
  };
  const double e0 = ev(i, j, k);
  const double ae = f.inv_h2 * (6.0 * e0 - ev(i - 1, j, k) - ev(i + 1, j, k) - ev(i, j - 1, k) - ev(i, j + 1, k) -
                                ev(i, j, k - 1) - ev(i, j, k + 1));
  f.e[q] = f.mask[q] ? e0 + s0 * (f.b[q] - ae) : 0.0;
}

// ---------------------------------------------------------------- tail
// Levels T..L (T >= 1) in LDS, one workgroup: restriction down to L, the
// Chebyshev iteration on L, prolongation and post-smoothing back up to T.
// Input b_T, output e_T (global).  Bound by latency: the levels of at most 4608
// cells together take one launch of 9.2 us instead of three of 3.2, 7.8 and
// 4.6 us (106^3 box: 14^3 and 7^3 cells; 13.9 us with cell coordinates divided
// out in the kernel instead of neighbour flags and parents from a table), and
// the Chebyshev steps' scalars come from the host instead of two divisions per
// step.
struct TailLev {
  int nx, ny, nz, cells, off;   // off: first cell of the level in the LDS arrays
  double inv_h2;
  const unsigned char* flags;   // bits 0..5: the x-, x+, y-, y+, z-, z+ neighbour is in the box; bit 6: active
  const unsigned short* par;    // cell of the next level over each cell
};
struct Tail {
  int nlev;                     // levels T..L = lev[0..nlev)
  int ncell;                    // cells of all of them
  TailLev lev[kMaxLev];
  const double* bT;
  double* eT;
  double d0;                    // first correction b / theta
  double cd[kCheb], cr[kCheb];  // Chebyshev: d = cd d + cr r
};
inline size_t tail_lds(int ncell) { return (size_t)ncell * (2 * sizeof(double) + 3) + 2 * kCoarsest * sizeof(double) + 8; }

__global__ __launch_bounds__(kTailThreads) void mg_tail(Tail tl, const double* sc) {
  extern __shared__ double lds[];
  double* bl = lds;
  double* el = bl + tl.ncell;
  double* xs = el + tl.ncell;   // [2][kCoarsest]
  unsigned short* pl = reinterpret_cast<unsigned short*>(xs + 2 * kCoarsest);
  unsigned char* ml = reinterpret_cast<unsigned char*>(pl + tl.ncell);
  constexpr int U = (kTailCells + kTailThreads - 1) / kTailThreads;
  const double done = sc[S_DONE];
  const int tid = threadIdx.x;
  for (int l = 0; l < tl.nlev; ++l) {
    const TailLev& f = tl.lev[l];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = tid + u * kTailThreads;
      if (q < f.cells) {
        ml[f.off + q] = f.flags[q];
        pl[f.off + q] = f.par[q];
        if (l == 0) bl[q] = tl.bT[q];
      }
    }
  }
  if (done != 0.0) return;
  __syncthreads();
  // the sum of a level array's six neighbours, cells outside the box zero
  auto nb6 = [&](const double* a, int sy, int sz, int q, unsigned fl) -> double {
    const double xm = a[fl & 1 ? q - 1 : q], xp = a[fl & 2 ? q + 1 : q], ym = a[fl & 4 ? q - sy : q];
    const double yp = a[fl & 8 ? q + sy : q], zm = a[fl & 16 ? q - sz : q], zp = a[fl & 32 ? q + sz : q];
    double s = fl & 1 ? xm : 0.0;
    s += fl & 2 ? xp : 0.0;
    s += fl & 4 ? ym : 0.0;
    s += fl & 8 ? yp : 0.0;
    s += fl & 16 ? zm : 0.0;
    s += fl & 32 ? zp : 0.0;
    return s;
  };
  // down: t = b - A omega b / D on the active cells (in the level's e array, free until the way up), b_{l+1} = R t
  for (int l = 0; l + 1 < tl.nlev; ++l) {
    const TailLev& f = tl.lev[l];
    const TailLev& c = tl.lev[l + 1];
    const int sy = f.nx, sz = f.nx * f.ny;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = tid + u * kTailThreads;
      if (q < f.cells) {
        const unsigned fl = ml[f.off + q];
        const double t = (1.0 - kOmegaC) * bl[f.off + q] + (kOmegaC / 6.0) * nb6(bl + f.off, sy, sz, q, fl);
        el[f.off + q] = fl & 64 ? t : 0.0;
      }
    }
    __syncthreads();
    for (int q = tid; q < c.cells; q += kTailThreads) {
      const int I = q % c.nx, J = (q / c.nx) % c.ny, K = q / (c.nx * c.ny);
      const int fq = f.off + (2 * K * f.ny + 2 * J) * f.nx + 2 * I;
      const bool x1 = 2 * I + 1 < f.nx, y1 = 2 * J + 1 < f.ny, z1 = 2 * K + 1 < f.nz;
      double s = 0.0;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const bool in = (!(d & 1) || x1) && (!(d & 2) || y1) && (!(d & 4) || z1);
        const double t = el[in ? fq + (d & 1) + (d & 2 ? sy : 0) + (d & 4 ? sz : 0) : fq];
        s += in ? t : 0.0;
      }
      bl[c.off + q] = 0.125 * s;
    }
    __syncthreads();
  }
  // coarsest: e = p(A) b, Chebyshev iteration on [lmin, lmax] from zero, one
  // barrier per step (x alternates between two LDS buffers)
  {
    const TailLev& c = tl.lev[tl.nlev - 1];
    const unsigned fl = tid < c.cells ? ml[c.off + tid] : 0;
    const bool act = fl & 64;
    const int sy = c.nx, sz = c.nx * c.ny;
    const double b = act ? bl[c.off + tid] : 0.0;
    double x = 0.0, d = b * tl.d0;
#pragma unroll
    for (int it = 0; it < kCheb; ++it) {
      x += d;
      double* xb = xs + (it & 1) * kCoarsest;
      if (tid < c.cells) xb[tid] = x;   // (d and x stay zero on inactive cells)
      __syncthreads();
      if (act) {
        const double r = b - c.inv_h2 * (6.0 * x - nb6(xb, sy, sz, tid, fl));
        d = tl.cd[it] * d + tl.cr[it] * r;
      }
    }
    x += d;
    if (tid < c.cells) {
      el[c.off + tid] = x;
      if (tl.nlev == 1) tl.eT[tid] = x;
    }
    __syncthreads();
  }
  // up: e_l = post-smooth(omega b_l / D_l + P e_{l+1}); the smoothed field first
  // replaces b, which the post-smoothing needs only at its own cell
  for (int l = tl.nlev - 2; l >= 0; --l) {
    const TailLev& f = tl.lev[l];
    const TailLev& c = tl.lev[l + 1];
    const double s0 = kOmegaC / (6.0 * f.inv_h2);
    const int sy = f.nx, sz = f.nx * f.ny;
    double bq[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = tid + u * kTailThreads;
      bq[u] = 0.0;
      if (q < f.cells) {
        bq[u] = bl[f.off + q];
        const double e0 = s0 * bq[u] + el[c.off + pl[f.off + q]];
        bl[f.off + q] = ml[f.off + q] & 64 ? e0 : 0.0;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = tid + u * kTailThreads;
      if (q < f.cells) {
        const unsigned fl = ml[f.off + q];
        const double e0 = bl[f.off + q];
        const double ae = f.inv_h2 * (6.0 * e0 - nb6(bl + f.off, sy, sz, q, fl));
        const double e = fl & 64 ? e0 + s0 * (bq[u] - ae) : 0.0;
        if (l == 0) tl.eT[q] = e;
        else el[f.off + q] = e;
      }
    }
    __syncthreads();
  }
}

__global__ void mg_reset(double* sc) {
  if (threadIdx.x < S_COUNT) sc[threadIdx.x] = 0.0;
}

// ---------------------------------------------------------------- host
struct MGCtx {
  void* grid;
  Fine g;
  ZMap zm;
  int radius;
  int nlev;                   // cube levels 1..nlev
  int tail;                   // first level held by mg_tail
  Cube lev[kMaxLev + 1];      // lev[1..nlev]
  Tail tl;
  std::vector<void*> allocs;
  double* t0;
  int first_check;            // iterations before the first state readback (0: check_every)
};

size_t work_bytes_for(long long n) {
  return (size_t)(5 * n + 2 * kNB + 2 * pcz::kMaxWG + S_COUNT) * sizeof(double);
}

template <int R, int SX>
struct FineLaunch {
  static dim3 grid(const MGCtx* c) { return dim3(8 * c->zm.nwg8); }
  static dim3 block() { return dim3(pcz::threads(SX, mg_rows(SX, R))); }
  static void res0(const MGCtx* c, hipStream_t st, const double* r, const double* sc) {
    const Cube& c1 = c->lev[1];
    const Res0Pass<R, SX> p{c->g.c0, r, c->t0, c1.b, c1.nx, c1.ny, c1.nz, sc, nullptr};
    hipLaunchKernelGGL((mg_res0<R, SX>), grid(c), block(), 0, st, c->zm, p);
    if (SX > 2)
      hipLaunchKernelGGL(mg_restrict0, dim3((unsigned)((c1.cells + kB - 1) / kB)), dim3(kB), 0, st, c->g, c->t0, c1, sc);
  }
  static void up0(const MGCtx* c, hipStream_t st, const double* r, double* z, double* prz, const double* sc) {
    const Cube& c1 = c->lev[1];
    const Up0Pass p{c->g.c0, r, c1.e, c1.nx, c1.ny, z, sc};
    hipLaunchKernelGGL((mg_up0<R, SX>), grid(c), block(), 0, st, c->zm, p, prz);
  }
  static void apply(const MGCtx* c, hipStream_t st, int t, int maxit, double tol, const double* z,
                    const double* p_old, double* p_new, double* ap, const double* prr, const double* prz, double* ppq,
                    double* sc) {
    const ApplyPass p{t, maxit, c->g.nb, c->zm.nwg, tol, z, p_old, p_new, ap, prr, prz, sc,
                      false, nullptr, nullptr, 0.0};
    hipLaunchKernelGGL((mg_apply<R, SX>), grid(c), block(), 0, st, c->zm, p, ppq);
  }
  static void init(const MGCtx* c, hipStream_t st, const double* x, const double* rhs, double* r, double* prr) {
    hipLaunchKernelGGL((mg_init<R>), dim3(8 * c->g.nb8), dim3(kB), 0, st, c->g, x, rhs, r, prr);
  }
};

struct FineOps {
  void (*res0)(const MGCtx*, hipStream_t, const double*, const double*);
  void (*up0)(const MGCtx*, hipStream_t, const double*, double*, double*, const double*);
  void (*apply)(const MGCtx*, hipStream_t, int, int, double, const double*, const double*, double*, double*,
                const double*, const double*, double*, double*);
  void (*init)(const MGCtx*, hipStream_t, const double*, const double*, double*, double*);
};

template <int R, int SX>
FineOps fine_ops_rs() {
  using F = FineLaunch<R, SX>;
  return {F::res0, F::up0, F::apply, F::init};
}

template <int R>
FineOps fine_ops_r(int sx) {
  if (sx == 1) return fine_ops_rs<R, 1>();
  if (sx == 2) return fine_ops_rs<R, 2>();
  return fine_ops_rs<R, 4>();
}

bool fine_ops(int radius, int sx, FineOps& ops) {
  switch (radius) {
    case 1: ops = fine_ops_r<1>(sx); return true;
    case 2: ops = fine_ops_r<2>(sx); return true;
    case 3: ops = fine_ops_r<3>(sx); return true;
    case 4: ops = fine_ops_r<4>(sx); return true;
    case 6: ops = fine_ops_r<6>(sx); return true;
    default: return false;
  }
}

}  // namespace

extern "C" {

// Builds the cube hierarchy for `grid` (spacing h): masks, right-hand-side and
// correction arrays on every level (a few MB for a 106^3 box).
int pc_mg_create(void* grid, double h, void** out_mg) {
  PC_CHECK_ARG(grid && out_mg && h > 0, "bad argument");
  MGCtx* c = new MGCtx();
  c->first_check = 0;
  c->grid = grid;
  Fine& g = c->g;
  double w8[8];
  pc_internal_grid_points(grid, &g.ny, &g.nz, &c->radius, &g.meta, &g.prow, w8);
  const int* zr;
  pc_internal_grid_zmap(grid, &g.nx, &zr);
  g.n = pc_internal_grid_npts(grid);
  const double inv_h2 = 1.0 / (h * h);
  for (int d = 0; d < 8; ++d) g.w[d] = w8[d] * inv_h2;
  g.w[0] *= 3.0;
  g.c0 = kOmega0 / g.w[0];
  const long long bp = (g.n + kB - 1) / kB;
  g.nb = (int)std::min<long long>(kNB, bp);
  g.chunk = ((bp + g.nb - 1) / g.nb) * kB;
  g.nb = (int)((g.n + g.chunk - 1) / g.chunk);
  g.nb8 = (g.nb + 7) / 8;
  int rz = 0;
  if (pcz::zmap_init(grid, g.w, c->zm, &rz, mg_rows(g.nx <= 64 ? 1 : (g.nx <= 128 ? 2 : 4), c->radius), 2)) {
    delete c;
    PC_CHECK_ARG(false, "nx > 256");
  }
  FineOps ops;
  if (!fine_ops(c->radius, c->zm.sx, ops)) {
    delete c;
    PC_CHECK_ARG(false, "unsupported stencil radius");
  }
  // domain mask on the full cube (host)
  int nx, ny, nz;
  const int *lo_d, *hi_d, *off_d;
  pc_internal_grid_view(grid, &nx, &ny, &nz, &lo_d, &hi_d, &off_d);
  std::vector<int> lo((size_t)ny * nz), hi((size_t)ny * nz);
  PC_HIP(hipMemcpy(lo.data(), lo_d, lo.size() * sizeof(int), hipMemcpyDeviceToHost));
  PC_HIP(hipMemcpy(hi.data(), hi_d, hi.size() * sizeof(int), hipMemcpyDeviceToHost));
  std::vector<unsigned char> prev((size_t)nx * ny * nz, 0);
  for (int k = 0; k < nz; ++k)
    for (int j = 0; j < ny; ++j)
      for (int i = lo[j + ny * k]; i < hi[j + ny * k]; ++i) prev[((size_t)k * ny + j) * nx + i] = 1;
  int pn[3] = {nx, ny, nz};
  double hl = h;
  c->nlev = 0;
  while (c->nlev < kMaxLev) {
    const int cn[3] = {(pn[0] + 1) / 2, (pn[1] + 1) / 2, (pn[2] + 1) / 2};
    std::vector<unsigned char> m((size_t)cn[0] * cn[1] * cn[2], 0);
    for (int k = 0; k < pn[2]; ++k)
      for (int j = 0; j < pn[1]; ++j)
        for (int i = 0; i < pn[0]; ++i)
          if (prev[((size_t)k * pn[1] + j) * pn[0] + i]) m[((size_t)(k / 2) * cn[1] + j / 2) * cn[0] + i / 2] = 1;
    hl *= 2.0;
    Cube& L = c->lev[++c->nlev];
    L.nx = cn[0]; L.ny = cn[1]; L.nz = cn[2];
    L.cells = (long long)cn[0] * cn[1] * cn[2];
    L.inv_h2 = 1.0 / (hl * hl);
    unsigned char* md = nullptr;
    double *bd = nullptr, *ed = nullptr;
    PC_HIP(hipMalloc(&md, L.cells));
    PC_HIP(hipMalloc(&bd, L.cells * sizeof(double)));
    PC_HIP(hipMalloc(&ed, L.cells * sizeof(double)));
    c->allocs.push_back(md); c->allocs.push_back(bd); c->allocs.push_back(ed);
    PC_HIP(hipMemcpy(md, m.data(), L.cells, hipMemcpyHostToDevice));
    PC_HIP(hipMemset(bd, 0, L.cells * sizeof(double)));
    PC_HIP(hipMemset(ed, 0, L.cells * sizeof(double)));
    L.mask = md; L.b = bd; L.e = ed;
    prev.swap(m);
    pn[0] = cn[0]; pn[1] = cn[1]; pn[2] = cn[2];
    if (L.cells <= kCoarsest) break;
  }
  PC_CHECK_ARG(c->lev[c->nlev].cells <= kCoarsest, "grid too large for the multigrid hierarchy");
  // tail: the deepest run of levels whose cells fit the LDS arrays
  c->tail = c->nlev;
  long long tcells = c->lev[c->nlev].cells;
  while (c->tail > 1 && tcells + c->lev[c->tail - 1].cells <= kTailCells) tcells += c->lev[--c->tail].cells;
  Tail& tl = c->tl;
  tl.nlev = c->nlev - c->tail + 1;
  int off = 0;
  for (int l = 0; l < tl.nlev; ++l) {
    const Cube& L = c->lev[c->tail + l];
    std::vector<unsigned char> m((size_t)L.cells);
    std::vector<unsigned short> par((size_t)L.cells);
    PC_HIP(hipMemcpy(m.data(), L.mask, m.size(), hipMemcpyDeviceToHost));
    const int px = (L.nx + 1) / 2, py = (L.ny + 1) / 2;
    for (int q = 0; q < (int)L.cells; ++q) {
      const int i = q % L.nx, j = (q / L.nx) % L.ny, k = q / (L.nx * L.ny);
      m[q] = (unsigned char)((i > 0) | (i + 1 < L.nx) << 1 | (j > 0) << 2 | (j + 1 < L.ny) << 3 | (k > 0) << 4 |
                             (k + 1 < L.nz) << 5 | (m[q] ? 64 : 0));
      par[q] = (unsigned short)((k / 2 * py + j / 2) * px + i / 2);
    }
    unsigned char* fd = nullptr;
    unsigned short* pd = nullptr;
    PC_HIP(hipMalloc(&fd, m.size()));
    c->allocs.push_back(fd);
    PC_HIP(hipMalloc(&pd, par.size() * sizeof(unsigned short)));
    c->allocs.push_back(pd);
    PC_HIP(hipMemcpy(fd, m.data(), m.size(), hipMemcpyHostToDevice));
    PC_HIP(hipMemcpy(pd, par.data(), par.size() * sizeof(unsigned short), hipMemcpyHostToDevice));
    tl.lev[l] = {L.nx, L.ny, L.nz, (int)L.cells, off, L.inv_h2, fd, pd};
    off += (int)L.cells;
  }
  tl.ncell = off;
  tl.bT = c->lev[c->tail].b;
  tl.eT = c->lev[c->tail].e;
  // Chebyshev interval of the coarsest 7-point operator: lambda_max <= 12/h^2
  // (Gershgorin); lambda_min >= that of the full box (Dirichlet on a subset)
  const Cube& C = c->lev[c->nlev];
  auto lam1 = [](int n) { return 2.0 * (1.0 - std::cos(M_PI / (n + 1))); };
  const double lmin = C.inv_h2 * (lam1(C.nx) + lam1(C.ny) + lam1(C.nz)), lmax = 12.0 * C.inv_h2;
  const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin), sigma = theta / delta;
  tl.d0 = 1.0 / theta;
  double rho = 1.0 / sigma;
  for (int it = 0; it < kCheb; ++it) {
    const double rho1 = 1.0 / (2.0 * sigma - rho);
    tl.cd[it] = rho1 * rho;
    tl.cr[it] = 2.0 * rho1 / delta;
    rho = rho1;
  }
  PC_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(mg_tail), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)tail_lds(kTailCells)));
  c->t0 = nullptr;
  if (c->zm.sx > 2) {
    PC_HIP(hipMalloc(&c->t0, g.n * sizeof(double)));
    c->allocs.push_back(c->t0);
  }
  *out_mg = c;
  return pc::PC_OK;
}

int pc_mg_destroy(void* mg) {
  MGCtx* c = static_cast<MGCtx*>(mg);
  if (!c) return pc::PC_OK;
  (void)hipDeviceSynchronize();   // queued V-cycles may still read the level arrays
  for (void* p : c->allocs) (void)hipFree(p);
  delete c;
  return pc::PC_OK;
}

int pc_mg_workspace(void* mg, size_t* out_bytes) {
  MGCtx* c = static_cast<MGCtx*>(mg);
  PC_CHECK_ARG(c && out_bytes, "null pointer");
  *out_bytes = work_bytes_for(c->g.n);
  return pc::PC_OK;
}

// Iterations before the first state readback of pc_pcg_solve_mg (0: its
// check_every); the results do not depend on it.
int pc_mg_set_first_check(void* mg, int first) {
  MGCtx* c = static_cast<MGCtx*>(mg);
  PC_CHECK_ARG(c && first >= 0, "bad argument");
  c->first_check = first;
  return pc::PC_OK;
}

// Multigrid-preconditioned CG: same arguments and stop rule as pc_pcg_solve
// (no first-iteration aliasing: this is the textbook preconditioned method).
int pc_pcg_solve_mg(void* mg, const double* rhs, double* x, int maxit, double tol, int check_every, void* work,
                    size_t work_bytes, int* its_out, double* res_out, void* stream) {
  MGCtx* c = static_cast<MGCtx*>(mg);
  PC_CHECK_ARG(c && rhs && x && work && its_out, "null pointer");
  PC_CHECK_ARG(work_bytes >= work_bytes_for(c->g.n), "workspace too small");
  PC_CHECK_ARG(((uintptr_t)work & 7) == 0, "workspace not 8-byte aligned");
  PC_CHECK_ARG(maxit >= 0, "maxit < 0");
  if (check_every < 1) check_every = 8;
  hipStream_t st = static_cast<hipStream_t>(stream);
  FineOps ops;
  fine_ops(c->radius, c->zm.sx, ops);
  const long long n = c->g.n;
  double* r = static_cast<double*>(work);
  double* z = r + n;
  double* p[2] = {z + n, z + 2 * n};
  double* ap = z + 3 * n;
  double* prr[2] = {ap + n, ap + n + kNB};
  double* prz = prr[1] + kNB;
  double* ppq = prz + pcz::kMaxWG;
  double* sc = ppq + pcz::kMaxWG;
  const int T = c->tail;
  auto vcycle = [&](const double* rr, double* zz) {
    ops.res0(c, st, rr, sc);
    for (int l = 1; l < T; ++l)
      hipLaunchKernelGGL(mg_down, dim3((unsigned)((8 * c->lev[l + 1].cells + kB - 1) / kB)), dim3(kB), 0, st,
                         c->lev[l], c->lev[l + 1], sc);
    hipLaunchKernelGGL(mg_tail, dim3(1), dim3(kTailThreads), tail_lds(c->tl.ncell), st, c->tl, sc);
    for (int l = T - 1; l >= 1; --l)
      hipLaunchKernelGGL(mg_up, dim3((unsigned)((c->lev[l].cells + kB - 1) / kB)), dim3(kB), 0, st, c->lev[l],
                         c->lev[l + 1], sc);
    ops.up0(c, st, rr, zz, prz, sc);
  };
  hipLaunchKernelGGL(mg_reset, dim3(1), dim3(64), 0, st, sc);
  ops.init(c, st, x, rhs, r, prr[0]);
  vcycle(r, z);
  PC_LAUNCH_CHECK();
  static thread_local double* host = nullptr;
  if (!host) PC_HIP(hipHostMalloc(&host, S_COUNT * sizeof(double), hipHostMallocDefault));
  int status = pc::PC_OK;
  // the state is read back after iteration first_check (when set), then every
  // check_every iterations; kernels queued past convergence return at once
  int t = 0;
  int next = c->first_check > 0 ? c->first_check : check_every;
  while (t <= maxit) {
    for (; t < next && t <= maxit; ++t) {
      // at t = 0 the direction is z itself: p_old = z with beta = 0
      const double* p_old = t == 0 ? z : p[t & 1];
      ops.apply(c, st, t, maxit, tol, z, p_old, p[(t + 1) & 1], ap, prr[t & 1], prz, ppq, sc);
      if (t < maxit) {
        hipLaunchKernelGGL(mg_update, dim3(8 * c->g.nb8), dim3(kB), 0, st, c->g, c->zm.nwg, t, sc, x, r,
                           p[(t + 1) & 1], ap, ppq, prr[(t + 1) & 1]);
        vcycle(r, z);
      }
      if (hipGetLastError() != hipSuccess) {
        pc::set_error("pc_pcg_solve_mg: kernel launch failed");
        status = pc::PC_ERR_HIP;
        break;
      }
    }
    if (status) break;
    if (hipMemcpyAsync(host, sc, S_COUNT * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
      pc::set_error("pc_pcg_solve_mg: readback failed");
      status = pc::PC_ERR_HIP;
      break;
    }
    if (host[S_DONE] != 0.0) break;
    next = t + check_every;
  }
  if (!status) {
    if (host[S_DONE] == 0.0) {
      pc::set_error("pc_pcg_solve_mg: internal error (no final state)");
      return pc::PC_ERR_HIP;
    }
    *its_out = (int)host[S_ITS];
    if (res_out) {
      res_out[0] = host[S_RES];
      res_out[1] = host[S_TOL1];
    }
  }
  return status;
}

}  // extern "C"
