// One FP64 application of the domain's stencil to a field that is formed on
// the fly, shared by the CG step, the multigrid fine level and the stencil of a
// single vector.
//
// A workgroup owns a slab of y-rows of the sphere-masked grid and a chunk of zc
// z-planes of them; a wavefront owns one row and 64 x-points of it (rows of at
// most 128 points; wider rows: the march at the end of this file).  These
// kernels move a few MB and are bound by latency, so every load of 6 planes
// (2R + 6 own planes, the halo rows, the values the output needs) goes out
// before the workgroup waits for anything but the row metadata; the scalars of
// the iteration (sums of partials) are formed meanwhile, and the planes are
// then computed from registers and LDS with one barrier each.  The order of
// every sum, the dot products' included, is the march's (one plane of loads in
// flight, which it replaces).  Plain CG step: H2O cube (140,608 points) 14.4 ->
// 9.7 us, same bits.  Values outside the domain are zero (Dirichlet).
//
// A pass P gives
//   Raw, Ext          what it loads per point, and per output point besides
//   DOT               whether it sums a product over its outputs
//   load(idx, in, i, j, z)   Raw of domain point idx = (i, j, z); where !in, of
//                     any valid place (the value is not used)
//   ext(idx)          Ext of an output point
//   pre()             run once by all threads after the first loads went out;
//                     false ends the pass (the same in every thread)
//   comb(raw)         the field's value
//   out(in, idx, raw, ext, qc, acc, a, b)   output: qc the centre value, acc =
//                     sum_d w_d (6 neighbours at distance d) + w_0 qc; where in,
//                     sets the product's factors a and b
//   POST, post(a, i, j, z, zend, row)   whether and how the workgroup treats the
//                     factors a of its planes z .. zend - 1 (0 outside the
//                     domain) together after them
#pragma once
#include "pc_common.h"

int pc_internal_grid_points(void* grid, int* ny, int* nz, int* radius, const int2** meta, const int** prow,
                            double* w8);
int pc_internal_grid_zmap(void* grid, int* nx, const int** zrange);

namespace pcz {

constexpr int kZW = 4;          // y-rows per workgroup unless a map says otherwise
constexpr int kMaxWG = 2048;    // workgroups of one march (= partials)

struct ZMap {
  const int2* meta;    // per row {off - lo, lo | hi << 16}
  const int* zrange;   // [2*ny]: z extent of each y-row column
  int nx, ny, nz;
  int nslab, nzc, zc;  // slabs of rows, z-chunks per slab, planes per chunk
  int nwg, nwg8;       // nslab * nzc workgroups, ceil(nwg / 8)
  int sx;              // 64-point x-strips per lane row (1, 2 or 4)
  double w[8];         // weights; w[0] is the 3D centre weight
};

// Fills the map for `grid` with weights w[0..7] (w[0] already the 3D centre
// weight) and slabs of zw rows.  zc = 6 planes per chunk (106^3 sphere, one plane
// of loads in flight: 38 us per CG iteration at 6 planes, 41 us at 2; 25 us with
// all of 6 planes in flight), raised in steps of zstep until the workgroups fit
// kMaxWG.
inline int zmap_init(void* grid, const double* w, ZMap& zm, int* radius, int zw = kZW, int zstep = 1) {
  int ny, nz;
  const int* prow;
  double w8[8];
  pc_internal_grid_points(grid, &ny, &nz, radius, &zm.meta, &prow, w8);
  zm.ny = ny;
  zm.nz = nz;
  pc_internal_grid_zmap(grid, &zm.nx, &zm.zrange);
  for (int d = 0; d < 8; ++d) zm.w[d] = w[d];
  zm.nslab = (zm.ny + zw - 1) / zw;
  zm.zc = 6;
  while ((long long)zm.nslab * ((zm.nz + zm.zc - 1) / zm.zc) > kMaxWG) zm.zc += zstep;
  zm.nzc = (zm.nz + zm.zc - 1) / zm.zc;
  zm.nwg = zm.nslab * zm.nzc;
  zm.nwg8 = (zm.nwg + 7) / 8;
  zm.sx = zm.nx <= 64 ? 1 : (zm.nx <= 128 ? 2 : 4);
  return zm.nx <= 256 ? 0 : 1;
}

// Block of launch-order workgroup b: consecutive blocks go to the same XCD
// (workgroup ids are dealt round-robin over the 8 XCDs), so the z-neighbour
// planes a block reads are mostly in that XCD's L2.
__device__ __forceinline__ int block_of(const ZMap& g) { return (blockIdx.x & 7) * g.nwg8 + (blockIdx.x >> 3); }

__device__ __forceinline__ int2 zrow(const ZMap& g, int j, int z) {
  return (j >= 0 && j < g.ny && z >= 0 && z < g.nz) ? g.meta[j + g.ny * z] : make_int2(0, 0);
}

constexpr int kZP = 6;          // planes whose loads are in flight together
constexpr int threads(int sx, int zw = kZW) { return sx <= 2 ? 64 * zw * sx : 256; }

// ORD: the products' factors of the second x-chunk, for the march's summation order
template <int R, int SX, int ZW = kZW, bool ORD = false>
struct Tile {
  static constexpr int LW = 64 * SX + 2 * R;
  static constexpr int LR = ZW + 2 * R;
  static constexpr int DOT = ORD && SX == 2 ? 2 * kZP * ZW * 64 : 0;
  static constexpr int SIZE = 2 * LR * LW + DOT;   // doubles
};
struct NoExt {};

// Rows of more than 128 points: each wavefront marches z with its row's SX
// chunks, the loads of plane z + 1 going out before plane z is computed.
template <int R, int SX, class P>
__device__ __forceinline__ void zmarch(const ZMap& g, int L, double* tile, P& p, double& sum) {
  constexpr int TY = kZW;
  constexpr int LW = Tile<R, SX>::LW;
  constexpr int LR = Tile<R, SX>::LR;
  constexpr int HT = (2 * R + kZW - 1) / kZW;
  const int slab = L % g.nslab;
  const int zci = L / g.nslab;
  const int j0 = slab * TY;
  int zb = g.nz, ze = 0;
  for (int q = 0; q < TY; ++q) {
    const int j = j0 + q;
    if (j < g.ny) {
      zb = min(zb, g.zrange[2 * j]);
      ze = max(ze, g.zrange[2 * j + 1]);
    }
  }
  const int z0 = zb + zci * g.zc;
  const int z1 = min(ze, z0 + g.zc);
  if (z0 >= z1) return;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = j0 + wv;
  auto load = [&](int2 m, int i, int jj, int z) -> double {
    const int lo = m.y & 0xffff, hi = m.y >> 16;
    return (i >= lo && i < hi) ? p.comb(p.load((long long)m.x + i, true, i, jj, z)) : 0.0;
  };
  // Row metadata windows: lane l holds meta(row, wb + l), so a plane's
  // lookups are register reads and its loads never wait for a metadata load;
  // a window is reloaded once every 64 planes.  The own row serves planes z
  // (output) and z + R (queue front).
  struct Win {
    int2 v;
    int wb;
  };
  auto win_load = [&](Win& w, int jj, int wb) {
    w.wb = wb;
    w.v = zrow(g, jj, wb + lane);
  };
  auto win_at = [&](const Win& w, int z) -> int2 {
    const int l = z - w.wb;
    return make_int2(__builtin_amdgcn_readlane(w.v.x, l), __builtin_amdgcn_readlane(w.v.y, l));
  };
  Win wown, whalo[HT];
  win_load(wown, j, z0 - R);
#pragma unroll
  for (int h = 0; h < HT; ++h) {
    const int hr = wv + kZW * h;
    const int tr = hr < R ? hr : hr + TY;
    win_load(whalo[h], j0 - R + tr, z0);
  }
  for (int e = threadIdx.x; e < 2 * LR * LW; e += 256) tile[e] = 0.0;
  __syncthreads();
  double q[SX][2 * R + 1];
  double nq[SX], hc[HT][SX], hn[HT][SX];
  int2 mcur, mnext;
#pragma unroll
  for (int s = 0; s < SX; ++s) {
    q[s][0] = 0.0;
#pragma unroll
    for (int h = 0; h < HT; ++h) hc[h][s] = hn[h][s] = 0.0;
  }
#pragma unroll
  for (int dz = 1; dz <= 2 * R; ++dz) {
    const int zz = z0 - R - 1 + dz;
    const int2 m = win_at(wown, zz);
#pragma unroll
    for (int s = 0; s < SX; ++s) q[s][dz] = load(m, lane + 64 * s, j, zz);
  }
  auto prefetch = [&](int z) {
    if (z + R >= wown.wb + 64) win_load(wown, j, z);
    const int2 mq = win_at(wown, z + R);
    mnext = win_at(wown, z);
#pragma unroll
    for (int s = 0; s < SX; ++s) nq[s] = load(mq, lane + 64 * s, j, z + R);
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const int hr = wv + kZW * h;
      if (hr < 2 * R) {
        const int tr = hr < R ? hr : hr + TY;
        const int jh = j0 - R + tr;
        if (z >= whalo[h].wb + 64) win_load(whalo[h], jh, z);
        const int2 mh = win_at(whalo[h], z);
#pragma unroll
        for (int s = 0; s < SX; ++s) hn[h][s] = load(mh, lane + 64 * s, jh, z);
      }
    }
  };
  prefetch(z0);
  for (int z = z0; z < z1; ++z) {
    double* tb = tile + ((z - z0) & 1) * (LR * LW);
    mcur = mnext;
#pragma unroll
    for (int s = 0; s < SX; ++s) {
#pragma unroll
      for (int d = 0; d < 2 * R; ++d) q[s][d] = q[s][d + 1];
      q[s][2 * R] = nq[s];
#pragma unroll
      for (int h = 0; h < HT; ++h) hc[h][s] = hn[h][s];
    }
    if (z + 1 < z1) prefetch(z + 1);
#pragma unroll
    for (int s = 0; s < SX; ++s) tb[(wv + R) * LW + R + lane + 64 * s] = q[s][R];
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const int hr = wv + kZW * h;
      if (hr < 2 * R) {
        const int tr = hr < R ? hr : hr + TY;
#pragma unroll
        for (int s = 0; s < SX; ++s) tb[tr * LW + R + lane + 64 * s] = hc[h][s];
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);   // LDS only: the prefetch stays in flight
    __builtin_amdgcn_s_barrier();
    const int lo = mcur.y & 0xffff, hi = mcur.y >> 16;
#pragma unroll
    for (int s = 0; s < SX; ++s) {
      const int i = lane + 64 * s;
      const double* trow = tb + (wv + R) * LW + R + i;
      double acc = g.w[0] * q[s][R];
#pragma unroll
      for (int d = 1; d <= R; ++d) {
        const double nb = trow[-d] + trow[d] + trow[-d * LW] + trow[d * LW] + q[s][R - d] + q[s][R + d];
        acc += g.w[d] * nb;
      }
      if (i >= lo && i < hi) {
        const long long idx = (long long)mcur.x + i;
        double a = 0.0, b = 0.0;
        p.out(true, idx, p.load(idx, true, i, j, z), p.ext(idx), q[s][R], acc, a, b);
        if constexpr (P::DOT) sum += a * b;
      }
    }
  }
}

// The pass over block L (0 <= L < g.nwg); `tile` holds Tile<R, SX, ZW,
// ORD>::SIZE doubles of LDS.  Every thread of the workgroup (threads(SX, ZW) of
// them) must call it.  sum: this thread's share of the DOT sum; ORD: in the
// march's order (plane by plane and x-chunk by x-chunk in one thread).  ZAL: the
// chunks start at multiples of zc instead of the slab's first plane.  EARLY:
// pre() before the loads, where two values per point would not fit the
// registers.  Returns false when pre() ended the pass.
template <int R, int SX, int ZW, bool ORD, bool ZAL, bool EARLY, class P>
__device__ __forceinline__ bool zpass(const ZMap& g, int L, double* tile, P& p, double& sum) {
  sum = 0.0;
  if constexpr (SX > 2) {
    static_assert(ZW == kZW && !ZAL, "the march takes 4 rows and unaligned chunks");
    if (!p.pre()) return false;
    zmarch<R, SX>(g, L, tile, p, sum);
    return true;
  } else {
    typedef typename P::Raw Raw;
    typedef typename P::Ext Ext;
    typedef Tile<R, SX, ZW, ORD> T;
    constexpr int LW = T::LW, LR = T::LR;
    constexpr int HT = (2 * R + ZW - 1) / ZW;
    constexpr int NQ = 2 * R + kZP;
    const int slab = L % g.nslab;
    const int zci = L / g.nslab;
    const int j0 = slab * ZW;
    int zb = g.nz, ze = 0;
#pragma unroll
    for (int q = 0; q < ZW; ++q) {
      const int j = min(j0 + q, g.ny - 1);
      zb = min(zb, g.zrange[2 * j]);
      ze = max(ze, g.zrange[2 * j + 1]);
    }
    const int z0 = ZAL ? zci * g.zc : zb + zci * g.zc;
    const int z1 = min(ze, z0 + g.zc);
    if (z0 >= z1 || (ZAL && z0 + g.zc <= zb)) return p.pre();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wv = wave % ZW, ck = wave / ZW;
    const int j = j0 + wv, i = lane + 64 * ck;
    // the R zero columns either side of both tiles
    for (int e = threadIdx.x; e < 2 * LR * 2 * R; e += threads(SX, ZW)) {
      const int row = e / (2 * R), c = e % (2 * R);
      tile[row * LW + (c < R ? c : 64 * SX + c)] = 0.0;
    }
    if (EARLY && !p.pre()) return false;
    for (int zs = z0; zs < z1; zs += kZP) {
      // lane l holds the own row's metadata at plane zs - R + l and the halo rows' at zs + l
      const int2 wown = zrow(g, j, zs - R + lane);
      int2 whalo[HT];
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        const int hr = wv + ZW * h;
        whalo[h] = zrow(g, j0 - R + (hr < R ? hr : hr + ZW), zs + lane);
      }
      Raw q[NQ], hq[HT][kZP];
      Ext ex[kZP];
      unsigned qin = 0, hin[HT];
      int own[kZP];
#pragma unroll
      for (int d = 0; d < NQ; ++d) {
        const int base = __builtin_amdgcn_readlane(wown.x, d), ext = __builtin_amdgcn_readlane(wown.y, d);
        const bool in = i >= (ext & 0xffff) && i < (ext >> 16);
        const int idx = in ? base + i : 0;
        qin |= (unsigned)in << d;
        q[d] = p.load(idx, in, i, j, zs - R + d);
        if (d >= R && d < R + kZP) {
          own[d - R] = idx;
          ex[d - R] = p.ext(idx);
        }
      }
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        const int hr = wv + ZW * h;
        const int jh = j0 - R + (hr < R ? hr : hr + ZW);
        hin[h] = 0;
        if (hr < 2 * R) {
#pragma unroll
          for (int pl = 0; pl < kZP; ++pl) {
            const int base = __builtin_amdgcn_readlane(whalo[h].x, pl);
            const int ext = __builtin_amdgcn_readlane(whalo[h].y, pl);
            const bool in = i >= (ext & 0xffff) && i < (ext >> 16);
            hin[h] |= (unsigned)in << pl;
            hq[h][pl] = p.load(in ? base + i : 0, in, i, jh, zs + pl);
          }
        }
      }
      if constexpr (!EARLY) {
        __builtin_amdgcn_sched_barrier(0);
        if (zs == z0 && !p.pre()) return false;
      }
      double v[NQ];
#pragma unroll
      for (int d = 0; d < NQ; ++d) v[d] = (qin >> d) & 1 ? p.comb(q[d]) : 0.0;
      double fa[kZP], fb[kZP];
#pragma unroll
      for (int pl = 0; pl < kZP; ++pl) {
        fa[pl] = fb[pl] = 0.0;
        if (zs + pl >= z1) continue;
        double* tb = tile + (pl & 1) * (LR * LW);
        tb[(wv + R) * LW + R + i] = v[R + pl];
#pragma unroll
        for (int h = 0; h < HT; ++h) {
          const int hr = wv + ZW * h;
          if (hr < 2 * R)
            tb[(hr < R ? hr : hr + ZW) * LW + R + i] = (hin[h] >> pl) & 1 ? p.comb(hq[h][pl]) : 0.0;
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);   // LDS only
        __builtin_amdgcn_s_barrier();
        const double* trow = tb + (wv + R) * LW + R + i;
        double acc = g.w[0] * v[R + pl];
#pragma unroll
        for (int d = 1; d <= R; ++d) {
          const double nb = trow[-d] + trow[d] + trow[-d * LW] + trow[d * LW] + v[R + pl - d] + v[R + pl + d];
          acc += g.w[d] * nb;
        }
        const bool in = (qin >> (R + pl)) & 1;
        p.out(in, own[pl], q[R + pl], ex[pl], v[R + pl], acc, fa[pl], fb[pl]);
      }
      if constexpr (P::DOT) {
        if constexpr (!ORD || SX == 1) {
#pragma unroll
          for (int pl = 0; pl < kZP; ++pl) sum += fa[pl] * fb[pl];
        } else {
          double* db = tile + 2 * LR * LW + (wv * 64 + lane) * 2;
          if (ck == 1) {
#pragma unroll
            for (int pl = 0; pl < kZP; ++pl) {
              db[pl * ZW * 128] = fa[pl];
              db[pl * ZW * 128 + 1] = fb[pl];
            }
          }
          __syncthreads();
          if (ck == 0) {
#pragma unroll
            for (int pl = 0; pl < kZP; ++pl) {
              sum += fa[pl] * fb[pl];
              sum += db[pl * ZW * 128] * db[pl * ZW * 128 + 1];
            }
          }
          if (zs + kZP < z1) __syncthreads();
        }
      }
      if constexpr (P::POST) {
        p.post(fa, i, j, zs, min(zs + kZP, z0 + g.zc), wv);
        if (zs + kZP < z1) __syncthreads();
      }
    }
    return true;
  }
}

}  // namespace pcz
