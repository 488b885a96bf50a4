// Kleinman-Bylander p-channel projectors in factored form.
//
// The reference stores V_nl = sum_a sum_{m=x,y,z} u_am u_am^T / (Zvalue/h^3) as
// dense outer products in a sparse matrix (src/V_ion/pseudoNL_original.py:
// 187-206).  Here each atom keeps its support points and the three u values,
// and V_nl*Y is applied as
//   gather : C[a, v, m] = sum_{p in supp(a)} u_am(p) * Y[p, v]          (FP64)
//   scatter: Out[p, v] += alpha * sum_{(a,m) covering p} scale_a u_am(p) C[a, v, m]
// C is atom-major, C[(a*nvec + v)*3 + m], so the scatter's 8 vectors of one
// entry read 24 consecutive doubles (two cache lines, not eight).
// The scatter runs over unique support points (no atomics, deterministic).
#include "pc_common.h"
#include <algorithm>
#include <numeric>
#include <vector>

namespace {

struct ProjDev {
  int natoms;
  int nent;
  int nupts;
  int* atom_ptr;   // [natoms+1]
  int* ent_pt;     // [nent]  point index of entry
  double* ent_u;   // [3*nent]
  int* ent_atom;   // [nent]
  double* scale;   // [natoms]
  int* upt;        // [nupts] unique point index
  int* upt_ptr;    // [nupts+1] into upt_ent
  int* upt_ent;    // [nent] entry ids grouped by point
  int* se_atom;    // [nent] atom of the t-th entry in point order
  double* se_u;    // [3*nent] scale[atom] * u of the t-th entry in point order
};

// C[a][v][m] = sum_e u_m[e] * Y[v][pt[e]] (FP64 accumulation).  GW wavefronts take
// one atom and 4 vectors, so the entry tables are read once for the 4: the atom's
// entries in rounds of 64 (wavefront w the rounds w, w + GW, ...), up to kGE rounds
// loaded together, their sums added in order.  A workgroup holds kGW / GW atoms.
// Small blocks are bound by the chain of dependent loads (the atom's range, its
// points, their values), large ones by the 128-byte lines that a support's short
// rows touch (5.6 points of 32 in FP32).  One wavefront per atom and 4
// vectors, round after round, atoms spread over the XCDs -> now: 3 atoms x 23
// vectors FP64 9.6 -> 4.4 us, 18 x 49 FP32 10.3 -> 5.0, 163 x 275 FP32 78 -> 61
// (83 without the XCD order, 65 with 8 vectors), 1,500 atoms of 20 points x 275
// FP32 157 -> 75 (222 with four wavefronts, each loading three rounds at any size).
constexpr int kGV = 4;   // vectors per wavefront in the gather
constexpr int kGE = 3;   // rounds in flight
constexpr int kGW = 4;   // wavefronts per workgroup
template <typename T, int GW>   // GW wavefronts per atom
__global__ __launch_bounds__(64 * kGW) void proj_gather(ProjDev P, const T* __restrict__ Y, long long ld, int nvec,
                                                        double* __restrict__ C) {
  constexpr int NA = kGW / GW;   // atoms per workgroup
  __shared__ double part[kGW][kGV * 3];
  // the atoms of one vector group follow each other on one XCD: atoms share lines
  const int na = (P.natoms + NA - 1) / NA;
  const int nb = na * ((nvec + kGV - 1) / kGV), L = (blockIdx.x & 7) * ((nb + 7) / 8) + (blockIdx.x >> 3);
  if (L >= nb) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wv = wave % GW, v0 = L / na * kGV, a0 = L % na * NA, a = a0 + wave / GW;
  double s[kGV][3];
#pragma unroll
  for (int u = 0; u < kGV; ++u) s[u][0] = s[u][1] = s[u][2] = 0.0;
  const int e0 = a < P.natoms ? P.atom_ptr[a] : 0, e1 = a < P.natoms ? P.atom_ptr[a + 1] : 0;
  const T* yv[kGV];
#pragma unroll
  for (int u = 0; u < kGV; ++u) yv[u] = Y + (long long)min(v0 + u, nvec - 1) * ld;
  // N rounds from entry eb on, of which only the last may be short: lanes past its
  // end take the last entry, with zeros (0 times an infinite value would be a NaN)
  auto rounds = [&](auto n, int eb) {
    constexpr int N = decltype(n)::value;
    int pt[N];
    double w[N][3];
    T y[N][kGV];
    const bool in = eb + 64 * GW * (N - 1) + lane < e1;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int e = eb + 64 * GW * k + lane, ec = k == N - 1 ? min(e, e1 - 1) : e;
      pt[k] = P.ent_pt[ec];
#pragma unroll
      for (int m = 0; m < 3; ++m) w[k][m] = P.ent_u[3 * (long long)ec + m];
    }
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int u = 0; u < kGV; ++u) y[k][u] = yv[u][pt[k]];
    __builtin_amdgcn_sched_barrier(0);   // every load first
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int u = 0; u < kGV; ++u) {
        const double yu = k == N - 1 && !in ? T(0) : y[k][u];
#pragma unroll
        for (int m = 0; m < 3; ++m) s[u][m] += (k == N - 1 && !in ? 0.0 : w[k][m]) * yu;
      }
  };
  for (int eb = e0 + 64 * wv; eb < e1; eb += 64 * GW * kGE) {
    if (eb + 64 * GW * 2 < e1) rounds(std::integral_constant<int, 3>{}, eb);
    else if (eb + 64 * GW < e1) rounds(std::integral_constant<int, 2>{}, eb);
    else rounds(std::integral_constant<int, 1>{}, eb);
  }
#pragma unroll
  for (int u = 0; u < kGV; ++u)
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double t = pc_wave_sum(s[u][m]);
      if (lane == 0) part[wave][3 * u + m] = t;
    }
  __syncthreads();
  const int t = threadIdx.x % (kGV * 3), q = threadIdx.x / (kGV * 3);
  if (q < NA && a0 + q < P.natoms && v0 + t / 3 < nvec) {
    double c = part[q * GW][t];
#pragma unroll
    for (int k = 1; k < GW; ++k) c += part[q * GW + k][t];
    C[((long long)(a0 + q) * nvec + v0) * 3 + t] = c;
  }
}

// Out[v][upt[q]] += alpha * sum over the entries e at point q of
// scale[atom] * (u[e] . C[atom][v]).  One thread per unique point and 8
// vectors: the point's entry list (atom and scaled u, in point order, so one
// dependent load instead of three) is read once for the 8.
constexpr int kSV = 8;   // vectors per thread in the scatter
template <typename T>
__global__ __launch_bounds__(256) void proj_scatter(ProjDev P, const double* __restrict__ C, T* Out, long long ld,
                                                    int nvec, double alpha) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  const int v0 = blockIdx.y * kSV;
  if (q >= P.nupts) return;
  const int t0 = P.upt_ptr[q], t1 = P.upt_ptr[q + 1];
  const long long pt = P.upt[q];
  // the read half of the read-modify-write goes out with the entry loads
  T ov[kSV];
#pragma unroll
  for (int u = 0; u < kSV; ++u) ov[u] = Out[(long long)min(v0 + u, nvec - 1) * ld + pt];
  double acc[kSV];
#pragma unroll
  for (int u = 0; u < kSV; ++u) acc[u] = 0.0;
  for (int t = t0; t < t1; ++t) {
    const int a = P.se_atom[t];
    const double u0 = P.se_u[3 * t], u1 = P.se_u[3 * t + 1], u2 = P.se_u[3 * t + 2];
#pragma unroll
    for (int u = 0; u < kSV; ++u) {
      const int v = min(v0 + u, nvec - 1);
      const double* c = C + ((long long)a * nvec + v) * 3;
      acc[u] += u0 * c[0] + u1 * c[1] + u2 * c[2];
    }
  }
#pragma unroll
  for (int u = 0; u < kSV; ++u) {
    if (v0 + u >= nvec) break;
    Out[(long long)(v0 + u) * ld + pt] = (T)((double)ov[u] + alpha * acc[u]);
  }
}

template <typename T>
int gather_impl(void* proj, const T* Y, long long ld, int nvec, double* C, void* stream) {
  const ProjDev* P = static_cast<const ProjDev*>(proj);
  PC_CHECK_ARG(P && Y && C, "null pointer");
  if (P->natoms == 0 || nvec == 0) return pc::PC_OK;
  const long long groups = (nvec + kGV - 1) / kGV;
  auto launch = [&](auto gw) -> int {
    constexpr int GW = decltype(gw)::value, NA = kGW / GW;
    const int step = (int)std::max<long long>(1, pc::kMaxGrid / groups) * NA;   // atoms per launch
    for (int a0 = 0; a0 < P->natoms; a0 += step) {
      ProjDev part = *P;
      part.atom_ptr += a0;
      part.natoms = std::min(step, P->natoms - a0);
      const dim3 grid((unsigned)(((part.natoms + NA - 1) / NA * groups + 7) / 8 * 8));
      hipLaunchKernelGGL((proj_gather<T, GW>), grid, dim3(64 * kGW), 0, static_cast<hipStream_t>(stream), part, Y, ld,
                         nvec, C + (long long)a0 * nvec * 3);
      PC_LAUNCH_CHECK();
    }
    return pc::PC_OK;
  };
  // As many wavefronts per atom as its support has rounds of 64, by the mean: more
  // only add sums and barriers, fewer wait for one round after the other.  FP32, 275
  // vectors, with 1, 2 and 4: 1,500 atoms of 20 points 75, 123, 223 us; 500 of 203
  // points 99, 97, 106; 163 of 478 points 75, 69, 65; of 905 points 126, 115, 107.
  const int mean = P->nent / P->natoms;
  return mean <= 64    ? launch(std::integral_constant<int, 1>{})
         : mean <= 256 ? launch(std::integral_constant<int, 2>{})
                       : launch(std::integral_constant<int, kGW>{});
}

template <typename T>
int scatter_impl(void* proj, const double* C, T* Out, long long ld, int nvec, double alpha, void* stream) {
  const ProjDev* P = static_cast<const ProjDev*>(proj);
  PC_CHECK_ARG(P && C && Out, "null pointer");
  if (P->nupts == 0 || nvec == 0) return pc::PC_OK;
  dim3 grid((P->nupts + 255) / 256, (nvec + kSV - 1) / kSV);
  hipLaunchKernelGGL(proj_scatter<T>, grid, dim3(256), 0, static_cast<hipStream_t>(stream), *P, C, Out, ld, nvec,
                     alpha);
  PC_LAUNCH_CHECK();
  return pc::PC_OK;
}

}  // namespace

extern "C" {

// atom_ptr[natoms+1] groups entries by atom; ent_pt[nent] are point indices in
// [0, npts); ent_u[3*nent] the (u_x,u_y,u_z) values; scale[natoms] = h^3/Zvalue.
int pc_proj_create(int natoms, const int* atom_ptr, const int* ent_pt, const double* ent_u, const double* scale,
                   long long npts, void** out_proj) {
  PC_CHECK_ARG(out_proj && atom_ptr && scale, "null pointer");
  PC_CHECK_ARG(natoms >= 0, "natoms < 0");
  const int nent = atom_ptr[natoms];
  PC_CHECK_ARG(nent >= 0 && (nent == 0 || (ent_pt && ent_u)), "bad entries");
  std::vector<int> ent_atom(nent);
  for (int a = 0; a < natoms; ++a) {
    PC_CHECK_ARG(atom_ptr[a] <= atom_ptr[a + 1], "atom_ptr not monotone");
    for (int e = atom_ptr[a]; e < atom_ptr[a + 1]; ++e) ent_atom[e] = a;
  }
  for (int e = 0; e < nent; ++e) PC_CHECK_ARG(ent_pt[e] >= 0 && ent_pt[e] < npts, "entry point out of range");
  std::vector<int> order(nent);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return ent_pt[x] < ent_pt[y]; });
  std::vector<int> upt, upt_ptr;
  for (int t = 0; t < nent; ++t) {
    if (t == 0 || ent_pt[order[t]] != ent_pt[order[t - 1]]) {
      upt.push_back(ent_pt[order[t]]);
      upt_ptr.push_back(t);
    }
  }
  upt_ptr.push_back(nent);
  ProjDev* P = new ProjDev();
  P->natoms = natoms; P->nent = nent; P->nupts = (int)upt.size();
  hipError_t e = hipSuccess;
  auto alloc_copy = [&](void** dst, const void* src, size_t bytes) {
    if (e != hipSuccess) return;
    e = hipMalloc(dst, std::max<size_t>(bytes, 8));
    if (e == hipSuccess && bytes) e = hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice);
  };
  alloc_copy((void**)&P->atom_ptr, atom_ptr, (natoms + 1) * sizeof(int));
  alloc_copy((void**)&P->ent_pt, ent_pt, nent * sizeof(int));
  alloc_copy((void**)&P->ent_u, ent_u, 3 * (size_t)nent * sizeof(double));
  alloc_copy((void**)&P->ent_atom, ent_atom.data(), nent * sizeof(int));
  alloc_copy((void**)&P->scale, scale, natoms * sizeof(double));
  alloc_copy((void**)&P->upt, upt.data(), upt.size() * sizeof(int));
  alloc_copy((void**)&P->upt_ptr, upt_ptr.data(), upt_ptr.size() * sizeof(int));
  alloc_copy((void**)&P->upt_ent, order.data(), nent * sizeof(int));
  std::vector<int> se_atom(nent);
  std::vector<double> se_u(3 * (size_t)nent);
  for (int t = 0; t < nent; ++t) {
    const int e = order[t], a = ent_atom[e];
    se_atom[t] = a;
    for (int m = 0; m < 3; ++m) se_u[3 * (size_t)t + m] = scale[a] * ent_u[3 * (size_t)e + m];
  }
  alloc_copy((void**)&P->se_atom, se_atom.data(), nent * sizeof(int));
  alloc_copy((void**)&P->se_u, se_u.data(), 3 * (size_t)nent * sizeof(double));
  if (e != hipSuccess) {
    pc::set_error(std::string("pc_proj_create: ") + hipGetErrorString(e));
    return pc::PC_ERR_HIP;
  }
  *out_proj = P;
  return pc::PC_OK;
}

int pc_proj_destroy(void* proj) {
  ProjDev* P = static_cast<ProjDev*>(proj);
  if (!P) return pc::PC_OK;
  (void)hipFree(P->atom_ptr); (void)hipFree(P->ent_pt); (void)hipFree(P->ent_u); (void)hipFree(P->ent_atom);
  (void)hipFree(P->scale); (void)hipFree(P->upt); (void)hipFree(P->upt_ptr); (void)hipFree(P->upt_ent);
  (void)hipFree(P->se_atom); (void)hipFree(P->se_u);
  delete P;
  return pc::PC_OK;
}

int pc_proj_ncols(void* proj, int* out_ncols) {
  const ProjDev* P = static_cast<const ProjDev*>(proj);
  PC_CHECK_ARG(P && out_ncols, "null pointer");
  *out_ncols = 3 * P->natoms;
  return pc::PC_OK;
}

int pc_proj_gather_f64(void* proj, const double* Y, long long ld, int nvec, double* C, void* stream) {
  return gather_impl<double>(proj, Y, ld, nvec, C, stream);
}
int pc_proj_gather_f32(void* proj, const float* Y, long long ld, int nvec, double* C, void* stream) {
  return gather_impl<float>(proj, Y, ld, nvec, C, stream);
}
int pc_proj_scatter_f64(void* proj, const double* C, double* Out, long long ld, int nvec, double alpha,
                        void* stream) {
  return scatter_impl<double>(proj, C, Out, ld, nvec, alpha, stream);
}
int pc_proj_scatter_f32(void* proj, const double* C, float* Out, long long ld, int nvec, double alpha,
                        void* stream) {
  return scatter_impl<float>(proj, C, Out, ld, nvec, alpha, stream);
}

}  // extern "C"
