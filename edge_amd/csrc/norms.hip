// FP64 reductions over a DOF array [nEl][9][N][R]: L2 norms, energies and the
// errors against plane waves.  Every block writes its partial sums; the last
// kernel adds them in an order that the block count fixes (sixteen strided
// sets of blocks, then the sixteen sums), so a result depends on the arrays and
// the sizes only.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <new>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"

namespace {

constexpr int kThreads = 256;

// Adds x over the lanes of a wave whose index is the same modulo n_crs (a
// power of two); every lane holds the sum.
__device__ __forceinline__ double add_lanes(double x, int n_crs) {
  for (int o = n_crs; o < 64; o *= 2) x += __shfl_xor(x, o);
  return x;
}

// Partial sums of |J| M_n (a - b)^2 and |J| M_n b^2 of quantity blockIdx.y
// over the block's elements, per run.  Bound by memory: consecutive threads
// read consecutive values of one quantity (a thread keeps its run, the run
// count divides the block), and all of them work at every run count; one
// thread per (quantity, run) that walked its values one after the other used
// 9 of 256 threads with one run.  24,576 tets, order 5, 16 runs: 0.42 -> 0.23
// ms.
template <typename TA, typename TB>
__global__ __launch_bounds__(kThreads) void k_l2(int64_t n_el, int n_md, int n_crs, const double* __restrict__ jdet,
                                                 const double* __restrict__ mass, const TA* __restrict__ a,
                                                 const TB* __restrict__ b, double* __restrict__ part) {
  __shared__ double sums[kThreads / 64][2][64];
  const int64_t per = (n_el + gridDim.x - 1) / gridDim.x;
  const int64_t e0 = min(n_el, blockIdx.x * per), e1 = min(n_el, e0 + per);
  const unsigned q = blockIdx.y, nr = n_md * n_crs, tot = (unsigned)(e1 - e0) * nr;
  double d2 = 0, r2 = 0;
#pragma unroll 4
  for (unsigned k = threadIdx.x; k < tot; k += kThreads) {
    const unsigned el = k / nr, rem = k - el * nr;
    const size_t at = ((size_t)(e0 + el) * 9 + q) * nr + rem;
    const double av = (double)a[at], bv = b ? (double)b[at] : av;
    const double w = fabs(jdet[e0 + el]) * mass[rem / n_crs];
    d2 += w * (av - bv) * (av - bv);
    r2 += w * bv * bv;
  }
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  sums[wave][0][lane] = add_lanes(d2, n_crs);
  sums[wave][1][lane] = add_lanes(r2, n_crs);
  __syncthreads();
  if (threadIdx.x < 2 * n_crs) {
    const int i = threadIdx.x / n_crs, r = threadIdx.x % n_crs;
    double s = 0;
    for (int w = 0; w < kThreads / 64; w++) s += sums[w][i][r];
    part[((size_t)blockIdx.x * 2 + i) * 9 * n_crs + q * n_crs + r] = s;
  }
}

// Partial sums per run of the kinetic energy 1/2 rho |v|^2 and the strain
// energy 1/2 sigma : C^-1 : sigma (isotropic compliance
// C^-1 sigma = sigma / (2 mu) - lambda / (2 mu (3 lambda + 2 mu)) tr(sigma) I),
// integrated exactly through |J| and the diagonal reference mass matrix.
// Threads take (element, mode, run) in memory order, as in k_l2 (same size: 0.33
// -> 0.093 ms).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_energy(int64_t n_el, int n_md, int n_crs,
                                                     const double* __restrict__ jdet, const double* __restrict__ mass,
                                                     const double* __restrict__ mat, const T* __restrict__ dofs,
                                                     double* __restrict__ part) {
  __shared__ double sums[kThreads / 64][2][64];
  const int64_t per = (n_el + gridDim.x - 1) / gridDim.x;
  const int64_t e0 = min(n_el, blockIdx.x * per), e1 = min(n_el, e0 + per);
  const unsigned nr = n_md * n_crs, tot = (unsigned)(e1 - e0) * nr;
  double ek = 0, es = 0;
  for (unsigned k = threadIdx.x; k < tot; k += kThreads) {
    const unsigned rel = k / nr, rem = k - rel * nr;
    const int64_t el = e0 + rel;
    double x[9];
#pragma unroll
    for (int q = 0; q < 9; q++) x[q] = (double)dofs[((size_t)el * 9 + q) * nr + rem];
    const double rho = mat[el], lam = mat[n_el + el], mu = mat[2 * n_el + el];
    const double c1 = 0.5 / mu, c2 = lam / (2 * mu * (3 * lam + 2 * mu));
    const double w = fabs(jdet[el]) * mass[rem / n_crs];
    const double tr = x[0] + x[1] + x[2];
    const double ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + 2 * (x[3] * x[3] + x[4] * x[4] + x[5] * x[5]);
    ek += w * 0.5 * rho * (x[6] * x[6] + x[7] * x[7] + x[8] * x[8]);
    es += w * 0.5 * (c1 * ss - c2 * tr * tr);
  }
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  sums[wave][0][lane] = add_lanes(ek, n_crs);
  sums[wave][1][lane] = add_lanes(es, n_crs);
  __syncthreads();
  if (threadIdx.x < 2 * n_crs) {
    const int i = threadIdx.x / n_crs, r = threadIdx.x % n_crs;
    double s = 0;
    for (int w = 0; w < kThreads / 64; w++) s += sums[w][i][r];
    part[((size_t)blockIdx.x * 2 + i) * n_crs + r] = s;
  }
}

// Partial L1, squared L2 and Linf errors per (quantity, run) at the
// quadrature points of every element against a sum of plane waves
// q(x, t) = sum_w r_w sin(k_w . x - omega_w t + phase_w) (per run:
// waves [R][n_waves][14] = r[9], k[3], omega, phase).
//
// A lane holds one (element, run) column, a workgroup 64 of them and three
// quantities (blockIdx.y), their DOFs in LDS.  A wave takes kPts points at a
// time: the points and the basis are the same for all lanes (scalar loads, a
// matrix entry is an operand of the FMA), one DOF read from LDS serves kPts
// FMAs, and a point's sine is taken once for the three quantities.  Bound by
// the FP64 FMAs (9 N per point and column) and sines, and by the scalar loads
// of the basis.  24,576 tets, order 5, 16 runs, 216 points: 3.0 ms; a thread
// per (quantity, run) that took the sine again for every quantity and read a
// DOF per FMA, 27.9 ms.
// Points per turn: 12 keep 36 sums in registers.
constexpr int kPts = 12, kQ = 3, kErrWaves = kThreads / 64;

template <typename T, int N>
__global__ __launch_bounds__(kThreads, 2) void k_err(int64_t n_el, int n_crs, int n_pts,
                                                     const double* __restrict__ geo, const double* __restrict__ jdet,
                                                     const double* __restrict__ pts,    // [groups][kPts][4]
                                                     const double* __restrict__ basis,  // [groups][N][kPts]
                                                     int n_waves, const double* __restrict__ waves, double time,
                                                     const T* __restrict__ dofs, double* __restrict__ part) {
  constexpr int LD = 65;  // columns per row: writes down a column go to different banks
  __shared__ double a[kQ * N * LD];
  __shared__ double sine[kErrWaves][kPts][64];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int els = 64 / n_crs, r = lane % n_crs, q0 = blockIdx.y * kQ;
  const int groups = (n_pts + kPts - 1) / kPts;
  const int64_t tiles = (n_el + els - 1) / els, per = (tiles + gridDim.x - 1) / gridDim.x;
  const int64_t t1 = min(tiles, (blockIdx.x + 1) * per);
  double l1[kQ] = {}, l2[kQ] = {}, li[kQ] = {};
  for (int64_t tile = blockIdx.x * per; tile < t1; tile++) {
    const int64_t first = tile * els;
    const int n = (int)min((int64_t)els, n_el - first);
    __syncthreads();  // the previous tile's DOFs have been read
    for (int k = threadIdx.x; k < n * kQ * N * n_crs; k += kThreads) {
      const int row = k / n_crs, e = row / (kQ * N);
      a[(row - e * kQ * N) * LD + e * n_crs + k % n_crs] =
          (double)dofs[((size_t)(first + e) * 9 + q0) * N * n_crs + (k - e * kQ * N * n_crs)];
    }
    __syncthreads();
    const bool on = lane < n * n_crs;
    const int64_t el = first + (on ? lane / n_crs : 0);
    double gm[12];
#pragma unroll
    for (int i = 0; i < 12; i++) gm[i] = geo[el * 12 + i];
    const double j = fabs(jdet[el]);
    for (int g = w; g < groups; g += kErrWaves) {
      double d[kQ][kPts] = {};
      const double* bs = basis + (size_t)g * N * kPts;
      const double* col = a + (on ? lane : 0);
#pragma unroll 5
      for (int m = 0; m < N; m++) {
        double v[kQ];
#pragma unroll
        for (int q = 0; q < kQ; q++) v[q] = col[(q * N + m) * LD];
#pragma unroll
        for (int p = 0; p < kPts; p++)
#pragma unroll
          for (int q = 0; q < kQ; q++) d[q][p] += bs[m * kPts + p] * v[q];
      }
      const double* pt = pts + (size_t)g * kPts * 4;
      for (int k = 0; k < n_waves; k++) {
        const double* wv = waves + ((size_t)r * n_waves + k) * 14;
        const double k0 = wv[9], k1 = wv[10], k2 = wv[11], wt = wv[12] * time, ph = wv[13];
#pragma unroll 2
        for (int p = 0; p < kPts; p++) {
          double x[3];
#pragma unroll
          for (int i = 0; i < 3; i++)
            x[i] = gm[i] + pt[4 * p] * gm[3 + i] + pt[4 * p + 1] * gm[6 + i] + pt[4 * p + 2] * gm[9 + i];
          sine[w][p][lane] = sin(k0 * x[0] + k1 * x[1] + k2 * x[2] - wt + ph);
        }
#pragma unroll
        for (int q = 0; q < kQ; q++) {
          const double amp = wv[q0 + q];
#pragma unroll
          for (int p = 0; p < kPts; p++) d[q][p] -= amp * sine[w][p][lane];
        }
      }
      if (on) {
#pragma unroll
        for (int p = 0; p < kPts; p++) {
          if (g * kPts + p >= n_pts) continue;
          const double wj = pt[4 * p + 3] * j;
#pragma unroll
          for (int q = 0; q < kQ; q++) {
            const double e = fabs(d[q][p]);
            l1[q] += wj * e;
            l2[q] += wj * e * e;
            li[q] = fmax(li[q], e);
          }
        }
      }
    }
  }
  __syncthreads();
  double* red = a;  // [kErrWaves][3][kQ][n_crs]
#pragma unroll
  for (int q = 0; q < kQ; q++) {
    l1[q] = add_lanes(l1[q], n_crs);
    l2[q] = add_lanes(l2[q], n_crs);
    for (int o = n_crs; o < 64; o *= 2) li[q] = fmax(li[q], __shfl_xor(li[q], o));
    if (lane < n_crs) {
      red[((w * 3 + 0) * kQ + q) * n_crs + lane] = l1[q];
      red[((w * 3 + 1) * kQ + q) * n_crs + lane] = l2[q];
      red[((w * 3 + 2) * kQ + q) * n_crs + lane] = li[q];
    }
  }
  __syncthreads();
  const int per_wave = 3 * kQ * n_crs;
  if ((int)threadIdx.x < per_wave) {
    const int i = threadIdx.x, kind = i / (kQ * n_crs);
    double s = red[i];
    for (int k = 1; k < kErrWaves; k++) s = kind == 2 ? fmax(s, red[k * per_wave + i]) : s + red[k * per_wave + i];
    part[((size_t)blockIdx.x * 3 + kind) * 9 * n_crs + q0 * n_crs + i % (kQ * n_crs)] = s;
  }
}

// out[i] = sum over k of part[k][i] (from `first_max` on: the largest), 64
// entries per block: sixteen rows at a time, then their sums in order.
constexpr int kRows = 16;
__global__ __launch_bounds__(64 * kRows) void k_sum(const double* __restrict__ part, unsigned nblk, int width,
                                                    int first_max, double* __restrict__ out) {
  __shared__ double s[kRows][64];
  const int c = threadIdx.x % 64, row = threadIdx.x / 64, i = blockIdx.x * 64 + c;
  const bool most = i >= first_max;
  double acc = 0;
  if (i < width) {
#pragma unroll 8
    for (unsigned k = row; k < nblk; k += kRows) {
      const double x = part[(size_t)k * width + i];
      acc = most ? fmax(acc, x) : acc + x;
    }
  }
  s[row][c] = acc;
  __syncthreads();
  if (row || i >= width) return;
  for (int k = 1; k < kRows; k++) acc = most ? fmax(acc, s[k][c]) : acc + s[k][c];
  out[i] = acc;
}

template <typename TA, typename TB>
void l2_launch(const edge::SolverRef& s, const void* a, const void* b, double* part, unsigned nblk, hipStream_t st) {
  hipLaunchKernelGGL((k_l2<TA, TB>), dim3(nblk, 9), dim3(kThreads), 0, st, s.n_el, s.n_modes, s.n_runs, s.jdet, s.mass,
                     (const TA*)a, (const TB*)b, part);
}

// Device scratch of one call, freed on every way out.
struct Scratch {
  double* p = nullptr;
  ~Scratch() { (void)hipFree(p); }
};

// Sums (of the last `n_max` of the `width` entries: the largest) of the
// partials in `part` on the device, to h.
int sum_to_host(const double* part, unsigned nblk, int width, int n_max, double* d_out, double* h, hipStream_t st) {
  if (int rc = edge::sum_partials(part, nblk, width, width - n_max, d_out, st)) return rc;
  EDGE_HIP_TRY(hipMemcpyAsync(h, d_out, sizeof(double) * width, hipMemcpyDeviceToHost, st));
  EDGE_HIP_TRY(hipStreamSynchronize(st));
  return EDGE_OK;
}

}  // namespace

namespace edge {
int l2_partials(edge_el_solver* h, const void* a, int prec_a, const void* b, int prec_b, double* part, unsigned nblk,
                hipStream_t st) {
  SolverRef s;
  if (int rc = solver_ref(h, &s)) return rc;
  const int pb = b ? prec_b : prec_a;
  if (prec_a == 64)
    pb == 64 ? l2_launch<double, double>(s, a, b, part, nblk, st) : l2_launch<double, float>(s, a, b, part, nblk, st);
  else
    pb == 64 ? l2_launch<float, double>(s, a, b, part, nblk, st) : l2_launch<float, float>(s, a, b, part, nblk, st);
  EDGE_HIP_TRY(hipGetLastError());
  return EDGE_OK;
}

int sum_partials(const double* part, unsigned nblk, int width, int first_max, double* out, hipStream_t st) {
  hipLaunchKernelGGL(k_sum, dim3((width + 63) / 64), dim3(64 * kRows), 0, st, part, nblk, width, first_max, out);
  EDGE_HIP_TRY(hipGetLastError());
  return EDGE_OK;
}
}  // namespace edge

extern "C" int edge_el_l2_norms(edge_el_solver* h, const void* a, int prec_a, const void* b, int prec_b,
                                double* diff_sq, double* ref_sq, void* stream) {
  edge::SolverRef s;
  if (int rc = edge::solver_ref(h, &s)) return rc;
  if (!s.jdet) return edge::fail(EDGE_ERR_UNSUPPORTED, "norms need a solver built from geometry");
  if (!a || (prec_a != 32 && prec_a != 64) || (b && prec_b != 32 && prec_b != 64))
    return edge::fail(EDGE_ERR_ARG, "norm arguments");
  hipStream_t st = (hipStream_t)stream;
  const int nqr = 9 * s.n_runs;
  const unsigned nblk = edge::kL2Blocks;
  Scratch d;
  EDGE_HIP_TRY(hipMalloc(&d.p, sizeof(double) * 2 * nqr * (nblk + 1)));
  double* out = d.p + (size_t)2 * nqr * nblk;
  std::vector<double> sums(2 * nqr);
  if (int rc = edge::l2_partials(h, a, prec_a, b, prec_b, d.p, nblk, st)) return rc;
  if (int rc = sum_to_host(d.p, nblk, 2 * nqr, 0, out, sums.data(), st)) return rc;
  if (diff_sq) std::copy_n(sums.data(), nqr, diff_sq);
  if (ref_sq) std::copy_n(sums.data() + nqr, nqr, ref_sq);
  return EDGE_OK;
}

extern "C" int edge_el_energy(edge_el_solver* h, const void* dofs, double* kinetic, double* strain, void* stream) {
  edge::SolverRef s;
  if (int rc = edge::solver_ref(h, &s)) return rc;
  if (!s.jdet || !s.mat) return edge::fail(EDGE_ERR_UNSUPPORTED, "the energy needs a solver built from materials");
  if (!dofs) return edge::fail(EDGE_ERR_ARG, "device DOFs missing");
  const int R = s.n_runs;
  hipStream_t st = (hipStream_t)stream;
  const unsigned nblk = 1024;
  Scratch d;
  EDGE_HIP_TRY(hipMalloc(&d.p, sizeof(double) * 2 * R * (nblk + 1)));
  if (s.precision == 64)
    hipLaunchKernelGGL(k_energy<double>, dim3(nblk), dim3(kThreads), 0, st, s.n_el, s.n_modes, R, s.jdet, s.mass, s.mat,
                       (const double*)dofs, d.p);
  else
    hipLaunchKernelGGL(k_energy<float>, dim3(nblk), dim3(kThreads), 0, st, s.n_el, s.n_modes, R, s.jdet, s.mass, s.mat,
                       (const float*)dofs, d.p);
  EDGE_HIP_TRY(hipGetLastError());
  std::vector<double> sums(2 * R);
  if (int rc = sum_to_host(d.p, nblk, 2 * R, 0, d.p + (size_t)2 * R * nblk, sums.data(), st)) return rc;
  if (kinetic) std::copy_n(sums.data(), R, kinetic);
  if (strain) std::copy_n(sums.data() + R, R, strain);
  return EDGE_OK;
}

extern "C" int edge_el_error_norms(edge_el_solver* h, const void* dofs, int32_t n1d, int32_t n_waves,
                                   const double* waves, double time, double* l1, double* l2sq, double* linf,
                                   void* stream) {
  edge::SolverRef s;
  if (int rc = edge::solver_ref(h, &s)) return rc;
  if (!s.jdet || !s.geo) return edge::fail(EDGE_ERR_UNSUPPORTED, "error norms need a solver built from geometry");
  if (!dofs || n_waves < 0 || (n_waves > 0 && !waves) || n1d < 0 || n1d > 32)
    return edge::fail(EDGE_ERR_ARG, "error-norm arguments");
  const int R = s.n_runs, nqr = 9 * R, N = s.n_modes;
  const int n1 = n1d ? n1d : s.order + 1, np = n1 * n1 * n1, groups = (np + kPts - 1) / kPts;
  std::vector<double> pts(3 * np), w(np), basis((size_t)np * N);
  int rc = edge_dg_quad_tet(n1, pts.data(), w.data());
  if (rc == EDGE_OK) rc = edge_dg_eval_basis(s.order, np, pts.data(), basis.data());
  if (rc) return rc;
  // one block: points and weights, basis (both in groups of kPts, the last
  // one filled up with zeros), waves; then the partial sums and the sums
  const size_t n_pt = (size_t)groups * kPts * 4, n_bs = (size_t)groups * kPts * N, n_wv = (size_t)R * n_waves * 14;
  const size_t n_in = n_pt + n_bs + n_wv;
  hipStream_t st = (hipStream_t)stream;
  const unsigned nblk = 1024;
  Scratch d;
  EDGE_HIP_TRY(hipMalloc(&d.p, sizeof(double) * (n_in + (size_t)3 * nqr * (nblk + 1))));
  // (the number of waves is the caller's: no allocation throws for it)
  const std::unique_ptr<double[]> in(new (std::nothrow) double[n_in]());
  if (!in) return edge::fail(EDGE_ERR_NOMEM, "error norms: waves");
  for (int p = 0; p < np; p++) {
    for (int i = 0; i < 3; i++) in[4 * (size_t)p + i] = pts[3 * p + i];
    in[4 * (size_t)p + 3] = w[p];
    for (int n = 0; n < N; n++)
      in[n_pt + ((size_t)(p / kPts) * N + n) * kPts + p % kPts] = basis[(size_t)p * N + n];
  }
  if (n_wv) std::copy_n(waves, n_wv, in.get() + n_pt + n_bs);
  double *part = d.p + n_in, *out = part + (size_t)3 * nqr * nblk;
  EDGE_HIP_TRY(hipMemcpyAsync(d.p, in.get(), sizeof(double) * n_in, hipMemcpyHostToDevice, st));
  const double *d_pt = d.p, *d_bs = d.p + n_pt, *d_wv = d_bs + n_bs;
  auto launch = [&](auto t, auto n) {
    using T = decltype(t);
    hipLaunchKernelGGL((k_err<T, decltype(n)::value>), dim3(nblk, 9 / kQ), dim3(kThreads), 0, st, s.n_el, R, np, s.geo,
                       s.jdet, d_pt, d_bs, n_waves, d_wv, time, (const T*)dofs, part);
  };
  auto by_order = [&](auto t) {
    if (s.order == 2) launch(t, std::integral_constant<int, 4>{});
    if (s.order == 3) launch(t, std::integral_constant<int, 10>{});
    if (s.order == 4) launch(t, std::integral_constant<int, 20>{});
    if (s.order == 5) launch(t, std::integral_constant<int, 35>{});
  };
  s.precision == 64 ? by_order(double{}) : by_order(float{});
  EDGE_HIP_TRY(hipGetLastError());
  std::vector<double> sums(3 * nqr);
  if ((rc = sum_to_host(part, nblk, 3 * nqr, nqr, out, sums.data(), st))) return rc;
  if (l1) std::copy_n(sums.data(), nqr, l1);
  if (l2sq) std::copy_n(sums.data() + nqr, nqr, l2sq);
  if (linf) std::copy_n(sums.data() + 2 * nqr, nqr, linf);
  return EDGE_OK;
}
