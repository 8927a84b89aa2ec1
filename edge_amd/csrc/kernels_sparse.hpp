// Element kernels that walk the non-zeros of the reference-element matrices
// (kernels_sparse_impl.hpp): data they need beside SolverDev, and the launchers.
#pragma once

#include "kernels.hpp"

namespace edge {
namespace phys {

// Per-element constants of the elastic update, [el / B][kSize][el % B] with
// B = block(runs): one run's lanes are different elements and read a constant
// of 64 of them at a time, the few elements of a tile of fused runs are
// contiguous.  In the solver's precision, each computed in FP64 and rounded
// once.  With J^-1
// the inverse Jacobian (j[k][d] = d xi_d / d x_k), n a face's outward normal,
// sc = -2 |A| / |J|, zp and zs the P and S impedances (1: the element's own
// side, 2: the other side):
//   0 + 3 k + d   j[k][d]
//   9 .. 12       -(lambda + 2 mu), -lambda, -mu, -1 / rho
//   13 + 14 f     n (3) | zs1 a_s, a_s, zp1 a_p - zs1 a_s, a_p - a_s
//                 with a_p = 1 / (zp1 + zp2), a_s = 1 / (zs1 + zs2) |
//                 sc n (3) | sc zs2 / rho, sc (zp2 - zs2) / rho |
//                 -sc zs1 / rho, -sc (zp1 - zs1) / rho
constexpr int kJinv = 0, kLam2 = 9, kLam = 10, kMu = 11, kIrho = 12, kFace = 13;
constexpr int kNrm = 0, kPrj = 3, kScN = 7, kOwn = 10, kOth = 12, kPerFace = 14;
constexpr int kSize = kFace + 4 * kPerFace;
constexpr int block(int n_runs) { return n_runs == 1 ? 64 : 1; }
inline int64_t values(int64_t n_el, int b) { return (n_el + b - 1) / b * b * kSize; }

// Face-orientation maps R_v (ec64_pack.hpp) as their diagonal blocks by
// face-basis degree p, row-major, padded: [4][kRotPad] (0: the identity).
constexpr int kRotPad = 56;
constexpr int rot_off(int p) { return p * (p + 1) * (2 * p + 1) / 6; }  // 0, 1, 5, 14, 30, 55

}  // namespace phys

// Vectors of four values per face projection (3 NF values, padded).
constexpr int sp_proj_vectors(int order) { return (3 * n_face_modes(order) + 3) / 4; }
// Values of the face projections per element.
constexpr int64_t sp_proj_values(int order, int n_runs) { return (int64_t)16 * sp_proj_vectors(order) * n_runs; }

template <typename T>
struct SpDev {
  const T* phys = nullptr;  // per-element constants
  const T* rot = nullptr;   // face-orientation maps
  // face projections [nEl][4][vectors][R][4] of this step (a local step
  // whose projections nothing reads: null)
  T* proj = nullptr;
  // tInt is written for every element, or only for those of need (a step
  // whose tInt nothing else reads)
  bool tint = true;
  const uint8_t* need = nullptr;  // [nEl], null: none
};

// One operation of one order (kernels_sparse_o*.hip).
constexpr int kSpLocal = 0, kSpNeigh = 1, kSpFused = 2;
template <typename T, int O>
int launch_sp(int op, const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
              const T* proj_in, hipStream_t st);

bool sp_supported(int order, int n_runs, int precision);
template <typename T>
int launch_local_sp(const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
                    hipStream_t st);
template <typename T>
int launch_neigh_sp(const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T* dofs, hipStream_t st);
// The neighbour step of step k - 1 (from proj_in) and the local step of step
// k (projections to x.proj) as one launch over all elements.
template <typename T>
int launch_fused_sp(const SolverDev<T>& s, const SpDev<T>& x, T dt, const T* proj_in, T* dofs, T* t_int,
                    hipStream_t st);

}  // namespace edge
