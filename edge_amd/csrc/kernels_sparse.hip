// The sparse element kernels' dispatch by order (the kernels:
// kernels_sparse_impl.hpp, one translation unit per order).
#include "kernels_sparse.hpp"

namespace edge {
namespace {

template <typename T>
int dispatch(int op, const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
             const T* proj_in, hipStream_t st) {
  switch (s.order) {
    case 2: return launch_sp<T, 2>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
    case 3: return launch_sp<T, 3>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
    case 4: return launch_sp<T, 4>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
    case 5: return launch_sp<T, 5>(op, s, x, first, n, dt, dofs, t_int, proj_in, st);
  }
  return fail(EDGE_ERR_UNSUPPORTED, "order");
}

}  // namespace

// Every order and run count but FP64 order 5 with one run: its registers and
// LDS leave one workgroup per CU, whose loads and stores nothing overlaps
// (7.77 ms per 4 steps of 196,608 tets against 7.83 for the element-batched
// kernels, 120 against 117 us per step of 1,296).  One order lower one run is
// faster here (897 -> 605 us per step of 131,712 tets, 68 -> 52 of 1,296).
// (Nor FP64 order 5 with 16 runs: no kernel that reads tInt, for the separate
// neighbour step, fits it, so the set-up refuses it.)
bool sp_supported(int order, int n_runs, int precision) {
  return (precision == 32 || (precision == 64 && !(order == 5 && n_runs != 8))) && order >= 2 && order <= 5 &&
         (n_runs == 1 || n_runs == 8 || n_runs == 16);
}

template <typename T>
int launch_local_sp(const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T dt, T* dofs, T* t_int,
                    hipStream_t st) {
  return dispatch<T>(kSpLocal, s, x, first, n, dt, dofs, t_int, nullptr, st);
}

template <typename T>
int launch_neigh_sp(const SolverDev<T>& s, const SpDev<T>& x, int64_t first, int64_t n, T* dofs, hipStream_t st) {
  return dispatch<T>(kSpNeigh, s, x, first, n, T(0), dofs, nullptr, x.proj, st);
}

template <typename T>
int launch_fused_sp(const SolverDev<T>& s, const SpDev<T>& x, T dt, const T* proj_in, T* dofs, T* t_int,
                    hipStream_t st) {
  return dispatch<T>(kSpFused, s, x, 0, s.n_el, dt, dofs, t_int, proj_in, st);
}

#define EDGE_SP(T)                                                                                                  \
  template int launch_local_sp<T>(const SolverDev<T>&, const SpDev<T>&, int64_t, int64_t, T, T*, T*, hipStream_t); \
  template int launch_neigh_sp<T>(const SolverDev<T>&, const SpDev<T>&, int64_t, int64_t, T*, hipStream_t);         \
  template int launch_fused_sp<T>(const SolverDev<T>&, const SpDev<T>&, T, const T*, T*, T*, hipStream_t);
EDGE_SP(float)
EDGE_SP(double)
#undef EDGE_SP

}  // namespace edge
