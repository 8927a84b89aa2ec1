// The sparse element kernels of order 4 in FP64.
#define EDGE_SP_WAVES 8
#define EDGE_SP_LOW_FIRST 1
#include "kernels_sparse_impl.hpp"

namespace edge {
template int launch_sp<double, 4>(int, const SolverDev<double>&, const SpDev<double>&, int64_t, int64_t, double,
                                  double*, double*, const double*, hipStream_t);
}  // namespace edge
