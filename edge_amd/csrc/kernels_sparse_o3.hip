// The sparse element kernels of order 3.
#include "kernels_sparse_impl.hpp"

namespace edge {
template int launch_sp<float, 3>(int, const SolverDev<float>&, const SpDev<float>&, int64_t, int64_t, float, float*,
                                 float*, const float*, hipStream_t);
}  // namespace edge
