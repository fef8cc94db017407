// The group-minimum selection for the Manhattan, Chebyshev and Minkowski arms.
// Their minima are of the arm's own values (launch_groupmin_tile), rounded to
// f32.
#include "knn_groupmin_select.hpp"

namespace mlrs {

template <typename T>
hipError_t launch_gm_select_metric(const GmSelectArgs<T>& a, int arm, hipStream_t s) {
    if (a.nq == 0) return hipSuccess;
    switch (arm) {
    case ARM_MANHATTAN: gm_select_k<T, T, ARM_MANHATTAN>(a, s); break;
    case ARM_CHEBYSHEV: gm_select_k<T, T, ARM_CHEBYSHEV>(a, s); break;
    case ARM_MINKOWSKI_INT: gm_select_k<T, T, ARM_MINKOWSKI_INT>(a, s); break;
    case ARM_MINKOWSKI_POW: gm_select_k<T, T, ARM_MINKOWSKI_POW>(a, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
template hipError_t launch_gm_select_metric<float>(const GmSelectArgs<float>&, int, hipStream_t);
template hipError_t launch_gm_select_metric<double>(const GmSelectArgs<double>&, int, hipStream_t);

}  // namespace mlrs
