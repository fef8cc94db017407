// The group-minimum scan's instances for cosine over rows in place: each value
// is scaled by its row's 1 / ||x||.
#include "knn_groupmin_scan.hpp"

namespace mlrs {

hipError_t launch_gm_scan_cosine(const GmScanArgs& a, hipStream_t s) { return gm_launch<true>(a, s); }

}  // namespace mlrs
