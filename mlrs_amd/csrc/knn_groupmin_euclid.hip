// The group-minimum scan's Euclidean instances (also the cosine searches over
// unit rows, which carry no per-row scale).
#include "knn_groupmin_scan.hpp"

namespace mlrs {

hipError_t launch_gm_scan_euclid(const GmScanArgs& a, hipStream_t s) { return gm_launch<false>(a, s); }

}  // namespace mlrs
