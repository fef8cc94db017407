// The group-minimum scan's instances.
#include "knn_groupmin_scan.hpp"

namespace mlrs {

hipError_t launch_gm_scan(const GmScanArgs& a, hipStream_t s) { return gm_launch(a, s); }

}  // namespace mlrs
