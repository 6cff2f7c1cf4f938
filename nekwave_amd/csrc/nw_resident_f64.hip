// nw_resident_f64.hip -- the resident multi-step kernel in FP64.
#include "nw_resident_kernel.hpp"

namespace nw {
ResidentKernel resident_kernel_f64(int n1, int em, bool affine) { return resident_pick_n1<double, double>(n1, em, affine); }
int resident_upload_f64(const GllTables& t) { return device_upload_tables(t); }
}  // namespace nw
