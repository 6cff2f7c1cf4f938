// nw_resident_f32.hip -- the resident multi-step kernel in FP32.
#include "nw_resident_kernel.hpp"

namespace nw {
ResidentKernel resident_kernel_f32(int n1, int em, bool affine) { return resident_pick_n1<float, float>(n1, em, affine); }
int resident_upload_f32(const GllTables& t) { return device_upload_tables(t); }
}  // namespace nw
