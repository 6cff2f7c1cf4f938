// nw_resident_f32k64.hip -- the resident multi-step kernel, FP32 fields and FP64 LSRK registers.
#include "nw_resident_kernel.hpp"

namespace nw {
ResidentKernel resident_kernel_f32k64(int n1, int em, bool affine) { return resident_pick_n1<float, double>(n1, em, affine); }
int resident_upload_f32k64(const GllTables& t) { return device_upload_tables(t); }
}  // namespace nw
