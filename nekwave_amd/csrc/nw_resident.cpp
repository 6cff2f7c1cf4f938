// nw_resident.cpp -- host side of the resident multi-step kernel: dispatch, capacity, face table.
#include "nw_resident.hpp"

#include <algorithm>

namespace nw {

namespace {
ResidentKernel resident_kernel(int n1, int prec, int em, bool affine) {
    if (prec == kFP64) return resident_kernel_f64(n1, em, affine);
    if (prec == kFP32) return resident_kernel_f32(n1, em, affine);
    if (prec == kFP32K64) return resident_kernel_f32k64(n1, em, affine);
    return {};
}
}  // namespace

ResidentCapacity resident_capacity(int n1, int prec, int em, bool affine, int max_per_cu) {
    const ResidentKernel k = resident_kernel(n1, prec, em, affine);
    if (!k.per_cu) return {};
    int dev = 0, cus = 0, per = k.per_cu();
    if (hipGetDevice(&dev) != hipSuccess) return {};
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return {};
    if (max_per_cu > 0) per = std::min(per, max_per_cu);
    const int most = resident_range(n1, prec, affine).per_cu;
    const long long groups = (long long)per * cus, fits = groups * resident_em(em);
    return {groups, most > 0 ? std::min(fits, (long long)most * cus) : fits};
}

hipError_t launch_resident(int n1, int prec, int em, bool affine, const ResidentArgs& a, hipStream_t s) {
    const ResidentKernel k = resident_kernel(n1, prec, em, affine);
    if (!k.launch || a.nelt <= 0 || a.per < 1 || a.per > resident_em(em) || a.nsteps < 1 ||
        resident_xchg_bytes(n1, prec, a.nelt) > (2ll << 30))
        return hipErrorInvalidValue;
    return k.launch(a, s);
}

int resident_upload_tables(const GllTables& t) {
    int st = resident_upload_f64(t);
    if (st == NW_OK) st = resident_upload_f32(t);
    if (st == NW_OK) st = resident_upload_f32k64(t);
    return st;
}

bool resident_face_table(const int* fcode, int nelt, int n1, int elem_base, int4* out) {
    for (int x = 0; x < nelt * 6; ++x) {
        const int code = fcode[x];
        if (code == -1) {
            out[x] = make_int4(-1, 0, 0, 0);
            continue;
        }
        if (code < 0) return false;  // ghost face
        const int e2 = code >> 6, f2 = (code >> 3) & 7, o = code & 7;
        const int back = fcode[e2 * 6 + f2];
        if (back < 0 || (back >> 6) * 6 + ((back >> 3) & 7) != x) return false;
        int p0, q0, p1, q1, p2, q2;
        orient_map(o, n1, 0, 0, p0, q0);
        orient_map(o, n1, 1, 0, p1, q1);
        orient_map(o, n1, 0, 1, p2, q2);
        const int at = p0 + n1 * q0;
        out[x] = make_int4((elem_base + e2) * 6 + f2, at, p1 + n1 * q1 - at, p2 + n1 * q2 - at);
    }
    return true;
}

}  // namespace nw
