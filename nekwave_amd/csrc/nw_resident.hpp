// nw_resident.hpp -- launch interface of the resident multi-step kernel.
//
// Where every element of a set of meshes fits on chip at once, one launch
// advances them any number of LSRK45 steps: a workgroup owns a few elements for
// the whole launch (fields in LDS, LSRK registers in VGPRs), and only the face
// traces travel, as self-validating 8-byte packets between workgroups.
#pragma once

#include "nw_fused.hpp"

namespace nw {

// Bytes of the exchange buffer of nelt elements: per face point and epoch parity
// six values in 8-byte packets, 4 of value and 4 of epoch.
constexpr long long resident_xchg_bytes(int n1, int prec, long long nelt) {
    return 2 * nelt * 6 * n1 * n1 * (prec == kFP64 ? 96 : 48);
}

// What one launch needs.  Element and face indices are relative to the segment.
struct ResidentArgs {
    const void* uin;          // node-major state (6 R per node), as the fused kernel's
    void* uout;               // another buffer: written only by a launch that completes
    const double* rec;        // per element: 26 words, as the fused kernel's
    const void* fw;           // per element face: 4 flux weights (R)
    const int4* nbr;          // per element face: resident_face_table
    unsigned long long* xchg; // trace packets by epoch parity: resident_xchg_bytes
    void* snap;               // fields of the probed elements after every step, or null
    const int* snap_slot;     // per element: its slot in snap, -1 none (snap != null)
    int nslots;
    long long node_base;      // first node of the segment
    int elem0, nelt;          // the elements of this launch
    int per;                  // elements per workgroup (<= EM)
    int nsteps;
    unsigned epoch;           // tag of the first stage; the launch uses 5 nsteps consecutive tags
    int* stop;                // device word: sequence number of a launch that gave up waiting (0: none)
    int* stop_host;           // the same in host memory
    int seq;                  // this launch's number (> 0)
    int spin_limit;           // polls before a workgroup gives up
    double dt;
    double a[5], b[5];
};

// Elements per workgroup the kernels are built for (registers and LDS sized
// for EM elements; a launch may use fewer).  em: index 0 .. kResidentSizes - 1.
constexpr int kResidentSizes = 4;
constexpr int resident_em(int em) { return 1 << em; }
// Elements of (n1, prec) on chip at once with EM elements per workgroup, at most
// `max_per_cu` workgroups per CU (0: as many as fit).  0: not built.
long long resident_capacity(int n1, int prec, int em, bool affine, int max_per_cu);
hipError_t launch_resident(int n1, int prec, int em, bool affine, const ResidentArgs& a, hipStream_t s);
int resident_upload_tables(const GllTables& t);

// Per element face: the plus side's face slot (e2 * 6 + f2; -1: PEC mirror), and
// its face point of (p, q) as y + p z + q w.  False where the faces do not pair
// up (face A's neighbour names another face back), or for ghost faces.
bool resident_face_table(const int* fcode, int nelt, int n1, int elem_base, int4* out);

// One kernel of the family, for the dispatch: workgroups per CU it allows.
struct ResidentKernel {
    hipError_t (*launch)(const ResidentArgs&, hipStream_t) = nullptr;
    int (*per_cu)() = nullptr;
};
ResidentKernel resident_kernel_f64(int n1, int em, bool affine);
ResidentKernel resident_kernel_f32(int n1, int em, bool affine);
ResidentKernel resident_kernel_f32k64(int n1, int em, bool affine);
int resident_upload_f64(const GllTables& t);
int resident_upload_f32(const GllTables& t);
int resident_upload_f32k64(const GllTables& t);

}  // namespace nw
