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
// Where resident launches beat the stage launches: the most elements per workgroup a
// kernel is built for, (per_cu > 0) the most elements per CU it is used for, and whether a
// segment of more meshes than fit at once takes several launches in turn.
//
// Measured over whole ranges, boxes of 27 elements up to the chip's capacity (us per
// stage, the stage kernel's tuned shape against this).  A kernel that spills registers
// loses: a reload waits for every packet in flight (FP64 jittered n1 = 4, four elements
// per workgroup, 8192 elements: 27.0 against 36.7; FP64 registers n1 = 5, eight, 10240:
// 35.9 against 64.1; those that spill and win have one or two elements).  So does one
// whose workgroups leave a CU with one wave per SIMD (FP64 n1 = 5, eight, 4096: no gain).
// Below n1 = 4 an element fills 8 or 27 lanes of a wave, where the stage kernel packs
// several elements into one (n1 = 2, FP32, 24576 elements: 10.9 against 42.7; n1 = 3,
// FP64, 16384: 26.5 against 50.8): only while a stage is bound by its launch.  At n1 = 4
// and 5, FP32 affine, the gain fades towards the capacity (20480 elements: 28.5 against
// 27.6) and a call of one step loses there (154 against 172 us: fields in and out of LDS).
// Every other range won or drew (n1 = 4, FP32, 12288 jittered: 18.7 against 17.0; n1 = 8,
// FP32, 2048: 22.4 against 15.2).
// Against several launches stands one stage launch over the whole segment, which then
// runs at its best rate: n1 = 5 lost throughout (124 elements per CU, FP32 affine 81.8
// against 83.7, jittered 87.5 against 97.7, FP64 184 against 188 to 293), as did n1 = 4
// with FP32 registers (78.9 against 85.5), n1 = 7 FP64 (202 against 211); the others won while
// the launches were nearly full (n1 = 8 FP32 affine 1.16 to 1.23x, n1 = 9 1.08 to 1.16x).
struct ResidentRange {
    int em, per_cu;
    bool several;
};
constexpr ResidentRange resident_range(int n1, int rbytes, int kbytes, bool affine) {
    const bool f64 = rbytes == 8, k32 = kbytes == 4;
    switch (n1) {
        case 2: return {f64 ? 0 : 1, 10, false};
        case 3: return {1, f64 ? 5 : 8, false};
        case 4: return {k32 ? (affine ? 8 : 4) : (affine ? 4 : 2), k32 && affine ? 60 : 0, !k32 && (affine || !f64)};
        case 5: return {k32 && affine ? 8 : (k32 || affine ? 4 : 2), k32 && affine ? 28 : 0, false};
        case 6: return {k32 ? 8 : 4, 0, true};
        case 7: return {f64 && affine ? 8 : 4, 0, !f64};
        case 8: return {!f64 && !k32 && !affine ? 2 : 4, 0, true};
        default: return {f64 ? 2 : (k32 ? 8 : 4), 0, true};
    }
}
constexpr ResidentRange resident_range(int n1, int prec, bool affine) {
    return resident_range(n1, prec == kFP64 ? 8 : 4, prec == kFP32 ? 4 : 8, affine);
}
// Several launches in turn: the share of their places that elements fill, at least (n1 =
// 8, FP32, launches of 1331 elements where 1536 have places: affine 64.9 against 65.6,
// jittered 65.1 against 70.0; n1 = 6, FP64 registers, affine, 1728 of 2048: 94.7 against 102.5).
constexpr double resident_fill(int n1, bool affine) { return affine && n1 != 6 ? 0.8 : 0.9; }

// Workgroups of (n1, prec) with EM elements each on chip at once, at most `max_per_cu` per
// CU (0: as many as fit), and the elements one launch takes.  0: not built (resident_range).
struct ResidentCapacity {
    long long groups = 0, elements = 0;
};
ResidentCapacity resident_capacity(int n1, int prec, int em, bool affine, int max_per_cu);
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
