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
// kernel is built for, (per_cu > 0) the most elements per CU it is used for, and the most
// launches in turn that a segment of more meshes than fit at once is cut into.
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
// Against several launches stands one stage launch over the whole segment, which runs at
// its best rate from three or four times the chip's capacity on.  Batches of equal and of
// mixed cavities, up to 40 launches: FP64 registers under FP32 fields won throughout
// (affine 1.1 to 1.4x, jittered 1.06 to 1.3x) but at n1 = 5 and 7 jittered (0.69 to 1.2x);
// affine FP64 won at n1 = 4, 6, 8, 9 (1.02 to 1.3x), affine FP32 from n1 = 6 on (1.0 to
// 1.23x).  The rest lost or drew beyond a few launches (n1 = 5 FP64 0.70 to 0.97x, n1 = 7
// jittered FP32 0.86 to 1.08x, at two launches 1.1 to 1.3x).
struct ResidentRange {
    int em, per_cu, launches;
};
constexpr ResidentRange resident_range(int n1, int rbytes, int kbytes, bool affine) {
    const bool f64 = rbytes == 8, k32 = kbytes == 4, mixed = !f64 && !k32;
    const int any = 1 << 30;
    switch (n1) {
        case 2: return {f64 ? 0 : 1, 10, 1};
        case 3: return {1, f64 ? 5 : 8, 1};
        case 4: return {k32 ? (affine ? 8 : 4) : (affine ? 4 : 2), k32 && affine ? 60 : 0, mixed || (f64 && affine) ? any : k32 ? 2 : 1};
        case 5: return {k32 && affine ? 8 : (k32 || affine ? 4 : 2), k32 && affine ? 28 : 0, mixed && affine ? any : 1};
        case 6: return {k32 ? 8 : 4, 0, affine || mixed ? any : 3};
        case 7: return {f64 && affine ? 8 : 4, 0, affine && !f64 ? any : 3};
        case 8: return {mixed && !affine ? 2 : 4, 0, affine || !k32 ? any : 3};
        default: return {f64 ? 2 : (k32 ? 8 : 4), 0, affine || mixed ? any : 3};
    }
}
constexpr ResidentRange resident_range(int n1, int prec, bool affine) {
    return resident_range(n1, prec == kFP64 ? 8 : 4, prec == kFP32 ? 4 : 8, affine);
}
// Several launches in turn, n1 > 3: any number where the batch has segments of other orders
// too and is larger than the Infinity Cache (`cold`), affine in FP32: a stage launch then
// reads its segment from HBM (256 cavities of n1 = 4 to 9, 2.4 GB: the n1 = 4 segment 34.5
// us per stage against 31.1).
constexpr int resident_launches(int n1, int prec, bool affine, bool cold) {
    return cold && affine && prec == kFP32 && n1 > 3 ? 1 << 30 : resident_range(n1, prec, affine).launches;
}
// And the share of their places that elements fill, at least (n1 = 8, FP32, launches of
// 1331 elements where 1536 have places: affine 64.9 against 65.6, jittered 65.1 against
// 70.0; FP64 registers, affine, n1 = 6, 1728 of 2048: 94.7 against 102.5, n1 = 5, 3456 of
// 3840: 102.7 against 114.5).
constexpr double resident_fill(int n1, bool affine) { return !affine ? 0.9 : n1 == 5 || n1 == 6 ? 0.91 : 0.8; }

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
