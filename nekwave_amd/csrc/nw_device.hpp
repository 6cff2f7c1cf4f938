// nw_device.hpp -- device code shared by the fused stage kernel and the resident
// multi-step kernel: GLL tables, element geometry, occupancy targets and buffer
// access.  Both kernels evaluate the same expressions, so their results are the
// same bits.  Each translation unit that includes it has its own constant
// tables, filled once per device by device_upload_tables.
#pragma once

#include "nw_fused.hpp"

namespace nw {
namespace {

__constant__ GllTables c_gll;
__constant__ float c_Df[kMaxN1 + 1][kMaxN1 * kMaxN1];

template <typename R> __device__ __forceinline__ R gD(int n1, int idx);
template <> __device__ __forceinline__ double gD<double>(int n1, int idx) { return c_gll.D[n1][idx]; }
template <> __device__ __forceinline__ float gD<float>(int n1, int idx) { return c_Df[n1][idx]; }

// Tangent vectors d x/dr, d x/ds, d x/dt of the trilinear map at (r, s, t), in
// arithmetic T, from the 24 coefficients c[d * 8 + x] (ElemGeom order).
template <typename T>
struct Tangents {
    T r[3], s[3], t[3];
};
template <typename T>
__device__ __forceinline__ Tangents<T> tangents(const T* cf, T r, T s, T t) {
    Tangents<T> G;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T* c = cf + 8 * d;
        G.r[d] = c[1] + c[4] * s + c[5] * t + c[7] * (s * t);
        G.s[d] = c[2] + c[4] * r + c[6] * t + c[7] * (r * t);
        G.t[d] = c[3] + c[5] * r + c[6] * s + c[7] * (r * s);
    }
    return G;
}

template <typename T>
__device__ __forceinline__ void cross3(const T* a, const T* b, T* o) {
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}

// Local node of face point (p, q) of face f (getFaceNodeVolIndex, mesh.cpp:955-981)
// as base + p*sp + q*sq.
template <int N1>
__device__ __forceinline__ int face_local_node(int f, int p, int q) {
    constexpr int N2 = N1 * N1;
    const int base = f == 1 ? N1 - 1 : f == 2 ? N1 * (N1 - 1) : f == 5 ? N2 * (N1 - 1) : 0;
    const int sp = (f == 1 || f == 3) ? N1 : 1;
    const int sq = (f >= 4) ? N1 : N2;
    return base + p * sp + q * sq;
}

// n1 = 8 in FP32: a line of 8 values lies in 8 consecutive lanes, each holding
// one value of the line's lower half (lo, position lane & 3) and one of its upper
// half (hi), so every lane reads any value of its line from its own quad, as the
// DPP operand of the fused multiply-add, instead of from LDS.  Lanes hold two
// values per line instead of reading eight (and D stays in registers: the lane's
// row is lane & 7 in every direction).  The sum runs over q in the same order as
// the plain loop: the same bits.
// Three lines at once, as independent chains (asm: the compiler leaves the DPP
// moves separate, one more VALU instruction per term; s_nop: two wait states
// between a VALU write of lo or hi and the first DPP read of it).
#define NW_QUAD(q) " quad_perm:[" #q "," #q "," #q "," #q "] row_mask:0xf bank_mask:0xf\n\t"
#define NW_LINE3(op, half0, half1, half2, q, d)                      \
    op " %0, %" #half0 ", %" #d NW_QUAD(q) op " %1, %" #half1 ", %" #d NW_QUAD(q) \
    op " %2, %" #half2 ", %" #d NW_QUAD(q)
__device__ __forceinline__ void line8x3(const float (&D)[8], const float (&lo)[3], const float (&hi)[3], float (&a)[3]) {
    asm("s_nop 1\n\t"
        NW_LINE3("v_mul_f32_dpp", 3, 4, 5, 0, 9)
        NW_LINE3("v_fmac_f32_dpp", 3, 4, 5, 1, 10)
        NW_LINE3("v_fmac_f32_dpp", 3, 4, 5, 2, 11)
        NW_LINE3("v_fmac_f32_dpp", 3, 4, 5, 3, 12)
        NW_LINE3("v_fmac_f32_dpp", 6, 7, 8, 0, 13)
        NW_LINE3("v_fmac_f32_dpp", 6, 7, 8, 1, 14)
        NW_LINE3("v_fmac_f32_dpp", 6, 7, 8, 2, 15)
        NW_LINE3("v_fmac_f32_dpp", 6, 7, 8, 3, 16)
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2])
        : "v"(lo[0]), "v"(lo[1]), "v"(lo[2]), "v"(hi[0]), "v"(hi[1]), "v"(hi[2]), "v"(D[0]), "v"(D[1]), "v"(D[2]),
          "v"(D[3]), "v"(D[4]), "v"(D[5]), "v"(D[6]), "v"(D[7]));
}
#undef NW_LINE3
#undef NW_QUAD

// An empty volatile asm that takes and returns v: the value must be computed
// before this point in program order (the scheduler otherwise sinks pure
// arithmetic below later loads and barriers, stretching live ranges).
template <typename T>
__device__ __forceinline__ void pin(T& v) {
    asm volatile("" : "+v"(v));
}

// Occupancy target (waves per SIMD) that the register budget is sized for.
// FP32 fields: a workgroup of two waves per SIMD gets 4 (two workgroups per CU
// in 128 VGPRs), any other shape 3 (168 VGPRs).  FP64 fields get 2 (256
// VGPRs): the doubled prefetch registers spill otherwise, and a spill reload
// inside the loop waits on every prefetch in flight (measured 1.8x slower).
template <int NT, int RBYTES>
struct WavesPerEU {
    static constexpr int value = RBYTES == 8 ? 2 : (((NT + 63) / 64 + 3) / 4 == 2 ? 4 : 3);
};

// 1/J: in FP32 the hardware reciprocal (1 ulp); in FP64 the IEEE quotient.
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }
// |N| and 1/|N| from |N|^2 with the reference's guard |N| > 1e-14
// (mesh.cpp:1032-1035): FP32 through the hardware reciprocal square root,
// FP64 through the IEEE square root and quotient.
__device__ __forceinline__ void norm_and_inverse(float n2, float& len, float& inv) {
    inv = n2 > 1e-28f ? __builtin_amdgcn_rsqf(n2) : 0.0f;
    len = n2 * inv;
}
__device__ __forceinline__ void norm_and_inverse(double n2, double& len, double& inv) {
    len = sqrt(n2);
    inv = len > 1e-14 ? 1.0 / len : 0.0;
}

// Geometry at reference point (r, s, t) of a trilinear element: the cofactors
// C = J J^-T (mesh.cpp:291-309 times J) and 1/J, in the field precision R (FP64
// fields: FP64 arithmetic; FP32 fields: FP32 arithmetic on the coefficients
// rounded once, relative error ~1e-7, below the FP32 fields' own rounding).  On
// an affine element (c4..c7 exactly 0) every product with them is an exact
// zero, so the result is the same bits at every node.
template <typename R>
__device__ __forceinline__ void node_geometry(const R* cf, R r, R s, R t, R (&C)[10]) {
    const Tangents<R> T = tangents(cf, r, s, t);
    R Cr[3], Cs[3], Ct[3];
    cross3(T.s, T.t, Cr);  // (rx, ry, rz) * J
    cross3(T.t, T.r, Cs);  // (sx, sy, sz) * J
    cross3(T.r, T.s, Ct);  // (tx, ty, tz) * J
    const R det = T.r[0] * Cr[0] + T.r[1] * Cr[1] + T.r[2] * Cr[2];
    C[0] = Cr[0]; C[1] = Cr[1]; C[2] = Cr[2];
    C[3] = Cs[0]; C[4] = Cs[1]; C[5] = Cs[2];
    C[6] = Ct[0]; C[7] = Ct[1]; C[8] = Ct[2];
    C[9] = recip(det);
}

// Global traffic goes through raw buffer instructions: the base address lives
// in a buffer resource (SGPRs), each lane supplies a 32-bit byte offset and the
// component stride rides in the scalar offset, so no lane computes a 64-bit
// address.  Offsets past num_records read 0 instead of faulting.  The
// launcher checks that every offset fits in 32 bits.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p) {
    // dword3 0x00020000: the raw-buffer format word of the gfx9 family
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffffu, 0x00020000);
}
__device__ __forceinline__ float bload(float*, __amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0));
}
__device__ __forceinline__ double bload(double*, __amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0));
}
template <typename T>
__device__ __forceinline__ T bld(__amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so) {
    return bload(static_cast<T*>(nullptr), r, vo, so);
}
__device__ __forceinline__ int4 bld_int4(__amdgpu_buffer_rsrc_t r, unsigned vo) {
    typedef __attribute__((ext_vector_type(4))) int i32x4;
    const i32x4 v = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, vo, 0, 0));
    return make_int4(v[0], v[1], v[2], v[3]);
}
// The six field values of one node (node-major state: 6 consecutive values
// per node) in as few accesses as the node's alignment allows: FP32 nodes sit
// 24 bytes apart (one 16-byte plus one 8-byte access; buffer accesses need only
// dword alignment), FP64 nodes 48 bytes apart (three 16-byte accesses).  Two
// instructions instead of three matter most for the neighbour-trace gathers,
// whose lanes each touch a different cache line.
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) double f64x2;
// (Each 8-byte word is reinterpreted whole as two floats: extracting single
// 32-bit lanes of the loaded vector before the reinterpretation let the
// compiler narrow the access to its first lane.)
// CP: the access's cache-policy bits (kNT: non-temporal -- no reuse expected,
// so the line is a first candidate for eviction from L2; kSC1: system scope --
// a store is written through L2 instead of left dirty in it).
constexpr int kNT = 2;
constexpr int kSC1 = 16;
template <int CP = 0>
__device__ __forceinline__ void ld6(__amdgpu_buffer_rsrc_t r, unsigned vo, float (&o)[6]) {
    const f32x4 a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, vo, 0, CP));
    const f32x2 b = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, vo + 16u, 0, CP));
    o[0] = a[0]; o[1] = a[1]; o[2] = a[2]; o[3] = a[3]; o[4] = b[0]; o[5] = b[1];
}
template <int CP = 0>
__device__ __forceinline__ void ld6(__amdgpu_buffer_rsrc_t r, unsigned vo, double (&o)[6]) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const f64x2 a = __builtin_bit_cast(f64x2, __builtin_amdgcn_raw_buffer_load_b128(r, vo + 16u * x, 0, CP));
        o[2 * x] = a[0];
        o[2 * x + 1] = a[1];
    }
}
__device__ __forceinline__ void ld4(__amdgpu_buffer_rsrc_t r, unsigned vo, float (&o)[4]) {
    const f32x4 a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, vo, 0, 0));
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = a[c];
}
__device__ __forceinline__ void ld4(__amdgpu_buffer_rsrc_t r, unsigned vo, double (&o)[4]) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const f64x2 a = __builtin_bit_cast(f64x2, __builtin_amdgcn_raw_buffer_load_b128(r, vo + 16u * x, 0, 0));
        o[2 * x] = a[0];
        o[2 * x + 1] = a[1];
    }
}
template <int CP = 0>
__device__ __forceinline__ void st6(__amdgpu_buffer_rsrc_t r, unsigned vo, const float (&v)[6]) {
    const f32x4 a = {v[0], v[1], v[2], v[3]};
    const f32x2 b = {v[4], v[5]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, a), r, vo, 0, CP);
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, b), r, vo + 16u, 0, CP);
}
template <int CP = 0>
__device__ __forceinline__ void st6(__amdgpu_buffer_rsrc_t r, unsigned vo, const double (&v)[6]) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const f64x2 a = {v[2 * x], v[2 * x + 1]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, a), r, vo + 16u * x, 0, CP);
    }
}

inline int device_upload_tables(const GllTables& t) {
    float df[kMaxN1 + 1][kMaxN1 * kMaxN1];
    for (int n = 0; n <= kMaxN1; ++n)
        for (int x = 0; x < kMaxN1 * kMaxN1; ++x) df[n][x] = static_cast<float>(t.D[n][x]);
    NW_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_gll), &t, sizeof(GllTables)));
    NW_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_Df), df, sizeof(df)));
    return NW_OK;
}

}  // namespace
}  // namespace nw
