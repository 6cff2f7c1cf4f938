// nw_plain_stage.hip -- one LSRK stage of the plain pipeline in one launch: FP64, any
// n1 in [2, 10], geometry from the reference's per-node and per-face-point arrays
// (dg_solver.cpp:114-236).  Every point operation is the reference's (volume curl
// dg_kernels.cu:41-155, flux :217-314, lift :316-338, inverse mass :340-366, LSRK
// :368-384), in the order of its kernels.
//
// Bound by memory: per node and stage the fields in (48 B) and out (48), the LSRK
// register (96; the first stage only writes it) and the metrics (80), per face point
// tables (48) and the plus trace (48).  As seven launches the stage also wrote and read
// the right-hand side four times, both traces and the flux.
//
// A workgroup takes EPW elements, KS planes of n1 x n1 threads each, so a thread has the
// nodes (i, j, ks + KS m): i and j, and with them its rows of D, are the same for all
// of them.  The fields of the element (48 n1^3 B) and its face fluxes (288 n1^2 B) lie
// in LDS; the plus traces are read from the input state, so the stage writes a second
// state (the fields node-major: a trace point is 48 consecutive bytes).
//
// Measured per stage, seven launches -> one (jittered box, media, 340 to 512 thousand
// nodes): n1 = 2 172.8 -> 42.3 us, 3 110.3 -> 30.6, 4 92.0 -> 27.5, 5 80.9 -> 26.3,
// 6 89.2 -> 27.6, 7 96.5 -> 26.4, 8 96.5 -> 26.2, 9 105.8 -> 27.1, 10 106.8 -> 31.1,
// 4.6 to 6.8 TB/s of the bytes above.
#include "nw_plain.hpp"

#include "nw_fused.hpp"
#include "nw_plain_device.hpp"

namespace nw {
namespace {

struct Node6 {
    double c[6];
};
template <typename I>
__device__ __forceinline__ Node6 load_node(const double* __restrict__ u, I v) {
    const double2* p = reinterpret_cast<const double2*>(u + 6 * v);
    const double2 a = p[0], b = p[1], c = p[2];
    return {{a.x, a.y, b.x, b.y, c.x, c.y}};
}

__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }

struct FacePoint {
    int v;  // plus node
    bool mirror;
    Vec3 n;
    Node6 u;  // plus fields
};
__device__ __forceinline__ void read_point(FacePoint& f, const PlainStageArgs& A, long long fg, unsigned p, bool on) {
    f.v = -1;
    f.mirror = true;
    if (on) {
        f.v = (A.vP + fg)[p];
        f.mirror = (A.bc + fg)[p] != 0 || f.v < 0;
        f.n = {(A.nx + fg)[p], (A.ny + fg)[p], (A.nz + fg)[p]};
    }
}
__device__ __forceinline__ void read_plus(FacePoint& f, const PlainStageArgs& A) {
    if (!f.mirror) f.u = load_node(A.uin, (long long)f.v);
}

template <int N1, int EPW, int KS, bool FIRST>
__global__ __launch_bounds__(EPW* KS* N1* N1) void k_plain_stage(const PlainStageArgs A) {
    constexpr int N2 = N1 * N1, NP = N1 * N2, T = KS * N2, NK = (N1 + KS - 1) / KS, F = 6 * N2;
    constexpr int FIT = (F + T - 1) / T;
    __shared__ double sU[EPW][6][NP];
    __shared__ double sF[EPW][6][F];  // flux of H (0..2) and E (3..5) per face point
    __shared__ double sD[N2];         // column-major D[i + q * N1]
    // consecutive groups of elements on one XCD: block b runs on XCD b mod 8
    const int per = gridDim.x >> 3;
    const int group = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (group * EPW >= A.nelt) return;
    const int es = threadIdx.x / T, l = threadIdx.x - es * T;
    const int ks = l / N2, ij = l - ks * N2, i = ij % N1, j = ij / N1;
    const bool live = group * EPW + es < A.nelt;
    const int e = live ? group * EPW + es : A.nelt - 1;
    // uniform base of the group's nodes and face points, 32-bit offsets within it
    const long long vg = (long long)group * EPW * NP, fg = (long long)group * EPW * F;
    const unsigned v0 = unsigned(e - group * EPW) * NP, f0 = unsigned(e - group * EPW) * F;
    const double* uin = A.uin + 6 * vg;
    for (int x = threadIdx.x; x < N2; x += EPW * T) sD[x] = A.D[x];

    // a face point's plus trace is a chain of two reads (table, then fields); the first
    // point of each thread is read ahead of the barrier
    FacePoint fp;
    read_point(fp, A, fg, f0 + l, l < F);
#pragma unroll
    for (int m = 0; m < NK; ++m) {
        const int x = l + m * T;
        if (x < NP) {
            const Node6 u = load_node(uin, v0 + x);
#pragma unroll
            for (int c = 0; c < 6; ++c) sU[es][c][x] = u.c[c];
        }
    }
    read_plus(fp, A);
    __syncthreads();

#pragma unroll
    for (int it = 0; it < FIT; ++it) {
        const int p = l + it * T;
        if (it > 0) {
            read_point(fp, A, fg, f0 + p, p < F);
            read_plus(fp, A);
        }
        if (p < F) {
            const int f = p / N2, pq = p - f * N2;
            const int x = face_local_node<N1>(f, pq % N1, pq / N1);
            Vec3 dE, dH, fE, fH;
            if (fp.mirror) {
                dE = {-2.0 * sU[es][0][x], -2.0 * sU[es][1][x], -2.0 * sU[es][2][x]};
                dH = {0.0, 0.0, 0.0};
            } else {
                dE = {fp.u.c[0] - sU[es][0][x], fp.u.c[1] - sU[es][1][x], fp.u.c[2] - sU[es][2][x]};
                dH = {fp.u.c[3] - sU[es][3][x], fp.u.c[4] - sU[es][4][x], fp.u.c[5] - sU[es][5][x]};
            }
            int ep = e;
            if (A.eps && !fp.mirror) ep = fp.v < A.npts ? fp.v / NP : A.ghost_elem[fp.v - A.npts];
            plain_flux(dE, dH, fp.n, A.c0, A.eps, A.mu, e, ep, fH, fE);
            sF[es][0][p] = fH.x; sF[es][1][p] = fH.y; sF[es][2][p] = fH.z;
            sF[es][3][p] = fE.x; sF[es][4][p] = fE.y; sF[es][5][p] = fE.z;
        }
    }

    // volume: +curl H into the rows of E, -curl E into the rows of H
    // (metrics and k read ahead of this loop take the registers of the second workgroup:
    // 34.2 -> 42.3 us at n1 = 10)
    double rhs[NK][6];
#pragma unroll
    for (int m = 0; m < NK; ++m) {
        const int k = NK * KS == N1 ? ks + KS * m : min(ks + KS * m, N1 - 1);
        const int x = ij + N2 * k;
        const unsigned v = v0 + x;
        double ar[6], as[6], at[6];
        plain_gradient<N1, 6>(sU[es], sD, i, j, k, ar, as, at);
        double met[9];
#pragma unroll
        for (int d = 0; d < 9; ++d) met[d] = (A.met[1 + d] + vg)[v];
        const double w = A.w3[x] * (A.met[0] + vg)[v];
        const Vec3 cH = plain_curl({ar[3], ar[4], ar[5]}, {as[3], as[4], as[5]}, {at[3], at[4], at[5]}, w, met);
        const Vec3 cE = plain_curl({ar[0], ar[1], ar[2]}, {as[0], as[1], as[2]}, {at[0], at[1], at[2]}, w, met);
        rhs[m][0] = cH.x; rhs[m][1] = cH.y; rhs[m][2] = cH.z;
        rhs[m][3] = -cE.x; rhs[m][4] = -cE.y; rhs[m][5] = -cE.z;
#pragma unroll
        for (int c = 0; c < 6; ++c) pin(rhs[m][c]);  // here, not sunk past the barrier with all its operands
    }
    __syncthreads();
    if (!live) return;

    const double dt = *A.dt;
    const double ep = A.eps ? A.eps[e] : 1.0, mu = A.mu ? A.mu[e] : 1.0;
#pragma unroll
    for (int m = 0; m < NK; ++m) {
        const int x = l + m * T, k = ks + KS * m;
        const unsigned v = v0 + x;
        if (x >= NP) break;
        // lift: faces in order 0..5
        const auto add = [&](bool on, int p) {
            if (!on) return;
            const double a = (A.dA + fg)[f0 + p];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                rhs[m][c] += a * sF[es][3 + c][p];
                rhs[m][3 + c] += a * sF[es][c][p];
            }
        };
        add(j == 0, 0 * N2 + i + N1 * k);
        add(i == N1 - 1, 1 * N2 + j + N1 * k);
        add(j == N1 - 1, 2 * N2 + i + N1 * k);
        add(i == 0, 3 * N2 + j + N1 * k);
        add(k == 0, 4 * N2 + ij);
        add(k == N1 - 1, 5 * N2 + ij);
        const double jac = (A.met[0] + vg)[v], w3 = A.w3[x];
        const double iE = 1.0 / (ep * jac * w3);
        const double iH = 1.0 / (mu * jac * w3);
        double out[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const double r = rhs[m][c] * (c < 3 ? iE : iH);
            double* kp = A.k + c * (long long)A.npts + vg + v;
            const double ki = FIRST ? dt * r : A.a * *kp + dt * r;
            *kp = ki;
            out[c] = sU[es][c][x] + A.b * ki;
        }
        double2* q = reinterpret_cast<double2*>(A.uout + 6 * vg + 6 * v);
        q[0] = {out[0], out[1]};
        q[1] = {out[2], out[3]};
        q[2] = {out[4], out[5]};
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <int N1>
hipError_t launch(const PlainStageArgs& a, hipStream_t s) {
    constexpr int EPW = PlainTile<N1>::EPW, KS = PlainTile<N1>::KS;
    const int groups = (a.nelt + EPW - 1) / EPW;
    const dim3 grid(8 * ((groups + 7) / 8)), block(EPW * KS * N1 * N1);
    if (a.a == 0.0) hipLaunchKernelGGL((k_plain_stage<N1, EPW, KS, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_plain_stage<N1, EPW, KS, false>), grid, block, 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_plain_stage(int n1, const PlainStageArgs& a, hipStream_t s) {
    if (a.nelt <= 0) return hipSuccess;
    switch (n1) {
        case 2: return launch<2>(a, s);
        case 3: return launch<3>(a, s);
        case 4: return launch<4>(a, s);
        case 5: return launch<5>(a, s);
        case 6: return launch<6>(a, s);
        case 7: return launch<7>(a, s);
        case 8: return launch<8>(a, s);
        case 9: return launch<9>(a, s);
        case 10: return launch<10>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace nw
