// nw_plain_device.hpp -- the point operations of the reference's stage kernels (FP64, in
// its expression order), shared by the kernel-level launchers and the plain pipeline's
// stage kernel.
#pragma once

#include <hip/hip_runtime.h>

namespace nw {
namespace {

// Elements per workgroup and thread planes per element.  The workgroups of a CU cover
// each other's barriers and loads: at n1 = 10 five planes of two nodes per thread (500
// threads, 110 registers, two workgroups per CU) take 31.1 us, ten planes (1000 threads,
// one workgroup) 34.8; n1 = 9 27.1 against 28.5; n1 = 8 four planes 26.2 against 27.9; from
// n1 = 7 down one node per thread.  Small elements: about two waves per workgroup (n1 = 5
// one element 26.3, two 26.9, four 29.0).
template <int N1> struct PlainTile;
template <> struct PlainTile<2> { static constexpr int EPW = 16, KS = 2; };
template <> struct PlainTile<3> { static constexpr int EPW = 4, KS = 3; };
template <> struct PlainTile<4> { static constexpr int EPW = 2, KS = 4; };
template <> struct PlainTile<5> { static constexpr int EPW = 1, KS = 5; };
template <> struct PlainTile<6> { static constexpr int EPW = 1, KS = 6; };
template <> struct PlainTile<7> { static constexpr int EPW = 1, KS = 7; };
template <> struct PlainTile<8> { static constexpr int EPW = 1, KS = 4; };
template <> struct PlainTile<9> { static constexpr int EPW = 1, KS = 5; };
template <> struct PlainTile<10> { static constexpr int EPW = 1, KS = 5; };

// Local node of face point (p, q) of face f, without branches.
template <int N1>
__device__ __forceinline__ int face_local_node(int f, int p, int q) {
    constexpr int N2 = N1 * N1;
    const int base = f == 1 ? N1 - 1 : f == 2 ? N1 * (N1 - 1) : f == 5 ? N2 * (N1 - 1) : 0;
    return base + p * ((f == 1 || f == 3) ? N1 : 1) + q * (f >= 4 ? N1 : N2);
}

struct Vec3 {
    double x, y, z;
};

// Derivatives along the reference axes of NC fields at node (i, j, k) of the element in
// u, from the column-major D.  (q rolled: unrolled, the reads ahead of their use take
// the registers of a second workgroup per CU.)
template <int N1, int NC>
__device__ __forceinline__ void plain_gradient(const double (&u)[NC][N1 * N1 * N1], const double* sD, int i, int j, int k,
                                               double (&r)[NC], double (&s)[NC], double (&t)[NC]) {
    constexpr int N2 = N1 * N1;
#pragma unroll
    for (int c = 0; c < NC; ++c) r[c] = s[c] = t[c] = 0.0;
#pragma unroll 1
    for (int q = 0; q < N1; ++q) {
        const double di = sD[i + q * N1], dj = sD[j + q * N1], dk = sD[k + q * N1];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            r[c] += di * u[c][q + N1 * j + N2 * k];
            s[c] += dj * u[c][i + N1 * q + N2 * k];
            t[c] += dk * u[c][i + N1 * j + N2 * q];
        }
    }
}

// W J (grad_ref u . J^-T) x of one node (dg_kernels.cu:106-154): r, s, t the derivatives
// of the three components along the reference axes, w = W J.
__device__ __forceinline__ Vec3 plain_curl(const double (&r)[3], const double (&s)[3], const double (&t)[3], double w,
                                           const double (&met)[9]) {
    const double u1rw = r[0] * w, u1sw = s[0] * w, u1tw = t[0] * w;
    const double u2rw = r[1] * w, u2sw = s[1] * w, u2tw = t[1] * w;
    const double u3rw = r[2] * w, u3sw = s[2] * w, u3tw = t[2] * w;
    const double Rx = met[0], Sx = met[1], Tx = met[2], Ry = met[3], Sy = met[4], Ty = met[5];
    const double Rz = met[6], Sz = met[7], Tz = met[8];
    Vec3 o;
    o.x = (u3rw * Ry + u3sw * Sy + u3tw * Ty) - (u2rw * Rz + u2sw * Sz + u2tw * Tz);
    o.y = (u1rw * Rz + u1sw * Sz + u1tw * Tz) - (u3rw * Rx + u3sw * Sx + u3tw * Tx);
    o.z = (u2rw * Rx + u2sw * Sx + u2tw * Tx) - (u1rw * Ry + u1sw * Sy + u1tw * Ty);
    return o;
}

// Upwind flux of one face point from the jumps (dg_kernels.cu:217-314); eps != null:
// the impedances of minus element em and plus element ep.
__device__ __forceinline__ void plain_flux(const Vec3& dE, const Vec3& dH, const Vec3& n, double c0,
                                           const double* __restrict__ eps, const double* __restrict__ mu, int em, int ep,
                                           Vec3& fH, Vec3& fE) {
    const double nxEx = n.y * dE.z - n.z * dE.y, nxEy = n.z * dE.x - n.x * dE.z, nxEz = n.x * dE.y - n.y * dE.x;
    const double nxHx = n.y * dH.z - n.z * dH.y, nxHy = n.z * dH.x - n.x * dH.z, nxHz = n.x * dH.y - n.y * dH.x;
    const double nnEx = n.y * nxEz - n.z * nxEy, nnEy = n.z * nxEx - n.x * nxEz, nnEz = n.x * nxEy - n.y * nxEx;
    const double nnHx = n.y * nxHz - n.z * nxHy, nnHy = n.z * nxHx - n.x * nxHz, nnHz = n.x * nxHy - n.y * nxHx;
    if (!eps) {
        fH.x = -0.5 * nxEx - 0.5 * c0 * nnHx; fH.y = -0.5 * nxEy - 0.5 * c0 * nnHy; fH.z = -0.5 * nxEz - 0.5 * c0 * nnHz;
        fE.x = 0.5 * nxHx - 0.5 * c0 * nnEx; fE.y = 0.5 * nxHy - 0.5 * c0 * nnEy; fE.z = 0.5 * nxHz - 0.5 * c0 * nnEz;
    } else {
        const double Zm = sqrt(mu[em] / eps[em]), Zp = sqrt(mu[ep] / eps[ep]);
        const double Ym = 1.0 / Zm, Yp = 1.0 / Zp;
        const double iz = 1.0 / (Zp + Zm), iy = 1.0 / (Yp + Ym);
        fH.x = (-Yp * nxEx - c0 * nnHx) * iy; fH.y = (-Yp * nxEy - c0 * nnHy) * iy; fH.z = (-Yp * nxEz - c0 * nnHz) * iy;
        fE.x = (Zp * nxHx - c0 * nnEx) * iz; fE.y = (Zp * nxHy - c0 * nnEy) * iz; fE.z = (Zp * nxHz - c0 * nnEz) * iz;
    }
}

}  // namespace
}  // namespace nw
