// nw_plain.hip -- the reference's stage decomposition, one gfx950 kernel per
// reference kernel (FP64), plus device-side geometry setup, diagnostics,
// precision conversion and the halo stand-in.
//
// The stage kernels take the same arrays as the reference launchers
// (dg_kernels.hpp:13-88) so every reference kernel has a counterpart that can
// be checked in isolation.  Design differences from the reference:
//   * volume curl: EPW elements per workgroup, KS thread planes per element;
//   * lift: one thread per node gathering its face contributions in face order
//     0..5 (deterministic; the reference uses FP64 atomics, dg_kernels.cu:329);
//   * elementwise kernels are grid-stride loops sized for 256 CUs.
#include <algorithm>
#include <mutex>

#include "nw_plain.hpp"

#include "nw_fused.hpp"
#include "nw_plain_device.hpp"

namespace nw {
namespace {

__constant__ GllTables c_gll;

constexpr int kBlock = 256;

inline int grid_for(long long n, int block = kBlock) {
    long long g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > 65536) g = 65536;
    return static_cast<int>(g);
}

// The block's place when neighbouring blocks are to share an XCD's L2: block b runs on
// XCD b mod 8.  The grid is a multiple of 8 (grid_for_xcd).  For the kernels that
// gather traces, where a line of the state holds points of several blocks: flux 27.0 ->
// 19.5 us at 593 thousand nodes, n1 = 7, 18.5 -> 14.0 at 512 thousand, n1 = 10; restrict
// 14.6 -> 12.4 and 13.2 -> 10.3.  For the kernels over nodes too: each then finds lines
// of the one before it in its L2 (a stage 104.4 -> 101.0 at n1 = 7, 68.2 -> 64.8 at 373
// thousand, n1 = 8, 80.2 -> 75.2 at 373 thousand, n1 = 4).
inline int grid_for_xcd(long long n) { return 8 * ((grid_for(n) + 7) / 8); }
__device__ __forceinline__ long long xcd_block() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// ---------------------------------------------------------------------------
// volume curl (dg_kernels.cu:41-155): w = sign * W*J * (grad_ref u . J^-T) x
// ---------------------------------------------------------------------------
// Bound by memory: fields in and out (48 B per node) and metrics (80).  The workgroups of
// k_plain_stage, the t-lines in LDS like the others: a thread per column with its line
// in registers had one or two waves per element and took 24.1 us at 593 thousand nodes,
// n1 = 7, 22.6 at 373 thousand, n1 = 8, 21.0 at 512 thousand, n1 = 10; now 16.5, 11.9
// and 15.2 (4.3 to 4.6 TB/s; launch to launch, the kernel itself 13.5 at n1 = 7).
template <int N1, int EPW, int KS>
__global__ __launch_bounds__(EPW* KS* N1* N1) void k_volume_curl(const PlainVolumeArgs A) {
    constexpr int N2 = N1 * N1, NP = N1 * N2, T = KS * N2, NK = (N1 + KS - 1) / KS;
    __shared__ double sU[EPW][3][NP];
    __shared__ double sD[N2];  // column-major D[i + q * N1]
    const int es = threadIdx.x / T, l = threadIdx.x - es * T;
    const int ks = l / N2, ij = l - ks * N2, i = ij % N1, j = ij / N1;
    const int group = static_cast<int>(xcd_block());
    if (group * EPW >= A.nelt) return;
    const bool live = group * EPW + es < A.nelt;
    // uniform base of the group's nodes, 32-bit offsets within it
    const long long vg = (long long)group * EPW * NP;
    const unsigned v0 = (live ? es : A.nelt - 1 - group * EPW) * NP;
    for (int x = threadIdx.x; x < N2; x += EPW * T) sD[x] = A.D[x];
#pragma unroll
    for (int m = 0; m < NK; ++m) {
        const int x = l + m * T;
        if (x < NP) {
            sU[es][0][x] = (A.u1 + vg)[v0 + x]; sU[es][1][x] = (A.u2 + vg)[v0 + x]; sU[es][2][x] = (A.u3 + vg)[v0 + x];
        }
    }
    __syncthreads();
    if (!live) return;
#pragma unroll
    for (int m = 0; m < NK; ++m) {
        const int k = ks + KS * m;
        if (NK * KS != N1 && k >= N1) break;
        const unsigned x = ij + N2 * k, v = v0 + x;
        double r[3], s[3], t[3];
        plain_gradient<N1, 3>(sU[es], sD, i, j, k, r, s, t);
        const double* const met[9] = {A.rx, A.sx, A.tx, A.ry, A.sy, A.ty, A.rz, A.sz, A.tz};
        double g[9];
#pragma unroll
        for (int d = 0; d < 9; ++d) g[d] = (met[d] + vg)[v];
        const Vec3 o = plain_curl(r, s, t, A.w3g[x] * (A.jac + vg)[v], g);
        (A.w1 + vg)[v] = A.sign * o.x; (A.w2 + vg)[v] = A.sign * o.y; (A.w3 + vg)[v] = A.sign * o.z;
    }
}

template <int N1>
hipError_t launch_vc(const PlainVolumeArgs& a, hipStream_t s) {
    constexpr int EPW = PlainTile<N1>::EPW, KS = PlainTile<N1>::KS;
    const int groups = (a.nelt + EPW - 1) / EPW;
    hipLaunchKernelGGL((k_volume_curl<N1, EPW, KS>), dim3(8 * ((groups + 7) / 8)), dim3(EPW * KS * N1 * N1), 0, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// restrict / flux / lift / inverse mass / LSRK / halo
// ---------------------------------------------------------------------------
__global__ void k_restrict(const double* __restrict__ st, double* __restrict__ fEN, double* __restrict__ fHN,
                           const int* __restrict__ vM, long long tfp, long long S) {
    for (long long p = xcd_block() * (long long)blockDim.x + threadIdx.x; p < tfp; p += (long long)gridDim.x * blockDim.x) {
        const long long v = vM[p];
        fEN[p] = st[v]; fEN[tfp + p] = st[S + v]; fEN[2 * tfp + p] = st[2 * S + v];
        fHN[p] = st[3 * S + v]; fHN[tfp + p] = st[4 * S + v]; fHN[2 * tfp + p] = st[5 * S + v];
    }
}

__global__ void k_flux(const double* __restrict__ st, const double* __restrict__ fEN, const double* __restrict__ fHN,
                       const int* __restrict__ vP, const int* __restrict__ bc, const double* __restrict__ nxa,
                       const double* __restrict__ nya, const double* __restrict__ nza, double* __restrict__ flux,
                       double c0, long long tfp, long long S, const int* __restrict__ vM, const double* __restrict__ eps,
                       const double* __restrict__ mu, const int* __restrict__ ghost_elem, int np, long long npts) {
    for (long long p = xcd_block() * (long long)blockDim.x + threadIdx.x; p < tfp; p += (long long)gridDim.x * blockDim.x) {
        const Vec3 Em = {fEN[p], fEN[tfp + p], fEN[2 * tfp + p]}, Hm = {fHN[p], fHN[tfp + p], fHN[2 * tfp + p]};
        const int v = vP[p];
        const bool mirror = bc[p] != 0 || v < 0;
        Vec3 dE, dH, fH, fE;
        if (mirror) {
            dE = {-2.0 * Em.x, -2.0 * Em.y, -2.0 * Em.z};
            dH = {0.0, 0.0, 0.0};
        } else {
            dE = {st[v] - Em.x, st[S + v] - Em.y, st[2 * S + v] - Em.z};
            dH = {st[3 * S + v] - Hm.x, st[4 * S + v] - Hm.y, st[5 * S + v] - Hm.z};
        }
        int em = 0, ep = 0;
        if (eps) {
            em = vM[p] / np;
            ep = mirror ? em : (v < npts ? v / np : ghost_elem[v - npts]);
        }
        plain_flux(dE, dH, {nxa[p], nya[p], nza[p]}, c0, eps, mu, em, ep, fH, fE);
        flux[p] = fH.x; flux[tfp + p] = fH.y; flux[2 * tfp + p] = fH.z;
        flux[3 * tfp + p] = fE.x; flux[4 * tfp + p] = fE.y; flux[5 * tfp + p] = fE.z;
    }
}

// Deterministic lift: node (i,j,k) of element e gathers dA*flux from the face
// points that map to it, faces in order 0..5 (the serial face-point order).  A
// face point counts here only if volIdxMinus names the node the element-major
// layout puts it at; k_lift_scatter adds the others.  A node lies on at most one
// face per axis: the reads of its (up to) three points are issued together, the
// additions follow in face order.  (With k_lift_scatter 21.2 us at 593 thousand
// nodes, n1 = 7, 14.9 at 373 thousand, n1 = 8, 32.9 at 512 thousand, n1 = 2; as a loop
// over the node's faces, each read waiting for the last and n1 a variable, 24.9, 16.2
// and 45.0.)
template <int N1>
__global__ __launch_bounds__(kBlock) void k_lift(const double* __restrict__ flux, const double* __restrict__ dA,
                                                 double* __restrict__ rhs, long long tfp, long long npts,
                                                 const int* __restrict__ vM) {
    constexpr int N2 = N1 * N1, NP = N2 * N1;
    for (long long v = xcd_block() * kBlock + threadIdx.x; v < npts; v += (long long)gridDim.x * kBlock) {
        const unsigned e = unsigned(v) / NP;  // volIdxMinus is 32-bit, so v is
        const int m = static_cast<int>(unsigned(v) - e * NP);
        const int i = m % N1, j = (m / N1) % N1, k = m / N2;
        const int pj = j == 0 ? i + N1 * k : (j == N1 - 1 ? 2 * N2 + i + N1 * k : -1);
        const int pi = i == N1 - 1 ? N2 + j + N1 * k : (i == 0 ? 3 * N2 + j + N1 * k : -1);
        const int pk = k == 0 ? 4 * N2 + i + N1 * j : (k == N1 - 1 ? 5 * N2 + i + N1 * j : -1);
        const bool j_first = pj >= 0 && (pi < 0 || pj < pi);
        const int pts[3] = {j_first ? pj : pi, j_first ? pi : pj, pk};
        if (pj < 0 && pi < 0 && pk < 0) continue;
        const long long fb = (long long)e * 6 * N2;
        double a[3], f[3][6], r[6];
        bool on[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const long long p = fb + pts[t];
            on[t] = pts[t] >= 0 && vM[p] == v;
            if (pts[t] >= 0) {
                a[t] = dA[p];
#pragma unroll
                for (int c = 0; c < 6; ++c) f[t][c] = flux[(c < 3 ? c + 3 : c - 3) * tfp + p];
            }
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) r[c] = rhs[c * npts + v];
#pragma unroll
        for (int t = 0; t < 3; ++t)
            if (on[t]) {
#pragma unroll
                for (int c = 0; c < 6; ++c) r[c] += a[t] * f[t][c];
            }
#pragma unroll
        for (int c = 0; c < 6; ++c) rhs[c * npts + v] = r[c];
    }
}

// The face points k_lift did not take (N1 > 0: those whose volIdxMinus is not
// the node the element-major layout puts them at; N1 == 0: all of them), added
// as the reference adds every point: rhs[vM] += dA * flux with FP64 atomics
// (dg_kernels.cu:316-338).  Points with vM outside [0, npts) are skipped.
template <int N1>
__global__ __launch_bounds__(kBlock) void k_lift_scatter(const double* __restrict__ flux, const double* __restrict__ dA,
                                                         double* __restrict__ rhs, long long tfp, long long npts,
                                                         const int* __restrict__ vM) {
    for (long long p = blockIdx.x * (long long)kBlock + threadIdx.x; p < tfp; p += (long long)gridDim.x * kBlock) {
        const long long v = vM[p];
        if constexpr (N1 > 0) {
            constexpr int N2 = N1 * N1;
            const long long e = p / (6 * N2);
            const int r = static_cast<int>(p - e * 6 * N2), f = r / N2, pq = r - f * N2;
            if (v == e * N2 * N1 + face_local_node<N1>(f, pq % N1, pq / N1)) continue;
        }
        if (v < 0 || v >= npts) continue;
        const double a = dA[p];
        atomicAdd(&rhs[v], a * flux[3 * tfp + p]);
        atomicAdd(&rhs[npts + v], a * flux[4 * tfp + p]);
        atomicAdd(&rhs[2 * npts + v], a * flux[5 * tfp + p]);
        atomicAdd(&rhs[3 * npts + v], a * flux[p]);
        atomicAdd(&rhs[4 * npts + v], a * flux[tfp + p]);
        atomicAdd(&rhs[5 * npts + v], a * flux[2 * tfp + p]);
    }
}

template <int N1>
void launch_lifts(const double* flux, const double* dA, double* rhs, long long tfp, long long npts, const int* vM,
                  hipStream_t s) {
    if constexpr (N1 > 0)
        hipLaunchKernelGGL(k_lift<N1>, dim3(grid_for_xcd(npts)), dim3(kBlock), 0, s, flux, dA, rhs, tfp, npts, vM);
    hipLaunchKernelGGL(k_lift_scatter<N1>, dim3(grid_for(tfp)), dim3(kBlock), 0, s, flux, dA, rhs, tfp, npts, vM);
}

__global__ void k_inv_mass(double* __restrict__ rhs, const double* __restrict__ jac, const double* __restrict__ w3,
                           int nxyz, long long npts, const double* __restrict__ eps, const double* __restrict__ mu) {
    for (long long idx = xcd_block() * blockDim.x + threadIdx.x; idx < npts; idx += (long long)gridDim.x * blockDim.x) {
        const long long e = npts <= 0x7fffffff ? unsigned(idx) / unsigned(nxyz) : idx / nxyz;
        const int i = static_cast<int>(idx - e * nxyz);
        const double ep = eps ? eps[e] : 1.0;
        const double iE = 1.0 / (ep * jac[idx] * w3[i]);
        const double iH = eps || mu ? 1.0 / ((mu ? mu[e] : 1.0) * jac[idx] * w3[i]) : iE;
        rhs[idx] *= iE; rhs[npts + idx] *= iE; rhs[2 * npts + idx] *= iE;
        rhs[3 * npts + idx] *= iH; rhs[4 * npts + idx] *= iH; rhs[5 * npts + idx] *= iH;
    }
}

__global__ void k_lsrk(double* __restrict__ st, double* __restrict__ k, const double* __restrict__ rhs, double a,
                       double b, double dt, long long npts, long long S) {
    const long long base = blockIdx.y * npts, sb = blockIdx.y * S;  // one component per grid row
    for (long long p = xcd_block() * blockDim.x + threadIdx.x; p < npts; p += (long long)gridDim.x * blockDim.x) {
        const double ki = a * k[base + p] + dt * rhs[base + p];
        k[base + p] = ki;
        st[sb + p] += b * ki;
    }
}

template <typename R>
__global__ void k_pack(const R* __restrict__ st, R* __restrict__ buf, const int* __restrict__ vol,
                       const int* __restrict__ off, const int* __restrict__ sizes, int nh, long long cs, long long ns) {
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < nh; x += gridDim.x * blockDim.x) {
        const long long v = vol[x];
        const int base = off[x], M = sizes[x];
#pragma unroll
        for (int c = 0; c < 6; ++c) buf[base + c * M] = st[c * cs + v * ns];
    }
}

template <typename R>
__global__ void k_unpack(const R* __restrict__ buf, R* __restrict__ st, const int* __restrict__ off,
                         const int* __restrict__ sizes, int nh, long long npts, long long cs, long long ns) {
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < nh; x += gridDim.x * blockDim.x) {
        const int base = off[x], M = sizes[x];
#pragma unroll
        for (int c = 0; c < 6; ++c) st[c * cs + (npts + x) * ns] = buf[base + c * M];
    }
}

// ---------------------------------------------------------------------------
// device geometry setup (computeMetricsFromCorners mesh.cpp:188-314 and
// setupFaceData mesh.cpp:985-1080, in the reference's expression order)
// ---------------------------------------------------------------------------
__global__ void k_metrics(const double* __restrict__ corners, int n1, long long npts, double* __restrict__ X,
                          double* __restrict__ Y, double* __restrict__ Z, double* __restrict__ jac, double* __restrict__ rx,
                          double* __restrict__ sx, double* __restrict__ tx, double* __restrict__ ry,
                          double* __restrict__ sy, double* __restrict__ ty, double* __restrict__ rz,
                          double* __restrict__ sz, double* __restrict__ tz) {
    const int n2 = n1 * n1, np = n2 * n1;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < npts; p += (long long)gridDim.x * blockDim.x) {
        const long long e = p / np;
        const int m = static_cast<int>(p - e * np);
        const double r = c_gll.z[n1][m % n1], s = c_gll.z[n1][(m / n1) % n1], t = c_gll.z[n1][m / n2];
        const double* c = corners + e * 24;
        const double sr[8] = {-1, 1, 1, -1, -1, 1, 1, -1}, ss[8] = {-1, -1, 1, 1, -1, -1, 1, 1};
        const double st[8] = {-1, -1, -1, -1, 1, 1, 1, 1};
        double x = 0, y = 0, z = 0, xr = 0, yr = 0, zr = 0, xs = 0, ys = 0, zs = 0, xt = 0, yt = 0, zt = 0;
#pragma unroll
        for (int a = 0; a < 8; ++a) {
            const double fr = 1.0 + sr[a] * r, fs = 1.0 + ss[a] * s, ft = 1.0 + st[a] * t;
            const double Nf = 0.125 * fr * fs * ft;
            const double dr = sr[a] * 0.125 * fs * ft, ds = ss[a] * 0.125 * fr * ft, dt = st[a] * 0.125 * fr * fs;
            const double vx = c[a * 3], vy = c[a * 3 + 1], vz = c[a * 3 + 2];
            x += Nf * vx; y += Nf * vy; z += Nf * vz;
            xr += dr * vx; yr += dr * vy; zr += dr * vz;
            xs += ds * vx; ys += ds * vy; zs += ds * vz;
            xt += dt * vx; yt += dt * vy; zt += dt * vz;
        }
        X[p] = x; Y[p] = y; Z[p] = z;
        const double det = xr * (ys * zt - yt * zs) - xs * (yr * zt - yt * zr) + xt * (yr * zs - ys * zr);
        jac[p] = det;
        const double iJ = 1.0 / det;
        rx[p] = iJ * (ys * zt - yt * zs); sx[p] = iJ * (yt * zr - yr * zt); tx[p] = iJ * (yr * zs - ys * zr);
        ry[p] = iJ * (xt * zs - xs * zt); sy[p] = iJ * (xr * zt - xt * zr); ty[p] = iJ * (xs * zr - xr * zs);
        rz[p] = iJ * (xs * yt - xt * ys); sz[p] = iJ * (xt * yr - xr * yt); tz[p] = iJ * (xr * ys - xs * yr);
    }
}

__global__ void k_face_data(const int* __restrict__ fcode, const int* __restrict__ fbc, int n1, long long tfp,
                            long long npts, const double* __restrict__ jac, const double* __restrict__ rx,
                            const double* __restrict__ sx, const double* __restrict__ tx, const double* __restrict__ ry,
                            const double* __restrict__ sy, const double* __restrict__ ty, const double* __restrict__ rz,
                            const double* __restrict__ sz, const double* __restrict__ tz, int* __restrict__ vP,
                            int* __restrict__ bc, double* __restrict__ nx, double* __restrict__ ny,
                            double* __restrict__ nz, double* __restrict__ dA) {
    const int n2 = n1 * n1, np = n2 * n1;
    for (long long P = blockIdx.x * (long long)blockDim.x + threadIdx.x; P < tfp; P += (long long)gridDim.x * blockDim.x) {
        const long long fi = P / n2;
        const int pq = static_cast<int>(P - fi * n2), p = pq % n1, q = pq / n1;
        const int e = static_cast<int>(fi / 6), f = static_cast<int>(fi % 6);
        int i, j, k;
        face_ijk(f, n1, p, q, i, j, k);
        const long long v = (long long)e * np + i + n1 * (j + n1 * k);
        const double J = jac[v], w2 = c_gll.w[n1][p] * c_gll.w[n1][q];
        double Nx, Ny, Nz;
        switch (f) {
            case 0: Nx = -J * sx[v]; Ny = -J * sy[v]; Nz = -J * sz[v]; break;
            case 1: Nx = J * rx[v]; Ny = J * ry[v]; Nz = J * rz[v]; break;
            case 2: Nx = J * sx[v]; Ny = J * sy[v]; Nz = J * sz[v]; break;
            case 3: Nx = -J * rx[v]; Ny = -J * ry[v]; Nz = -J * rz[v]; break;
            case 4: Nx = -J * tx[v]; Ny = -J * ty[v]; Nz = -J * tz[v]; break;
            default: Nx = J * tx[v]; Ny = J * ty[v]; Nz = J * tz[v]; break;
        }
        const double L = sqrt(Nx * Nx + Ny * Ny + Nz * Nz);
        nx[P] = L > 1e-14 ? Nx / L : 0.0; ny[P] = L > 1e-14 ? Ny / L : 0.0; nz[P] = L > 1e-14 ? Nz / L : 0.0;
        dA[P] = L * w2;
        const int code = fcode[fi];
        int plus;
        if (code >= 0) {
            const int e2 = code >> 6, f2 = (code >> 3) & 7, o = code & 7;
            int p2, q2, i2, j2, k2;
            orient_map(o, n1, p, q, p2, q2);
            face_ijk(f2, n1, p2, q2, i2, j2, k2);
            plus = e2 * np + i2 + n1 * (j2 + n1 * k2);
        } else if (code == -1) {
            plus = -1;
        } else {
            plus = static_cast<int>(npts) + (-(code + 2)) * n2 + pq;
        }
        vP[P] = plus;
        int b = fbc[fi];
        if (plus < 0 && b == 0) b = 1;
        bc[P] = b;
    }
}

// ---------------------------------------------------------------------------
// diagnostics: energy (FP64), max |E|, max |H|; two-pass deterministic reduce
// ---------------------------------------------------------------------------
// Quadrature weight of node p: J w_i w_j w_k, J from the metric array when
// given, else from the element's trilinear map (mesh.cpp:291-295).
__device__ __forceinline__ double node_dv(long long p, int n1, const double* __restrict__ jac,
                                          const ElemGeom* __restrict__ geom) {
    const int n2 = n1 * n1, np = n2 * n1;
    const long long e = p / np;
    const int m = static_cast<int>(p - e * np);
    const int i = m % n1, j = (m / n1) % n1, k = m / n2;
    double J;
    if (jac) {
        J = jac[p];
    } else {
        const double r = c_gll.z[n1][i], s = c_gll.z[n1][j], t = c_gll.z[n1][k];
        const double* c0 = geom[e].c[0];
        const double* c1 = geom[e].c[1];
        const double* c2 = geom[e].c[2];
        const double xr = c0[1] + c0[4] * s + c0[5] * t + c0[7] * (s * t);
        const double xs = c0[2] + c0[4] * r + c0[6] * t + c0[7] * (r * t);
        const double xt = c0[3] + c0[5] * r + c0[6] * s + c0[7] * (r * s);
        const double yr = c1[1] + c1[4] * s + c1[5] * t + c1[7] * (s * t);
        const double ys = c1[2] + c1[4] * r + c1[6] * t + c1[7] * (r * t);
        const double yt = c1[3] + c1[5] * r + c1[6] * s + c1[7] * (r * s);
        const double zr = c2[1] + c2[4] * s + c2[5] * t + c2[7] * (s * t);
        const double zs = c2[2] + c2[4] * r + c2[6] * t + c2[7] * (r * t);
        const double zt = c2[3] + c2[5] * r + c2[6] * s + c2[7] * (r * s);
        J = xr * (ys * zt - yt * zs) - xs * (yr * zt - yt * zr) + xt * (yr * zs - ys * zr);
    }
    return J * c_gll.w[n1][i] * c_gll.w[n1][j] * c_gll.w[n1][k];
}

template <typename R>
__global__ void k_diag_partial(const R* __restrict__ u, long long cs, long long ns, long long npts, int n1,
                               const double* __restrict__ jac,
                               const ElemGeom* __restrict__ geom, const ElemMat* __restrict__ mat,
                               double* __restrict__ part) {
    __shared__ double sh[3][kBlock];
    const int np = n1 * n1 * n1;
    double en = 0.0, me = 0.0, mh = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < npts; p += (long long)gridDim.x * blockDim.x) {
        const long long e = p / np;
        const double dV = node_dv(p, n1, jac, geom);
        const R* up = u + p * ns;
        const double ex = up[0], ey = up[cs], ez = up[2 * cs];
        const double hx = up[3 * cs], hy = up[4 * cs], hz = up[5 * cs];
        const double e2 = ex * ex + ey * ey + ez * ez, h2 = hx * hx + hy * hy + hz * hz;
        const double ep = mat ? 1.0 / mat[e].ieps : 1.0, mu = mat ? 1.0 / mat[e].imu : 1.0;
        en += 0.5 * (ep * e2 + mu * h2) * dV;
        me = fmax(me, e2);
        mh = fmax(mh, h2);
    }
    sh[0][threadIdx.x] = en; sh[1][threadIdx.x] = me; sh[2][threadIdx.x] = mh;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] = fmax(sh[1][threadIdx.x], sh[1][threadIdx.x + w]);
            sh[2][threadIdx.x] = fmax(sh[2][threadIdx.x], sh[2][threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x] = sh[0][0]; part[3 * blockIdx.x + 1] = sh[1][0]; part[3 * blockIdx.x + 2] = sh[2][0];
    }
}

// The partial triples of the blocks, reduced by one workgroup: kFinal threads stride
// over them, then a tree in LDS.  (One thread walking 1024 triples was a serial chain
// of dependent additions and reads: 121 us; this 4 us, most of it the launch.)
constexpr int kFinal = 256;
__global__ __launch_bounds__(kFinal) void k_diag_final(const double* __restrict__ part, int n, double* __restrict__ out) {
    __shared__ double sh[3][kFinal];
    const int t = threadIdx.x;
    double en = 0.0, me = 0.0, mh = 0.0;
    for (int b = t; b < n; b += kFinal) {
        en += part[3 * b]; me = fmax(me, part[3 * b + 1]); mh = fmax(mh, part[3 * b + 2]);
    }
    sh[0][t] = en; sh[1][t] = me; sh[2][t] = mh;
    __syncthreads();
    for (int w = kFinal / 2; w > 0; w >>= 1) {
        if (t < w) {
            sh[0][t] += sh[0][t + w];
            sh[1][t] = fmax(sh[1][t], sh[1][t + w]);
            sh[2][t] = fmax(sh[2][t], sh[2][t + w]);
        }
        __syncthreads();
    }
    if (t == 0) {
        out[0] = sh[0][0]; out[1] = sqrt(sh[1][0]); out[2] = sqrt(sh[2][0]);
    }
}

// Case::computeTotalEnergy, getMaxE, getMaxH (case.cpp:733-794) on a device
// state in the reference layout (component c of node p at c S + p): per block
// the sum of 1/2 (eps |E|^2 + mu |H|^2) J w_i w_j w_k (the reference's
// J[p] * w[i] * w[j] * w[k]) and the largest |E|^2, |H|^2; eps/mu per element
// or NULL (the reference's 1/2 (|E|^2 + |H|^2) dV).
__global__ void k_energy_partial(const double* __restrict__ st, long long S, long long npts, int n1,
                                 const double* __restrict__ jac, const double* __restrict__ w,
                                 const double* __restrict__ eps, const double* __restrict__ mu,
                                 double* __restrict__ part) {
    __shared__ double sh[3][kBlock];
    const int n2 = n1 * n1, np = n2 * n1;
    double en = 0.0, me = 0.0, mh = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < npts; p += (long long)gridDim.x * blockDim.x) {
        const long long e = p / np;
        const int m = static_cast<int>(p - e * np);
        const int i = m % n1, j = (m / n1) % n1, k = m / n2;
        const double dV = jac[p] * w[i] * w[j] * w[k];
        const double ex = st[p], ey = st[S + p], ez = st[2 * S + p];
        const double hx = st[3 * S + p], hy = st[4 * S + p], hz = st[5 * S + p];
        const double e2 = ex * ex + ey * ey + ez * ez, h2 = hx * hx + hy * hy + hz * hz;
        if (eps || mu)
            en += 0.5 * ((eps ? eps[e] : 1.0) * e2 + (mu ? mu[e] : 1.0) * h2) * dV;
        else
            en += 0.5 * (e2 + h2) * dV;
        me = fmax(me, e2);
        mh = fmax(mh, h2);
    }
    sh[0][threadIdx.x] = en; sh[1][threadIdx.x] = me; sh[2][threadIdx.x] = mh;
    __syncthreads();
    for (int r = blockDim.x / 2; r > 0; r >>= 1) {
        if (threadIdx.x < r) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + r];
            sh[1][threadIdx.x] = fmax(sh[1][threadIdx.x], sh[1][threadIdx.x + r]);
            sh[2][threadIdx.x] = fmax(sh[2][threadIdx.x], sh[2][threadIdx.x + r]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x] = sh[0][0]; part[3 * blockIdx.x + 1] = sh[1][0]; part[3 * blockIdx.x + 2] = sh[2][0];
    }
}

// Relative L2 distance to a reference state (3dboxpec_test.cpp:76-119):
// sum over components and nodes of (u - ref)^2 dV and ref^2 dV, in FP64.
// ref is in the reference's host layout (component blocks of npts).
template <typename R>
__global__ void k_l2_partial(const R* __restrict__ u, long long cs, long long ns, const double* __restrict__ ref,
                             long long npts, int n1, const double* __restrict__ jac,
                             const ElemGeom* __restrict__ geom, double* __restrict__ part) {
    __shared__ double sh[2][kBlock];
    double num = 0.0, den = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < npts; p += (long long)gridDim.x * blockDim.x) {
        const double dV = node_dv(p, n1, jac, geom);
        const R* up = u + p * ns;
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const double r = ref[c * npts + p], d = double(up[c * cs]) - r;
            a += d * d;
            b += r * r;
        }
        num += a * dV;
        den += b * dV;
    }
    sh[0][threadIdx.x] = num; sh[1][threadIdx.x] = den;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sh[0][0]; part[2 * blockIdx.x + 1] = sh[1][0];
    }
}

__global__ __launch_bounds__(kFinal) void k_l2_final(const double* __restrict__ part, int n, double* __restrict__ out) {
    __shared__ double sh[2][kFinal];
    const int t = threadIdx.x;
    double num = 0.0, den = 0.0;
    for (int b = t; b < n; b += kFinal) {
        num += part[2 * b]; den += part[2 * b + 1];
    }
    sh[0][t] = num; sh[1][t] = den;
    __syncthreads();
    for (int w = kFinal / 2; w > 0; w >>= 1) {
        if (t < w) {
            sh[0][t] += sh[0][t + w];
            sh[1][t] += sh[1][t + w];
        }
        __syncthreads();
    }
    if (t == 0) {
        out[0] = sh[0][0]; out[1] = sh[1][0];
    }
}

// Probe records (ProbeManager::record, probe.cpp:192-216) on the device, one
// workgroup per probe and step: the threads form the rounded products w_p *
// u_c(p), w_p = (Lr[i] Ls[j]) Lt[k], of all the element's nodes at once into LDS;
// then one thread per component adds them in node order -- the reference's
// operations in its order, in FP64, so the record is bit for bit the host's --
// into record slot (*slot + step) mod cap.  The sum is one serial chain: its LDS
// reads are issued eight at a time ahead of the additions.  `stop`
// (may be null): nonzero where the steps' launch gave up, no record then.
// k_probe_advance moves the slot afterwards (stream order), so every workgroup
// reads the same slot.
template <typename R>
__global__ void __launch_bounds__(256) k_probe(const R* __restrict__ u, long long cs, long long ns, int nprobes,
                                               const long long* __restrict__ base, const double* __restrict__ lw,
                                               int n1, double* __restrict__ hist, const int* __restrict__ slot,
                                               int cap, long long step_stride, const int* __restrict__ stop) {
    constexpr int kAhead = 8;
    __shared__ double prod[6][kMaxN1 * kMaxN1 * kMaxN1];
    if (stop && *stop) return;
    const int q = blockIdx.x, step = blockIdx.y;
    const int np = n1 * n1 * n1;
    const double* Lr = lw + size_t(q) * 3 * n1;
    const double* Ls = Lr + n1;
    const double* Lt = Ls + n1;
    const R* up = u + step * step_stride + base[q] * ns;
    for (int p = threadIdx.x; p < np; p += blockDim.x) {
        const int i = p % n1, j = (p / n1) % n1, kk = p / (n1 * n1);
        const double w = __dmul_rn(__dmul_rn(Lr[i], Ls[j]), Lt[kk]);
#pragma unroll
        for (int c = 0; c < 6; ++c) prod[c][p] = __dmul_rn(w, double(up[p * ns + c * cs]));
    }
    __syncthreads();
    // past the capacity the history is lost either way (the host reports it)
    const long long at = (long long)*slot + step;
    if (threadIdx.x < 6 && (gridDim.y == 1 || at < cap)) {
        const int c = threadIdx.x;
        double acc = 0.0;
        int p = 0;
        for (; p + kAhead <= np; p += kAhead) {
            double v[kAhead];
#pragma unroll
            for (int x = 0; x < kAhead; ++x) v[x] = prod[c][p + x];
#pragma unroll
            for (int x = 0; x < kAhead; ++x) acc = __dadd_rn(acc, v[x]);  // no contraction: the host sum's roundings
        }
        for (; p < np; ++p) acc = __dadd_rn(acc, prod[c][p]);
        hist[(size_t(at % cap) * nprobes + q) * 6 + c] = acc;
    }
}

// Counts records up to cap + 1 (the overflow the host reports), so a run that
// never fetches its history cannot wrap the counter.
__global__ void k_probe_advance(int* p, int cap, int n, const int* __restrict__ stop) {
    if (threadIdx.x == 0 && blockIdx.x == 0 && !(stop && *stop)) *p = min(*p + n, cap + 1);
}

// Sets *slot = 0 with a kernel (no memset node if a caller captures it).
__global__ void k_zero_int(int* p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}
// ---------------------------------------------------------------------------
// conversions and plain copy (HBM calibration)
// ---------------------------------------------------------------------------
// Nodes p0 .. p0 + n - 1 of a device state (component c of node p at c cs + p ns) from
// a pinned host slot of six blocks of n doubles, or to one of six blocks of n device
// values: the slot's side is coalesced and crosses the link once; bound by the link
// (55 GB/s).  Rounding to FP32 is done here on the way in: on the host, values below
// FP32's normal range take an assist each (12.6 MB of a pulse: 3.4 ms instead of 0.3).
template <typename R>
__global__ void k_state_in(R* __restrict__ u, long long cs, long long ns, long long p0, long long n,
                           const double* __restrict__ slot) {
    for (long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x < n; x += (long long)gridDim.x * blockDim.x) {
        R* q = u + (p0 + x) * ns;
#pragma unroll
        for (int c = 0; c < 6; ++c) q[c * cs] = static_cast<R>(slot[c * n + x]);
    }
}
template <typename R>
__global__ void k_state_out(const R* __restrict__ u, long long cs, long long ns, long long p0, long long n,
                            R* __restrict__ slot) {
    for (long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x < n; x += (long long)gridDim.x * blockDim.x) {
        const R* q = u + (p0 + x) * ns;
#pragma unroll
        for (int c = 0; c < 6; ++c) slot[c * n + x] = q[c * cs];
    }
}

__global__ void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, long long n4) {
    for (long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x < n4; x += (long long)gridDim.x * blockDim.x)
        dst[x] = src[x];
}

__global__ void k_fill(double* __restrict__ p, long long n, double v) {
    for (long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x < n; x += (long long)gridDim.x * blockDim.x)
        p[x] = v;
}

}  // namespace

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
int plain_upload_tables(const GllTables& t) {
    NW_TRY_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_gll), &t, sizeof(GllTables)));
    return NW_OK;
}

hipError_t launch_volume_curl(const PlainVolumeArgs& a, hipStream_t s) {
    if (a.nelt <= 0) return hipSuccess;
    switch (a.n1) {
        case 2: return launch_vc<2>(a, s);
        case 3: return launch_vc<3>(a, s);
        case 4: return launch_vc<4>(a, s);
        case 5: return launch_vc<5>(a, s);
        case 6: return launch_vc<6>(a, s);
        case 7: return launch_vc<7>(a, s);
        case 8: return launch_vc<8>(a, s);
        case 9: return launch_vc<9>(a, s);
        case 10: return launch_vc<10>(a, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_restrict(const double* st, double* fEN, double* fHN, const int* vM, long long tfp, long long S,
                           hipStream_t s) {
    if (tfp <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_restrict, dim3(grid_for_xcd(tfp)), dim3(kBlock), 0, s, st, fEN, fHN, vM, tfp, S);
    return hipGetLastError();
}

hipError_t launch_flux(const double* st, const double* fEN, const double* fHN, const int* vP, const int* bc,
                       const double* nx, const double* ny, const double* nz, double* flux, double c0, long long tfp,
                       long long S, const int* vM, const double* eps, const double* mu, const int* ghost_elem, int np,
                       long long npts, hipStream_t s) {
    if (tfp <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_flux, dim3(grid_for_xcd(tfp)), dim3(kBlock), 0, s, st, fEN, fHN, vP, bc, nx, ny, nz, flux, c0,
                       tfp, S, vM, eps, mu, ghost_elem, np, npts);
    return hipGetLastError();
}

hipError_t launch_add_flux(const double* flux, const int* vM, const double* dA, double* rhs, long long tfp,
                           long long npts, hipStream_t s) {
    if (tfp <= 0) return hipSuccess;
    // n1 of the element-major layout, when the sizes admit one: tfp = 6 n1^2 nelt,
    // npts = n1^3 nelt
    int n1 = 0;
    if (npts > 0 && (6 * npts) % tfp == 0) {
        const long long c = 6 * npts / tfp;
        if (c >= kMinN1 && c <= kMaxN1 && npts % (c * c * c) == 0 && tfp == 6 * c * c * (npts / (c * c * c)))
            n1 = static_cast<int>(c);
    }
    switch (n1) {
        case 2: launch_lifts<2>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 3: launch_lifts<3>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 4: launch_lifts<4>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 5: launch_lifts<5>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 6: launch_lifts<6>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 7: launch_lifts<7>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 8: launch_lifts<8>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 9: launch_lifts<9>(flux, dA, rhs, tfp, npts, vM, s); break;
        case 10: launch_lifts<10>(flux, dA, rhs, tfp, npts, vM, s); break;
        default: launch_lifts<0>(flux, dA, rhs, tfp, npts, vM, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_inv_mass(double* rhs, const double* jac, const double* w3, int nxyz, long long npts,
                           const double* eps, const double* mu, hipStream_t s) {
    if (npts <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_inv_mass, dim3(grid_for_xcd(npts)), dim3(kBlock), 0, s, rhs, jac, w3, nxyz, npts, eps, mu);
    return hipGetLastError();
}

hipError_t launch_lsrk(double* st, double* k, const double* rhs, double a, double b, double dt,
                       long long npts, long long S, hipStream_t s) {
    if (npts <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_lsrk, dim3(grid_for_xcd(npts), 6), dim3(kBlock), 0, s, st, k, rhs, a, b, dt, npts, S);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_pack(const R* st, R* buf, const int* vol, const int* off, const int* sizes, int nh, long long cs,
                       long long ns, hipStream_t s) {
    if (nh <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pack<R>, dim3(grid_for(nh)), dim3(kBlock), 0, s, st, buf, vol, off, sizes, nh, cs, ns);
    return hipGetLastError();
}
template <typename R>
hipError_t launch_unpack(const R* buf, R* st, const int* off, const int* sizes, int nh, long long npts, long long cs,
                         long long ns, hipStream_t s) {
    if (nh <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_unpack<R>, dim3(grid_for(nh)), dim3(kBlock), 0, s, buf, st, off, sizes, nh, npts, cs, ns);
    return hipGetLastError();
}
template hipError_t launch_pack<double>(const double*, double*, const int*, const int*, const int*, int, long long,
                                        long long, hipStream_t);
template hipError_t launch_pack<float>(const float*, float*, const int*, const int*, const int*, int, long long, long long,
                                       hipStream_t);
template hipError_t launch_unpack<double>(const double*, double*, const int*, const int*, int, long long, long long,
                                          long long, hipStream_t);
template hipError_t launch_unpack<float>(const float*, float*, const int*, const int*, int, long long, long long,
                                         long long, hipStream_t);

hipError_t launch_metrics(const double* corners, int n1, long long npts, double* const* out13, hipStream_t s) {
    if (npts <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_metrics, dim3(grid_for(npts)), dim3(kBlock), 0, s, corners, n1, npts, out13[0], out13[1],
                       out13[2], out13[3], out13[4], out13[5], out13[6], out13[7], out13[8], out13[9], out13[10],
                       out13[11], out13[12]);
    return hipGetLastError();
}

hipError_t launch_face_data(const int* fcode, const int* fbc, int n1, long long tfp, long long npts,
                            const double* const* met10, int* vP, int* bc, double* nx, double* ny, double* nz,
                            double* dA, hipStream_t s) {
    if (tfp <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_face_data, dim3(grid_for(tfp)), dim3(kBlock), 0, s, fcode, fbc, n1, tfp, npts, met10[0],
                       met10[1], met10[2], met10[3], met10[4], met10[5], met10[6], met10[7], met10[8], met10[9], vP,
                       bc, nx, ny, nz, dA);
    return hipGetLastError();
}

int diag_blocks() { return 1024; }

template <typename R>
hipError_t launch_diag(const R* u, long long cs, long long ns, long long npts, int n1, const double* jac,
                       const ElemGeom* geom, const ElemMat* mat, double* part, double* out, hipStream_t s) {
    const int nb = diag_blocks();
    hipLaunchKernelGGL(k_diag_partial<R>, dim3(nb), dim3(kBlock), 0, s, u, cs, ns, npts, n1, jac, geom, mat, part);
    hipLaunchKernelGGL(k_diag_final, dim3(1), dim3(kFinal), 0, s, part, nb, out);
    return hipGetLastError();
}
// Partial sums of nw_launch_diagnostics_noalloc: a fixed device array (one
// copy per GPU, each at its own address, held until the process ends) instead
// of an allocation.  Host code must use the address energy_scratch() returns,
// never this name.  Every call on a GPU shares that GPU's copy: calls that
// overlap on one GPU race.
static __device__ __align__(256) double scratch[3 * kEnergyScratchBlocks];
static_assert(kEnergyScratchBlocks >= kEnergyMaxBlocks, "the scratch holds every block of the largest grid");

int energy_scratch(double** out) {
    static std::mutex mu;
    static double* addr[kMaxDevices] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return -1;
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return -2;
        addr[dev] = static_cast<double*>(p);
    }
    *out = addr[dev];
    return 0;
}

int energy_blocks(long long npts) {
    const long long b = (npts + kBlock - 1) / kBlock;
    return static_cast<int>(b < 1 ? 1 : (b > kEnergyMaxBlocks ? kEnergyMaxBlocks : b));
}

hipError_t launch_energy(const double* st, long long S, long long npts, int n1, const double* jac, const double* w,
                         const double* eps, const double* mu, double* part, double* out, hipStream_t s) {
    const int nb = energy_blocks(npts);
    hipLaunchKernelGGL(k_energy_partial, dim3(nb), dim3(kBlock), 0, s, st, S, npts, n1, jac, w, eps, mu, part);
    hipLaunchKernelGGL(k_diag_final, dim3(1), dim3(kFinal), 0, s, part, nb, out);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_l2(const R* u, long long cs, long long ns, const double* ref, long long npts, int n1, const double* jac,
                     const ElemGeom* geom, double* part, double* out, hipStream_t s) {
    const int nb = diag_blocks();
    hipLaunchKernelGGL(k_l2_partial<R>, dim3(nb), dim3(kBlock), 0, s, u, cs, ns, ref, npts, n1, jac, geom, part);
    hipLaunchKernelGGL(k_l2_final, dim3(1), dim3(kFinal), 0, s, part, nb, out);
    return hipGetLastError();
}
template hipError_t launch_l2<double>(const double*, long long, long long, const double*, long long, int, const double*,
                                      const ElemGeom*, double*, double*, hipStream_t);
template hipError_t launch_l2<float>(const float*, long long, long long, const double*, long long, int, const double*,
                                     const ElemGeom*, double*, double*, hipStream_t);
template hipError_t launch_diag<double>(const double*, long long, long long, long long, int, const double*,
                                        const ElemGeom*, const ElemMat*, double*, double*, hipStream_t);
template hipError_t launch_diag<float>(const float*, long long, long long, long long, int, const double*, const ElemGeom*,
                                       const ElemMat*, double*, double*, hipStream_t);

static dim3 state_grid(long long n) { return dim3(static_cast<unsigned>(std::min<long long>(256, (n + kBlock - 1) / kBlock))); }
template <typename R>
hipError_t launch_state_in(R* u, long long cs, long long ns, long long p0, long long n, const double* slot, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_state_in<R>, state_grid(n), dim3(kBlock), 0, s, u, cs, ns, p0, n, slot);
    return hipGetLastError();
}
template <typename R>
hipError_t launch_state_out(const R* u, long long cs, long long ns, long long p0, long long n, R* slot, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_state_out<R>, state_grid(n), dim3(kBlock), 0, s, u, cs, ns, p0, n, slot);
    return hipGetLastError();
}
#define NW_STATE_MOVE(R)                                                                                                   \
    template hipError_t launch_state_in<R>(R*, long long, long long, long long, long long, const double*, hipStream_t);    \
    template hipError_t launch_state_out<R>(const R*, long long, long long, long long, long long, R*, hipStream_t);
NW_STATE_MOVE(float)
NW_STATE_MOVE(double)
#undef NW_STATE_MOVE

hipError_t launch_copy(const void* src, void* dst, long long bytes, hipStream_t s) {
    const long long n4 = bytes / 16;
    hipLaunchKernelGGL(k_copy, dim3(grid_for(n4, 256) > 8192 ? 8192 : grid_for(n4, 256)), dim3(256), 0, s,
                       static_cast<const float4*>(src), static_cast<float4*>(dst), n4);
    return hipGetLastError();
}

hipError_t launch_fill(double* p, long long n, double v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(kBlock), 0, s, p, n, v);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_probe(const R* u, long long cs, long long ns, int nprobes, const long long* base, const double* lw,
                        int n1, double* hist, int* slot, int cap, hipStream_t s, int nsteps, long long step_stride,
                        const int* stop) {
    if (nprobes <= 0 || nsteps <= 0) return hipSuccess;
    if (n1 < 2 || n1 > kMaxN1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_probe<R>, dim3(nprobes, nsteps), dim3(256), 0, s, u, cs, ns, nprobes, base, lw, n1, hist, slot, cap,
                       step_stride, stop);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_probe_advance, dim3(1), dim3(64), 0, s, slot, cap, nsteps, stop);
    return hipGetLastError();
}
template hipError_t launch_probe<double>(const double*, long long, long long, int, const long long*, const double*, int,
                                         double*, int*, int, hipStream_t, int, long long, const int*);
template hipError_t launch_probe<float>(const float*, long long, long long, int, const long long*, const double*, int,
                                        double*, int*, int, hipStream_t, int, long long, const int*);

hipError_t launch_zero_int(int* p, hipStream_t s) {
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, s, p);
    return hipGetLastError();
}


}  // namespace nw
