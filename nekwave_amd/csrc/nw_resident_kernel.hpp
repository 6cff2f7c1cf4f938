// nw_resident_kernel.hpp -- the resident multi-step kernel (gfx950), included by
// one translation unit per precision.
#pragma once

#include <algorithm>
#include <atomic>

#include "nw_device.hpp"
#include "nw_resident.hpp"

namespace nw {
namespace {

constexpr int kLdsGranule = 1280;  // LDS is handed out in 128ths of a CU's 160 KB

// LDS bytes of one workgroup, as k_resident declares them, without LSRK registers.
constexpr int resident_lds(int n1, int em, int rsz, bool affine) {
    const int n2 = n1 * n1;
    const int plane = n1 == 8 && rsz == 4 ? 72 : n2, sent = n1 == 8 && rsz == 4 ? 1 : 0;
    return rsz * ((em + sent) * 6 * plane * n1 + (6 * n2 + 1) * 6 + n2 + n1 + em * (affine ? 12 : 26)) + 32;
}
// VGPRs a thread may have, and the workgroups per CU that they and LDS allow.
template <int NT, int RBYTES>
constexpr int resident_budget() {
    constexpr int waves = (NT + 63) / 64, eu = WavesPerEU<NT, RBYTES>::value, own = (waves + 3) / 4;
    return 512 / (eu > own ? eu : own) / 8 * 8;
}
template <int NT, int RBYTES>
constexpr int resident_fit(int lds) {
    constexpr int waves = (NT + 63) / 64, eu = WavesPerEU<NT, RBYTES>::value;
    constexpr int regs = 4 * eu / waves > 1 ? 4 * eu / waves : 1;
    const int held = 160 * 1024 / ((lds + kLdsGranule - 1) / kLdsGranule * kLdsGranule);
    return regs < held ? regs : held;
}
// Elements whose LSRK registers lie in LDS instead of VGPRs: enough that nothing spills (a
// reload inside the stage waits for every packet in flight), as far as they fit beside
// the fields without costing a workgroup per CU.  The need is what the compiler reports
// for kernels that do not spill: a base by face points per thread, field type and
// geometry, and per element its LSRK registers and packet offsets.  Measured per stage,
// all in VGPRs -> this: FP32 jittered n1 = 5, 2744 elements 14.9 -> 10.9 us; FP64 jittered
// n1 = 5, 1000 13.6 -> 9.6; FP32 with FP64 registers jittered n1 = 7, 1287 16.8 -> 15.1,
// n1 = 5, 1728 10.2 -> 7.9.  Where nothing spills LDS costs 1-3 % (n1 = 9, 1000 elements
// 16.2 -> 16.5), so the registers stay there.  (tests/test_resident_registers.py reads the
// spills from the built library, so that a compiler that spills more is noticed.)
template <int N1, int EM, int RBYTES, int KBYTES, bool AFF>
constexpr int resident_lds_k() {
    constexpr int NT = N1 * N1 * N1, fpt = (6 * N1 * N1 + NT - 1) / NT, kregs = 6 * KBYTES / 4;
    constexpr int base = fpt == 1 ? (RBYTES == 4 ? (AFF ? 98 : 112) : (AFF ? 147 : 190))
                                  : (RBYTES == 4 ? (AFF ? 106 : 151) : (AFF ? 182 : 272));
    constexpr int lds = resident_lds(N1, EM, RBYTES, AFF), per = 6 * NT * KBYTES, budget = resident_budget<NT, RBYTES>();
    int n = 0;
    while (EM > 1 && n < EM && base + EM * fpt + (EM - n) * kregs > budget && lds + (n + 1) * per <= 160 * 1024 &&
           resident_fit<NT, RBYTES>(lds + (n + 1) * per) >= resident_fit<NT, RBYTES>(lds)) ++n;
    return n;
}

// A uniform base and a 32-bit offset per lane: no 64-bit address arithmetic.
__device__ __forceinline__ void packet_store(char* base, unsigned off, unsigned ep, unsigned v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(base + size_t(off)),
                       (static_cast<unsigned long long>(ep) << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long packet_load(const char* base, unsigned off) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(base + size_t(off)), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// One launch = nsteps LSRK45 steps of the elements of `nelt`, all on chip at once: a
// workgroup owns up to EM elements, one thread per node (as k_fused_stage with one
// element per workgroup, whose expressions it repeats: the same bits), fields in
// LDS, LSRK registers in VGPRs (or LDS: resident_lds_k).  HBM is touched at the launch's ends only; per stage
// an element's six traces go out and its neighbours' come in.
//
// Why: a stage of a small mesh is bound by its launch (3-4 us for dispatch and the
// boundary's L2 write-back) and the chain of dependent first reads, not by
// bandwidth.  Here the chain per stage is publish -> one trip of the fabric ->
// flux -> two barriers.  Measured per stage, stage launches against this kernel:
//   n1 = 5,   64 elements, FP64              6.5 ->  2.6 us
//   n1 = 8,  216 / 512 elements, FP32        7.6 ->  2.5 / 10.3 -> 3.9 us
//   n1 = 6, 1000 elements, FP64             14.2 ->  8.5 us
//   n1 = 8, 1728 elements, FP32             21.7 -> 14.3 us (uniform), 23.3 -> 18.0 us (jittered)
//   n1 = 9, 1728 elements, FP32             36.7 -> 27.4 us (uniform), 37.7 -> 29.6 us (jittered)
//   n1 = 4, 5832 elements, FP32             11.8 ->  8.3 us
// (where it is slower: resident_range).
// Up to one element per workgroup the stage is bound by that chain (packets alone:
// 1.3 us for 64 workgroups, 2.5 for 256, 4.3 for 512 at 384 points each); beyond, by
// the vector ALUs (54-60 % busy) and LDS (55-60 %; n1 = 8 in FP32 77 % before QB).
// Traces as plain values behind a per-wave flag (half the bytes) were slower
// everywhere (n1 = 8, 512 elements 6.0 us, 1728 elements 17.9): two trips of the
// fabric instead of one.  So were packets stored by a node's own thread at once after its
// update (partly filled waves: 512 elements 5.1).
template <int N1, int EM, typename R, typename KR, bool AFF>
__global__ __launch_bounds__(N1* N1* N1) __attribute__((amdgpu_waves_per_eu(WavesPerEU<N1 * N1 * N1, sizeof(R)>::value)))
void k_resident(ResidentArgs A) {
    constexpr int N2 = N1 * N1, NP = N1 * N2, NF = 6 * N2, NT = NP;
    constexpr int FPT = (NF + NT - 1) / NT;     // face points per thread
    constexpr int PC = 6 * int(sizeof(R)) / 4;  // packets per face point
    constexpr int GW = AFF ? 10 : 24;           // geometry words per element
    // QB: contractions by quad broadcast (line8x3); wave k holds plane k.  Rows are 9
    // and planes 72 words apart there, so that lines in every direction and the nodes
    // of every face fall into different banks.  A third less
    // LDS time (n1 = 8, 512 elements: 423 -> 285 LDS cycles per wave and stage): against
    // this kernel without it 4.6 -> 4.2 us per stage, 1728 uniform elements 17.0 -> 15.6.
    constexpr bool QB = N1 == 8 && sizeof(R) == 4;
    constexpr int RS = QB ? 9 : N1, PL = QB ? 72 : N2;  // row and plane strides of sU
    __shared__ R sU[EM][6][PL * N1];
    __shared__ R sT[QB ? 6 : 1][QB ? PL * N1 : 1];  // QB: t-derivatives, handed across waves
    __shared__ R sF[NF + 1][6];  // face terms dA*F; the last row stays zero
    __shared__ __attribute__((aligned(16))) R sD[N2];
    __shared__ R sZ[N1];         // GLL nodes
    __shared__ R sG[EM][GW];
    __shared__ R sM[EM][2];      // 1/eps, 1/mu
    constexpr int KL = resident_lds_k<N1, EM, sizeof(R), sizeof(KR), AFF>();
    // LSRK registers of elements 0 .. KL - 1, [element][component][node].  Dynamic LDS: as
    // static LDS it would count in the compiler's occupancy, which then spends the
    // registers of a second workgroup
    extern __shared__ double sKdyn[];
    KR* const sK = reinterpret_cast<KR*>(sKdyn);
    __shared__ int sStop;

    const int tid = threadIdx.x, m = tid;
    const int i = m % N1, j = (m / N1) % N1, k = m / N2;
    const int at = i + RS * j + PL * k;  // the node's place in sU
    const int el0 = A.elem0 + static_cast<int>(blockIdx.x) * A.per;  // first element of this workgroup
    const int cnt = min(A.per, A.elem0 + A.nelt - el0);
    const R* uin = static_cast<const R*>(A.uin);
    R* uout = static_cast<R*>(A.uout);

    // a launch before this one gave up: leave the buffers as they are
    if (tid == 0) sStop = __hip_atomic_load(A.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int x = tid; x < N2; x += NT) sD[x] = gD<R>(N1, x);
    for (int x = tid; x < N1; x += NT) sZ[x] = R(c_gll.z[N1][x]);
    for (int x = tid; x < 6; x += NT) sF[NF][x] = R(0);
    for (int w = tid; w < EM * 26; w += NT) {
        const int x = w / 26, c = w - 26 * x;
        if (x < cnt) {
            const R v = R(A.rec[size_t(el0 + x) * 26 + c]);
            if (c >= 24) sM[x][c - 24] = v;
            else if (c < GW) sG[x][c] = v;
        }
    }
    for (int x = 0; x < cnt; ++x) {
        const R* q = uin + (A.node_base + (long long)(el0 + x) * NP + m) * 6;
#pragma unroll
        for (int c = 0; c < 6; ++c) sU[x][c][at] = q[c];
    }
    const R Winv = R(c_gll.iw[N1][i] * c_gll.iw[N1][j] * c_gll.iw[N1][k]);

    // this thread's face points: local node, weight, own slot and plus-side slot
    int fnode[FPT], ff[FPT], fpq[FPT];
    unsigned own[FPT];  // byte offset of its packets in element 0 of the workgroup
    R wpq[FPT];
#pragma unroll
    for (int t = 0; t < FPT; ++t) {
        const int fp = min(tid + t * NT, NF - 1);
        const int f = fp / N2, pq = fp - f * N2, p = pq % N1, q = pq / N1;
        ff[t] = f;
        fpq[t] = pq;
        own[t] = 8u * (unsigned((el0 - A.elem0) * 6 + f) * (PC * N2) + unsigned(pq));
        const int ln = face_local_node<N1>(f, p, q);
        fnode[t] = ln % N1 + RS * (ln / N1 % N1) + PL * (ln / N2);
        wpq[t] = R(c_gll.w[N1][p] * c_gll.w[N1][q]);
    }
    __syncthreads();
    // uniform over the workgroup: the second barrier, so that a wave that gives up later
    // stores sStop only after every wave has read the entry value
    const bool gone = sStop != 0;
    __syncthreads();
    if (gone) return;

    // Traces travel as 8-byte packets of 4 bytes of value and the epoch, stored and
    // read whole: a reader that sees the tag has the value, in one trip of the
    // fabric, and no flag, fence or barrier orders anything.  Two buffers by the
    // epoch's parity suffice: element A writes epoch e + 2 after it has read B's
    // e + 1, which B wrote after it had read A's e (faces pair up).
    const unsigned half = unsigned(A.nelt) * 6u * (PC * N2) * 8u;
    auto buffer_of = [&](unsigned e) { return reinterpret_cast<char*>(A.xchg) + (e & 1u ? half : 0u); };
    auto publish = [&](int x, unsigned ep) {
        char* const xb = buffer_of(ep);
#pragma unroll
        for (int t = 0; t < FPT; ++t) {
            if (tid + t * NT < NF) {
                const unsigned o = own[t] + unsigned(x) * (48u * PC * N2);
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    const R v = sU[x][c][fnode[t]];
                    if constexpr (sizeof(R) == 4) {
                        packet_store(xb, o + 8 * c * N2, ep, __builtin_bit_cast(unsigned, v));
                    } else {
                        const unsigned long long w = __builtin_bit_cast(unsigned long long, v);
                        packet_store(xb, o + 16 * c * N2, ep, static_cast<unsigned>(w));
                        packet_store(xb, o + (16 * c + 8) * N2, ep, static_cast<unsigned>(w >> 32));
                    }
                }
            }
        }
    };

    // Per element: LSRK registers (in LDS for the first KL), and the byte offset of the
    // plus side's packets of the thread's face points (-1: mirror; the exchange buffer is
    // below 2 GiB, the launcher's limit).  The element in hand has them in kc and slot; the others
    // stay in registers, moved by uniform branches (pinned: as selects, every
    // element would cost moves of all of them).
    KR kk[EM > KL ? EM - KL : 1][6], kc[6];
    int slots[EM][FPT], slot[FPT];
#pragma unroll
    for (int x = 0; x < EM; ++x) {
        for (int c = 0; c < 6 && x >= KL; ++c) kk[x - KL][c] = KR(0);
#pragma unroll
        for (int t = 0; t < FPT; ++t) {
            slots[x][t] = -1;
            if (x < cnt) {
                const int4 b = A.nbr[(el0 + x) * 6 + ff[t]];
                const int p = fpq[t] % N1, q = fpq[t] / N1;
                if (b.x >= 0) slots[x][t] = 8 * ((b.x - A.elem0 * 6) * (PC * N2) + b.y + p * b.z + q * b.w);
            }
        }
    }
    auto take_slots = [&](int x) {
#pragma unroll
        for (int y = 0; y < EM; ++y)
            if (EM == 1 || x == y) {
#pragma unroll
                for (int t = 0; t < FPT; ++t) { slot[t] = slots[y][t]; if (EM > 1) pin(slot[t]); }
            }
    };
    // taken at the update (six registers fewer live through the volume work: n1 = 8,
    // 1728 jittered elements 18.5 against 20.4 us per stage)
    auto take_k = [&](int x) {
        if (KL > 0 && x < KL) {
#pragma unroll
            for (int c = 0; c < 6; ++c) kc[c] = sK[(x * 6 + c) * NP + m];
        }
#pragma unroll
        for (int y = KL; y < EM; ++y)
            if (EM == 1 || x == y) {
#pragma unroll
                for (int c = 0; c < 6; ++c) { kc[c] = kk[y - KL][c]; if (EM > 1) pin(kc[c]); }
            }
    };
    auto keep_k = [&](int x) {
        if (KL > 0 && x < KL) {
#pragma unroll
            for (int c = 0; c < 6; ++c) sK[(x * 6 + c) * NP + m] = kc[c];
        }
#pragma unroll
        for (int y = KL; y < EM; ++y)
            if (EM == 1 || x == y) {
#pragma unroll
                for (int c = 0; c < 6; ++c) { kk[y - KL][c] = kc[c]; if (EM > 1) pin(kk[y - KL][c]); }
            }
    };

    // with one element per workgroup its geometry stays in registers
    constexpr bool KEEP = EM == 1;
    R geo[10];
    R fN[FPT][4];  // unit normal, dA
    R fw[FPT][4];
    auto face_geometry = [&](int x) {
#pragma unroll
        for (int t = 0; t < FPT; ++t) {
            const int f = ff[t];
            const int dir = (f == 1 || f == 3) ? 0 : ((f == 0 || f == 2) ? 1 : 2);  // r-, s-, t-face
            // outward Nanson vector: +-(cofactor row of the face's direction)
            const R sg = (f == 1 || f == 2 || f == 5) ? R(1) : R(-1);
            R C[3];
            if constexpr (AFF) {
#pragma unroll
                for (int c = 0; c < 3; ++c) C[c] = sG[x][3 * dir + c];
            } else {
                // the row alone: the cross product of the two other directions'
                // tangents, in node_geometry's expressions (node_geometry computes
                // nine tangents and three rows)
                int ln = fnode[t];
                if constexpr (!KEEP) pin(ln);
                const R r = sZ[ln % PL % RS], q = sZ[ln % PL / RS], w = sZ[ln / PL];
                R T[2][3];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int a = (dir + 1 + h) % 3;  // tangent along direction a
                    const R u = a == 0 ? q : r, v = a == 2 ? q : w;
                    const int cu = a == 2 ? 5 : 4, cv = a == 0 ? 5 : 6;
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const R* c = &sG[x][8 * d];
                        T[h][d] = c[1 + a] + c[cu] * u + c[cv] * v + c[7] * (u * v);
                    }
                }
                cross3(T[0], T[1], C);
            }
            const R Nx = sg * C[0], Ny = sg * C[1], Nz = sg * C[2];
            R Ln, il;
            norm_and_inverse(Nx * Nx + Ny * Ny + Nz * Nz, Ln, il);
            fN[t][0] = Nx * il;
            fN[t][1] = Ny * il;
            fN[t][2] = Nz * il;
            fN[t][3] = Ln * wpq[t];
        }
    };
    auto flux_weights = [&](int x) {
#pragma unroll
        for (int t = 0; t < FPT; ++t) {
            const R* w = static_cast<const R*>(A.fw) + unsigned((el0 + x) * 24 + ff[t] * 4);
#pragma unroll
            for (int c = 0; c < 4; ++c) fw[t][c] = w[c];
        }
    };
    // The plus side's packets of epoch e, into pk; whether they carry the tag is
    // checked where they are used.
    unsigned long long pk[FPT][PC];
    auto read_plus = [&](int t, unsigned e) {
        const char* const xb = buffer_of(e);
        const unsigned o = unsigned(max(slot[t], 0));
#pragma unroll
        for (int c = 0; c < PC; ++c) pk[t][c] = packet_load(xb, o + 8 * c * N2);
    };
    auto read_all = [&](unsigned e) {
#pragma unroll
        for (int t = 0; t < FPT; ++t)
            if (tid + t * NT < NF) read_plus(t, e);
    };
    // What a poll that is not answered does: false once the wait is given up
    // (bounded, or another workgroup gave up), and the launch with it.
    int spin = 0;
    auto wait_on = [&]() -> bool {
        ++spin;
        if (spin <= A.spin_limit &&
            ((spin & 63) != 0 || __hip_atomic_load(A.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0))
            return true;
        int none = 0;
        if (__hip_atomic_compare_exchange_strong(A.stop, &none, A.seq, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            __hip_atomic_store(A.stop_host, A.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        sStop = 1;
        return false;
    };
    auto node_geo = [&](int x) {
        if constexpr (AFF) {
#pragma unroll
            for (int c = 0; c < 10; ++c) geo[c] = sG[x][c];
        } else {
            // pinned: recomputed per stage where several elements share the
            // workgroup (hoisted out of the stage loop, it would spill)
            int a = i, b = j, c = k;
            if constexpr (!KEEP) { pin(a); pin(b); pin(c); }
            node_geometry(&sG[x][0], sZ[a], sZ[b], sZ[c], geo);
        }
    };
    if constexpr (KEEP) {
        face_geometry(0);
        flux_weights(0);
        node_geo(0);
    }

    // QB: the lane's row of D (kept with one element per workgroup, else read per
    // element: the registers are wanted for the other elements' LSRK registers)
    float Dq[8];
    auto row_of_D = [&]() {
        int r = i * N1;
        if constexpr (!KEEP) pin(r);
#pragma unroll
        for (int q = 0; q < 8; ++q) Dq[q] = sD[r + q];
    };
    if constexpr (QB && KEEP) row_of_D();
    unsigned ep = A.epoch;
    for (int x = 0; x < cnt; ++x) publish(x, ep);
    for (int step = 0; step < A.nsteps; ++step) {
        for (int s = 0; s < 5; ++s, ++ep) {
            const bool last = step == A.nsteps - 1 && s == 4;
            const KR ca = KR(A.a[s]), cb = KR(A.b[s]), cdt = KR(A.dt);
#pragma unroll 1
            for (int x = 0; x < (KEEP ? 1 : cnt); ++x) {
                take_slots(x);
                // With several elements per workgroup a neighbour's traces were mostly
                // published an element or more ago: they are read before the volume
                // work, which hides their latency.  Else in the middle of it.
                if constexpr (!KEEP) {
                    node_geo(x);
                    __builtin_amdgcn_sched_barrier(0);  // its temporaries and the packets are not live at once
                    read_all(ep);
                    flux_weights(x);
                }
                // ---- volume: reference derivatives folded straight into J * curl ----
                R cE[3] = {R(0), R(0), R(0)}, cH[3] = {R(0), R(0), R(0)};
                // a[3] = derivatives of E (h = 0) or H along d: J d/dx_e of component c gets a * C_d,e;
                // curl u = (dy u_z - dz u_y, dz u_x - dx u_z, dx u_y - dy u_x)
                auto fold = [&](int d, int h, const R (&a)[3]) {
                    const R Cx = geo[3 * d], Cy = geo[3 * d + 1], Cz = geo[3 * d + 2];
                    R* cv = h == 0 ? cE : cH;
                    cv[1] += a[0] * Cz; cv[2] -= a[0] * Cy;
                    cv[0] -= a[1] * Cz; cv[2] += a[1] * Cx;
                    cv[0] += a[2] * Cy; cv[1] -= a[2] * Cx;
                };
                if constexpr (QB) {
                    // lane = (line, position): r lines (j, k), s lines (i, k) -- both in the
                    // wave's own plane -- and t lines (i, j = wave) across the planes
                    if constexpr (!KEEP) row_of_D();
                    const int lr = (i & 3) + RS * j + PL * k, ls = j + RS * (i & 3) + PL * k, lt = j + RS * k + PL * (i & 3);
                    auto lines = [&](int h, int lo, int hi, R (&a)[3]) {
                        const R l[3] = {sU[x][3 * h][lo], sU[x][3 * h + 1][lo], sU[x][3 * h + 2][lo]};
                        const R u[3] = {sU[x][3 * h][hi], sU[x][3 * h + 1][hi], sU[x][3 * h + 2][hi]};
                        line8x3(Dq, l, u, a);
                    };
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        R a[3];
                        lines(h, lr, lr + 4, a);
                        fold(0, h, a);
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        R a[3];
                        lines(h, ls, ls + 4 * RS, a);
#pragma unroll
                        for (int c = 0; c < 3; ++c)  // lane (position j, line i) -> the node's lane (i, j)
                            a[c] = __builtin_bit_cast(R, __builtin_amdgcn_ds_bpermute(4 * (j + 8 * i), __builtin_bit_cast(int, a[c])));
                        fold(1, h, a);
                    }
                    if constexpr (KEEP) read_all(ep);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        R a[3];
                        lines(h, lt, lt + 4 * PL, a);
#pragma unroll
                        for (int c = 0; c < 3; ++c) sT[3 * h + c][j + RS * k + PL * i] = a[c];
                    }
                    pin(cE[0]); pin(cE[1]); pin(cE[2]); pin(cH[0]); pin(cH[1]); pin(cH[2]);
                } else {
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    if (KEEP && d == 2) read_all(ep);
                    const int row = d == 0 ? i : (d == 1 ? j : k);
                    R Dr[N1];
#pragma unroll
                    for (int q = 0; q < N1; ++q) Dr[q] = sD[row * N1 + q];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        R a[3] = {R(0), R(0), R(0)};
#pragma unroll
                        for (int q = 0; q < N1; ++q) {
                            const int lq = d == 0 ? q + N1 * j + N2 * k : (d == 1 ? i + N1 * q + N2 * k : i + N1 * j + N2 * q);
#pragma unroll
                            for (int c = 0; c < 3; ++c) a[c] += Dr[q] * sU[x][3 * h + c][lq];
                        }
                        fold(d, h, a);
                    }
                    pin(cE[0]); pin(cE[1]); pin(cE[2]); pin(cH[0]); pin(cH[1]); pin(cH[2]);
                }
                }
                // ---- face terms ----
                if constexpr (!KEEP) face_geometry(x);
#pragma unroll
                for (int t = 0; t < FPT; ++t) {
                    const int fp = tid + t * NT;
                    if (fp < NF) {
                        R mine[6];
#pragma unroll
                        for (int c = 0; c < 6; ++c) mine[c] = sU[x][c][fnode[t]];
                        R jE[3], jH[3];
                        if (slot[t] < 0) {  // PEC mirror
#pragma unroll
                            for (int c = 0; c < 3; ++c) { jE[c] = R(-2) * mine[c]; jH[c] = R(0); }
                        } else {
                            spin = 0;
                            for (;;) {
                                unsigned other = 0;
#pragma unroll
                                for (int c = 0; c < PC; ++c) other |= static_cast<unsigned>(pk[t][c] >> 32) ^ ep;
                                if (other == 0 || !wait_on()) break;
                                read_plus(t, ep);
                            }
                            R plus[6];
#pragma unroll
                            for (int c = 0; c < 6; ++c) {
                                if constexpr (sizeof(R) == 4)
                                    plus[c] = __builtin_bit_cast(R, static_cast<unsigned>(pk[t][c]));
                                else
                                    plus[c] = __builtin_bit_cast(R, (pk[t][2 * c] & 0xffffffffull) | (pk[t][2 * c + 1] << 32));
                            }
#pragma unroll
                            for (int c = 0; c < 3; ++c) {
                                jE[c] = plus[c] - mine[c];
                                jH[c] = plus[c + 3] - mine[c + 3];
                            }
                        }
                        const R nx = fN[t][0], ny = fN[t][1], nz = fN[t][2], dA = fN[t][3];
                        const R nxEx = ny * jE[2] - nz * jE[1], nxEy = nz * jE[0] - nx * jE[2], nxEz = nx * jE[1] - ny * jE[0];
                        const R nxHx = ny * jH[2] - nz * jH[1], nxHy = nz * jH[0] - nx * jH[2], nxHz = nx * jH[1] - ny * jH[0];
                        const R nnEx = ny * nxEz - nz * nxEy, nnEy = nz * nxEx - nx * nxEz, nnEz = nx * nxEy - ny * nxEx;
                        const R nnHx = ny * nxHz - nz * nxHy, nnHy = nz * nxHx - nx * nxHz, nnHz = nx * nxHy - ny * nxHx;
                        const R wEh = fw[t][0], wEe = fw[t][1], wHe = fw[t][2], wHh = fw[t][3];
                        R* out = sF[fp];
                        out[0] = dA * (wEh * nxHx - wEe * nnEx);
                        out[1] = dA * (wEh * nxHy - wEe * nnEy);
                        out[2] = dA * (wEh * nxHz - wEe * nnEz);
                        out[3] = dA * (-wHe * nxEx - wHh * nnHx);
                        out[4] = dA * (-wHe * nxEy - wHh * nnHy);
                        out[5] = dA * (-wHe * nxEz - wHh * nnHz);
                    }
                }
                __syncthreads();
                if (sStop) return;  // uniform: written before the barrier, and next only after the one below
                if constexpr (QB) {  // the t-derivatives, complete since the barrier
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const R a[3] = {sT[3 * h][at], sT[3 * h + 1][at], sT[3 * h + 2][at]};
                        fold(2, h, a);
                    }
                }
                // ---- lift, inverse mass, LSRK update ----
                {
                    const int sj = j == 0 ? 0 * N2 + i + N1 * k : (j == N1 - 1 ? 2 * N2 + i + N1 * k : NF);
                    const int si = i == N1 - 1 ? 1 * N2 + j + N1 * k : (i == 0 ? 3 * N2 + j + N1 * k : NF);
                    const int sk = k == 0 ? 4 * N2 + i + N1 * j : (k == N1 - 1 ? 5 * N2 + i + N1 * j : NF);
                    R LE[3], LH[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        LE[c] = (sF[sj][c] + sF[si][c]) + sF[sk][c];
                        LH[c] = (sF[sj][c + 3] + sF[si][c + 3]) + sF[sk][c + 3];
                    }
                    take_k(x);
                    const R iJ = geo[9];
                    const R sE_ = sM[x][0] * iJ, sH_ = sM[x][1] * iJ;
#pragma unroll
                    for (int c = 0; c < 6; ++c) {
                        const R rhs = c < 3 ? sE_ * (cH[c] + LE[c] * Winv) : sH_ * (-cE[c - 3] + LH[c - 3] * Winv);
                        const KR kn = s == 0 ? cdt * KR(rhs) : ca * kc[c] + cdt * KR(rhs);
                        kc[c] = kn;
                        sU[x][c][at] = R(KR(sU[x][c][at]) + cb * kn);
                    }
                    keep_k(x);
                }
                __syncthreads();
                if (!last) publish(x, ep + 1);
            }
        }
        if (A.snap) {  // the probed elements' fields after this step
            for (int x = 0; x < cnt; ++x) {
                const int q = A.snap_slot[el0 + x];
                if (q < 0) continue;
                R* o = static_cast<R*>(A.snap) + (size_t(step) * A.nslots + q) * (6 * NP) + m;
#pragma unroll
                for (int c = 0; c < 6; ++c) o[c * NP] = sU[x][c][at];
            }
        }
    }
    for (int x = 0; x < cnt; ++x) {
        R* q = uout + (A.node_base + (long long)(el0 + x) * NP + m) * 6;
#pragma unroll
        for (int c = 0; c < 6; ++c) q[c] = sU[x][c][at];
    }
}

template <int N1, int EM, typename R, typename KR, bool AFF>
struct ResidentFamily {
    static constexpr int lds_k = resident_lds_k<N1, EM, sizeof(R), sizeof(KR), AFF>() * 6 * N1 * N1 * N1 * int(sizeof(KR));
    static hipError_t launch(const ResidentArgs& a, hipStream_t s) {
        const int grid = (a.nelt + a.per - 1) / a.per;
        hipLaunchKernelGGL((k_resident<N1, EM, R, KR, AFF>), dim3(grid), dim3(N1 * N1 * N1), lds_k, s, a);
        return hipGetLastError();
    }
    // Workgroups per CU that the hardware places wherever its waves start.  The
    // occupancy query divides the LDS by the bytes a workgroup asks for, but a workgroup
    // is given whole granules (n1 = 4, eight elements: 15536 bytes take 16640, nine
    // workgroups and not ten).  It counts wave slots, but a workgroup whose waves are no
    // multiple of the four SIMDs loads them unevenly (six waves: 2 2 1 1), and two such
    // may not fit where 12 slots are free.
    static int per_cu() {
        static std::atomic<int> known{-1};
        int n = known.load(std::memory_order_relaxed);
        if (n >= 0) return n;
        hipFuncAttributes fa;
        const void* fn = reinterpret_cast<const void*>(&k_resident<N1, EM, R, KR, AFF>);
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_resident<N1, EM, R, KR, AFF>, N1 * N1 * N1, lds_k) != hipSuccess ||
            hipFuncGetAttributes(&fa, fn) != hipSuccess)
            return 0;
        const int lds = (static_cast<int>(fa.sharedSizeBytes) + lds_k + kLdsGranule - 1) / kLdsGranule * kLdsGranule;
        n = std::min(n, 160 * 1024 / std::max(lds, kLdsGranule));
        constexpr int W = (N1 * N1 * N1 + 63) / 64;
        const int slots = 512 / ((std::max(fa.numRegs, 1) + 7) / 8 * 8);  // waves per SIMD
        if (W > 4 && W % 4 != 0) n = std::min(n, std::max(1, slots / ((W + 3) / 4)));
        if (W == 2 || W == 3) n = std::min(n, std::max(1, 4 * slots / W - 1));
        known.store(n, std::memory_order_relaxed);
        return n;
    }
};

template <int N1, int EM, typename R, typename KR>
ResidentKernel resident_pick(bool affine) {
    if constexpr (EM <= resident_range(N1, sizeof(R), sizeof(KR), true).em) {
        using A = ResidentFamily<N1, EM, R, KR, true>;
        if (affine) return {&A::launch, &A::per_cu};
    }
    if constexpr (EM <= resident_range(N1, sizeof(R), sizeof(KR), false).em) {
        using G = ResidentFamily<N1, EM, R, KR, false>;
        if (!affine) return {&G::launch, &G::per_cu};
    }
    return {};
}

template <int N1, typename R, typename KR>
ResidentKernel resident_pick_em(int em, bool affine) {
    switch (em) {
        case 0: return resident_pick<N1, 1, R, KR>(affine);
        case 1: return resident_pick<N1, 2, R, KR>(affine);
        case 2: return resident_pick<N1, 4, R, KR>(affine);
        case 3: return resident_pick<N1, 8, R, KR>(affine);
        default: return {};
    }
}

template <typename R, typename KR>
ResidentKernel resident_pick_n1(int n1, int em, bool affine) {
    switch (n1) {
        case 2: return resident_pick_em<2, R, KR>(em, affine);
        case 3: return resident_pick_em<3, R, KR>(em, affine);
        case 4: return resident_pick_em<4, R, KR>(em, affine);
        case 5: return resident_pick_em<5, R, KR>(em, affine);
        case 6: return resident_pick_em<6, R, KR>(em, affine);
        case 7: return resident_pick_em<7, R, KR>(em, affine);
        case 8: return resident_pick_em<8, R, KR>(em, affine);
        case 9: return resident_pick_em<9, R, KR>(em, affine);
        default: return {};
    }
}

}  // namespace
}  // namespace nw
