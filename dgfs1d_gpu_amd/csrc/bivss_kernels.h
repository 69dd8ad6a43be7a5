// Binary-mixture VSS fast-spectral collision operator, one species pair
// (p, q), batched over collision tasks.
//
// Reference behaviour (jaisw7/dgfs1D_gpu): DGFSBiVSSScatteringModel.fs
// (bi/scattering.py:261-321) with kernels bi/kernels/scattering/vss.mako:
// 96-285.  Per node the reference runs 10 launches and batched M*N_rho cuFFT
// transforms, nodes one after another.  Here every node of a pair shares one
// launch of each of five kernels:
//
//   A  fwd   : F = FFT3(f_p)/n, G = FFT3(f_q)/n per task (the forward kernels
//              of the single-species operator, collision_kernels.h)
//   B  gain  : per (task, radius x, direction y):
//                u1 = IFFT3(exp(+i m_q/(m_p+m_q) a_xy) F),
//                u2 = IFFT3(exp(-i m_p/(m_p+m_q) a_xy) G)  (Fft3Engine, complex),
//              and the forward transform along x of u1 u2 in registers
//   C  plane : per (task, k1-plane, xy group): partial sums
//              G^_g = sum_{xy in g} W_xy FFT2_{y,z}(acc_xy), summed in fixed
//              order by a second kernel, which also does the inverses:
//              W_xy = qw_x sw / n * b_pq[x,y] (complex, per direction: the VSS
//              kernel depends on the direction, so the sum over y cannot be
//              taken in physical space as the single-species gain does);
//              then IFFT2 of G^ and of c_pq G
//   D  line  : inverse along k1 and Q[out] += prefac (Re gain - f_p Re loss)
//              (k_line_output of the single-species operator)
//
// This engine needs a product's whole cube in a work-group's LDS and keeps
// both sides and the product complex.  Larger grids and larger task sets take
// the streaming form of B to D (bi_pipeline.h).
#pragma once
#include "bi_pipeline.h"

#include <algorithm>

namespace dgfs {

template <typename T, int N>
constexpr int bi_split() { return pick_split<T>(N); }

// Which grids take the streaming kernels of bi_pipeline.h: all whose product
// cube does not fit a work-group's LDS whole (FP64 N >= 24, FP32 N >= 32), and
// N = 20 and FP32 N = 24 once a plan's products fill the chip.  Below that the
// engine's fewer launches win, and at N <= 16 at every size that matters.
// Microseconds for the four pairs, engine against streaming, M = 12, N_rho = 6
// and 2, 8, 50 tasks: N = 16 FP32 160/205, 186/246, 503/526; N = 20 FP32
// 223/293, 329/394, 1175/1008; N = 20 FP64 288/318, 603/531, 2499/1810; N = 24
// FP32 253/283, 511/439, 2281/1438.
template <typename T, int N>
constexpr bool bi_engine() { return N <= 24 && bi_split<T, N>() == 1; }
constexpr bool bi_streams(int N) { return N >= 20; }
constexpr size_t kBiStreamBytes = size_t(48) << 20;    // of a plan's product cubes

// B: one work-group per (task, xy); acc[t][xy][k1][y][z].
template <typename T, int N>
__global__ void __launch_bounds__(round64(N * N))
k_bi_gain(const cplx<T>* __restrict__ Fhat, const cplx<T>* __restrict__ phase, int NXY,
          cplx<T>* __restrict__ acc_out) {
    using E = Fft3Engine<T, N, 1, round64(N * N), +1>;
    constexpr int n = N * N * N, NN = N * N;
    __shared__ cplx<T> V[E::LDS_ELEMS];
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int xy = lb % NXY, t = lb / NXY;
    typename E::Split sp;
    sp.init(0);
    const cplx<T>* ph = phase + size_t(xy) * 2 * 3 * N;     // [side][axis][l]
    auto map1 = [](int pp, int& i1, int& i2) { i1 = pp / N; i2 = pp - (pp / N) * N; };
    auto map3 = [](int P, int& o2, int& j) { o2 = P / N; j = P - (P / N) * N; };
    cplx<T> R1[N];
    sfor<0, 2>([&](auto Si) {
        constexpr int side = Si;
        const cplx<T>* F = Fhat + (size_t(t) * 2 + side) * n;     // [l3][l1][l2]
        const cplx<T>* e = ph + side * 3 * N;
        // the separable phase exp(i th_1 l1) exp(i th_2 l2) exp(i th_3 l3) is
        // applied per axis just before that axis' transform: l3 in the load,
        // l2 in pass 2 and l1 in pass 3
        E::run(V, sp, map1,
               [&](int i1, int i2, int i3) { return e[2 * N + i3] * F[(size_t(i3) * N + i1) * N + i2]; },
               [&](auto I, cplx<T> v) { return e[N + int(I)] * v; }, map3,
               [&](auto I, cplx<T> v) { return e[int(I)] * v; },
               [&](int o2, int j, const cplx<T>* o) {
                   if constexpr (side == 0) {
                       sfor<0, N>([&](auto I) { R1[I] = o[I]; });
                   } else {
                       cplx<T> pr[N];
                       sfor<0, N>([&](auto I) { pr[I] = R1[I] * o[I]; });
                       RegDFT<T, N, -1>::template run<1, 0>(pr, R1);
                       cplx<T>* dst = acc_out + (size_t(t) * NXY + xy) * n;
                       sfor<0, N>([&](auto I) {
                           dst[size_t(I) * NN + o2 * N + j] = R1[I];
                       });
                   }
               });
    });
}

// C1: one work-group per (t, k1, xy-group g): slot s of PL takes the group's
// xy = xy0 + s, xy0 + s + PL, ...; the group's partial
// G^_g(k1, :, :) = sum_xy W_xy FFT2_{y,z}(acc_xy(k1)) goes to
// Gp[t][g][k1][k2][k3].
template <typename T, int N>
__global__ void __launch_bounds__(planes_per_wg(N) * N)
k_bi_plane_part(const cplx<T>* __restrict__ acc_in, const cplx<T>* __restrict__ wtab, int NXY,
                int XG, cplx<T>* __restrict__ Gp) {
    constexpr int PL = planes_per_wg(N), NN = N * N, n = N * NN, PS = N * (N + 1);
    __shared__ cplx<T> L[PL * PS];
    const int g = blockIdx.x % XG;
    const int k1 = (blockIdx.x / XG) % N, t = blockIdx.x / (XG * N);
    const int slot = threadIdx.x / N, c = threadIdx.x - slot * N;
    cplx<T>* P = L + slot * PS;
    const int per = (NXY + XG - 1) / XG;
    const int xy0 = g * per < NXY ? g * per : NXY;
    const int xy1 = xy0 + per < NXY ? xy0 + per : NXY;
    cplx<T> G[N];
    sfor<0, N>([&](auto I) { G[I] = mk(T(0), T(0)); });
    const int nround = (xy1 - xy0 + PL - 1) / PL;
    for (int rd = 0; rd < nround; ++rd) {
        const int xy = xy0 + rd * PL + slot;
        const bool live = xy < xy1;
        __syncthreads();
        if (live) {
            const cplx<T>* src = acc_in + (size_t(t) * NXY + xy) * n + size_t(k1) * NN;
            for (int y = 0; y < N; ++y) P[y * (N + 1) + c] = src[y * N + c];
        }
        __syncthreads();
        if (live) lds_fft_row<T, N, -1>(P, c);     // z -> k3
        __syncthreads();
        if (live) {
            lds_fft_col<T, N, -1>(P, c);            // y -> k2 (column c = k3)
            const cplx<T>* w = wtab + size_t(xy) * n + size_t(k1) * NN + c;   // [k1][k2][k3]
            sfor<0, N>([&](auto K2) { G[K2] = G[K2] + w[size_t(K2) * N] * P[K2 * (N + 1) + c]; });
        }
    }
    __syncthreads();
    sfor<0, N>([&](auto K2) { P[K2 * (N + 1) + c] = G[K2]; });
    __syncthreads();
    if (slot == 0) {
        for (int o = 1; o < PL; ++o)
            sfor<0, N>([&](auto K2) { G[K2] = G[K2] + L[o * PS + K2 * (N + 1) + c]; });
        cplx<T>* dst = Gp + ((size_t(t) * XG + g) * N + k1) * NN + c;
        sfor<0, N>([&](auto K2) { dst[size_t(K2) * N] = G[K2]; });
    }
}

// C2: one work-group per plane (t, k1): G^ = sum_g Gp[t][g][k1] (fixed
// order), IFFT2 of G^ (slot 0) and of c_pq G_q (slot 1) ->
// H[t][0 = loss | 1 = gain][k1][y][z], as k_line_output reads it.
template <typename T, int N>
__global__ void __launch_bounds__(planes_per_wg(N) * N)
k_bi_plane_fin(const cplx<T>* __restrict__ Gp, int XG, const cplx<T>* __restrict__ Fhat,
               const cplx<T>* __restrict__ ctab, cplx<T>* __restrict__ H) {
    constexpr int PL = planes_per_wg(N), NT = PL * N, NN = N * N, n = N * NN, PS = N * (N + 1);
    static_assert(PL >= 2, "plane kernel needs two slots");
    __shared__ cplx<T> L[PL * PS];
    const int k1 = blockIdx.x % N, t = blockIdx.x / N;
    const int slot = threadIdx.x / N, c = threadIdx.x - slot * N;
    cplx<T>* P = L + slot * PS;
    if (slot == 0) {
        cplx<T> G[N];
        sfor<0, N>([&](auto K2) { G[K2] = mk(T(0), T(0)); });
        for (int g = 0; g < XG; ++g) {
            const cplx<T>* src = Gp + ((size_t(t) * XG + g) * N + k1) * NN + c;
            sfor<0, N>([&](auto K2) { G[K2] = G[K2] + src[size_t(K2) * N]; });
        }
        sfor<0, N>([&](auto K2) { P[K2 * (N + 1) + c] = G[K2]; });
    } else if (slot == 1) {
        // loss plane: c_pq * G_q at l1 = k1, column c = l3
        const cplx<T>* Fg = Fhat + (size_t(t) * 2 + 1) * n;
        sfor<0, N>([&](auto L2) {
            P[L2 * (N + 1) + c] = ctab[size_t(k1) * NN + L2 * N + c] *
                                  Fg[(size_t(c) * N + k1) * N + L2];
        });
    }
    __syncthreads();
    if (slot < 2) lds_fft_col<T, N, +1>(P, c);      // k2 -> y
    __syncthreads();
    if (slot < 2) lds_fft_row<T, N, +1>(P, c);      // k3 -> z
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * NN; i += NT) {
        const int which = i / NN, rr = i - which * NN;    // slot 0 = gain, slot 1 = loss
        H[((size_t(t) * 2 + (which == 0 ? 1 : 0)) * N + k1) * NN + rr] =
            L[which * PS + (rr / N) * (N + 1) + rr % N];
    }
}

// xy groups of the plane stage: enough work-groups to fill the chip, at
// least one slot round per group
template <int N>
inline int bi_xgroups(int nt, int NXY) {
    constexpr int PL = planes_per_wg(N);
    const int maxg = (NXY + PL - 1) / PL;
    int g = (2048 + nt * N - 1) / (nt * N);
    return g < 1 ? 1 : (g > maxg ? maxg : g);
}
template <int N>
constexpr int bi_xgroups_max(int NXY) { return (NXY + planes_per_wg(N) - 1) / planes_per_wg(N); }

// ================================================================ the plan
struct BiPlan {
    int N, M, Nrho, Mpre, dtype, ntask_max;
    int chunk;              // tasks whose products the scratch holds
    int like_chunk;         // the same for calls that share products (bi_launch)
    double prefac, mp, mq;
    size_t n;
    bool stream = false;    // the streaming kernels (bi_pipeline.h)
    bool antipodal = false; // the streaming form's products come in opposite pairs (2u, 2u + 1)
    // a species with itself: the products of an opposite pair are one
    bool shares() const { return antipodal && mp == mq; }
    size_t nspec = 0;       // planes of spec
    size_t ngrp = 0;        // partial G^ that Gp holds
    void* phase = nullptr;  // [Nrho*M][2][3][N] cplx<T>, in product order
    void* wtab = nullptr;   // [Nrho*M][k1][k2][k3] cplx<T>  qw sw / n * b_pq; streaming: k_bi_wtab
    void* wspec = nullptr;  // streaming: the weights at k1 = N/2 (k_bi_wtab)
    void* ctab = nullptr;   // [l1][l2][l3] cplx<T>  c_pq; streaming: k_bi_chtab
    void* Fhat = nullptr;   // [like_chunk][2][n] cplx<T>
    void* Iw = nullptr;     // [like_chunk][2][n] cplx<T>
    void* Y = nullptr;      // streaming: [chunk][Nrho*M][n] cplx<T>, before and after k_bi_plane
    void* nyq = nullptr;    // streaming: [chunk][Nrho*M][3][N*N] cplx<T>
    void* spec = nullptr;   // streaming: [chunk][Nrho*M][XS][NPH] cplx<T>
    void* acc = nullptr;    // [chunk][Nrho*M][n] cplx<T>
    void* H = nullptr;      // [ntask_max][2][n] cplx<T>: loss, gain
    void* norm = nullptr;   // streaming: [like_chunk][2][2][bi_norm_blocks] FP64
    void* Gp = nullptr;     // [chunk][groups][n] cplx<T>  partial G^; streaming: [ngrp][H][NPT][2]
};

// x-ranges of k_bi_plane and weight groups of k_bi_sum for nt tasks of ND
// products, NU weights: the split with the shortest longest CU.  A CU's share
// is its ceil(blocks / 256) work-groups, but no less than the eight waves that
// it needs to be busy, times the length of one; finer splits even the shares
// out and pay per piece (a range its k1 = N/2 plane, about half a plane's
// transforms; a group the write and the read of its partial sums, about two
// weights).  Against the first split of at least 2048 waves, same chunks: N = 20
// FP64 8.11 -> 7.83 ms, N = 48 FP32 41.9 -> 38.0, N = 32 FP64 29.7 both, the
// 6-task N = 24 set 536/538 us (at 4096 waves it took 591).
// A group also costs k_bi_pen a step of its serial sum (0.3 weights): one task
// of 96 directions, N = 24 FP64, 374 us without that term, 356 with it.  More
// than 12 ranges only where four work-groups per CU or fewer come of it, because
// k_bi_sum adds their k1 = N/2 planes up: N = 32 FP32, one task of 30 directions
// 270 -> 252 us, but of 216 directions 465 -> 504.
constexpr int kBiCU = 256;
inline double bi_share(long blocks, int wg, double length) {
    const long per = (blocks + kBiCU - 1) / kBiCU;
    return std::max(double(per), 512.0 / wg) * length;
}
template <typename T, int N>
inline int bi_xranges(int nt, int ND) {
    using Pl = BiPlane<T, N>;
    int XS = 1;
    double least = 0.0;
    for (int d = 1; d <= kBiXSMax; ++d) {
        const long blocks = (long(nt) * ND * d + Pl::PW - 1) / Pl::PW;
        if (N % d || (d > 12 && blocks > 4 * kBiCU)) continue;
        const double c = bi_share(blocks, Pl::WG, N / d + 0.5);
        if (d == 1 || c < least) XS = d, least = c;
    }
    return XS;
}
template <int N>
inline int bi_sum_groups(int nt, int NU) {
    constexpr int QB = (BiGeo<N>::NPT + kBiSumWG / 2 - 1) / (kBiSumWG / 2);
    constexpr int QF = (BiGeo<N>::NPH + 31) / 32;
    int XG = 1;
    double least = 0.0;
    for (int per = NU; per >= 1; --per) {
        const int g = (NU + per - 1) / per;
        if (g > 64) break;
        const double c = bi_share(long(nt) * QB * g, kBiSumWG, per + 2.0) +
                         bi_share(long(nt) * QF, kBiPenWG, 0.3 * g);
        if (per == NU || c < least) XG = g, least = c;
    }
    return XG;
}
// the most planes of spec and partial sums of Gp that a chunk takes, with or
// without the shared products of `like`
template <typename T, int N>
inline void bi_stream_sizes(BiPlan* pl) {
    const int NXY = pl->Nrho * pl->M, us = pl->antipodal ? 2 : 1;
    auto take = [&](int chunk, int ND) {
        for (int nt = 1; nt <= chunk; ++nt) {
            pl->nspec = std::max(pl->nspec, size_t(nt) * ND * bi_xranges<T, N>(nt, ND));
            pl->ngrp = std::max(pl->ngrp, size_t(nt) * bi_sum_groups<N>(nt, NXY / us));
        }
    };
    take(pl->chunk, NXY);
    take(pl->like_chunk, NXY / us);
}

// The streaming form for nt tasks: forward plane transforms of f, g in Iw ->
// the x-planes of loss and gain in Z.
template <typename T, int N>
int bi_stream_chunk(BiPlan* pl, int nt, bool like, cplx<T>* Z, hipStream_t st) {
    using Gm = BiGeo<N>;
    using Pl = BiPlane<T, N>;
    const int dstride = like ? 2 : 1;
    const int ND = pl->Nrho * pl->M / dstride;
    const int NU = pl->antipodal ? pl->Nrho * pl->M / 2 : ND;
    const cplx<T>* F = (const cplx<T>*)pl->Fhat;
    const cplx<T>* ph = (const cplx<T>*)pl->phase;
    double* norm = (double*)pl->norm;
    hipLaunchKernelGGL((k_bi_fwd_line<T, N>), dim3(nt * 2 * bi_norm_blocks(N)), dim3(256), 0, st,
                       (const cplx<T>*)pl->Iw, (cplx<T>*)pl->Fhat, norm);
    DGFS_HIP_CHECK(hipGetLastError());
    const int PB = (Gm::NN + kBiXWG / 2 - 1) / (kBiXWG / 2);
    // 8192 waves (at 2048: N = 20 8.30, N = 32 30.4, N = 48 43.8 against 8.11, 29.7,
    // 41.9 ms); a group reloads F and G, so it has two products or more
    const long xb = long(nt) * PB * (kBiXWG / 64);
    const int XGX = int(std::max(1L, std::min((8192 + xb - 1) / xb, long(ND + 1) / 2)));
    const int nxb = nt * PB * XGX;
    const long nny = long(nt) * ND * 3;
    constexpr int NPW = BiNyq<T, N>::PW;
    hipLaunchKernelGGL((k_bi_x<T, N>), dim3(nxb + (nny + NPW - 1) / NPW), dim3(kBiXWG), 0, st, F, ph,
                       norm, ND, dstride, PB, XGX, nxb, (cplx<T>*)pl->Y, nny, (cplx<T>*)pl->nyq);
    DGFS_HIP_CHECK(hipGetLastError());
    const int XS = bi_xranges<T, N>(nt, ND);
    const long ns = long(nt) * ND * XS;
    hipLaunchKernelGGL((k_bi_plane<T, N>), dim3((ns + Pl::PW - 1) / Pl::PW), dim3(Pl::WG), 0, st,
                       (cplx<T>*)pl->Y, (const cplx<T>*)pl->nyq, ns, XS, (cplx<T>*)pl->spec);
    DGFS_HIP_CHECK(hipGetLastError());
    const int QB = (Gm::NPT + kBiSumWG / 2 - 1) / (kBiSumWG / 2);
    const int XG = bi_sum_groups<N>(nt, NU);
    auto* sum = like ? k_bi_sum<T, N, kBiReal>
                     : (pl->antipodal ? k_bi_sum<T, N, kBiPair> : k_bi_sum<T, N, kBiComplex>);
    hipLaunchKernelGGL(sum, dim3(nt * QB * XG), dim3(kBiSumWG), 0, st, (const cplx<T>*)pl->Y,
                       (const cplx<T>*)pl->spec, (const cplx<T>*)pl->wtab,
                       (const cplx<T>*)pl->wspec, nt, ND, XS, NU, XG, QB, (cplx<T>*)pl->Gp);
    DGFS_HIP_CHECK(hipGetLastError());
    const int QF = (Gm::NPH + 31) / 32;
    hipLaunchKernelGGL((k_bi_pen<T, N>), dim3(nt * QF), dim3(kBiPenWG), 0, st, (const cplx<T>*)pl->Gp,
                       XG, QF, F, norm, (const cplx<T>*)pl->ctab, Z);
    DGFS_HIP_CHECK(hipGetLastError());
    return 0;
}

// like: up = uq and each output's tasks add up to a form symmetric in f and g
template <typename T, int N>
int bi_launch(BiPlan* pl, const void* up, const void* uq, void* Q, TaskView tv, int ntask,
              int ngroup, const int* gstart, const int* gslice, bool like, hipStream_t st) {
    constexpr long NN = long(N) * N;
    const int NXY = pl->Nrho * pl->M;
    const size_t n = pl->n;
    like = like && pl->shares();
    // even chunks: a short last one would leave the chip idle at each kernel's end
    const int most = like ? pl->like_chunk : pl->chunk;
    const int nchunk = (ntask + most - 1) / most;
    const int per = nchunk ? (ntask + nchunk - 1) / nchunk : 0;
    for (int c0 = 0; c0 < ntask; c0 += per) {
        const int nt = ntask - c0 < per ? ntask - c0 : per;
        TaskView tc = tv;
        tc.nterm = tv.nterm + 2 * size_t(c0);
        tc.slice = tv.slice + size_t(c0) * 2 * tv.K;
        tc.coef = static_cast<const T*>(tv.coef) + size_t(c0) * 2 * tv.K;
        const long npl = long(nt) * 2 * N;
        constexpr int FP = fwd_planes_per_wg(N);
        hipLaunchKernelGGL((k_fwd_plane<T, N, false>), dim3((npl + FP - 1) / FP), dim3(FP * N),
                           0, st, (const T*)up, (const T*)uq, tc, 2, npl, (cplx<T>*)pl->Iw);
        DGFS_HIP_CHECK(hipGetLastError());
        bool done = false;
        if constexpr (bi_streams(N)) if (pl->stream) {
            if (int rc = bi_stream_chunk<T, N>(pl, nt, like, (cplx<T>*)pl->H + size_t(c0) * 2 * n,
                                               st))
                return rc;
            done = true;
        }
        if constexpr (bi_engine<T, N>()) if (!done) {
            constexpr int PL = planes_per_wg(N);
            const int XG = bi_xgroups<N>(nt, NXY);
            const long nli = long(nt) * 2 * NN;
            hipLaunchKernelGGL((k_fwd_line<T, N>), dim3((nli + 255) / 256), dim3(256), 0, st, nli,
                               2, (const cplx<T>*)pl->Iw, (cplx<T>*)pl->Fhat, (cplx<T>*)nullptr);
            DGFS_HIP_CHECK(hipGetLastError());
            hipLaunchKernelGGL((k_bi_gain<T, N>), dim3(nt * NXY), dim3(round64(N * N)), 0, st,
                               (const cplx<T>*)pl->Fhat, (const cplx<T>*)pl->phase, NXY,
                               (cplx<T>*)pl->acc);
            DGFS_HIP_CHECK(hipGetLastError());
            hipLaunchKernelGGL((k_bi_plane_part<T, N>), dim3(nt * N * XG), dim3(PL * N), 0, st,
                               (const cplx<T>*)pl->acc, (const cplx<T>*)pl->wtab, NXY, XG,
                               (cplx<T>*)pl->Gp);
            DGFS_HIP_CHECK(hipGetLastError());
            hipLaunchKernelGGL((k_bi_plane_fin<T, N>), dim3(nt * N), dim3(PL * N), 0, st,
                               (const cplx<T>*)pl->Gp, XG, (const cplx<T>*)pl->Fhat,
                               (const cplx<T>*)pl->ctab, (cplx<T>*)pl->H + size_t(c0) * 2 * n);
            DGFS_HIP_CHECK(hipGetLastError());
        }
    }
    if constexpr (bi_streams(N)) if (pl->stream) {
        using Pl = BiPlane<T, N>;
        const long ns = long(ngroup) * N;
        hipLaunchKernelGGL((k_bi_out<T, N>), dim3((ns + Pl::PW - 1) / Pl::PW), dim3(Pl::WG), 0, st,
                           (const T*)up, tv, (const cplx<T>*)pl->H, ns, gstart, gslice,
                           T(pl->prefac), (T*)Q);
        DGFS_HIP_CHECK(hipGetLastError());
        return 0;
    }
    if constexpr (bi_engine<T, N>()) {
        const long nlo = long(ngroup) * NN;
        hipLaunchKernelGGL((k_line_output<T, N, false>),
                           dim3((nlo * line_lanes(N) + kLineWG - 1) / kLineWG), dim3(kLineWG), 0,
                           st, (const T*)up, (const T*)nullptr, (const double*)nullptr, tv,
                           (const cplx<T>*)pl->H, nlo, gstart, gslice, T(pl->prefac), (T*)Q);
        DGFS_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

// the streaming form's weight tables (FP64 device inputs, see k_bi_wtab)
template <typename T, int N>
int bi_stream_tables(BiPlan* pl, const int* ylist, const double* fac, const double* wx,
                     const double* szpre, const double* Bt, const double* wc, const double* Bsum,
                     double mqf) {
    if constexpr (bi_streams(N)) {
        using Gm = BiGeo<N>;
        hipLaunchKernelGGL((k_bi_chtab<T, N>), dim3((N * Gm::NPH + 31) / 32), dim3(256), 0, 0,
                           pl->Nrho, pl->Mpre, fac, wc, szpre, Bsum, (cplx<T>*)pl->ctab);
        const int us = pl->antipodal ? 2 : 1, NU = pl->Nrho * pl->M / us;
        const long per = long(N) * Gm::NPT + Gm::NPH;
        hipLaunchKernelGGL((k_bi_wtab<T, N>), dim3((NU * per + 255) / 256), dim3(256), 0, 0,
                           pl->M, NU, us, pl->Mpre, ylist, fac, wx, szpre, Bt, mqf,
                           (cplx<T>*)pl->wtab, (cplx<T>*)pl->wspec);
        return hipGetLastError() == hipSuccess ? 0 : 1;
    }
    return 1;
}

#define DGFS_BI_SIG(T, N)                                                                  \
    template int bi_launch<T, N>(BiPlan*, const void*, const void*, void*, TaskView, int, int, \
                                 const int*, const int*, bool, hipStream_t);               \
    template int bi_stream_tables<T, N>(BiPlan*, const int*, const double*, const double*, \
                                        const double*, const double*, const double*, \
                                        const double*, double);
#define DGFS_BI_EXTERN(T, N)                                                               \
    extern template int bi_launch<T, N>(BiPlan*, const void*, const void*, void*, TaskView, int, \
                                        int, const int*, const int*, bool, hipStream_t);   \
    extern template int bi_stream_tables<T, N>(BiPlan*, const int*, const double*, const double*, \
                                               const double*, const double*, const double*, \
                                               const double*, double);
#define DGFS_BI_INST(T, N) DGFS_BI_SIG(T, N)

DGFS_COLLIDE_SIZES(DGFS_BI_EXTERN, float)
DGFS_BI_EXTERN(float, 48)
DGFS_COLLIDE_SIZES(DGFS_BI_EXTERN, double)

}  // namespace dgfs
