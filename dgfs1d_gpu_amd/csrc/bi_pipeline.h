// Streaming form of the binary-mixture gain (bivss_kernels.h): the gain sum
//   G^(k) = sum_d W_d(k) FFT3(u1_d u2_d)(k),
//   u1_d = IFFT3(exp(+i m_q' a_d) F),  u2_d = IFFT3(exp(-i m_p' a_d) G)
// over the products d = (radius, direction), of which the result keeps the
// real part of IFFT3(G^), in three kernels that each transform along the axes
// they hold in registers:
//
//   k_bi_x      per (l2, l3) pencil: phases and the inverse along l1
//   k_bi_plane  per x-plane: inverses along l3, l2, the product, forwards
//               along y, z
//   k_bi_sum    per (k2, k3) pencil: forward along x, weight, sum over d
//
// Three identities halve the work against transforming both sides and the
// product as complex fields:
//
// * f, g are real, so u1, u2 are real except for the Nyquist set (some index
//   equal to N/2, which has no +N/2 partner), and one transform of
//   X1 + i X2 carries both: w = IFFT3(X1 + i X2) = u1 + i u2.  With
//   beta = Im u1, delta = Im u2 (from the Nyquist planes alone, BiNyq),
//   Re u1 = Re w + delta, Re u2 = Im w - beta.  The spectrum of
//   beta + i delta is K = kap1 F + i kap2 G, kap = (e - e~)/(2i), e the
//   phase and e~ the phase with the conjugate factor on every Nyquist axis.
// * Only the Hermitian part of G^ reaches the real result, so P = u1 u2 needs
//   the half k3 <= N/2: with R = (P^(k) + conj P^(-k))/2 = FFT(Re P),
//   J = (P^(k) - conj P^(-k))/2 = i FFT(Im P), and the Hermitian and
//   anti-Hermitian parts Ws, Wa of W (Wa vanishes off the Nyquist set),
//   G^_h = Ws R + Wa J.  J is kept on the Nyquist set only: the lines
//   k2 = N/2 and k3 = N/2 of every x-plane travel as extra pencils, and
//   k1 = N/2 is the plane transform of sum_x (-1)^x Im P.
// * For an antipodally symmetric direction rule (and pre-rule)
//   W_-s = conj W_s, so an opposite pair shares one weight; and with equal
//   masses P_-s(f, g) = P_s(g, f), so where an output's tasks add up to a form
//   symmetric in f and g (a species with itself) the pair shares its product:
//   one product per pair with the weight 2 Re W.
//
// Measured (FP64 N = 32, M = 12, N_rho = 8, 216 tasks per pair, four pairs; one
// call): 101.9 ms as complex transforms of both sides and the product, 29.9 ms
// here.  Shares: k_bi_plane 44 %, k_bi_x 26 % and k_bi_sum 23 % (near the HBM
// rate of the products they write and read), k_bi_pen 2 %.  N = 20: 12.9 -> 7.8
// ms; FP32 N = 48: 157 -> 38 ms.  k_bi_plane by counters, N = 32, 20, 48: vector
// units busy 52, 53, 62 %, LDS 36, 22, 22 % of the busy cycles, of its cycles
// 50, 16, 37 % bank conflicts of the exchanges; three waves per SIMD spill (N =
// 32: 28 -> 33 ms).
//
// Layouts: pencil p(l2, l3) = (l3 / 2) 2N + 2 l2 + (l3 & 1), the order in
// which k_bi_plane's lanes hold a plane; F[which][l1][p]; Y[d][x][p], whose
// planes k_bi_plane overwrites with its results: Y[d][x][q], q < NPT <= N^2,
// with q the regular pencils k3 <= N/2 (same formula), then the lines
// (k2 = N/2, k3 = 0..N/2) and (k2, k3 = N/2).  In place a product takes 0.57
// instead of 0.9 MB (FP64 N = 32), so a chunk of the scratch budget holds 1.6
// times the tasks.  spec[d][s][q]: the k1 = N/2 plane of x-range s.  Every
// length-N transform is shared by a lane pair (pair_dft_*), but for k_bi_plane's
// at N = 20: half the registers per lane.
#pragma once
#include "collision_kernels.h"

namespace dgfs {

template <int N>
struct BiGeo {
    static constexpr int H = N / 2, NN = N * N, n = N * NN;
    static constexpr int MH = H / 2 + 1;            // k3 slots of a lane that hold k3 <= N/2
    static constexpr int NPH = MH * 2 * N;          // regular half pencils
    static constexpr int NE = H + 1 + N;            // line pencils
    static constexpr int NPT = NPH + NE;
    static_assert(N % 2 == 0 && N >= 4, "even grids");
    static_assert(N < 20 || NPT <= NN, "a plane's results fit its place in Y");
    static DGFS_HD int pen(int l2, int l3) { return (l3 / 2) * 2 * N + 2 * l2 + (l3 & 1); }
};
constexpr int kBiXSMax = 16;                        // most x-ranges of a product

// F[t][which][k1][p] = FFT_x(Iw)/n, one thread per (t, which, p), and
// norm[t][which][0][blk] = the work-group's sum of |F|^2, 0 only where F is zero.
// FP64 sums whose squares could leave the range (FP32's fit an FP64 sum) are
// taken again, scaled by the largest component: -s there and e in
// norm[t][which][1][blk] stand for s 4^e.
constexpr int bi_norm_blocks(int N) { return (N * N + 255) / 256; }
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_bi_fwd_line(const cplx<T>* __restrict__ Iw, cplx<T>* __restrict__ F, double* __restrict__ norm) {
    constexpr int NN = N * N, NB = bi_norm_blocks(N);
    __shared__ double sh[4];
    const int blk = blockIdx.x % NB, tw = blockIdx.x / NB;
    const int p = blk * 256 + int(threadIdx.x);
    const bool live = p < NN;
    cplx<T>* dst = F + tw * size_t(N) * NN + p;
    double s = 0.0;
    if (live) {
        const int l3 = 2 * (p / (2 * N)) + (p & 1), l2 = (p % (2 * N)) >> 1;
        const cplx<T>* src = Iw + tw * size_t(N) * NN + l3 * N + l2;
        cplx<T> a[N], o[N];
        sfor<0, N>([&](auto X) { a[X] = src[size_t(X) * NN]; });
        RegDFT<T, N, -1>::template run<1, 0>(a, o);
        const T inv_n = T(1) / T(N * NN);
        sfor<0, N>([&](auto K1) {
            const cplx<T> v = inv_n * o[K1];
            dst[size_t(K1) * NN] = v;
            s += double(v.x) * double(v.x) + double(v.y) * double(v.y);
        });
    }
    auto total = [&](double v) {
        for (int o = 32; o; o >>= 1) v += __shfl_down(v, o);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
        __syncthreads();
        return (sh[0] + sh[1]) + (sh[2] + sh[3]);
    };
    s = total(s);
    double* out = norm + size_t(tw) * 2 * NB + blk;
    if constexpr (sizeof(T) == 8) if (!(s > 1e-200 && s < 1e200)) {
        double m = 0.0;
        if (live)
            for (int k = 0; k < N; ++k) {
                const cplx<T> v = dst[size_t(k) * NN];
                m = fmax(m, fmax(fabs(v.x), fabs(v.y)));
            }
        for (int o = 32; o; o >>= 1) m = fmax(m, __shfl_xor(m, o));
        __syncthreads();
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
        __syncthreads();
        m = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
        const int e = m > 0.0 && !isinf(m) ? max(ilogb(m), -1000) : 0;   // 2^-e is finite
        const double r = ldexp(1.0, -e);
        s = 0.0;
        if (live)
            for (int k = 0; k < N; ++k) {
                const cplx<T> v = r * dst[size_t(k) * NN];
                s += v.x * v.x + v.y * v.y;
            }
        __syncthreads();
        s = -total(s);
        if (threadIdx.x == 0) out[NB] = double(e);
    }
    if (threadIdx.x == 0) *out = s;
}

// The two sides of task t share one complex transform, whose rounding is
// relative to the larger of them: F enters as 2^f F and G as 2^g G (the factors
// go with the phases), of sizes near 1 and at most a factor of 2 apart, and the
// gain is multiplied by 2^-(f + g).  All three are exact, so each side keeps the
// range and the relative precision of a transform of its own.  zero: a side is
// exactly zero (and the other finite), and so is the gain, which the shared
// transform would leave at the other side's rounding (eps |g|^2).  Sides that
// are not finite enter as they are.
struct BiScale {
    int f, g;
    bool zero;
};
template <typename T, int N>
DGFS_DEV BiScale bi_scale(const double* norm, int t) {
    constexpr int NB = bi_norm_blocks(N);
    const double* p = norm + size_t(t) * 4 * NB;
    double s[2];
    int e[2];
    for (int w = 0; w < 2; ++w, p += 2 * NB) {
        s[w] = 0.0;
        e[w] = 0;
        bool scaled = false;
        for (int i = 0; i < NB; ++i) {
            s[w] += p[i];
            if constexpr (sizeof(T) == 8) scaled = scaled || p[i] < 0.0;
        }
        if (scaled) {
            s[w] = 0.0;
            e[w] = -1000;                             // the largest of the blocks that are not zero
            for (int i = 0; i < NB; ++i)
                if (p[i] != 0.0) e[w] = max(e[w], p[i] < 0.0 ? int(p[NB + i]) : 0);
            for (int i = 0; i < NB; ++i)
                s[w] += ldexp(fabs(p[i]), 2 * ((p[i] < 0.0 ? int(p[NB + i]) : 0) - e[w]));
        }
    }
    BiScale c{0, 0, false};
    if (!(s[0] < 1e300 && s[1] < 1e300)) return c;
    c.zero = s[0] == 0.0 || s[1] == 0.0;
    // log2 |F|^2, |G|^2, rounded down
    const int lf = s[0] > 0.0 ? ilogb(s[0]) + 2 * e[0] : 0;
    const int lg = s[1] > 0.0 ? ilogb(s[1]) + 2 * e[1] : 0;
    constexpr int most = sizeof(T) == 8 ? 1000 : 120;      // times a phase: still normal
    auto clamp = [](int x) { return x > most ? most : (x < -most ? -most : x); };
    c.f = clamp(-(lf / 2));
    c.g = clamp((lf - lg) / 2 - lf / 2);
    return c;
}

constexpr int kBiXWG = 128, kBiXD = 8;             // threads; products staged at a time

// The Nyquist planes of beta + i delta, one plane per slot (t, d, s) of 2N
// threads:
//   (-1)^x A(y, z) + (-1)^y B(x, z) + (-1)^z C(x, y)
// s = A: l1 = N/2; B: l2 = N/2, l1 != N/2; C: l3 = N/2, l1, l2 != N/2.
// nyq[t][d][3][NN]: A as p(z, .) orders it with y = (N/2) h + k at
// k 2N + 2z + h, B as [x][z], C as [x][y].
template <typename T, int N>
struct BiNyq {
    static constexpr int PW = kBiXWG / (2 * N) ? kBiXWG / (2 * N) : 1;   // slots per work-group
    static constexpr int LDS = PW * N * (N + 1);
    static DGFS_DEV void run(cplx<T>* L, int blk, long nslot, const cplx<T>* F, const cplx<T>* phase,
                             const double* norm, int ND, int dstride, cplx<T>* nyq) {
        using Gm = BiGeo<N>;
        constexpr int H = Gm::H, NN = Gm::NN, n = Gm::n;
        const int sl = threadIdx.x / (2 * N), u = threadIdx.x - sl * 2 * N, r = u >> 1, h = u & 1;
        const long slot = long(blk) * PW + sl;
        const bool live = sl < PW && slot < nslot;
        const int s = live ? int(slot % 3) : 0;
        const long td = live ? slot / 3 : 0;
        const long t = td / ND;
        const int d = int(td - t * ND);
        const cplx<T>* Ff = F + size_t(t) * 2 * n;
        const cplx<T>* Fg = Ff + n;
        const cplx<T>* e1 = phase + size_t(d) * dstride * 6 * N;  // [side][axis][l]
        const cplx<T>* e2 = e1 + 3 * N;
        // the (row, column) axes of the plane; s is its fixed axis
        const int ra = s == 0 ? 1 : 0, ca = s == 2 ? 1 : 2;
        auto kap = [&](const cplx<T>* e, int a, int b, T hs) {   // 2 hs kap
            const cplx<T> E = e[s * N + H], ea = e[ra * N + a], eb = e[ca * N + b];
            const cplx<T> p = ea * eb;
            const cplx<T> pt = (a == H ? conj(ea) : ea) * (b == H ? conj(eb) : eb);
            const cplx<T> v = E * p - conj(E) * pt;
            return mk(hs * v.y, -hs * v.x);                       // 2 hs v / (2i)
        };
        cplx<T>* P = L + sl * N * (N + 1);
        cplx<T> x[H], o[H];
        if (live) {
            const BiScale sc = bi_scale<T, N>(norm, int(t));
            const T hf = T(ldexp(0.5, sc.f)), hg = T(ldexp(0.5, sc.g));
            sfor<0, H>([&](auto K) {
                const int c = 2 * int(K) + h;                     // column index of this load
                const int l1 = s == 0 ? H : r, l2 = s == 0 ? r : (s == 1 ? H : c);
                const int l3 = s == 2 ? H : c;
                const bool zero = (s == 1 && r == H) || (s == 2 && (r == H || c == H));
                const size_t at = size_t(l1) * NN + Gm::pen(l2, l3);
                const cplx<T> a = kap(e1, r, c, hf) * Ff[at], b = kap(e2, r, c, hg) * Fg[at];
                x[K] = zero ? mk(T(0), T(0)) : mk(a.x - b.y, a.y + b.x);
            });
            pair_dft_dit<T, N, +1>(x, o, h);
            sfor<0, H>([&](auto K) { P[r * (N + 1) + H * h + K] = o[K]; });
        }
        __syncthreads();
        if (live) {
            sfor<0, H>([&](auto K) { x[K] = P[(2 * int(K) + h) * (N + 1) + r]; });
            pair_dft_dit<T, N, +1>(x, o, h);
            cplx<T>* dst = nyq + size_t(td) * 3 * NN + size_t(s) * NN;
            sfor<0, H>([&](auto K) {
                const int a = H * h + int(K);                     // y (A) or x (B, C), column r
                dst[s == 0 ? int(K) * 2 * N + 2 * r + h : a * N + r] = o[K];
            });
        }
    }
};

// Work-groups below nxb: Y[t][d][x][p] = sum_l1 e^{2 pi i l1 x / N}
// (2^f e1 F + i 2^g e2 G)(l1, p), a lane pair per pencil holds its F and G in
// registers over a group of products.  The others: the Nyquist planes.
template <typename T, int N>
__global__ void __launch_bounds__(kBiXWG, 2)
k_bi_x(const cplx<T>* __restrict__ F, const cplx<T>* __restrict__ phase,
       const double* __restrict__ norm, int ND, int dstride, int PB, int XG, int nxb,
       cplx<T>* __restrict__ Y, long nslot, cplx<T>* __restrict__ nyq) {
    using Gm = BiGeo<N>;
    using Ny = BiNyq<T, N>;
    constexpr int H = Gm::H, NN = Gm::NN, n = Gm::n, EX = kBiXD * 2 * N;
    __shared__ cplx<T> sh[EX > Ny::LDS ? EX : Ny::LDS];
    __shared__ T scl[2];                              // 2^f, 2^g
    if (int(blockIdx.x) >= nxb) {
        Ny::run(sh, int(blockIdx.x) - nxb, nslot, F, phase, norm, ND, dstride,
                nyq);
        return;
    }
    cplx<T>(*ex)[2][N] = reinterpret_cast<cplx<T>(*)[2][N]>(sh);
    const int lb = xcd_remap(blockIdx.x, nxb);
    const int pb = lb % PB, g = (lb / PB) % XG, t = lb / (PB * XG);
    const int per = (ND + XG - 1) / XG;
    const int d0 = g * per, d1 = d0 + per < ND ? d0 + per : ND;
    const int h = threadIdx.x & 1;
    int p = pb * (kBiXWG / 2) + int(threadIdx.x >> 1);
    const bool live = p < NN;
    p = live ? p : 0;
    const int l3 = 2 * (p / (2 * N)) + (p & 1), l2 = (p % (2 * N)) >> 1;
    cplx<T> f[H], gg[H];
    const cplx<T>* Ff = F + size_t(t) * 2 * n + size_t(h) * NN + p;
    sfor<0, H>([&](auto K) { f[K] = Ff[size_t(2 * int(K)) * NN]; });
    sfor<0, H>([&](auto K) { gg[K] = Ff[n + size_t(2 * int(K)) * NN]; });
    if (threadIdx.x == 0) {                           // in LDS: registers are short here
        const BiScale sc = bi_scale<T, N>(norm, t);
        scl[0] = T(ldexp(1.0, sc.f));
        scl[1] = T(ldexp(1.0, sc.g));
    }
    for (int db = d0; db < d1; db += kBiXD) {
        const int nd = d1 - db < kBiXD ? d1 - db : kBiXD;
        __syncthreads();
        for (int i = threadIdx.x; i < nd * 2 * N; i += kBiXWG) {
            const int dd = i / (2 * N), k = i - dd * 2 * N, sd = k / N;
            ex[dd][sd][k - sd * N] = scl[sd] *
                phase[(size_t(db + dd) * dstride * 2 + sd) * 3 * N + k - sd * N];
        }
        __syncthreads();
        for (int dd = 0; dd < nd; ++dd) {
            const int d = db + dd;
            const cplx<T>* e = phase + size_t(d) * dstride * 6 * N;
            const cplx<T> s1 = e[N + l2] * e[2 * N + l3];
            const cplx<T> s2 = mul_i<1>(e[4 * N + l2] * e[5 * N + l3]);
            cplx<T> a[H], o[H];
            sfor<0, H>([&](auto K) {
                const int l1 = 2 * int(K) + h;
                a[K] = (s1 * ex[dd][0][l1]) * f[K] + (s2 * ex[dd][1][l1]) * gg[K];
            });
            pair_dft_dit<T, N, +1>(a, o, h);
            if (live) {
                cplx<T>* dst = Y + ((size_t(t) * ND + d) * N + H * h) * NN + p;
                sfor<0, H>([&](auto K) { dst[size_t(int(K)) * NN] = o[K]; });
            }
        }
    }
}

// How k_bi_plane and k_bi_out share planes among threads: LN lanes per row.
//   LN = 1: a lane holds a row; 64 / N planes per one-wave work-group (the
//           lanes beyond repeat the first plane's rows in step with them);
//   LN = 2: a lane pair holds a row (pair_dft_*), the fewest planes that fill
//           whole waves.
// A lane (r, h) of an inverse (forward) transform holds the inputs in(k)
// (out(k)) and receives the outputs out(k) (in(k)), k < PN.
constexpr int bi_lanes(int N) { return N <= 20 ? 1 : 2; }
template <typename T, int N>
struct BiPlane {
    static constexpr int LN = bi_lanes(N), PN = N / LN, H = N / 2, PT = LN * N;
    static constexpr int PW = LN == 1 ? 64 / N
                                      : (PT % 64 == 0 ? 1 : PT % 32 == 0 ? 2 : 4);
    static constexpr int WG = LN == 1 ? 64 : PW * PT;
    static_assert(WG % 64 == 0 && PW >= 1, "whole waves");
    static constexpr int PI = N + 1, ELEMS = N * PI;
    static constexpr int MH = LN == 1 ? H + 1 : H / 2 + 1;    // in(k), k < MH, covers 0 .. N/2
    static DGFS_DEV constexpr int in(int k, int h) { return LN == 1 ? k : 2 * k + h; }
    static DGFS_DEV constexpr int out(int k, int h) { return LN == 1 ? k : H * h + k; }
    static DGFS_DEV void inverse(const cplx<T>* a, cplx<T>* o, int h) {
        if constexpr (LN == 1)
            RegDFT<T, N, +1>::template run<1, 0>(a, o);
        else
            pair_dft_dit<T, N, +1>(a, o, h);
    }
    static DGFS_DEV void forward(const cplx<T>* a, cplx<T>* o, int h) {
        if constexpr (LN == 1)
            RegDFT<T, N, -1>::template run<1, 0>(a, o);
        else
            pair_dft_dif<T, N, -1>(a, o, h);
    }
    // hand CW values in the lanes' order w(k) over to r(k); no barrier follows
    // the reads
    template <int CW, int CR, class W, class R>
    static DGFS_DEV void exchange(cplx<T>* P, const cplx<T>* o, cplx<T>* a, W&& w, R&& r) {
        sfor<0, CW>([&](auto K) { P[w(K)] = o[K]; });
        __syncthreads();
        sfor<0, CR>([&](auto K) { a[K] = P[r(K)]; });
    }
};

// Slot (t, d, s) takes x-range s of product d: per plane the inverses along
// l3 and l2, the product, the forward transforms along y and z and the split
// into R and the Nyquist lines of J, over the plane it read: no other live slot
// reads that plane, and the slot's lanes have theirs before the first barrier.
template <typename T, int N>
__global__ void __launch_bounds__((BiPlane<T, N>::WG), 2)
k_bi_plane(cplx<T>* Y, const cplx<T>* __restrict__ nyq, long nslot, int XS,
           cplx<T>* __restrict__ spec) {
    using Gm = BiGeo<N>;
    using Pl = BiPlane<T, N>;
    constexpr int H = Gm::H, NN = Gm::NN, NPH = Gm::NPH;
    constexpr int PI = Pl::PI, PN = Pl::PN, PW = Pl::PW, MH = Pl::MH;
    __shared__ cplx<T> L[PW * Pl::ELEMS];
    __shared__ cplx<T> Cs[PW * N];                    // row x of C
    int sl = threadIdx.x / Pl::PT;
    sl = sl < PW ? sl : 0;
    const int u = (threadIdx.x - sl * Pl::PT) % Pl::PT, r = u / Pl::LN, h = u % Pl::LN;
    const long sid = long(blockIdx.x) * PW + sl;
    const bool live = sid < nslot;                    // the others repeat the last slot, unstored
    const long slot = live ? sid : nslot - 1;
    const long td = slot / XS;
    const int s = int(slot - td * XS);
    cplx<T>* P = L + sl * Pl::ELEMS;
    cplx<T>* Cr = Cs + sl * N;
    cplx<T>* Yp = Y + td * size_t(N) * NN;
    const cplx<T>* A = nyq + td * size_t(3) * NN;
    const cplx<T>* B = A + NN;
    const cplx<T>* C = B + NN;
    const int nx = N / XS, x0 = s * nx;
    const int rm = r ? N - r : 0;                     // row of -k2
    const T sz = (r & 1) ? T(-1) : T(1);              // (-1)^z of this column
    auto row_in = [&](int k) { return r * PI + Pl::in(k, h); };
    auto row_out = [&](int k) { return r * PI + Pl::out(k, h); };
    auto col_in = [&](int k) { return Pl::in(k, h) * PI + r; };
    auto row_mirror = [&](int m) {                    // (-k2, -k3) of (r, in(m))
        const int c = Pl::in(m, h);
        return rm * PI + (c ? N - c : 0);
    };
    T lc[PN];                                         // sum_x (-1)^x Im P(x, y, z = r)
    sfor<0, PN>([&](auto K) { lc[K] = T(0); });
    for (int x = x0; x < x0 + nx; ++x) {
        cplx<T> a[PN], o[PN];
        sfor<0, PN>([&](auto K) { a[K] = Yp[size_t(x) * NN + Gm::pen(r, Pl::in(K, h))]; });
        const cplx<T> b = B[x * N + r], c = C[x * N + r];
        Pl::inverse(a, o, h);                         // row l2 = r -> z
        if (h == 0) Cr[r] = c;
        Pl::template exchange<PN, PN>(P, o, a, row_out, col_in);
        Pl::inverse(a, o, h);                         // column z = r -> y
        const T sx = (x & 1) ? T(-1) : T(1);
        sfor<0, PN>([&](auto K) {
            // A is read here, eight values at a time, not kept over the loop
            if constexpr (int(K) % 8 == 0) asm volatile("" ::: "memory");
            const int y = Pl::out(K, h);
            const T sy = (y & 1) ? T(-1) : T(1);
            const cplx<T> va = A[(y % H) * 2 * N + 2 * r + y / H], vc = Cr[y];
            const T be = sx * va.x + sy * b.x + sz * vc.x;
            const T de = sx * va.y + sy * b.y + sz * vc.y;
            const T r1 = o[K].x + de, r2 = o[K].y - be;
            a[K] = mk(r1 * r2 - be * de, r1 * de + be * r2);
            lc[K] += sx * a[K].y;
        });
        Pl::forward(a, o, h);                         // column z = r -> k2
        // these lanes read the column they now write
        Pl::template exchange<PN, PN>(P, o, a, col_in, row_out);
        Pl::forward(a, o, h);                         // row k2 = r -> k3
        Pl::template exchange<PN, MH>(P, o, a, row_in, row_mirror);
        if (live) {
            cplx<T>* dst = Yp + size_t(x) * NN;
            sfor<0, MH>([&](auto M) {
                const int k3 = Pl::in(M, h);
                const cplx<T> c = conj(a[M]);
                dst[Gm::pen(r, k3)] = mk(T(0.5) * (o[M].x + c.x), T(0.5) * (o[M].y + c.y));
                const cplx<T> J = mk(T(0.5) * (o[M].x - c.x), T(0.5) * (o[M].y - c.y));
                if (r == H && k3 <= H) dst[NPH + k3] = J;
                if (k3 == H) dst[NPH + H + 1 + r] = J;
            });
        }
        __syncthreads();
    }
    // the k1 = N/2 plane: J = i FFT2(lc)
    cplx<T> a[PN], o[PN];
    sfor<0, PN>([&](auto K) { a[K] = mk(lc[K], T(0)); });
    Pl::forward(a, o, h);
    Pl::template exchange<PN, PN>(P, o, a, col_in, row_out);
    Pl::forward(a, o, h);
    if (live) {
        cplx<T>* dst = spec + size_t(slot) * NPH;
        sfor<0, MH>([&](auto M) { dst[Gm::pen(r, Pl::in(M, h))] = mul_i<1>(o[M]); });
    }
}

enum BiWeight { kBiComplex = 0, kBiPair = 1, kBiReal = 2 };

// Gp[t][g][m][q][h] = sum over the weights u of group g of
//   kBiComplex: W_u P_u,  kBiPair: W_u P_2u + conj(W_u) P_(2u+1),
//   kBiReal: 2 Re(W_u) P_u,
// P_d the forward transform along x of pencil q (k1 = 2 m + h).
constexpr int kBiSumWG = 64;
template <typename T, int N, int MODE>
__global__ void __launch_bounds__(kBiSumWG, 2)
k_bi_sum(const cplx<T>* __restrict__ Y, const cplx<T>* __restrict__ spec,
         const cplx<T>* __restrict__ wtab, const cplx<T>* __restrict__ wspec, int nt, int ND, int XS, int NU, int XG, int QB,
         cplx<T>* __restrict__ Gp) {
    using Gm = BiGeo<N>;
    constexpr int H = Gm::H, NN = Gm::NN, NPT = Gm::NPT, NPH = Gm::NPH;
    constexpr int NP = MODE == kBiPair ? 2 : 1;
    // consecutive work-groups (one XCD) take the tasks of one weight block
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int t = lb % nt, qb = (lb / nt) % QB, g = lb / (nt * QB);
    const int h = threadIdx.x & 1;
    int q = qb * (kBiSumWG / 2) + int(threadIdx.x >> 1);
    const bool live = q < NPT;
    q = live ? q : NPT - 1;
    const int per = (NU + XG - 1) / XG;
    const int u0 = g * per, u1 = u0 + per < NU ? u0 + per : NU;
    cplx<T> G[H];
    sfor<0, H>([&](auto M) { G[M] = mk(T(0), T(0)); });
    for (int u = u0; u < u1; ++u) {
        const cplx<T>* w = wtab + (size_t(u) * H * NPT + q) * 2 + h;
#pragma unroll 1
        for (int sgn = 0; sgn < NP; ++sgn) {              // one product's pencil at a time
            const T cj = sgn ? T(-1) : T(1);              // the second one's weight is conj(W_u)
            const size_t td = size_t(t) * ND + NP * u + sgn;
            const cplx<T>* src = Y + td * N * NN + q;
            cplx<T> a[H], o[H];
            sfor<0, H>([&](auto K) { a[K] = src[size_t(H * h + int(K)) * NN]; });
            pair_dft_dif<T, N, -1>(a, o, h);
            sfor<0, H>([&](auto M) {
                const cplx<T> v = w[size_t(int(M)) * NPT * 2];
                if constexpr (MODE == kBiReal)
                    G[M] = G[M] + (v.x + v.x) * o[M];
                else
                    G[M] = G[M] + mk(v.x, cj * v.y) * o[M];
            });
            if (q < NPH && h == (H & 1)) {
                cplx<T> sp = mk(T(0), T(0));
                for (int s = 0; s < XS; ++s) sp = sp + spec[(td * XS + s) * NPH + q];
                cplx<T> v = wspec[size_t(u) * NPH + q];
                if constexpr (MODE == kBiReal) v = mk(v.x + v.x, T(0));
                G[H / 2] = G[H / 2] + mk(v.x, cj * v.y) * sp;     // k1 = N/2
            }
        }
    }
    if (live) {
        cplx<T>* dst = Gp + ((size_t(t) * XG + g) * H * NPT + q) * 2 + h;
        sfor<0, H>([&](auto M) { dst[size_t(int(M)) * NPT * 2] = G[M]; });
    }
}

// Z[t][0 = loss | 1 = gain][x][p] = IFFT along k1 of (c_pq G)_h and G^_h, a
// lane pair per regular pencil of a task; k3 > N/2 are the conjugates at
// (-k2, -k3).  The groups' sums (line pencils added to their regular ones) are
// dealt out to the four waves and added in wave order by wave 0, which inverts
// the gain; wave 1 inverts the loss meanwhile.  (One transform of gain + i loss
// would round the gain relative to the loss field, an order larger.)
constexpr int kBiPenWG = 256;
template <typename T, int N>
__global__ void __launch_bounds__(kBiPenWG)
k_bi_pen(const cplx<T>* __restrict__ Gp, int XG, int QB, const cplx<T>* __restrict__ F,
         const double* __restrict__ norm, const cplx<T>* __restrict__ ctab,
         cplx<T>* __restrict__ Z) {
    using Gm = BiGeo<N>;
    constexpr int H = Gm::H, NN = Gm::NN, n = Gm::n, NPT = Gm::NPT, NPH = Gm::NPH;
    constexpr int NW = kBiPenWG / 64;
    __shared__ cplx<T> sh[(NW - 1) * H * 64];
    const int qb = blockIdx.x % QB, t = blockIdx.x / QB;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane & 1;
    int q = qb * 32 + (lane >> 1);
    bool live = q < NPH;
    q = live ? q : 0;
    const int k3 = 2 * (q / (2 * N)) + (q & 1), k2 = (q % (2 * N)) >> 1;
    live = live && k3 <= H;
    const int ql = k2 == H ? NPH + k3 : (k3 == H ? NPH + H + 1 + k2 : -1);
    cplx<T> g[H], o[H];
    sfor<0, H>([&](auto M) { g[M] = mk(T(0), T(0)); });
    for (int x = wave; x < XG; x += NW) {
        const cplx<T>* src = Gp + (size_t(t) * XG + x) * H * NPT * 2 + h;
        sfor<0, H>([&](auto M) { g[M] = g[M] + src[(size_t(int(M)) * NPT + q) * 2]; });
        if (live && ql >= 0)
            sfor<0, H>([&](auto M) { g[M] = g[M] + src[(size_t(int(M)) * NPT + ql) * 2]; });
    }
    if (wave) sfor<0, H>([&](auto M) { sh[((wave - 1) * H + int(M)) * 64 + lane] = g[M]; });
    __syncthreads();
    if (wave > 1) return;
    if (wave == 0) {
        for (int w = 0; w < NW - 1; ++w)
            sfor<0, H>([&](auto M) { g[M] = g[M] + sh[(w * H + int(M)) * 64 + lane]; });
        const BiScale sc = bi_scale<T, N>(norm, t);
        const int back = -(sc.f + sc.g);
        sfor<0, H>([&](auto M) {
            g[M] = sc.zero ? T(0) * g[M] : mk(T(ldexp(g[M].x, back)), T(ldexp(g[M].y, back)));
        });
    } else {
        const cplx<T>* Fg = F + (size_t(t) * 2 + 1) * n + size_t(h) * NN + (k3 <= H ? q : 0);
        sfor<0, H>([&](auto M) {
            g[M] = ctab[(size_t(int(M)) * NPH + q) * 2 + h] * Fg[size_t(2 * int(M)) * NN];
        });
    }
    pair_dft_dit<T, N, +1>(g, o, h);                  // x = H h + k
    if (!live) return;
    const int qm = Gm::pen(k2 ? N - k2 : 0, (N - k3) % N);
    cplx<T>* dst = Z + ((size_t(t) * 2 + 1 - wave) * N + H * h) * NN;
    sfor<0, H>([&](auto K) {
        dst[size_t(int(K)) * NN + q] = o[K];
        if (k3 > 0 && k3 < H) dst[size_t(int(K)) * NN + qm] = conj(o[K]);
    });
}

// Q[gslice[g]](x, y, z) += prefac sum_{t in g} (gain_t - f_t loss_t), slot
// (g, x) a plane: the inverse plane transforms of Z.
template <typename T, int N>
__global__ void __launch_bounds__((BiPlane<T, N>::WG))
k_bi_out(const T* __restrict__ u, TaskView tv, const cplx<T>* __restrict__ Z, long nslot,
         const int* __restrict__ gstart, const int* __restrict__ gslice, T prefac,
         T* __restrict__ Q) {
    using Gm = BiGeo<N>;
    using Pl = BiPlane<T, N>;
    constexpr int NN = Gm::NN, n = Gm::n, PI = Pl::PI, PN = Pl::PN;
    __shared__ cplx<T> L[Pl::PW * Pl::ELEMS];
    __shared__ int most;
    int sl = threadIdx.x / Pl::PT;
    const bool own = sl < Pl::PW;                     // not a repeated lane
    sl = own ? sl : 0;
    const int w = (threadIdx.x - sl * Pl::PT) % Pl::PT, r = w / Pl::LN, h = w % Pl::LN;
    const long sid = long(blockIdx.x) * Pl::PW + sl;
    const bool live = own && sid < nslot;
    const long slot = sid < nslot ? sid : nslot - 1;
    const int g = int(slot / N), x = int(slot - long(g) * N);
    cplx<T>* P = L + sl * Pl::ELEMS;
    const int ta = gstart[g], nt = gstart[g + 1] - ta;
    if (threadIdx.x == 0) most = 0;
    __syncthreads();
    atomicMax(&most, nt);                             // tasks of the work-group's longest slot
    __syncthreads();
    T s[PN];
    sfor<0, PN>([&](auto K) { s[K] = T(0); });
    const int rounds = most;
    for (int i = 0; i < rounds; ++i) {
        // a shorter slot repeats its last task, one of an empty group task 0
        const int t = nt ? ta + (i < nt ? i : nt - 1) : 0;
        cplx<T> a[PN], o[PN];
        auto field = [&](int which) {                 // Re o = the field of column z = r
            const cplx<T>* Zp = Z + ((size_t(t) * 2 + which) * N + x) * NN;
            sfor<0, PN>([&](auto K) { a[K] = Zp[Gm::pen(r, Pl::in(K, h))]; });
            Pl::inverse(a, o, h);
            Pl::template exchange<PN, PN>(P, o, a,
                [&](int k) { return r * PI + Pl::out(k, h); },
                [&](int k) { return Pl::in(k, h) * PI + r; });
            Pl::inverse(a, o, h);                     // -> y
            __syncthreads();
        };
        field(1);
        if (i < nt) sfor<0, PN>([&](auto K) { s[K] += o[K].x; });
        field(0);
        const int nterm = tv.nterm[2 * t];
        const int* slc = tv.slice + size_t(t) * 2 * tv.K;
        const T* cf = static_cast<const T*>(tv.coef) + size_t(t) * 2 * tv.K;
        T f[PN];
        sfor<0, PN>([&](auto K) { f[K] = T(0); });
        for (int k = 0; k < nterm; ++k) {
            const T* p = u + size_t(slc[k]) * n + size_t(x) * NN + r;
            sfor<0, PN>([&](auto K) { f[K] += cf[k] * p[Pl::out(K, h) * N]; });
        }
        if (i < nt) sfor<0, PN>([&](auto K) { s[K] -= f[K] * o[K].x; });
    }
    if (live) {
        T* dst = Q + size_t(gslice[g]) * n + size_t(x) * NN + r;
        sfor<0, PN>([&](auto K) { dst[Pl::out(K, h) * N] += prefac * s[K]; });
    }
}

// ctab[m][q][h] = the Hermitian part of c_pq at k1 = 2 m + h and the regular
// pencil q (c_pq as k_bi_ctab): FFT(g) is Hermitian, so this is the part of
// c_pq FFT(g) that reaches the real loss.  Eight lanes share an entry's radii.
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_bi_chtab(int Nrho, int Mpre, const double* __restrict__ fac, const double* __restrict__ wc,
           const double* __restrict__ szpre, const double* __restrict__ Bsum,
           cplx<T>* __restrict__ ctab) {
    using Gm = BiGeo<N>;
    constexpr int H = Gm::H, NPH = Gm::NPH;
    const int e0 = blockIdx.x * 32 + int(threadIdx.x >> 3), e = e0 < N * NPH ? e0 : 0;
    const int q = (e >> 1) % NPH;
    const int kk[3] = {2 * ((e >> 1) / NPH) + (e & 1), (q % (2 * N)) >> 1,
                       (2 * (q / (2 * N)) + (q & 1)) % N};
    double l[3], lt[3];
    for (int a = 0; a < 3; ++a) {
        l[a] = kk[a] < H ? double(kk[a]) : double(kk[a] - N);
        lt[a] = kk[a] == H ? -l[a] : l[a];
    }
    const bool nyq = kk[0] == H || kk[1] == H || kk[2] == H;
    double cr = 0.0, ci = 0.0;
    for (int x = threadIdx.x & 7; x < Nrho; x += 8) {
        double sr = 0.0, si = 0.0, tr = 0.0, ti = 0.0;
        for (int pp = 0; pp < Mpre; ++pp) {
            double s, c;
            sincos(fac[x] * ((szpre[3 * pp] * l[0]) + (szpre[3 * pp + 1] * l[1]) +
                             (szpre[3 * pp + 2] * l[2])), &s, &c);
            sr += Bsum[pp] * c;
            si -= Bsum[pp] * s;
            if (nyq) {
                sincos(fac[x] * ((szpre[3 * pp] * lt[0]) + (szpre[3 * pp + 1] * lt[1]) +
                                 (szpre[3 * pp + 2] * lt[2])), &s, &c);
                tr += Bsum[pp] * c;
                ti -= Bsum[pp] * s;
            }
        }
        cr += wc[x] * (nyq ? 0.5 * (sr + tr) : sr);
        ci += wc[x] * (nyq ? 0.5 * (si + ti) : si);
    }
    for (int o = 4; o; o >>= 1) {
        cr += __shfl_xor(cr, o);
        ci += __shfl_xor(ci, o);
    }
    if ((threadIdx.x & 7) == 0 && e0 < N * NPH) ctab[e0] = mk(T(cr), T(ci));
}

// The weights of unit u = (x, y): Ws on the regular pencils, Wa on the line
// pencils (zero at k1 = N/2) and, in wspec, Wa at k1 = N/2 on the regular
// ones; W as k_bi_btab.  FP64 sums over the pre-rule, one thread per entry.
// ylist[j] is the direction of the j-th product of a radius, ustride the
// products per unit.
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_bi_wtab(int M, int NU, int ustride, int Mpre, const int* __restrict__ ylist,
          const double* __restrict__ fac, const double* __restrict__ wx,
          const double* __restrict__ szpre, const double* __restrict__ Bt, double mpq,
          cplx<T>* __restrict__ wtab, cplx<T>* __restrict__ wspec) {
    using Gm = BiGeo<N>;
    constexpr int H = Gm::H, NPT = Gm::NPT, NPH = Gm::NPH;
    constexpr long PER = long(N) * NPT + NPH;
    const long gid = long(blockIdx.x) * 256 + threadIdx.x;
    if (gid >= NU * PER) return;
    const int u = int(gid / PER);
    const long e = gid - u * PER;
    const bool spec = e >= long(N) * NPT;
    int q, k1;
    if (spec) {
        q = int(e - long(N) * NPT);
        k1 = H;
    } else {
        const long mq = e >> 1;
        k1 = int(2 * (mq / NPT) + (e & 1));
        q = int(mq % NPT);
    }
    const bool line = q >= NPH;
    int k2, k3;
    bool none = false;
    if (!line) {
        k3 = 2 * (q / (2 * N)) + (q & 1);
        k2 = (q % (2 * N)) >> 1;
        none = k3 > H;                              // an unused slot
    } else if (q - NPH <= H) {
        k2 = H;
        k3 = q - NPH;
    } else {
        k2 = q - NPH - H - 1;
        k3 = H;
        none = k2 == H;                             // on the first line already
    }
    const bool nyq = k1 == H || k2 == H || k3 == H;
    if (line && k1 == H) none = true;               // in wspec
    if (spec && !nyq) none = true;
    cplx<T> out = mk(T(0), T(0));
    if (!none) {
        const int d = u * ustride, x = d / M, y = ylist[d - x * M];
        const int kk[3] = {k1, k2, k3};
        double l[3], lt[3];                         // l and l with Nyquist components negated
        for (int a = 0; a < 3; ++a) {
            l[a] = kk[a] < H ? double(kk[a]) : double(kk[a] - N);
            lt[a] = kk[a] == H ? -l[a] : l[a];
        }
        double sr = 0.0, si = 0.0, tr = 0.0, ti = 0.0;
        for (int pp = 0; pp < Mpre; ++pp) {
            const double B = Bt[size_t(y) * Mpre + pp];
            double s, c;
            sincos(mpq * (fac[x] * ((szpre[3 * pp] * l[0]) + (szpre[3 * pp + 1] * l[1]) +
                                    (szpre[3 * pp + 2] * l[2]))), &s, &c);
            sr += B * c;
            si -= B * s;
            if (nyq) {                              // conj W(-k)
                sincos(mpq * (fac[x] * ((szpre[3 * pp] * lt[0]) + (szpre[3 * pp + 1] * lt[1]) +
                                        (szpre[3 * pp + 2] * lt[2]))), &s, &c);
                tr += B * c;
                ti -= B * s;
            }
        }
        if (nyq) {
            const double sg = line || spec ? -1.0 : 1.0;
            sr = 0.5 * (sr + sg * tr);
            si = 0.5 * (si + sg * ti);
        }
        out = mk(T(wx[x] * sr), T(wx[x] * si));
    }
    if (spec)
        wspec[size_t(u) * NPH + q] = out;
    else
        wtab[size_t(u) * N * NPT + e] = out;
}

}  // namespace dgfs
