// Binary-mixture VSS collision plan (kernel tables, scratch) and its C ABI.
// The kernels live in bivss_kernels.h; each (dtype, N) instance is compiled
// in its own translation unit (bi_<dtype>_<N>.hip).
#include "bivss_kernels.h"

#include <cmath>
#include <cstdlib>
#include <vector>

namespace dgfs {

DGFS_DEV double l_of(int i, int N) { return i < N / 2 ? double(i) : double(i - N); }

// b_pq tables times the gain weight (vss.mako:50-93, bi/scattering.py:193-206):
// W[xy][k] = wx[x] sum_pre B[y][pre] exp(-i mpq fac_x szpre . l_k),
// wx = qw_x sw / n * swpre qz_x^(gamma+2).  FP64, one thread per (xy, k).
template <typename T>
__global__ void __launch_bounds__(256)
k_bi_btab(int N, int M, int NXY, int Mpre, const double* __restrict__ fac,
          const double* __restrict__ wx, const double* __restrict__ szpre,
          const double* __restrict__ Bt, double mpq, cplx<T>* __restrict__ wtab) {
    const long n = long(N) * N * N;
    const long gid = long(blockIdx.x) * 256 + threadIdx.x;
    if (gid >= NXY * n) return;
    const int xy = int(gid / n), k = int(gid - long(xy) * n);
    const int x = xy / M, y = xy - x * M;
    const double l1 = l_of(k / (N * N), N), l2 = l_of((k / N) % N, N), l3 = l_of(k % N, N);
    double sr = 0.0, si = 0.0;
    for (int pp = 0; pp < Mpre; ++pp) {
        const double d = fac[x] * ((szpre[3 * pp] * l1) + (szpre[3 * pp + 1] * l2) +
                                   (szpre[3 * pp + 2] * l3));
        double s, c;
        sincos(mpq * d, &s, &c);
        const double B = Bt[size_t(y) * Mpre + pp];
        sr += B * c;
        si -= B * s;
    }
    wtab[gid] = mk(T(wx[x] * sr), T(wx[x] * si));
}

// c_pq (vss.mako:81-89): c[k] = sum_x wc[x] sum_pre Bsum[pre] exp(-i fac_x szpre . l_k),
// wc = qw_x sw swpre qz_x^(gamma+2), Bsum[pre] = sum_y B[y][pre].
template <typename T>
__global__ void __launch_bounds__(256)
k_bi_ctab(int N, int Nrho, int Mpre, const double* __restrict__ fac,
          const double* __restrict__ wc, const double* __restrict__ szpre,
          const double* __restrict__ Bsum, cplx<T>* __restrict__ ctab) {
    const long n = long(N) * N * N;
    const long k = long(blockIdx.x) * 256 + threadIdx.x;
    if (k >= n) return;
    const double l1 = l_of(int(k / (N * N)), N), l2 = l_of(int((k / N) % N), N),
                 l3 = l_of(int(k % N), N);
    double cr = 0.0, ci = 0.0;
    for (int x = 0; x < Nrho; ++x) {
        double sr = 0.0, si = 0.0;
        for (int pp = 0; pp < Mpre; ++pp) {
            const double d = fac[x] * ((szpre[3 * pp] * l1) + (szpre[3 * pp + 1] * l2) +
                                       (szpre[3 * pp + 2] * l3));
            double s, c;
            sincos(d, &s, &c);
            sr += Bsum[pp] * c;
            si -= Bsum[pp] * s;
        }
        cr += wc[x] * sr;
        ci += wc[x] * si;
    }
    ctab[k] = mk(T(cr), T(ci));
}

// f(std::integral_constant<int, N>) for the plan's grid; N = 48 is FP32 only
template <typename T, typename Fn>
static int bi_for_grid(int N, Fn&& f) {
    switch (N) {
        case 4: return f(std::integral_constant<int, 4>{});
        case 6: return f(std::integral_constant<int, 6>{});
        case 8: return f(std::integral_constant<int, 8>{});
        case 12: return f(std::integral_constant<int, 12>{});
        case 16: return f(std::integral_constant<int, 16>{});
        case 20: return f(std::integral_constant<int, 20>{});
        case 24: return f(std::integral_constant<int, 24>{});
        case 32: return f(std::integral_constant<int, 32>{});
        case 48:
            if constexpr (sizeof(T) == 4) return f(std::integral_constant<int, 48>{});
            break;
        default: break;
    }
    set_error("bi_collide: unsupported velocity grid N=%d", N);
    return 2;
}

static void bi_free(BiPlan* pl) {
    for (void* p : {pl->phase, pl->wtab, pl->wspec, pl->ctab, pl->Fhat, pl->Iw, pl->Y, pl->nyq,
                    pl->spec, pl->acc, pl->H, pl->norm, pl->Gp})
        if (p) (void)hipFree(p);
    delete pl;
}

// element counts of a grid's device arrays
struct BiSizes {
    size_t wtab = 0, wspec = 0;             // weight tables
    size_t Y = 0, nyq = 0, acc = 0;         // per task
    size_t group = 0;                       // one group's partial G^ of a task
    int groups = 1;                         // groups per task (streaming: BiPlan::ngrp in all)
    size_t ctab = 0;                        // c_pq
    size_t spec = 0;                        // a plane of spec
};
template <int N>
static BiSizes bi_sizes(bool stream, int NXY, int NU) {
    using Gm = BiGeo<N>;
    BiSizes z;
    if (stream) {
        z.wtab = size_t(NU) * N * Gm::NPT;
        z.wspec = size_t(NU) * Gm::NPH;
        z.Y = size_t(NXY) * Gm::n;
        z.nyq = size_t(NXY) * 3 * Gm::NN;
        z.group = size_t(N) * Gm::NPT;
        z.spec = Gm::NPH;
        z.ctab = size_t(N) * Gm::NPH;
    } else {
        z.wtab = z.acc = size_t(NXY) * Gm::n;
        z.group = Gm::n;
        z.groups = bi_xgroups_max<N>(NXY);
        z.ctab = Gm::n;
    }
    return z;
}
static BiSizes bi_sizes_of(const BiPlan* pl) {
    BiSizes z;
    const int NXY = pl->Nrho * pl->M;
    (void)bi_for_grid<float>(pl->N, [&](auto n) {
        z = bi_sizes<int(n)>(pl->stream, NXY, pl->antipodal ? NXY / 2 : NXY);
        return 0;
    });
    return z;
}

// opp[i] = the index of the exactly opposite point of a rule, -1 without one
static std::vector<int> opposite(const double* p, int n) {
    std::vector<int> o(n, -1);
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n && o[i] < 0; ++j)
            if (j != i && p[3 * j] == -p[3 * i] && p[3 * j + 1] == -p[3 * i + 1] &&
                p[3 * j + 2] == -p[3 * i + 2])
                o[i] = j;
    for (int i = 0; i < n; ++i)             // repeated points pair up one to one or not at all
        if (o[i] >= 0 && o[o[i]] != i) o[i] = -1;
    return o;
}

// scratch budget of the gain products (streaming: with their Nyquist planes):
// tasks are processed in chunks whose products fit in it.  Larger ones
// (3 GiB and more) take up to seconds to allocate.
constexpr size_t kBiAccBudget = size_t(2) << 30;

}  // namespace dgfs

using dgfs::BiPlan;

extern "C" int dgfs_bi_collision_plan_create(int N, int M, int Nrho, double L, const double* qz,
                                             const double* qw, const double* sz, double sw,
                                             int Mpre, const double* szpre, double mp, double mq,
                                             double alpha, double omega, double prefac,
                                             int dtype, int ntask_max,
                                             dgfs_bi_collision_plan_t* out) {
    DGFS_REQUIRE(out != nullptr, "bi_collision_plan_create: null output handle");
    *out = nullptr;
    DGFS_REQUIRE(N == 4 || N == 6 || N == 8 || N == 12 || N == 16 || N == 20 || N == 24 ||
                     N == 32 || N == 48,
                 "bi_collision_plan_create: unsupported N=%d", N);
    DGFS_REQUIRE(N != 48 || dtype == DGFS_F32,
                 "bi_collision_plan_create: N=48 is built for DGFS_F32 only");
    DGFS_REQUIRE(M > 0 && Nrho > 0 && Mpre > 0 && ntask_max > 0,
                 "bi_collision_plan_create: bad sizes");
    DGFS_REQUIRE(dtype == DGFS_F64 || dtype == DGFS_F32, "bi_collision_plan_create: bad dtype");
    DGFS_REQUIRE(qz && qw && sz && szpre, "bi_collision_plan_create: null table");
    DGFS_REQUIRE(mp > 0 && mq > 0, "bi_collision_plan_create: masses must be positive");
    const double eta = alpha - 1.0, gam = 2.0 * (1.0 - omega);
    const size_t n = size_t(N) * N * N;
    const int NXY = Nrho * M;
    const size_t es = dtype == DGFS_F64 ? 8 : 4, cs = 2 * es;

    // ---- host parts of the tables (own code; formulas of vss.mako:29-93)
    std::vector<double> Bt(size_t(M) * Mpre), Bsum(Mpre, 0.0);
    for (int y = 0; y < M; ++y)
        for (int pp = 0; pp < Mpre; ++pp) {
            const double base = 1.0 + sz[3 * y] * szpre[3 * pp] + sz[3 * y + 1] * szpre[3 * pp + 1] +
                                sz[3 * y + 2] * szpre[3 * pp + 2];
            // an exactly antipodal pair (1 + s.s' = 0) can round below zero,
            // where pow with a fractional exponent is NaN: clamp at its exact value
            Bt[size_t(y) * Mpre + pp] = std::pow(base > 0.0 ? base : 0.0, eta);
        }
    for (int pp = 0; pp < Mpre; ++pp)
        for (int y = 0; y < M; ++y) Bsum[pp] += Bt[size_t(y) * Mpre + pp];
    const double swpre = 4.0 * M_PI / Mpre;
    std::vector<double> fac(Nrho), wx(Nrho), wc(Nrho);
    for (int x = 0; x < Nrho; ++x) {
        fac[x] = M_PI / L * qz[x];
        const double fb = swpre * std::pow(qz[x], gam + 2.0);
        wx[x] = qw[x] * sw / double(n) * fb;
        wc[x] = qw[x] * sw * fb;
    }
    const double mqf = mq / (mp + mq), mpf = mp / (mp + mq);
    const bool stream =
        dgfs::bi_streams(N) &&
        ((dtype == DGFS_F64 ? dgfs::pick_split<double>(N) : dgfs::pick_split<float>(N)) > 1 ||
         size_t(ntask_max) * NXY * n * cs >= dgfs::kBiStreamBytes);
    // the direction of the j-th product of a radius: opposite points next to
    // each other where both rules are antipodally symmetric
    std::vector<int> ylist;
    const std::vector<int> oy = dgfs::opposite(sz, M), op = dgfs::opposite(szpre, Mpre);
    bool antipodal = stream && M % 2 == 0;
    for (int v : oy) antipodal = antipodal && v >= 0;
    for (int v : op) antipodal = antipodal && v >= 0;
    for (int y = 0; y < M; ++y) {
        if (antipodal && oy[y] < y) continue;
        ylist.push_back(y);
        if (antipodal) ylist.push_back(oy[y]);
    }
    std::vector<double> ph(size_t(NXY) * 2 * 3 * N * 2);
    for (int x = 0; x < Nrho; ++x)
        for (int j = 0; j < M; ++j)
            for (int side = 0; side < 2; ++side)
                for (int ax = 0; ax < 3; ++ax)
                    for (int i = 0; i < N; ++i) {
                        const double l = i < N / 2 ? double(i) : double(i - N);
                        const double th =
                            (side == 0 ? mqf : -mpf) * fac[x] * sz[3 * ylist[j] + ax] * l;
                        const size_t o = ((((size_t(x) * M + j) * 2 + side) * 3 + ax) * N + i) * 2;
                        ph[o] = std::cos(th);
                        ph[o + 1] = std::sin(th);
                    }

    auto* pl = new BiPlan();
    pl->N = N; pl->M = M; pl->Nrho = Nrho; pl->Mpre = Mpre; pl->dtype = dtype;
    pl->ntask_max = ntask_max; pl->prefac = prefac; pl->mp = mp; pl->mq = mq; pl->n = n;
    pl->stream = stream;
    pl->antipodal = antipodal;
    const dgfs::BiSizes sizes = dgfs::bi_sizes_of(pl);
    const size_t per_task = (sizes.Y + sizes.nyq + sizes.acc + size_t(NXY) * sizes.spec) * cs;
    size_t budget = dgfs::kBiAccBudget;
    if (const char* mb = std::getenv("DGFS_BI_SCRATCH_MB")) {
        const long v = std::atol(mb);
        if (v > 0) budget = size_t(v) << 20;
    }
    size_t chunk = budget / per_task;
    if (chunk < 1) chunk = 1;
    if (chunk > size_t(ntask_max)) chunk = size_t(ntask_max);
    pl->chunk = int(chunk);
    // a call that shares products takes half of them per task
    const size_t lchunk = pl->shares() ? std::min(2 * chunk, size_t(ntask_max)) : chunk;
    pl->like_chunk = int(lchunk);

    pl->ngrp = chunk * size_t(sizes.groups);
    if (stream) {
        auto more = [&](auto zero) {
            using T = decltype(zero);
            return dgfs::bi_for_grid<T>(N, [&](auto g) {
                if constexpr (dgfs::bi_streams(int(g))) dgfs::bi_stream_sizes<T, int(g)>(pl);
                return 0;
            });
        };
        (void)(dtype == DGFS_F64 ? more(0.0) : more(0.0f));
    }

    void *d_fac = nullptr, *d_wx = nullptr, *d_wc = nullptr, *d_sp = nullptr, *d_B = nullptr,
         *d_Bs = nullptr, *d_yl = nullptr;
    auto fail = [&](int rc) {
        for (void* p : {d_fac, d_wx, d_wc, d_sp, d_B, d_Bs, d_yl})
            if (p) (void)hipFree(p);
        dgfs::bi_free(pl);
        return rc;
    };
    auto up64 = [&](void** d, const double* h, size_t cnt) -> bool {
        return hipMalloc(d, cnt * 8) == hipSuccess &&
               hipMemcpy(*d, h, cnt * 8, hipMemcpyHostToDevice) == hipSuccess;
    };
    if (!up64(&d_fac, fac.data(), Nrho) || !up64(&d_wx, wx.data(), Nrho) ||
        !up64(&d_wc, wc.data(), Nrho) || !up64(&d_sp, szpre, size_t(Mpre) * 3) ||
        !up64(&d_B, Bt.data(), Bt.size()) || !up64(&d_Bs, Bsum.data(), Mpre) ||
        hipMalloc(&d_yl, size_t(M) * sizeof(int)) != hipSuccess ||
        hipMemcpy(d_yl, ylist.data(), size_t(M) * sizeof(int), hipMemcpyHostToDevice) !=
            hipSuccess) {
        dgfs::set_error("bi_collision_plan_create: table upload failed");
        return fail(1);
    }
    if (hipMalloc(&pl->phase, ph.size() / 2 * cs) != hipSuccess ||
        hipMalloc(&pl->wtab, sizes.wtab * cs) != hipSuccess ||
        (sizes.wspec && hipMalloc(&pl->wspec, sizes.wspec * cs) != hipSuccess) ||
        (sizes.Y && hipMalloc(&pl->Y, chunk * sizes.Y * cs) != hipSuccess) ||
        (sizes.nyq && hipMalloc(&pl->nyq, chunk * sizes.nyq * cs) != hipSuccess) ||
        hipMalloc(&pl->ctab, sizes.ctab * cs) != hipSuccess ||
        hipMalloc(&pl->Fhat, lchunk * 2 * n * cs) != hipSuccess ||
        hipMalloc(&pl->Iw, lchunk * 2 * n * cs) != hipSuccess ||
        hipMalloc(&pl->norm, lchunk * 4 * dgfs::bi_norm_blocks(N) * sizeof(double)) != hipSuccess ||
        (sizes.acc && hipMalloc(&pl->acc, chunk * sizes.acc * cs) != hipSuccess) ||
        (pl->nspec && hipMalloc(&pl->spec, pl->nspec * sizes.spec * cs) != hipSuccess) ||
        hipMalloc(&pl->H, size_t(ntask_max) * 2 * n * cs) != hipSuccess ||
        hipMalloc(&pl->Gp, pl->ngrp * sizes.group * cs) != hipSuccess) {
        dgfs::set_error("bi_collision_plan_create: allocation failed");
        return fail(1);
    }
    if (es == 8) {
        if (hipMemcpy(pl->phase, ph.data(), ph.size() * 8, hipMemcpyHostToDevice) != hipSuccess) {
            dgfs::set_error("bi_collision_plan_create: phase upload failed");
            return fail(1);
        }
    } else {
        std::vector<float> f(ph.begin(), ph.end());
        if (hipMemcpy(pl->phase, f.data(), f.size() * 4, hipMemcpyHostToDevice) != hipSuccess) {
            dgfs::set_error("bi_collision_plan_create: phase upload failed");
            return fail(1);
        }
    }
    auto tables = [&](auto zero) -> int {
        using T = decltype(zero);
        if (pl->stream)
            return dgfs::bi_for_grid<T>(N, [&](auto g) {
                return dgfs::bi_stream_tables<T, int(g)>(
                    pl, (const int*)d_yl, (const double*)d_fac, (const double*)d_wx,
                    (const double*)d_sp, (const double*)d_B, (const double*)d_wc,
                    (const double*)d_Bs, mqf);
            });
        hipLaunchKernelGGL(dgfs::k_bi_ctab<T>, dim3((long(n) + 255) / 256), dim3(256), 0, 0, N, Nrho,
                           Mpre, (const double*)d_fac, (const double*)d_wc, (const double*)d_sp,
                           (const double*)d_Bs, (dgfs::cplx<T>*)pl->ctab);
        hipLaunchKernelGGL(dgfs::k_bi_btab<T>, dim3((long(NXY) * long(n) + 255) / 256), dim3(256), 0,
                           0, N, M, NXY, Mpre, (const double*)d_fac, (const double*)d_wx,
                           (const double*)d_sp, (const double*)d_B, mqf,
                           (dgfs::cplx<T>*)pl->wtab);
        return 0;
    };
    if (es == 8 ? tables(0.0) : tables(0.0f)) {
        dgfs::set_error("bi_collision_plan_create: table kernels failed");
        return fail(1);
    }
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
        dgfs::set_error("bi_collision_plan_create: table kernels failed");
        return fail(1);
    }
    for (void* p : {d_fac, d_wx, d_wc, d_sp, d_B, d_Bs, d_yl}) (void)hipFree(p);
    *out = pl;
    return 0;
}

extern "C" int dgfs_bi_collision_plan_query(dgfs_bi_collision_plan_t plan, int* split,
                                            int* chunk, size_t* scratch_bytes) {
    auto* pl = static_cast<BiPlan*>(plan);
    DGFS_REQUIRE(pl, "bi_collision_plan_query: null plan");
    const size_t cs = pl->dtype == DGFS_F64 ? 16 : 8;
    if (split) *split = pl->dtype == DGFS_F64 ? dgfs::pick_split<double>(pl->N)
                                              : dgfs::pick_split<float>(pl->N);
    if (chunk) *chunk = pl->chunk;
    if (scratch_bytes) {
        const dgfs::BiSizes z = dgfs::bi_sizes_of(pl);
        *scratch_bytes = (size_t(pl->chunk) * (z.Y + z.nyq + z.acc) +
                          size_t(pl->like_chunk) * 4 * pl->n +
                          pl->nspec * z.spec + pl->ngrp * z.group +
                          size_t(pl->ntask_max) * 2 * pl->n) * cs;
    }
    return 0;
}

extern "C" int dgfs_bi_collision_plan_form(dgfs_bi_collision_plan_t plan, int* streaming,
                                           int* like_chunk) {
    auto* pl = static_cast<BiPlan*>(plan);
    DGFS_REQUIRE(pl, "bi_collision_plan_form: null plan");
    if (streaming) *streaming = pl->stream;
    if (like_chunk) *like_chunk = pl->shares() ? pl->like_chunk : 0;
    return 0;
}

extern "C" int dgfs_bi_collision_plan_destroy(dgfs_bi_collision_plan_t plan) {
    if (plan) dgfs::bi_free(static_cast<BiPlan*>(plan));
    return 0;
}

static int bi_collide(dgfs_bi_collision_plan_t plan, const void* up, const void* uq, void* Q,
                      int K, int Ne, int ntask, const int* task_nterm, const int* task_slice,
                      const void* task_coef, int ngroup, const int* group_start,
                      const int* group_slice, bool like, hipStream_t stream) {
    auto* pl = static_cast<BiPlan*>(plan);
    DGFS_REQUIRE(pl, "bi_collide: null plan");
    DGFS_REQUIRE(ntask >= 0 && ntask <= pl->ntask_max, "bi_collide: ntask=%d exceeds plan max %d",
                 ntask, pl->ntask_max);
    DGFS_REQUIRE(ngroup >= 0 && ngroup <= ntask, "bi_collide: bad ngroup=%d", ngroup);
    DGFS_REQUIRE(K > 0 && Ne > 0, "bi_collide: bad K/Ne");
    if (ntask == 0) return 0;
    DGFS_REQUIRE(up && uq && Q && task_nterm && task_slice && task_coef && group_start &&
                     group_slice,
                 "bi_collide: null pointer argument");
    dgfs::TaskView tv{K, Ne, int(pl->n), task_nterm, task_slice, task_coef};
    auto run = [&](auto zero) {
        using T = decltype(zero);
        return dgfs::bi_for_grid<T>(pl->N, [&](auto g) {
            return dgfs::bi_launch<T, int(g)>(pl, up, uq, Q, tv, ntask, ngroup, group_start,
                                              group_slice, like, stream);
        });
    };
    return pl->dtype == DGFS_F64 ? run(0.0) : run(0.0f);
}

extern "C" int dgfs_bi_collide(dgfs_bi_collision_plan_t plan, const void* up, const void* uq,
                               void* Q, int K, int Ne, int ntask, const int* task_nterm,
                               const int* task_slice, const void* task_coef, int ngroup,
                               const int* group_start, const int* group_slice,
                               hipStream_t stream) {
    return bi_collide(plan, up, uq, Q, K, Ne, ntask, task_nterm, task_slice, task_coef, ngroup,
                      group_start, group_slice, false, stream);
}

extern "C" int dgfs_bi_collide_like(dgfs_bi_collision_plan_t plan, const void* u, void* Q, int K,
                                    int Ne, int ntask, const int* task_nterm,
                                    const int* task_slice, const void* task_coef, int ngroup,
                                    const int* group_start, const int* group_slice,
                                    hipStream_t stream) {
    return bi_collide(plan, u, u, Q, K, Ne, ntask, task_nterm, task_slice, task_coef, ngroup,
                      group_start, group_slice, true, stream);
}
