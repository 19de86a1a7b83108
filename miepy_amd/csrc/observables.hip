// Observables of a solved cluster: scattered/interior coefficients,
// per-particle cross-sections, force and torque, cluster totals.
//
// Replaces, for all particles and sources in one launch:
//   p_scat = p_inc * mie_scat[:, :, n_idx], p_int = p_inc * mie_int[:, ::-1, n_idx]
//       (src/miepy/sphere_cluster.py:715-717)
//   particle_cross_sections           (cpp/src/flux.cpp:5-30)
//   force / force_all                 (cpp/src/forces.cpp:7-86, 139-154)
//   torque / torque_all               (cpp/src/forces.cpp:88-137, 156-171)
//   cross_sections() cluster sums     (src/miepy/sphere_cluster.py:442-454)
// All in FP64.  A group of lanes per (particle, source); totals are reduced in a
// fixed order by one workgroup per source.

#include <algorithm>

#include "common.hpp"

namespace {

constexpr int kThreads = 256;
// GSL_CONST_MKSA_VACUUM_PERMITTIVITY, the constant compiled into the
// reference's force/torque (cpp/src/forces.cpp:12)
constexpr double kEps0 = 8.854187817e-12;
constexpr double kPi = 3.14159265358979323846;

__device__ inline double re_mulc(double2 a, double2 b) {  // Re(a * conj(b))
    return a.x * b.x + a.y * b.y;
}
// a * conj(b)
__device__ inline double2 mulc2(double2 a, double2 b) { return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y); }

// 2 P[r] conj(Q[r1]) - P[r] conj(Qi[r1]) - Pi[r] conj(Q[r1])
__device__ inline double2 fterm(int r, int r1, const double2* P, const double2* Pi, const double2* Q,
                                const double2* Qi) {
    double2 t = cscale(mulc2(P[r], Q[r1]), 2.0);
    t = csub(t, mulc2(P[r], Qi[r1]));
    return csub(t, mulc2(Pi[r], Q[r1]));
}

// mode index r -> (n, m): r = n^2 + n + m - 1
__device__ __forceinline__ void mode_nm(int r, int& n, int& m) {
    n = (int)sqrtf((float)(r + 1) + 0.5f);
    m = r + 1 - n * n - n;
}

// mode (n, m)'s terms of the force on one particle (forces.cpp:7-86); ps_/pi_ are [2 rmax]
__device__ __forceinline__ void force_terms(int lmax, int n, int m, const double2* ps_, const double2* pi_, double k,
                                            double eps_b, double2& Fxy, double2& Fz) {
    const int rmax = lmax_to_rmax(lmax);
    const double2* p = ps_;
    const double2* q = ps_ + rmax;
    const double2* pi = pi_;
    const double2* qi = pi_ + rmax;
    const double Axy = kPi / (k * k) * kEps0 * eps_b;
    const double Az = -2 * Axy;
    const int r = n * n + n + m - 1;
    if (m != n) {
        const double f = Axy * sqrt((double)((n + m + 1) * (n - m))) / (double)(n * (n + 1));
        const int r1 = r + 1;
        Fxy = cadd(Fxy, cscale(cadd(fterm(r, r1, p, pi, q, qi), fterm(r, r1, q, qi, p, pi)), f));
    }
    Fz = cadd(Fz, cscale(fterm(r, r, p, pi, q, qi), Az * m / (double)(n * (n + 1))));
    if (n < lmax) {
        const double den = (double)((2 * n + 3) * (2 * n + 1));
        double f = -Axy * sqrt((double)((n + m + 2) * (n + m + 1) * n * (n + 2)) / den) / (n + 1);
        int r1 = (n + 1) * (n + 1) + (n + 1) + m;
        Fxy = cadd(Fxy, cscale(cadd(fterm(r, r1, p, pi, p, pi), fterm(r, r1, q, qi, q, qi)), f));
        f = Axy * sqrt((double)((n - m + 1) * (n - m + 2) * n * (n + 2)) / den) / (n + 1);
        r1 = (n + 1) * (n + 1) + (n + 1) + m - 2;
        Fxy = cadd(Fxy, cscale(cadd(fterm(r1, r, p, pi, p, pi), fterm(r1, r, q, qi, q, qi)), f));
        f = Az * sqrt((double)((n - m + 1) * (n + m + 1) * n * (n + 2)) / den) / (n + 1);
        r1 = (n + 1) * (n + 1) + (n + 1) + m - 1;
        Fz = cadd(Fz, cscale(cadd(fterm(r1, r, p, pi, p, pi), fterm(r1, r, q, qi, q, qi)), f));
    }
}

// mode (n, m)'s terms of the torque on one particle (forces.cpp:88-137)
__device__ __forceinline__ void torque_terms(int lmax, int n, int m, const double2* ps_, const double2* pi_, double k,
                                             double eps_b, double (&T)[3]) {
    const int rmax = lmax_to_rmax(lmax);
    const double2* p = ps_;
    const double2* q = ps_ + rmax;
    const double2* pi = pi_;
    const double2* qi = pi_ + rmax;
    const double A = -2 * kPi / (k * k * k) * kEps0 * eps_b;
    const int r = n * n + n + m - 1;
    if (m != n) {
        const double f = -A * sqrt((double)((n - m) * (n + m + 1)));
        const int r1 = r + 1;
        const double2 pp = cadd(mulc2(p[r], p[r1]), mulc2(q[r], q[r1]));
        const double2 x1 = cadd(cadd(mulc2(p[r1], pi[r]), mulc2(p[r], pi[r1])),
                                cadd(mulc2(q[r1], qi[r]), mulc2(q[r], qi[r1])));
        const double2 y1 = cadd(csub(mulc2(p[r1], pi[r]), mulc2(p[r], pi[r1])),
                                csub(mulc2(q[r1], qi[r]), mulc2(q[r], qi[r1])));
        T[0] += f * (pp.x - 0.5 * x1.x);
        T[1] += f * (pp.y + 0.5 * y1.y);
    }
    T[2] += A * m * ((p[r].x * p[r].x + p[r].y * p[r].y) + (q[r].x * q[r].x + q[r].y * q[r].y) -
                     (re_mulc(p[r], pi[r]) + re_mulc(q[r], qi[r])));
}

// ---- a group of lanes per particle and source -------------------------------------
//
// The lanes of a group read the particle's coefficients together (consecutive
// modes, coalesced) into LDS; lane l then forms the cross-section terms of
// the modes l, l + lanes, ..., and the force and torque terms of the same
// modes, which the group adds by shuffles.  With one thread per (particle,
// source) the 2000 threads of 500 spheres and 4 sources filled 8 workgroups
// whose lanes read 64 rows at once: 57 us, 7.5 us with 16 lanes each.
// One kernel body serves the entry points: p_scat given or formed from the Mie
// coefficients, and whichever outputs are asked for (null: not).

__host__ __device__ inline int obs_lanes(int lmax) { return lmax <= 3 ? 16 : 32; }  // rmax 15 and 24 .. 48
__host__ __device__ inline int obs_per_group(int lmax) { return kThreads / obs_lanes(lmax); }
// LDS of one particle: p_scat and p_inc [2 rmax] c128, absorption and extinction terms [2 rmax] f64
__host__ __device__ inline size_t obs_lds(int lmax) {
    return (size_t)obs_per_group(lmax) * 2 * lmax_to_rmax(lmax) * (2 * sizeof(double2) + 2 * sizeof(double));
}

__device__ __forceinline__ void observables_group(const mpa_obs_cluster& C, bool given, int wg, double2* lds) {
    const int lmax = C.lmax, rmax = lmax_to_rmax(lmax), bs = 2 * rmax;
    const int lanes = obs_lanes(lmax), lane = threadIdx.x & (lanes - 1), slot = threadIdx.x / lanes;
    const int per = kThreads / lanes, item = wg * per + slot;  // item = source * N + particle
    const bool live = item < C.N * C.nsrc;
    double2* ps = lds + (size_t)slot * 2 * bs;
    double2* pi = ps + bs;
    double* ca = (double*)(lds + (size_t)per * 2 * bs) + (size_t)slot * 2 * bs;
    double* ce = ca + bs;
    const size_t base = (size_t)item * bs;
    const double factor = 4 * kPi / (C.k * C.k);
    if (live) {
        const int i = item % C.N;
        const double2 *inc = (const double2*)C.p_inc, *src = (const double2*)C.p_src;
        for (int e = lane; e < bs; e += lanes) {
            const int a = e >= rmax ? 1 : 0;
            const double2 pv = inc[base + e];
            double2 sc;
            if (given) {
                sc = ((const double2*)C.p_scat)[base + e];
            } else {
                int n, m;
                mode_nm(e - a * rmax, n, m);
                sc = cmul(pv, ((const double2*)C.mie_scat)[((size_t)i * 2 + a) * lmax + n - 1]);
                ((double2*)C.p_scat)[base + e] = sc;
                if (C.p_int)
                    ((double2*)C.p_int)[base + e] =
                        cmul(pv, ((const double2*)C.mie_int)[((size_t)i * 2 + (1 - a)) * lmax + n - 1]);
            }
            ps[e] = sc;
            pi[e] = pv;
            if (C.C_part) {
                ca[e] = factor * (re_mulc(sc, pv) - (sc.x * sc.x + sc.y * sc.y));
                ce[e] = factor * re_mulc(sc, src[base + e]);
            }
        }
    }
    __syncthreads();
    if (live && C.C_part) {  // cross-sections per multipole (flux.cpp:5-30): [3][2][lmax]
        double* Cp = C.C_part + (size_t)item * 6 * lmax;
        for (int q = lane; q < 2 * lmax; q += lanes) {
            const int a = q / lmax, n = q - a * lmax + 1;
            double cabs = 0, cext = 0;
            for (int m = -n; m <= n; m++) {
                cabs += ca[a * rmax + mode_r(n, m)];
                cext += ce[a * rmax + mode_r(n, m)];
            }
            Cp[q] = cext - cabs;
            Cp[2 * lmax + q] = cabs;
            Cp[4 * lmax + q] = cext;
        }
    }
    double2 Fxy = make_double2(0, 0), Fz = make_double2(0, 0);
    double T[3] = {0, 0, 0};
    if (live)
        for (int r = lane; r < rmax; r += lanes) {
            int n, m;
            mode_nm(r, n, m);
            if (C.F) force_terms(lmax, n, m, ps, pi, C.k, C.eps_b, Fxy, Fz);
            if (C.T) torque_terms(lmax, n, m, ps, pi, C.k, C.eps_b, T);
        }
    double v[6] = {Fxy.x, Fxy.y, Fz.x, T[0], T[1], T[2]};
    for (int off = lanes / 2; off > 0; off >>= 1)
#pragma unroll
        for (int e = 0; e < 6; e++) v[e] += __shfl_xor(v[e], off);
    if (live && lane == 0)
#pragma unroll
        for (int e = 0; e < 3; e++) {
            if (C.F) C.F[(size_t)item * 3 + e] = v[e];
            if (C.T) C.T[(size_t)item * 3 + e] = v[3 + e];
        }
}

__global__ __launch_bounds__(kThreads) void k_observables(mpa_obs_cluster C, int given) {
    extern __shared__ double2 lds[];
    observables_group(C, given != 0, blockIdx.x, lds);
}

int obs_workgroups(int lmax, long long items) {
    const int per = obs_per_group(lmax);
    return (int)((items + per - 1) / per);
}

void launch_observables(const mpa_obs_cluster& C, bool given, hipStream_t st) {
    hipLaunchKernelGGL(k_observables, dim3(obs_workgroups(C.lmax, (long long)C.N * C.nsrc)), dim3(kThreads),
                       obs_lds(C.lmax), st, C, given ? 1 : 0);
}

// ---- many clusters per launch: descriptors travel by value in the kernel
// arguments (up to kObsBatchMax clusters per launch), workgroups dealt to the
// clusters in order; each cluster's arithmetic is that of its own launch.
constexpr int kObsBatchMax = 32;

struct ObsBatch {
    int count;
    int first[kObsBatchMax + 1];  // prefix of each cluster's workgroups
    mpa_obs_cluster c[kObsBatchMax];
};

__device__ __forceinline__ int obs_cluster_of(const ObsBatch& B, int v) {
    int q = 0;
    while (q + 1 < B.count && v >= B.first[q + 1]) q++;
    return q;
}

__global__ __launch_bounds__(kThreads) void k_observables_b(ObsBatch B) {
    extern __shared__ double2 lds[];
    const int q = obs_cluster_of(B, blockIdx.x);
    observables_group(B.c[q], false, blockIdx.x - B.first[q], lds);
}

// cluster totals per source: sum over particles (fixed order) of the
// per-particle sums over multipoles; out [S][3] (scat, abs, ext)
__device__ void totals_one(int N, int lmax, int s, const double* __restrict__ C_part, double* __restrict__ C_total) {
    const int L = 2 * lmax;
    double acc[3] = {0, 0, 0};
    for (int i = threadIdx.x; i < N; i += kThreads) {
        const double* Cp = C_part + ((size_t)s * N + i) * 3 * L;
        for (int c = 0; c < 3; c++) {
            double t = 0;
            for (int e = 0; e < L; e++) t += Cp[c * L + e];
            acc[c] += t;
        }
    }
    __shared__ double red[3][kThreads];
    for (int c = 0; c < 3; c++) red[c][threadIdx.x] = acc[c];
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int c = 0; c < 3; c++) red[c][threadIdx.x] += red[c][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 3; c++) C_total[s * 3 + c] = red[c][0];
}

__global__ __launch_bounds__(kThreads) void k_totals(int N, int lmax, const double* __restrict__ C_part,
                                                     double* __restrict__ C_total) {
    totals_one(N, lmax, blockIdx.x, C_part, C_total);
}

// one workgroup per (cluster, source) of the batch with C_total set; first[] counts sources
__global__ __launch_bounds__(kThreads) void k_totals_b(ObsBatch B) {
    const int q = obs_cluster_of(B, blockIdx.x);
    const mpa_obs_cluster& C = B.c[q];
    totals_one(C.N, C.lmax, blockIdx.x - B.first[q], C.C_part, C.C_total);
}

// y_j = Tm_j x_j for every particle and right-hand side (block-diagonal
// product): p_scat = T p_inc of cpp's `cluster` path (src/miepy/cluster.py:657,
// einsum "naibj,nbj->nai").  One thread per output entry; Tm_j rows are read
// through the caches.
__global__ __launch_bounds__(256) void k_tmatrix_apply(int N, int bs, int S, const double2* __restrict__ tm,
                                                       const double2* __restrict__ x, double2* __restrict__ y) {
    const size_t n = (size_t)bs * N;
    const size_t total = (size_t)S * n;
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (size_t)gridDim.x * 256) {
        const size_t s = idx / n, rest = idx - s * n;
        const size_t j = rest / bs, e = rest - j * bs;
        const double2* trow = tm + (j * bs + e) * bs;
        const double2* xj = x + s * n + j * bs;
        double2 acc = make_double2(0.0, 0.0);
        for (int c = 0; c < bs; c++) cfma(acc, trow[c], xj[c]);
        y[idx] = acc;
    }
}

}  // namespace

int mpa_internal_tmatrix_apply(int N, int lmax, int nrhs, const double* tmatrix, const void* x, void* y,
                               hipStream_t st) {
    const int bs = 2 * lmax_to_rmax(lmax);
    const size_t total = (size_t)nrhs * bs * N;
    const unsigned blocks = (unsigned)std::min<size_t>(4096, (total + 255) / 256);
    hipLaunchKernelGGL(k_tmatrix_apply, dim3(blocks), dim3(256), 0, st, N, bs, nrhs, (const double2*)tmatrix,
                       (const double2*)x, (double2*)y);
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}

extern "C" int mpa_tmatrix_apply(int N, int lmax, int nrhs, const double* tmatrix, const void* x, void* y,
                                 void* stream) {
    if (N < 1 || nrhs < 1 || lmax < 1 || lmax > MPA_LMAX_MAX || !tmatrix || !x || !y || x == y) {
        mpa_set_error("tmatrix_apply: bad argument");
        return MPA_ERR_ARG;
    }
    return mpa_internal_tmatrix_apply(N, lmax, nrhs, tmatrix, x, y, (hipStream_t)stream);
}

extern "C" int mpa_cluster_observables(int N, int lmax, int nsrc, const double* p_inc, const double* p_src,
                                       const double* mie_scat, const double* mie_int, double k, double eps_b,
                                       double* p_scat, double* p_int, double* C_part, double* C_total, double* F,
                                       double* T, void* stream) {
    if (N < 1 || nsrc < 1 || lmax < 1 || lmax > MPA_LMAX_MAX || !p_inc || !p_src || !mie_scat || !p_scat || !C_part ||
        !F || !(k > 0) || (p_int && !mie_int)) {
        mpa_set_error("cluster_observables: bad argument");
        return MPA_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    launch_observables(mpa_obs_cluster{N, lmax, nsrc, 0, p_inc, p_src, mie_scat, mie_int, k, eps_b, p_scat, p_int,
                                       C_part, C_total, F, T},
                       false, st);
    if (C_total) hipLaunchKernelGGL(k_totals, dim3(nsrc), dim3(kThreads), 0, st, N, lmax, C_part, C_total);
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}

extern "C" int mpa_cluster_observables_batched(int count, const mpa_obs_cluster* clusters, void* stream) {
    if (count < 0 || (count > 0 && !clusters)) {
        mpa_set_error("cluster_observables_batched: bad argument");
        return MPA_ERR_ARG;
    }
    for (int q = 0; q < count; q++) {
        const mpa_obs_cluster& C = clusters[q];
        if (C.N < 1 || C.nsrc < 1 || C.lmax < 1 || C.lmax > MPA_LMAX_MAX || !C.p_inc || !C.p_src || !C.mie_scat ||
            !C.p_scat || !C.C_part || !C.F || !(C.k > 0) || (C.p_int && !C.mie_int) ||
            (long long)C.N * C.nsrc > 0x7fffffffLL - kThreads) {
            mpa_set_error("cluster_observables_batched: bad cluster %d", q);
            return MPA_ERR_ARG;
        }
    }
    hipStream_t st = (hipStream_t)stream;
    for (int b = 0; b < count; b += kObsBatchMax) {
        const int cnt = std::min(kObsBatchMax, count - b);
        ObsBatch Bo{}, Bt{};
        Bo.count = cnt;
        long long wg = 0;
        size_t lds = 0;
        for (int q = 0; q < cnt; q++) {
            const mpa_obs_cluster& C = clusters[b + q];
            Bo.c[q] = C;
            const int groups = obs_workgroups(C.lmax, (long long)C.N * C.nsrc);
            wg += groups;
            if (wg <= 0x7fffffffLL) Bo.first[q + 1] = Bo.first[q] + groups;
            lds = std::max(lds, obs_lds(C.lmax));
            if (C.C_total) {
                Bt.c[Bt.count] = C;
                Bt.first[Bt.count + 1] = Bt.first[Bt.count] + C.nsrc;
                Bt.count++;
            }
        }
        if (wg > 0x7fffffffLL) {
            mpa_set_error("cluster_observables_batched: batch too large for one launch");
            return MPA_ERR_ARG;
        }
        hipLaunchKernelGGL(k_observables_b, dim3((unsigned)Bo.first[cnt]), dim3(kThreads), lds, st, Bo);
        if (Bt.count) hipLaunchKernelGGL(k_totals_b, dim3((unsigned)Bt.first[Bt.count]), dim3(kThreads), 0, st, Bt);
        MPA_LAUNCH_CHECK();
    }
    return MPA_OK;
}

extern "C" int mpa_force_torque(int M, int lmax, const double* p_scat, const double* p_inc, double k, double eps_b,
                                double* F, double* T, void* stream) {
    if (M < 1 || lmax < 1 || lmax > MPA_LMAX_MAX || !p_scat || !p_inc || (!F && !T) || !(k > 0)) {
        mpa_set_error("force_torque: bad argument");
        return MPA_ERR_ARG;
    }
    mpa_obs_cluster C{};
    C.N = M;
    C.lmax = lmax;
    C.nsrc = 1;
    C.p_inc = p_inc;
    C.p_scat = const_cast<double*>(p_scat);  // given: read only
    C.k = k;
    C.eps_b = eps_b;
    C.F = F;
    C.T = T;
    launch_observables(C, true, (hipStream_t)stream);
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}

extern "C" int mpa_particle_cross_sections(int M, int lmax, const double* p_scat, const double* p_inc,
                                           const double* p_src, double k, double* C_part, void* stream) {
    if (M < 1 || lmax < 1 || lmax > MPA_LMAX_MAX || !p_scat || !p_inc || !p_src || !C_part || !(k > 0)) {
        mpa_set_error("particle_cross_sections: bad argument");
        return MPA_ERR_ARG;
    }
    mpa_obs_cluster C{};
    C.N = M;
    C.lmax = lmax;
    C.nsrc = 1;
    C.p_inc = p_inc;
    C.p_src = p_src;
    C.p_scat = const_cast<double*>(p_scat);  // given: read only
    C.k = k;
    C.C_part = C_part;
    launch_observables(C, true, (hipStream_t)stream);
    MPA_LAUNCH_CHECK();
    return MPA_OK;
}
