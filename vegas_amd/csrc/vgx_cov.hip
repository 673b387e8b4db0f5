// vgx_cov.hip -- per-hcube sums of multi-component integrands (fcn_size > 1):
// the mean vector and the covariance (or the variances) of one iteration,
// src/vegas/_vegas.pyx:2136-2183 with correlate_integrals on or off.
//
// Work item: (hcube h, component pair q, or all pairs for m <= 6).  A thread
// owns a strided set of the batch's hcubes (longer ones are shared by its wave or
// workgroup); for each hcube it makes the reference's two passes over the
// hcube's points: S = sum w f (per component), then the deviations
// d = w f - S/n with the EPSILON guard (a guarded deviation adds
// (EPSILON |S/n|)^2 to its own diagonal entry and is 0 in every other sum).
// Diagonal pairs also contribute S + D to the mean (Neely's correction).
// Sums over hcubes are double-double, reduced in a fixed order (partials per
// workgroup, then one thread per pair), so results do not depend on timing.
#include "vgx_internal.h"

namespace vgx {

constexpr int kCovThreads = 256;
constexpr int kCovWaves = kCovThreads / 64;
constexpr int kCovMaxBlocks = 8192;  // workgroups per pair (one thread per hcube up to 2M hcubes)
// A hcube of up to kCovShort points is summed by a thread, of up to kCovLong by
// a wave, a longer one by the workgroup.  (Everything above 32 by the workgroup
// in turn: up to 375 us a batch of 2e6 points in adapted strata, 8 axes, four
// components, now up to 170.  From 16 by a wave: 5-15 % slower where most
// hcubes are that short; from 8 twice the time.)
constexpr uint32_t kCovShort = 32, kCovLong = 2048;
// A batch of hcubes that are long on average (above kCovShort) has few of them:
// with a workgroup for 256 they would be the work of a few waves.  As long as
// that gives fewer workgroups than CUs, it has a workgroup for each hcube, up to
// kCovFew in all, the hcubes of a workgroup are spread over its waves, and a
// workgroup with one hcube sums it together from kCovAlone points on.  (56
// hcubes of 2000 points, six components: 1306 us by one wave, 361 by one
// workgroup in turn, 36 so.  kCovFew = 2048: 40,000 hcubes of 40, 231 us for 178.)
constexpr int kCovFew = 1024;
constexpr uint32_t kCovAlone = 128;
// Five and six components: pair by pair for few points or hcubes, where the
// kernel of all pairs is one long chain.  (us a call, all pairs / pair by pair:
// 256 hcubes of 4 points 25 / 17, 56 of 500 33 / 17, one of 100,000 349 / 299.)
constexpr int64_t kCovPairPoints = 32768, kCovPairHcubes = 4;

struct CovPlan {
    uint32_t lng;  // hcubes with more points are summed by the workgroup
    uint32_t few;  // spread a workgroup's hcubes over its waves
};

// Pair q of the lower triangle (t <= s), row-major: (0,0) (1,0) (1,1) (2,0) ...
__device__ inline void cov_pair(int q, int correlate, int& s, int& t) {
    if (!correlate) {
        s = t = q;
        return;
    }
    int r = (int)((sqrt(8.0 * q + 1.0) - 1.0) * 0.5);
    while ((r + 1) * (r + 2) / 2 <= q) ++r;
    while (r * (r + 1) / 2 > q) --r;
    s = r;
    t = q - r * (r + 1) / 2;
}

// Workgroup sum of K values per thread, in a fixed order (wave butterflies,
// then waves 0..3); every thread receives the totals.  red: K * kCovWaves.
template <int K>
__device__ inline void block_sum(double (&v)[K], double* red) {
    const int wv = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double r = wave_sum_fixed(v[k]);
        if ((threadIdx.x & 63) == 0) red[wv * K + k] = r;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double r = red[k];
#pragma unroll
        for (int u = 1; u < kCovWaves; ++u) r += red[u * K + k];
        v[k] = r;
    }
    __syncthreads();
}

__device__ inline double lane_value(double v, int lane) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane), hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// v from lane (l & ~15) | ((l + N) & 15): a rotation within 16 lanes.
template <int N>
__device__ inline double row_ror(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (uint32_t)u, 0x120 + N, 0xF, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (uint32_t)(u >> 32), 0x120 + N, 0xF, 0xF, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// a + b of the halves (SIXTEEN: the odd and even rows of 16 lanes) of the wave:
// the lower (even) lanes receive a's, the upper (odd) lanes b's.
template <bool SIXTEEN>
__device__ inline double fold2(double a, double b) {
    const uint64_t ua = (uint64_t)__double_as_longlong(a), ub = (uint64_t)__double_as_longlong(b);
    uint32_t x[2], y[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t wa = (uint32_t)(ua >> (32 * i)), wb = (uint32_t)(ub >> (32 * i));
        const auto r = SIXTEEN ? __builtin_amdgcn_permlane16_swap(wa, wb, false, false)
                               : __builtin_amdgcn_permlane32_swap(wa, wb, false, false);
        x[i] = r[0];
        y[i] = r[1];
    }
    return __longlong_as_double((long long)(((uint64_t)x[1] << 32) | x[0])) +
           __longlong_as_double((long long)(((uint64_t)y[1] << 32) | y[0]));
}
// Wave sum of K values per lane, in a fixed order; every lane receives the
// totals.  Two foldings leave a quarter of the values in each 16 lanes, which
// add theirs: a third of the instructions of K butterflies.
template <int K>
__device__ inline void wave_total(double (&v)[K]) {
    constexpr int Q = (K + 3) / 4;
    double z[4 * Q];
#pragma unroll
    for (int k = 0; k < 4 * Q; ++k) z[k] = k < K ? v[k] : 0.0;
#pragma unroll
    for (int k = 0; k < 2 * Q; ++k) z[k] = fold2<false>(z[k], z[2 * Q + k]);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        z[k] = fold2<true>(z[k], z[Q + k]);
        z[k] += row_ror<8>(z[k]);
        z[k] += row_ror<4>(z[k]);
        z[k] += row_ror<2>(z[k]);
        z[k] += row_ror<1>(z[k]);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = lane_value(z[k % Q], 16 * (k / Q));
}

// The hcubes [h0, h1) in rounds of gridDim.x * blockDim.x: thread t of
// workgroup b takes hcube h0 + r0 + t * gridDim.x + b (neighbouring hcubes,
// which tend to be large together near a peak, land in different
// workgroups; with `few` also in different waves).  A hcube of at most kCovShort points is summed by its thread
// (wk.thread_hcube), a longer one after that by the thread's wave
// (wk.wave_hcube), and those of more than pl.lng points after the round by
// the whole workgroup, in thread order (wk.block_hcube), so the work per
// thread stays bounded however the points are spread.  A hcube whose points are not the
// batch's [p0, p1) (or that has fewer than two) sets VGX_ERANGE and is not read.
template <class Work>
__device__ inline void cov_rounds(const uint32_t* off, uint32_t h0, uint32_t h1, uint32_t p0, uint32_t p1,
                                  CovPlan pl, int32_t* status, Work& wk) {
    __shared__ uint64_t lmask[kCovWaves];
    __shared__ uint32_t la[kCovThreads], lb[kCovThreads];
    const uint32_t nh = h1 - h0, stride = gridDim.x * blockDim.x;
    for (uint32_t r0 = 0; r0 < nh; r0 += stride) {
        const uint32_t slot = pl.few ? (threadIdx.x & 63) * kCovWaves + (threadIdx.x >> 6) : threadIdx.x;
        const uint32_t idx = r0 + slot * gridDim.x + blockIdx.x;
        bool block = false, mid = false;
        uint32_t oa = 0, ob = 0;
        if (idx < nh) {
            oa = off[h0 + idx];
            ob = off[h0 + idx + 1];
            if (oa < p0 || ob > p1 || ob < oa + 2) {
                if (status) atomicOr(status, VGX_ERANGE);
            } else if (ob - oa > pl.lng) {
                block = true;
                la[threadIdx.x] = oa - p0;
                lb[threadIdx.x] = ob - p0;
            } else if (ob - oa > kCovShort) {
                mid = true;
            } else {
                wk.thread_hcube(oa - p0, ob - p0);
            }
        }
        for (uint64_t mk = __ballot(mid); mk; mk &= mk - 1) {
            const int src = __builtin_ctzll(mk);
            wk.wave_hcube(__builtin_amdgcn_readlane(oa, src) - p0, __builtin_amdgcn_readlane(ob, src) - p0, src);
        }
        const uint64_t bal = __ballot(block);
        if ((threadIdx.x & 63) == 0) lmask[threadIdx.x >> 6] = bal;
        __syncthreads();
        for (int wv = 0; wv < kCovWaves; ++wv) {
            uint64_t mk = lmask[wv];
            while (mk) {
                const int src = wv * 64 + __builtin_ctzll(mk);
                mk &= mk - 1;
                wk.block_hcube(la[src], lb[src]);
            }
        }
        __syncthreads();
    }
}

// One component pair (s, t) per workgroup row blockIdx.y, any m.
struct PairWork {
    const double* w;
    const double* f;
    int m, s, t;
    double eps;
    DD am, av;
    double* red;

    // the reference's two passes over one hcube's points, [a, b)
    __device__ void thread_hcube(uint32_t a, uint32_t b) {
        const double n = (double)(b - a);
        double Ss = 0.0, St = 0.0;
        for (uint32_t j = a; j < b; ++j) Ss += w[j] * f[(size_t)j * m + s];
        if (s != t)
            for (uint32_t j = a; j < b; ++j) St += w[j] * f[(size_t)j * m + t];
        double v[3] = {0.0, 0.0, 0.0};
        pass2(a, b, 1, Ss / n, St / n, v);
        close(n, Ss, v);
    }
    // by the wave, into lane src's sums
    __device__ void wave_hcube(uint32_t a, uint32_t b, int src) {
        const int lane = threadIdx.x & 63;
        const double n = (double)(b - a);
        double S[2] = {0.0, 0.0};
        for (uint32_t j = a + lane; j < b; j += 64) {
            S[0] += w[j] * f[(size_t)j * m + s];
            S[1] += w[j] * f[(size_t)j * m + t];
        }
        wave_total<2>(S);
        double v[3] = {0.0, 0.0, 0.0};
        pass2(a + lane, b, 64, S[0] / n, S[1] / n, v);
        wave_total<3>(v);
        if (lane == src) close(n, S[0], v);
    }
    __device__ void block_hcube(uint32_t a, uint32_t b) {
        const double n = (double)(b - a);
        double S[2] = {0.0, 0.0};
        for (uint32_t j = a + threadIdx.x; j < b; j += blockDim.x) {
            S[0] += w[j] * f[(size_t)j * m + s];
            S[1] += w[j] * f[(size_t)j * m + t];
        }
        block_sum<2>(S, red);
        double v[3] = {0.0, 0.0, 0.0};
        pass2(a + threadIdx.x, b, blockDim.x, S[0] / n, S[1] / n, v);
        block_sum<3>(v, red);
        if (threadIdx.x == 0) close(n, S[0], v);
    }
    // v = {Q, Ds, Dt} over points a, a + step, ... < b
    __device__ void pass2(uint32_t a, uint32_t b, uint32_t step, double ms, double mt, double (&v)[3]) {
        const double gs = eps * fabs(ms), gt = eps * fabs(mt);
        for (uint32_t j = a; j < b; j += step) {
            double ds = w[j] * f[(size_t)j * m + s] - ms;
            if (s == t) {
                if (fabs(ds) < gs) {
                    v[0] += gs * gs;
                    ds = 0.0;
                } else {
                    v[0] += ds * ds;
                }
                v[1] += ds;
            } else {
                double dt = w[j] * f[(size_t)j * m + t] - mt;
                if (fabs(ds) < gs) ds = 0.0;
                if (fabs(dt) < gt) dt = 0.0;
                v[0] += ds * dt;
                v[1] += ds;
                v[2] += dt;
            }
        }
    }
    __device__ void close(double n, double Ss, const double (&v)[3]) {
        double Dt = v[2];
        if (s == t) {
            dd_add(am, Ss + v[1]);
            Dt = v[1];
        }
        dd_add(av, (n * v[0] - v[1] * Dt) / (n - 1.));
    }
};

__global__ __launch_bounds__(kCovThreads) void cov_hcube_kernel(const uint32_t* off, uint32_t h0, uint32_t h1,
                                                                 uint32_t p0, uint32_t p1, const double* w,
                                                                 const double* f, int m, int correlate, CovPlan pl,
                                                                 double* part, int32_t* status) {
    __shared__ double red[4 * kCovWaves];
    PairWork wk{w, f, m, 0, 0, kEpsilon, DD{0, 0}, DD{0, 0}, red};
    cov_pair((int)blockIdx.y, correlate, wk.s, wk.t);
    cov_rounds(off, h0, h1, p0, p1, pl, status, wk);
    DD am = wave_sum_dd(wk.am);
    DD av = wave_sum_dd(wk.av);
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[4 * wv + 0] = am.hi;
        red[4 * wv + 1] = am.lo;
        red[4 * wv + 2] = av.hi;
        red[4 * wv + 3] = av.lo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        DD m2{0, 0}, v2{0, 0};
        for (int k = 0; k < kCovWaves; ++k) {
            m2 = dd_sum(m2, DD{red[4 * k], red[4 * k + 1]});
            v2 = dd_sum(v2, DD{red[4 * k + 2], red[4 * k + 3]});
        }
        double* o = part + 4 * ((size_t)blockIdx.y * gridDim.x + blockIdx.x);
        o[0] = m2.hi;
        o[1] = m2.lo;
        o[2] = v2.hi;
        o[3] = v2.lo;
    }
}

// Up to kCovAllMax components: every pair at once from the hcube's
// contiguous rows of f (each row read once per pass), then the same fixed-order double-double reduction and partial
// layout as cov_hcube_kernel.
// (Pair by pair, six components took 980-4400 us a batch of 2e6 points, 12
// axes, now 142-324; 250 registers.)
constexpr int kCovAllMax = 6;

template <int M>
struct AllWork {
    static constexpr int NP = M * (M + 1) / 2;
    const double* w;
    const double* f;
    double eps;
    DD am[M], av[NP];
    double* red;

    __device__ void thread_hcube(uint32_t a, uint32_t b) {
        double S[M];
#pragma unroll
        for (int s = 0; s < M; ++s) S[s] = 0.0;
        pass1(a, b, 1, S);
        double v[M + NP];
        pass2(a, b, 1, S, (double)(b - a), v);
        close((double)(b - a), S, v);
    }
    // by the wave, into lane src's sums
    __device__ void wave_hcube(uint32_t a, uint32_t b, int src) {
        const int lane = threadIdx.x & 63;
        double S[M];
#pragma unroll
        for (int s = 0; s < M; ++s) S[s] = 0.0;
        pass1(a + lane, b, 64, S);
        wave_total<M>(S);
        double v[M + NP];
        pass2(a + lane, b, 64, S, (double)(b - a), v);
        wave_total<M + NP>(v);
        if (lane == src) close((double)(b - a), S, v);
    }
    __device__ void block_hcube(uint32_t a, uint32_t b) {
        double S[M];
#pragma unroll
        for (int s = 0; s < M; ++s) S[s] = 0.0;
        pass1(a + threadIdx.x, b, blockDim.x, S);
        block_sum<M>(S, red);
        double v[M + NP];
        pass2(a + threadIdx.x, b, blockDim.x, S, (double)(b - a), v);
        block_sum<M + NP>(v, red);
        if (threadIdx.x == 0) close((double)(b - a), S, v);
    }
    __device__ void pass1(uint32_t a, uint32_t b, uint32_t step, double (&S)[M]) {
        for (uint32_t j = a; j < b; j += step) {
            const double wj = w[j];
#pragma unroll
            for (int s = 0; s < M; ++s) S[s] += wj * f[(size_t)j * M + s];
        }
    }
    // v = {D[M], Q[NP]} over points a, a + step, ... < b; S = the hcube's sums
    __device__ void pass2(uint32_t a, uint32_t b, uint32_t step, const double (&S)[M], double n,
                          double (&v)[M + NP]) {
        double mu[M], g[M];
#pragma unroll
        for (int s = 0; s < M; ++s) {
            mu[s] = S[s] / n;
            g[s] = eps * fabs(mu[s]);
        }
#pragma unroll
        for (int k = 0; k < M + NP; ++k) v[k] = 0.0;
        for (uint32_t j = a; j < b; j += step) {
            const double wj = w[j];
            double d[M];
#pragma unroll
            for (int s = 0; s < M; ++s) {
                d[s] = wj * f[(size_t)j * M + s] - mu[s];
                double& qss = v[M + s * (s + 1) / 2 + s];
                if (fabs(d[s]) < g[s]) {
                    qss += g[s] * g[s];
                    d[s] = 0.0;
                } else {
                    qss += d[s] * d[s];
                }
                v[s] += d[s];
            }
#pragma unroll
            for (int s = 1; s < M; ++s)
#pragma unroll
                for (int t = 0; t < s; ++t) v[M + s * (s + 1) / 2 + t] += d[s] * d[t];
        }
    }
    // double-double beyond four components, as PairWork; plain up to four
    static __device__ void add(DD& a, double v) {
        if constexpr (M > 4)
            dd_add(a, v);
        else
            a.hi += v;
    }
    __device__ void close(double n, const double (&S)[M], const double (&v)[M + NP]) {
#pragma unroll
        for (int s = 0; s < M; ++s) {
            add(am[s], S[s] + v[s]);
#pragma unroll
            for (int t = 0; t <= s; ++t) {
                const int q = s * (s + 1) / 2 + t;
                add(av[q], (n * v[M + q] - v[s] * v[t]) / (n - 1.));
            }
        }
    }
};

template <int M>
__global__ __launch_bounds__(kCovThreads) void cov_hcube_all_kernel(const uint32_t* off, uint32_t h0, uint32_t h1,
                                                                     uint32_t p0, uint32_t p1, const double* w,
                                                                     const double* f, int correlate, CovPlan pl,
                                                                     double* part, int32_t* status) {
    constexpr int NP = M * (M + 1) / 2;
    __shared__ double red[kCovWaves * 2 * (M + NP)];
    AllWork<M> wk;
    wk.w = w;
    wk.f = f;
    wk.eps = kEpsilon;
    wk.red = red;
#pragma unroll
    for (int s = 0; s < M; ++s) wk.am[s] = DD{0, 0};
#pragma unroll
    for (int q = 0; q < NP; ++q) wk.av[q] = DD{0, 0};
    cov_rounds(off, h0, h1, p0, p1, pl, status, wk);
    // workgroup partials: mean entries then pair entries, DD per wave
    const int wv = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < M + NP; ++k) {
        const DD r = wave_sum_dd(k < M ? wk.am[k] : wk.av[k - M]);
        if ((threadIdx.x & 63) == 0) {
            red[2 * ((size_t)wv * (M + NP) + k)] = r.hi;
            red[2 * ((size_t)wv * (M + NP) + k) + 1] = r.lo;
        }
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)(correlate ? NP : M)) {
        // output pair q (the layout of cov_hcube_kernel: npairs x blocks x 4)
        const int q = threadIdx.x;
        int s, t;
        cov_pair(q, correlate, s, t);
        const int kq = s * (s + 1) / 2 + t;
        DD m2{0, 0}, v2{0, 0};
        for (int k = 0; k < kCovWaves; ++k) {
            if (s == t) m2 = dd_sum(m2, DD{red[2 * ((size_t)k * (M + NP) + s)], red[2 * ((size_t)k * (M + NP) + s) + 1]});
            v2 = dd_sum(v2, DD{red[2 * ((size_t)k * (M + NP) + M + kq)], red[2 * ((size_t)k * (M + NP) + M + kq) + 1]});
        }
        double* o = part + 4 * ((size_t)q * gridDim.x + blockIdx.x);
        o[0] = m2.hi;
        o[1] = m2.lo;
        o[2] = v2.hi;
        o[3] = v2.lo;
    }
}

// acc: mean[m] then cov entries [npairs], each a DD (hi, lo) pair.  One
// workgroup per pair sums that pair's workgroup partials (thread k takes
// partials k, k + 256, ..., then a fixed tree) and adds them to acc.
__global__ __launch_bounds__(kCovThreads) void cov_reduce_kernel(const double* part, int nbx, int npairs, int m,
                                                                 int correlate, double* acc) {
    __shared__ double red[4 * (kCovThreads / 64)];
    const int q = blockIdx.x;
    int s, t;
    cov_pair(q, correlate, s, t);
    DD mm{0, 0}, vv{0, 0};
    for (int b = threadIdx.x; b < nbx; b += blockDim.x) {
        const double* p = part + 4 * ((size_t)q * nbx + b);
        mm = dd_sum(mm, DD{p[0], p[1]});
        vv = dd_sum(vv, DD{p[2], p[3]});
    }
    mm = wave_sum_dd(mm);
    vv = wave_sum_dd(vv);
    const int wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[4 * wv] = mm.hi;
        red[4 * wv + 1] = mm.lo;
        red[4 * wv + 2] = vv.hi;
        red[4 * wv + 3] = vv.lo;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    mm = DD{0, 0};
    vv = DD{0, 0};
    for (int k = 0; k < nw; ++k) {
        mm = dd_sum(mm, DD{red[4 * k], red[4 * k + 1]});
        vv = dd_sum(vv, DD{red[4 * k + 2], red[4 * k + 3]});
    }
    if (s == t) {
        const DD r = dd_sum(DD{acc[2 * s], acc[2 * s + 1]}, mm);
        acc[2 * s] = r.hi;
        acc[2 * s + 1] = r.lo;
    }
    double* cv = acc + 2 * m;
    const DD r = dd_sum(DD{cv[2 * q], cv[2 * q + 1]}, vv);
    cv[2 * q] = r.hi;
    cv[2 * q + 1] = r.lo;
}

}  // namespace vgx

using namespace vgx;

extern "C" int vgx_iter_accumulate_cov(vgx_ctx* ctx, const vgx_config* c, int64_t h0, int64_t h1, int64_t p0,
                                       int64_t p1, const double* f, const double* wgt, int m, int correlate,
                                       double* acc, int32_t* status, void* stream) {
    if (!ctx || !c || !f || !wgt || !acc || m < 1 || m > VGX_MAXCOMP) return VGX_EINVAL;
    if (h0 < 0 || h1 > c->nhcube || h0 >= h1 || p0 < 0 || p1 <= p0 || p1 > 0xFFFFFFFFll) return VGX_EINVAL;
    if (!ctx->off.ptr || ctx->off.bytes < (size_t)(h1 + 1) * sizeof(uint32_t)) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const int npairs = correlate ? m * (m + 1) / 2 : m;
    const int64_t nh = h1 - h0;
    const int64_t np = p1 - p0;
    const bool all = m <= kCovAllMax && (m <= 4 || (np > kCovPairPoints && nh > kCovPairHcubes));
    const int rows = all ? 1 : npairs;  // workgroups per block of hcubes
    int64_t blocks = std::min<int64_t>(kCovMaxBlocks, (nh + kCovThreads - 1) / kCovThreads);
    CovPlan pl{kCovLong, 0};
    if (np > nh * (int64_t)kCovShort && blocks * rows < ctx->info.cus) {
        blocks = std::min<int64_t>(nh, std::max<int64_t>(blocks, kCovFew / rows));
        pl = CovPlan{blocks == nh ? kCovAlone : kCovLong, 1};
    }
    const int nbx = (int)blocks;
    int rc;
    if ((rc = ctx->cov_part.ensure((size_t)npairs * nbx * 4 * sizeof(double)))) return rc;
    const uint32_t* off = (const uint32_t*)ctx->off.ptr;
    double* part = (double*)ctx->cov_part.ptr;
    // timed as one span: per-hcube sums and their reduction (events around both)
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const bool timed = timed_slot(ctx, kTimedCov, &e0, &e1);
    if (timed) VGX_HIP(hipEventRecord(e0, s));
    switch (all ? m : 0) {
        case 1: hipLaunchKernelGGL(cov_hcube_all_kernel<1>, dim3(nbx), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                                   (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, correlate, pl, part, status); break;
        case 2: hipLaunchKernelGGL(cov_hcube_all_kernel<2>, dim3(nbx), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                                   (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, correlate, pl, part, status); break;
        case 3: hipLaunchKernelGGL(cov_hcube_all_kernel<3>, dim3(nbx), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                                   (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, correlate, pl, part, status); break;
        case 4: hipLaunchKernelGGL(cov_hcube_all_kernel<4>, dim3(nbx), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                                   (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, correlate, pl, part, status); break;
        case 5: hipLaunchKernelGGL(cov_hcube_all_kernel<5>, dim3(nbx), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                                   (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, correlate, pl, part, status); break;
        case 6: hipLaunchKernelGGL(cov_hcube_all_kernel<6>, dim3(nbx), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                                   (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, correlate, pl, part, status); break;
        default:
            hipLaunchKernelGGL(cov_hcube_kernel, dim3(nbx, npairs), dim3(kCovThreads), 0, s, off, (uint32_t)h0,
                               (uint32_t)h1, (uint32_t)p0, (uint32_t)p1, wgt, f, m, correlate, pl, part, status);
    }
    hipLaunchKernelGGL(cov_reduce_kernel, dim3(npairs), dim3(kCovThreads), 0, s,
                       (const double*)ctx->cov_part.ptr, nbx, npairs, m, correlate, acc);
    if (timed) VGX_HIP(hipEventRecord(e1, s));
    return check_launch();
}
