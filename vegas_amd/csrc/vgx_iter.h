// vgx_iter.h -- shared definitions of the vegas+ iteration kernels.
#pragma once
#include <type_traits>

#include "vgx_internal.h"

namespace vgx {

constexpr int kK = 4;               // points per lane in a wave tile
constexpr int kT = 64 * kK;         // points per wave tile
constexpr int kNoff = kT / 2 + 4;   // offsets slice: hcubes touching a tile (+1 end, +pad)
constexpr int kFusedThreads = 1024; // 16 waves per workgroup, one workgroup per CU
constexpr int kAllocThreads = 256;
constexpr int kAllocItems = 8;
constexpr int kAllocPerBlock = kAllocThreads * kAllocItems;
constexpr uint32_t kCntFlushTiles = 224; // u16 LDS counts: (224 + 15) tiles x 256 < 65536
constexpr int kStradThreads = 256;  // straddler kernel: one lane per tile slot
constexpr int kLaneParts = 8;       // cut hcubes of up to this many tiles: one lane; more: the wave
constexpr int kKeySentinel = 0x7fff;

// Register-array bound of a dimension template argument: DIM > 0 is exact;
// DIM <= 0 is a runtime dimension of at most -DIM (all 64 for DIM = 0).
__host__ __device__ constexpr int nd_max(int DIM) { return DIM > 0 ? DIM : (DIM < 0 ? -DIM : VGX_MAXDIM); }

// Kernel-argument copy of the iteration geometry (Integrator.set, pyx:1331-1446).
struct IterGeom {
    int dim, ld, nb;
    int adaptive_sampler;  // beta > 0 && nhcube > 1 && !adapt_to_errors  (pyx:1675)
    int adaptive_strat;    // ... && adapt                              (pyx:2052-2055)
    int train_points;      // !adapt_to_errors && adapt && alpha > 0      (pyx:2196)
    int train_errors;      // adapt_to_errors && adapt                    (pyx:2187)
    int rng32;             // 24-bit uniforms (FP32 integrand) else 53-bit
    int exact_div;         // y = (c+u)/s by IEEE division
    int hist_lds, grid_lds;
    int split;             // few tiles: split_kernel instead of fused_kernel
    int hist_unordered;    // hist_lds: LDS atomics in timing order (VGX_FLAG_UNORDERED_HIST)
    int weighted;
    int adapt;
    int fast_pow;          // sigf = |var|^(beta/2) in the sampler, FP32 log2/exp2
                           // (else FP64 pow in a separate pass)
    int per_all;           // rng32, no exact division, and ninc a multiple of
                           // nstrat on every axis: the integer stratum->bin path
    int32_t ninc[VGX_MAXDIM];
    int32_t nstrat[VGX_MAXDIM];
    double inv_nstrat[VGX_MAXDIM];
    DivMagic dm[VGX_MAXDIM];
    int64_t nhcube;
    double neval;
    double neval_frac;
    double beta_half;
    double beta;
    double dv_y;
    double jn;             // product over the axes of (double)ninc
    int32_t nmin, nmax, avg_nh, pad2;
    uint32_t seed_lo, seed_hi;
    uint32_t iteration;  // RNG stream of this iteration
    uint32_t itn;        // index within the run
    uint32_t nitn;
    uint32_t pad3;
    const double* uext;  // caller's uniforms [total][dim] (53-bit path), or null: Philox
};

// Device-resident scalars of one run.
struct Scalars {
    uint32_t total;       // points this iteration (off[nhcube])
    uint32_t overflow;
    int32_t nh_min, nh_max;
    // current batch (whole iteration for device integrands)
    uint32_t b_p0, b_p1, b_h0, b_h1, b_ntiles, pad0;
    double acc[6];          // iteration sums (DD): mean, var, sum_sigf
    int32_t status;         // 0 or VGX_ENAN
    int32_t reset_sigf;
    double pad1[2];
};

// The part of an hcube cut by a tile edge that lies in one tile: its point
// count and its two-pass sums about the part's own mean S/n (the straddler
// kernel combines the parts exactly, Chan-Golub-LeVeque style).
struct Slot {
    int32_t h;      // hcube, or -1
    uint32_t n;     // points of h in this tile
    double S;       // sum of w f over them
    double Q;       // sum of guarded (w f - S/n)^2
    double D;       // sum of guarded (w f - S/n)
};

struct AxisC;
struct FusedPtrs {
    const AxisC* axes;  // dim per-axis sampler constants (device)
    const double* grid;
    const uint32_t* off;
    const int32_t* tile_h;
    double* sigf;
    Slot* slots;        // [2 * tile]: part of the hcube cut by the tile's start / end
    double* tile_part;  // [tile][3]: the tile's sums (mean, variance, sigf), summed in tile order
    double* blk_part;   // [gridDim.x][6]
    double* sum_f;
    double* n_f;
    double* hpart_s;    // LDS histogram (fast mode): [gridDim.x][dim * nb] sums and counts
    uint32_t* hpart_c;  //   of each workgroup, summed in workgroup order after the launch
    uint32_t* rec_bins; // training records, one per point of the batch (index i = point
    double* rec_c2;     //   index - b_p0): the bins of axes 2k, 2k+1 as the u16 halves of
                        //   rec_bins[k * rec_stride + i] (kNoBin where the point is not
                        //   trained on the axis, pyx:459-463), (w f n)^2 (pyx:2173) at rec_c2[i]
    uint32_t rec_stride; // a multiple of the tile size (whole tiles per row)
    double* errv;       // adapt_to_errors: |variance| per hcube
    Scalars* sc;
};

// ---------------------------------------------------------------------------
// Integrands (device functors).  eval() receives x in FP64 and returns f in
// FP64; the arithmetic precision is the functor's.

// Reads a parameter that no kernel writes while the integrand runs, through
// the constant address space: at a wave-uniform index (the component loop)
// this is a scalar load into SGPRs rather than a vector load with its full
// memory latency per component.
template <class T>
__device__ __forceinline__ T ldc(const T* p, int i) {
    return ((const __attribute__((address_space(4))) T*)p)[i];
}

// f(x) = sum_k A_k exp(-B_k |x - c_k|^2)
struct GaussMix64 {
    static constexpr bool kRng32 = false;
    int ncomp;
    const double* A;
    const double* B;
    const double* c;
    template <int DIM, bool FEW>
    __device__ double eval(const double* x, int dim, uint32_t) const {
        const int nd = DIM > 0 ? DIM : dim;
        double acc = 0.0;
        for (int k = 0; k < ncomp; ++k) {
            double r2 = 0.0;
#pragma unroll
            for (int d = 0; d < nd_max(DIM); ++d) {
                if (DIM <= 0 && d >= nd) break;
                double t = x[d] - ldc(c, k * nd + d);
                r2 += t * t;
            }
            acc += ldc(A, k) * exp(-ldc(B, k) * r2);
        }
        return acc;
    }
};

// A * 2^y for y <= 0 in FP32 arithmetic with the FP64 exponent range: y = n + f
// (n = floor(y), f in [0,1), an exact split), A * 2^f by the FP32 hardware
// exp2, and the scaling by 2^n exact in FP64.  FP32 exp flushes e^-104 and
// below to 0; here a point far from a narrow peak keeps its tiny value (down
// to 2^-1074) as the reference's FP64 evaluation does -- the training signal
// that leads the map to the peak in the first iterations.  NaN propagates.
__device__ __forceinline__ double scaled_exp2(float A, float y) {
    y = y < -1100.0f ? -1100.0f : y;  // 2^-1100 is 0 in FP64 as well
    const float fl = floorf(y);
    return ldexp((double)(A * __builtin_amdgcn_exp2f(y - fl)), (int)fl);
}

// An integrand's eval: FEW where the sampler has fewer than 16 waves.
// STEPS: four components at a time there, their constants loaded first (one
// wait for scalar loads instead of one per component): 16 waves cover those
// waits, and a short mixture pays for the registers (8 axes, two components:
// 1-2 % of its launch).
// 1e7 points, 250 components of 10 axes, two iterations: 4155 us one by one
// (3523 with 16 waves, which spilled), 3297 so; two or three at a time 3469,
// 3409.  (FP64 two at a time: short mixtures of 12 and 13 axes lose 10 %.  7
// axes with 12 waves: short ones lose 10-15 %, 8 axes 0-3 %, more axes none.)
template <bool STEPS>
struct GaussMix32T {
    static constexpr bool kRng32 = true;
    int ncomp;
    const float* A;
    const float* B;
    const float* c;
    template <int DIM, bool FEW>
    __device__ double eval(const double* x, int dim, uint32_t) const {
        const int nd = DIM > 0 ? DIM : dim;
        float xf[nd_max(DIM)];
#pragma unroll
        for (int d = 0; d < nd_max(DIM); ++d) {
            if (DIM <= 0 && d >= nd) break;
            xf[d] = (float)x[d];
        }
        // the components' values, each with the FP64 exponent range, summed in
        // FP64 in component order
        double acc = 0.0;
        int k = 0;
        if constexpr (STEPS && FEW && DIM >= 8) {
            constexpr int kStep = 4;
            for (; k + kStep <= ncomp; k += kStep) {
                float cc[kStep][DIM], aa[kStep], bb[kStep];
#pragma unroll
                for (int i = 0; i < kStep; ++i) {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) cc[i][d] = ldc(c, (k + i) * DIM + d);
                    aa[i] = ldc(A, k + i);
                    bb[i] = ldc(B, k + i);
                }
#pragma unroll
                for (int i = 0; i < kStep; ++i) {
                    float r2 = 0.0f;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const float t = xf[d] - cc[i][d];
                        r2 = __builtin_fmaf(t, t, r2);
                    }
                    acc += scaled_exp2(aa[i], (-bb[i] * r2) * 1.44269504088896341f);
                }
            }
        }
        for (; k < ncomp; ++k) {
            float r2 = 0.0f;
#pragma unroll
            for (int d = 0; d < nd_max(DIM); ++d) {
                if (DIM <= 0 && d >= nd) break;
                float t = xf[d] - ldc(c, k * nd + d);
                r2 = __builtin_fmaf(t, t, r2);
            }
            acc += scaled_exp2(ldc(A, k), (-ldc(B, k) * r2) * 1.44269504088896341f);
        }
        return acc;
    }
};
using GaussMix32 = GaussMix32T<true>;
using GaussOne32 = GaussMix32T<false>;  // the batched sampler's (16 waves for every dimension)

// GaussMix32 for long mixtures (many_pays below): the same operations in the
// same order, so the same bits, but two components at a time, and a pair whose
// terms are all below 2^-56 of the sum on every lane of the wave is not added:
// each would round away (its exponential, scaling and FP64 addition cost as
// much as its distance), and the constants' scalar loads are waited for once
// a pair.  VALU bound.  8 axes, 1000 components on a diagonal, 1.8e7 points:
// 11.3 -> 8.2 ms.  (Four at a time, or eight: slower, their registers cost
// waves in flight.)
struct GaussMany32 {
    static constexpr bool kRng32 = true;
    int ncomp;
    const float* A;
    const float* B;
    const float* c;
    const float* ea;  // [1]: an integer, every A[k] < 2^ea (max_exponent_kernel)
    template <int DIM, bool FEW>
    __device__ double eval(const double* x, int dim, uint32_t) const {
        const int nd = DIM > 0 ? DIM : dim;
        float xf[nd_max(DIM)];
#pragma unroll
        for (int d = 0; d < nd_max(DIM); ++d) {
            if (DIM <= 0 && d >= nd) break;
            xf[d] = (float)x[d];
        }
        const float e0 = ldc(ea, 0) + (1023.0f + 56.0f);
        double acc = 0.0;
        // A term A 2^y with y < skip is below 2^-56 of acc (a quarter of the
        // spacing of doubles just below a power of two); acc = 0 counts as
        // 2^-1023, beside which such a term is 0 itself.  ea is infinite, and
        // nothing skipped, unless every A is finite and none negative: then
        // acc only grows, and an older skip is merely lower.
        float skip = -INFINITY;
        auto pair = [&](int k) {
            float aa[2], y[2];
            bool add = false;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float r2 = 0.0f;
#pragma unroll
                for (int d = 0; d < nd_max(DIM); ++d) {
                    if (DIM <= 0 && d >= nd) break;
                    const float t = xf[d] - ldc(c, (k + i) * nd + d);
                    r2 = __builtin_fmaf(t, t, r2);
                }
                aa[i] = ldc(A, k + i);
                y[i] = (-ldc(B, k + i) * r2) * 1.44269504088896341f;
                add |= !(y[i] < skip);  // (a NaN is added)
            }
            if (!__any(add)) return;
#pragma unroll
            for (int i = 0; i < 2; ++i) acc += scaled_exp2(aa[i], y[i]);
        };
        int k = 0;
        for (; k + 4 <= ncomp; k += 4) {
            pair(k);
            pair(k + 2);
            const uint32_t hi = (uint32_t)((uint64_t)__double_as_longlong(acc) >> 32);
            skip = (float)((hi >> 20) & 0x7FFu) - e0;
        }
        for (; k < ncomp; ++k) {
            float r2 = 0.0f;
#pragma unroll
            for (int d = 0; d < nd_max(DIM); ++d) {
                if (DIM <= 0 && d >= nd) break;
                const float t = xf[d] - ldc(c, k * nd + d);
                r2 = __builtin_fmaf(t, t, r2);
            }
            acc += scaled_exp2(ldc(A, k), (-ldc(B, k) * r2) * 1.44269504088896341f);
        }
        return acc;
    }
};

// Where GaussMany32 takes GaussMix32's place (one pair against the other, 256
// to 1000 components, FP32 samples): with 5 to 9 axes and 4.2e6 or 8e6 points
// it is 1.00-1.11 times as fast where every term counts (sigma 0.2) and
// 1.05-1.18 where few do (0.02).  Where GaussMix32 takes four at a time itself
// (few waves: from 10 axes on, from 8 off the integer strata) that is faster.
// With 4 axes wide mixtures lose 2-5 %, with 1.2e6 points (few tiles to a wave)
// up to 11 %; a short mixture loses its whole kernel 1-2 % (two components, 8
// axes, 9.8e6 points: 259 -> 261-265 us).
inline bool many_pays(int ncomp, int dim, int64_t neval, bool per) {
    return ncomp >= 256 && dim >= 5 && dim <= (per ? 9 : 7) && neval >= (1 << 22);
}

// Mixture with centres t_k (1,...,1): |x - c_k|^2 = P + dim (xbar - t_k)^2,
// P = sum_d (x_d - xbar)^2 (exact algebra, no cancellation).
struct DiagRidge32 {
    static constexpr bool kRng32 = true;
    int ncomp;
    const float* A;
    const float* B;
    const float* c;  // t_k
    template <int DIM, bool FEW>
    __device__ double eval(const double* x, int dim, uint32_t) const {
        const int nd = DIM > 0 ? DIM : dim;
        float xf[nd_max(DIM)];
        float s = 0.0f;
#pragma unroll
        for (int d = 0; d < nd_max(DIM); ++d) {
            if (DIM <= 0 && d >= nd) break;
            xf[d] = (float)x[d];
            s += xf[d];
        }
        const float xbar = s / (float)nd;
        float P = 0.0f;
#pragma unroll
        for (int d = 0; d < nd_max(DIM); ++d) {
            if (DIM <= 0 && d >= nd) break;
            float t = xf[d] - xbar;
            P = __builtin_fmaf(t, t, P);
        }
        const float fd = (float)nd;
        float acc = 0.0f;
        // eight components per step with their constants loaded first (wide
        // scalar loads, one wait instead of two per component); the sum runs
        // in component order as in the remainder loop.  Sixteen, then eight, on
        // 10 to 12 axes, where the sampler has 12 waves (4e6 points, 1000
        // components of 11 axes: 1900 us with eight, 1684; with 16 waves, which
        // spilled, 1716).
        int k = 0;
        auto step = [&](auto n) {
            constexpr int kStep = decltype(n)::value;
            float cc[kStep], aa[kStep], bb[kStep];
#pragma unroll
            for (int i = 0; i < kStep; ++i) {
                cc[i] = ldc(c, k + i);
                aa[i] = ldc(A, k + i);
                bb[i] = ldc(B, k + i);
            }
#pragma unroll
            for (int i = 0; i < kStep; ++i) {
                float t = xbar - cc[i];
                float r2 = __builtin_fmaf(fd * t, t, P);
                acc = __builtin_fmaf(aa[i], __expf(-bb[i] * r2), acc);
            }
            k += kStep;
        };
        if constexpr (DIM >= 10 && DIM <= 12)
            while (k + 16 <= ncomp) step(std::integral_constant<int, 16>{});
        while (k + 8 <= ncomp) step(std::integral_constant<int, 8>{});
        for (; k < ncomp; ++k) {
            float t = xbar - ldc(c, k);
            float r2 = __builtin_fmaf(fd * t, t, P);
            acc = __builtin_fmaf(ldc(A, k), __expf(-ldc(B, k) * r2), acc);
        }
        return (double)acc;
    }
};

struct DiagRidge64 {
    static constexpr bool kRng32 = false;
    int ncomp;
    const double* A;
    const double* B;
    const double* c;
    template <int DIM, bool FEW>
    __device__ double eval(const double* x, int dim, uint32_t) const {
        const int nd = DIM > 0 ? DIM : dim;
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < nd_max(DIM); ++d) {
            if (DIM <= 0 && d >= nd) break;
            s += x[d];
        }
        const double xbar = s / (double)nd;
        double P = 0.0;
#pragma unroll
        for (int d = 0; d < nd_max(DIM); ++d) {
            if (DIM <= 0 && d >= nd) break;
            double t = x[d] - xbar;
            P += t * t;
        }
        double acc = 0.0;
        for (int k = 0; k < ncomp; ++k) {
            double t = xbar - ldc(c, k);
            acc += ldc(A, k) * exp(-ldc(B, k) * (P + (double)nd * t * t));
        }
        return acc;
    }
};

// f supplied by the caller for global point p (host-driven integrands).
template <bool R32>
struct BufferFcn {
    static constexpr bool kRng32 = R32;
    const double* f;
    int64_t base;
    template <int DIM, bool FEW>
    __device__ double eval(const double*, int, uint32_t p) const {
        return f[(int64_t)p - base];
    }
};

// AdaptiveMap.adapt for the integrator loop (vgx_adapt.hip): in place, a
// no-op once *status != 0, clears sum_f/n_f after reading them.
int adapt_in_place(vgx_ctx* ctx, int dim, const int32_t* ninc, double* grid, int ld, double* sum_f,
                   double* n_f, int has_training, double alpha, int exact, const int32_t* status,
                   hipStream_t st);
// Its set-up alone: fills *args and sets *parallel when the workgroup-per-
// axis kernel applies (the caller then runs adapt_parallel_axis itself).
struct AdaptArgs;
int adapt_in_place_setup(vgx_ctx* ctx, int dim, const int32_t* ninc, double* grid, int ld, double* sum_f,
                         double* n_f, int has_training, double alpha, int exact, const int32_t* status,
                         AdaptArgs* args, int* parallel);

// Launchers, one per (integrand, dim) instantiation (vgx_fused_*.hip).
// ev0/ev1 (may be null): events that take the launch's own start and end
// timestamps (hipExtLaunchKernel), so timing adds no packets to the stream.
template <class Fcn>
int launch_fused(const IterGeom& g, const FusedPtrs& io, const Fcn& fcn, int grid_blocks,
                 size_t lds, hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);

}  // namespace vgx
