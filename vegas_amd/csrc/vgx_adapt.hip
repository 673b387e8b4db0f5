// vgx_adapt.hip -- AdaptiveMap.adapt (src/vegas/_vegas.pyx:467-594) on device.
//
// Per axis: average the training data, smooth and compress it (alpha > 0),
// then invert the cumulative distribution onto new_ninc equal-weight
// increments.  Two implementations:
//   exact     one lane walks each axis with the reference's order of
//             operations (sequential sums, the while-loop CDF walk);
//   parallel  one 1024-lane workgroup per axis: tree reductions, an LDS
//             prefix sum and a binary search per new node.  Node i lands in
//             the first old increment j with prefix P_j >= i*F, exactly the
//             increment the sequential walk stops in (its running
//             accumulator equals P_j - i*F); only rounding differs.
#include "vgx_adapt.h"

namespace vgx {

// Fill the padding of one output row and nothing else.
__device__ inline void pad_row(double* ng, int nn, int new_ld) {
    for (int i = nn + 1; i < new_ld; ++i) ng[i] = ng[nn];
}

__device__ void adapt_axis_exact(const AdaptArgs& a, int d, double* avg, double* tmp, const double* g) {
    const int old = a.ninc[d], nn = a.new_ninc[d];
    double* ng = a.new_grid + (int64_t)d * a.new_ld;
    if (a.alpha != 0 && old > 1) {
        if (a.has_training) {
            for (int i = 0; i < old; ++i) {
                double nf = a.n_f[(int64_t)d * a.nb + i];
                avg[i] = nf > 0 ? a.sum_f[(int64_t)d * a.nb + i] / nf : 0.;
            }
        }
        if (a.alpha > 0) {
            tmp[0] = fabs(7. * avg[0] + avg[1]) / 8.;
            tmp[old - 1] = fabs(7. * avg[old - 1] + avg[old - 2]) / 8.;
            double s = tmp[0] + tmp[old - 1];
            for (int i = 1; i < old - 1; ++i) {
                tmp[i] = fabs(6. * avg[i] + avg[i - 1] + avg[i + 1]) / 8.;
                s += tmp[i];
            }
            if (s > 0) {
                for (int i = 0; i < old; ++i) avg[i] = tmp[i] / s + kTiny;
            } else {
                for (int i = 0; i < old; ++i) avg[i] = kTiny;
            }
            for (int i = 0; i < old; ++i)
                if (avg[i] > 0 && avg[i] <= 0.99999999)
                    avg[i] = pow(-(1 - avg[i]) / log(avg[i]), a.alpha);
        }
    }
    ng[0] = g[0];
    ng[nn] = g[old];
    double acc = 0., f_ninc = 0.;
    int j = -1;
    for (int i = 0; i < old; ++i) f_ninc += avg[i];
    f_ninc /= (double)nn;
    int i = 1;
    for (; i < nn; ++i) {
        bool stopped = false;
        while (acc < f_ninc) {
            j += 1;
            if (j < old) acc += avg[j];
            else { stopped = true; break; }
        }
        if (stopped) break;
        acc -= f_ninc;
        ng[i] = g[j + 1] - (acc / avg[j]) * (g[j + 1] - g[j]);
    }
    // The reference leaves nodes after an early stop unset (round-off only);
    // pin them to the upper limit.
    for (; i < nn; ++i) ng[i] = g[old];
    pad_row(ng, nn, a.new_ld);
}

__global__ void adapt_exact_kernel(AdaptArgs a) {
    if (a.status && *a.status) return;
    if (a.chain) {
        for (int d = 0; d < a.dim; ++d) source_row(a, d, blockDim.x);
        __syncthreads();
        if (threadIdx.x == 0) {
            double* avg = a.buf;
            double* tmp = a.buf + a.nb;
            for (int i = 0; i < a.nb; ++i) avg[i] = 1.0;
            for (int d = 0; d < a.dim; ++d)
                adapt_axis_exact(a, d, avg, tmp, a.old_rows ? a.old_rows + (int64_t)d * a.ld
                                                            : a.grid + (int64_t)d * a.ld);
        }
        __syncthreads();
        for (int d = 0; d < a.dim; ++d) clear_row(a, d, blockDim.x);
    } else {
        const int d = blockIdx.x;
        const double* g = source_row(a, d, blockDim.x);
        __syncthreads();
        if (threadIdx.x == 0) {
            double* avg = a.buf + (int64_t)d * 2 * a.nb;
            double* tmp = avg + a.nb;
            for (int i = 0; i < a.nb; ++i) avg[i] = 1.0;
            adapt_axis_exact(a, d, avg, tmp, g);
        }
        __syncthreads();
        clear_row(a, d, blockDim.x);
    }
}

// The exact adapt with one workgroup per axis and the axis in LDS: the same
// operations on the same values as adapt_axis_exact, so the same bits.
// What is independent per increment (averages, smoothing, the compression's
// log and pow, the new nodes' divisions) is spread over the threads; the
// reference's sequential sums and its CDF walk stay sequential, in one wave
// that reads the values from LDS 8 ahead (sums) or keeps 64 of them in its
// lanes (walk, one branch-free step per addition).  The chain of dependent
// operations bounds it.  5 axes of 400 increments: 732 us with one lane doing
// everything from global memory, 108 us so with a branching walk, 48 us with
// the walk branch-free (14 instructions a step).
constexpr int kExactThreads = 256;
constexpr int kExactLds = 60 * 1024;  // bytes: av[old], tmp/acc[max(old, nn)], jj[nn]
inline size_t exact_lds_bytes(int old, int nn) {
    return (size_t)old * 8 + (size_t)(old > nn ? old : nn) * 8 + (size_t)nn * 4;
}

// s + v[0] + v[1] + ... in order (every lane of the calling wave alike).
__device__ inline double seq_sum(double s, const double* v, int n) {
    int i = 0;
    for (; i + 8 <= n; i += 8) {
        double t[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) t[k] = v[i + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) s += t[k];
    }
    for (; i < n; ++i) s += v[i];
    return s;
}

__device__ inline double read_lane(double v, int l) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

__global__ __launch_bounds__(kExactThreads) void adapt_exact_lds_kernel(AdaptArgs a) {
    extern __shared__ double el[];
    __shared__ double s_sum;
    __shared__ int s_last;  // nodes 1..s_last-1 were placed by the walk
    if (a.status && *a.status) return;
    const int d = blockIdx.x, T = kExactThreads;
    const int old = a.ninc[d], nn = a.new_ninc[d];
    double* av = el;
    double* tmp = el + old;  // smoothed values, then the walk's accumulator per node
    int* jj = reinterpret_cast<int*>(tmp + (old > nn ? old : nn));
    double* ng = a.new_grid + (int64_t)d * a.new_ld;
    const double* g = source_row(a, d, T);
    const bool wave0 = threadIdx.x < 64;
    for (int i = threadIdx.x; i < old; i += T) {
        double v = 1.0;
        if (a.alpha != 0 && old > 1 && a.has_training) {
            const double nf = a.n_f[(int64_t)d * a.nb + i];
            v = nf > 0 ? a.sum_f[(int64_t)d * a.nb + i] / nf : 0.;
        }
        av[i] = v;
    }
    __syncthreads();
    if (a.alpha > 0 && old > 1) {
        for (int i = threadIdx.x; i < old; i += T) {
            double t;
            if (i == 0) t = fabs(7. * av[0] + av[1]) / 8.;
            else if (i == old - 1) t = fabs(7. * av[old - 1] + av[old - 2]) / 8.;
            else t = fabs(6. * av[i] + av[i - 1] + av[i + 1]) / 8.;
            tmp[i] = t;
        }
        __syncthreads();
        if (wave0) {
            const double s = seq_sum(tmp[0] + tmp[old - 1], tmp + 1, old - 2);
            if (threadIdx.x == 0) s_sum = s;
        }
        __syncthreads();
        const double s = s_sum;
        for (int i = threadIdx.x; i < old; i += T) {
            double v = s > 0 ? tmp[i] / s + kTiny : kTiny;
            if (v > 0 && v <= 0.99999999) v = pow(-(1 - v) / log(v), a.alpha);
            av[i] = v;
        }
        __syncthreads();
    }
    if (wave0) {
        const int lane = threadIdx.x;
        const double f = read_lane(seq_sum(0., av, old) / (double)nn, 0);
        // The walk, one addition a step: the next increment's weight while
        // acc < f, else -f for a node placed (i and j are scalars, and
        // acc + (-f) is acc - f).  In a window of kWalk steps lane l holds
        // increment j0 + 1 + l, and collects the accumulator and increment of
        // node i0 + l: every step writes the node it may have placed, a step
        // that placed none is overwritten by the one that does.
        constexpr int kWalk = 32;
        int j = -1, i = 1;
        double acc = 0.;
        bool walking = true;
        while (walking) {
            const int j0 = j, i0 = i;
            const double cur = j0 + 1 + lane < old ? av[j0 + 1 + lane] : 0.0;
            double rec = 0.0;
            int recj = 0, taken = 0;
            // step s of the window: after it i - i0 = s + 1 - taken
            auto step = [&](int s) {
                const double next = read_lane(cur, taken);
                const bool take = acc < f;
                acc += take ? next : -f;
                const bool mine = lane == s - taken;  // the node being placed
                rec = mine ? acc : rec;
                recj = mine ? s : recj;  // its increment is j0 + s - (i - i0)
                taken += (int)(__ballot(take) & 1);
            };
            int steps = 0;
            if (i0 + kWalk <= nn && j0 + kWalk < old) {
#pragma unroll
                for (int s = 0; s < kWalk; ++s) step(s);
                steps = kWalk;
            } else {
                for (; steps < kWalk; ++steps) {
                    if (i0 + steps - taken >= nn || (j0 + taken + 1 >= old && (__ballot(acc < f) & 1))) {
                        walking = false;
                        break;
                    }
                    step(steps);
                }
            }
            j = j0 + taken;
            i = i0 + steps - taken;
            if (lane < i - i0) {
                tmp[i0 + lane] = rec;
                jj[i0 + lane] = j0 + recj - lane;
            }
        }
        if (lane == 0) s_last = i;
    }
    __syncthreads();
    // node i from the increment the walk stopped in; nodes after an early
    // stop (round-off only) at the upper limit, as adapt_axis_exact
    const int last = s_last;
    const double glo = g[0], ghi = g[old];
    for (int i = 1 + threadIdx.x; i < nn; i += T) {
        double xv = ghi;
        if (i < last) {
            const int j = jj[i];  // -1 only when the weights sum to 0 or NaN
            xv = j >= 0 ? g[j + 1] - (tmp[i] / av[j]) * (g[j + 1] - g[j]) : glo - 0.0 * tmp[i];
        }
        ng[i] = xv;
    }
    if (threadIdx.x == 0) ng[0] = glo;
    for (int i = nn + (int)threadIdx.x; i < a.new_ld; i += T) ng[i] = ghi;
    clear_row(a, d, T);
}

// The exact adapt of every axis on stream st: by adapt_exact_lds_kernel
// where each axis fits its LDS (up to 3072 increments to as many: the bins
// and nodes of one axis in 60 KiB), else, or when the axes are chained
// (pyx:534), by one lane per axis.
static void launch_adapt_exact(const AdaptArgs& a, hipStream_t st) {
    size_t need = 0;
    for (int d = 0; d < a.dim; ++d) {
        const size_t b = exact_lds_bytes(a.ninc[d], a.new_ninc[d]);
        need = b > need ? b : need;
    }
    if (!a.chain && need <= (size_t)kExactLds)
        hipLaunchKernelGGL(adapt_exact_lds_kernel, dim3(a.dim), dim3(kExactThreads), need, st, a);
    else
        hipLaunchKernelGGL(adapt_exact_kernel, dim3(a.chain ? 1 : a.dim), dim3(64), 0, st, a);
}

__global__ __launch_bounds__(1024) void adapt_parallel_kernel(AdaptArgs a) {
    __shared__ double av[kAdaptLdsMax];
    __shared__ double P[kAdaptLdsMax];
    __shared__ double red[40];
    if (a.status && *a.status) return;
    adapt_parallel_axis(a, blockIdx.x, av, P, red);
}

// The integrator's adapt: in place on `grid`, skipped when *status != 0.
// The training data are left as they are (the next iteration's allocation
// kernel clears them).
int adapt_in_place_setup(vgx_ctx* ctx, int dim, const int32_t* ninc, double* grid, int ld, double* sum_f,
                         double* n_f, int has_training, double alpha, int exact, const int32_t* status,
                         AdaptArgs* out, int* parallel) {
    AdaptArgs& a = *out;
    a = AdaptArgs{};
    a.dim = dim;
    a.ld = ld;
    a.nb = ld - 1;
    a.new_ld = ld;
    a.has_training = has_training;
    a.alpha = alpha;
    a.grid = grid;
    a.sum_f = sum_f;
    a.n_f = n_f;
    a.new_grid = grid;
    a.status = status;
    a.clear_sum_f = nullptr;
    a.clear_n_f = nullptr;
    int max_old = 0;
    for (int d = 0; d < dim; ++d) {
        a.ninc[d] = ninc[d];
        a.new_ninc[d] = ninc[d];
        max_old = ninc[d] > max_old ? ninc[d] : max_old;
    }
    a.chain = (!has_training && alpha > 0) ? 1 : 0;
    if (!exact && max_old > kAdaptLdsMax) exact = 1;
    size_t rows = (size_t)dim * ld;
    size_t bufs = (size_t)(a.chain ? 1 : dim) * 2 * (size_t)a.nb;
    int rc = ctx->adapt_tmp.ensure((rows + bufs) * sizeof(double));
    if (rc) return rc;
    a.old_rows = (double*)ctx->adapt_tmp.ptr;
    a.buf = a.old_rows + rows;
    *parallel = !(exact || a.chain);
    return VGX_OK;
}

int adapt_in_place(vgx_ctx* ctx, int dim, const int32_t* ninc, double* grid, int ld, double* sum_f,
                   double* n_f, int has_training, double alpha, int exact, const int32_t* status,
                   hipStream_t st) {
    AdaptArgs a;
    int parallel = 0;
    int rc = adapt_in_place_setup(ctx, dim, ninc, grid, ld, sum_f, n_f, has_training, alpha, exact, status,
                                  &a, &parallel);
    if (rc) return rc;
    if (parallel)
        hipLaunchKernelGGL(adapt_parallel_kernel, dim3(dim), dim3(1024), 0, st, a);
    else
        launch_adapt_exact(a, st);
    return check_launch();
}

}  // namespace vgx

using namespace vgx;

extern "C" int vgx_adapt(vgx_ctx* ctx, int dim, const int32_t* ninc, const double* grid, int ld,
                         int has_training, const double* sum_f, const double* n_f, double alpha,
                         const int32_t* new_ninc, double* new_grid, int new_ld, int exact,
                         void* stream) {
    if (dim < 1 || dim > VGX_MAXDIM || !ninc || !new_ninc || !grid || !new_grid) return VGX_EINVAL;
    if (grid == new_grid) return VGX_EINVAL;
    if (has_training && (!sum_f || !n_f)) return VGX_EINVAL;
    AdaptArgs a{};
    a.dim = dim;
    a.ld = ld;
    a.nb = ld - 1;
    a.new_ld = new_ld;
    a.has_training = has_training;
    a.alpha = alpha;
    a.grid = grid;
    a.sum_f = sum_f;
    a.n_f = n_f;
    a.new_grid = new_grid;
    int max_new = 0, min_new = 1 << 30, max_old = 0;
    for (int d = 0; d < dim; ++d) {
        if (ninc[d] < 1 || ninc[d] + 1 > ld) return VGX_EINVAL;
        a.ninc[d] = ninc[d];
        a.new_ninc[d] = new_ninc[d];
        max_new = new_ninc[d] > max_new ? new_ninc[d] : max_new;
        min_new = new_ninc[d] < min_new ? new_ninc[d] : min_new;
        max_old = ninc[d] > max_old ? ninc[d] : max_old;
    }
    if (min_new < 1) return VGX_EINVAL;
    if (max_new + 1 > new_ld) return VGX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    // pyx:519-530: every axis collapses to its end points
    if (max_new == 1) {
        a.alpha = 0.0;  // the CDF walk with one increment writes only the ends
        exact = 1;
    }
    // pyx:534: with alpha > 0 and no training data the shared buffer carries
    // one axis' smoothed weights into the next; only the chained walk
    // reproduces that, and only when axes differ in ninc does it matter.
    a.chain = (!has_training && alpha > 0) ? 1 : 0;
    if (!exact && max_old > kAdaptLdsMax) exact = 1;
    if (exact || a.chain) {
        if (!ctx) return VGX_EINVAL;
        size_t need = (size_t)(a.chain ? 1 : dim) * 2 * (size_t)a.nb * sizeof(double);
        int rc = ctx->adapt_tmp.ensure(need);
        if (rc) return rc;
        a.buf = (double*)ctx->adapt_tmp.ptr;
        launch_adapt_exact(a, st);
    } else {
        hipLaunchKernelGGL(adapt_parallel_kernel, dim3(dim), dim3(1024), 0, st, a);
    }
    return check_launch();
}
