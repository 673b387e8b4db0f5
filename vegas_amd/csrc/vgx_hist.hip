// vgx_hist.hip -- AdaptiveMap.add_training_data (src/vegas/_vegas.pyx:421-464).
//
// Fast mode: each workgroup privatises the (dim x ninc) histogram in LDS
// (FP64 sums via ds_add_f64, u32 counts), then flushes it with one global
// FP64 atomic per touched bin.  Counts are exact; sums equal the
// reference's up to the order of additions.
//
// Ordered mode: bit-for-bit the reference's sequential loop.  A stable
// counting sort groups |f| by (axis, bin) keeping point order, then one lane
// per bin adds the group in point order onto the existing sum:
//   1 hist_count    per-tile, per-bin counts (LDS)
//   2 hist_scan     exclusive scan over tiles per bin; hist_start over bins
//   3 hist_scatter  one wave per (tile, axis); stable ranks from ballots
//   4 hist_sum      sequential per-bin sums in point order
#include <algorithm>
#include <mutex>

#include "vgx_internal.h"

namespace vgx {

constexpr int kHistTile = 1024;  // points per tile (ordered mode)

struct HistArgs {
    int dim;
    int nb;  // ld - 1: row stride of sum_f / n_f
    int use_lds;
    int ntiles;
    int32_t ninc[VGX_MAXDIM];
    const double* y;
    const double* f;
    int64_t n;
    double* sum_f;
    double* n_f;
    uint32_t* cnt;     // ordered: dim x ntiles x nb
    uint32_t* start;   // ordered: dim x nb bin starts
    uint32_t* total;   // ordered: dim x nb bin totals
    double* sorted;    // ordered: dim x n
    // training records of the fused sampler instead of y and f: the bin of
    // point i on axis d in the (d & 1) half of rbins[(d >> 1) * rstride + i],
    // the values in f, the point count read on the device as nrange[1] -
    // nrange[0] (n is then the capacity)
    const uint32_t* rbins;
    int64_t rstride;
    const uint32_t* nrange;
};

__device__ inline int64_t npoints(const HistArgs& a) {
    return a.nrange ? (int64_t)(a.nrange[1] - a.nrange[0]) : a.n;
}

// Bin of y for axis d, or -1 when y is not strictly inside (0, 1).
__device__ inline int train_bin(double yv, int ni) {
    if (!(yv > 0 && yv < 1)) return -1;
    int k = (int)floor(yv * (double)ni);
    // y*ninc can round up to ninc for y within an ulp of 1; the reference
    // would then write one slot past the row.  Keep it in the last bin.
    return k < ni ? k : ni - 1;
}

// Bin of point i on axis d: from its record, or from y (pyx:459-463).
__device__ inline int point_bin(const HistArgs& a, int64_t i, int d, int ni) {
    if (a.rbins) {
        const uint32_t b = (a.rbins[(d >> 1) * a.rstride + i] >> (16 * (d & 1))) & 0xFFFFu;
        return (b == kNoBin || (int)b >= ni) ? -1 : (int)b;  // (a bin >= ninc is never written)
    }
    return train_bin(a.y[i * a.dim + d], ni);
}

__global__ __launch_bounds__(256) void hist_fast_kernel(HistArgs a) {
    extern __shared__ double lds[];
    double* s = lds;
    uint32_t* c = reinterpret_cast<uint32_t*>(lds + (a.use_lds ? a.dim * a.nb : 0));
    const int tot = a.dim * a.nb;
    if (a.use_lds) {
        for (int i = threadIdx.x; i < tot; i += blockDim.x) {
            s[i] = 0.0;
            c[i] = 0u;
        }
        __syncthreads();
    }
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const double fa = fabs(a.f[i]);
        for (int d = 0; d < a.dim; ++d) {
            int k = train_bin(a.y[i * a.dim + d], a.ninc[d]);
            if (k < 0) continue;
            if (a.use_lds) {
                unsafeAtomicAdd(&s[d * a.nb + k], fa);
                atomicAdd(&c[d * a.nb + k], 1u);
            } else {
                unsafeAtomicAdd(&a.sum_f[d * a.nb + k], fa);
                unsafeAtomicAdd(&a.n_f[d * a.nb + k], 1.0);
            }
        }
    }
    if (!a.use_lds) return;
    __syncthreads();
    for (int i = threadIdx.x; i < tot; i += blockDim.x) {
        if (c[i]) {
            unsafeAtomicAdd(&a.sum_f[i], s[i]);
            unsafeAtomicAdd(&a.n_f[i], (double)c[i]);
        }
    }
}

// ---- ordered mode ---------------------------------------------------------
constexpr size_t kCountLds = 32 * 1024;  // bytes of LDS counts of one hist_count workgroup

// One workgroup per tile and group of axes (as many as have LDS counts in
// kCountLds): the workgroups of a tile read its rows of y once per group.
__global__ __launch_bounds__(256) void hist_count_kernel(HistArgs a, int daxes) {
    extern __shared__ uint32_t cl[];
    const int tile = blockIdx.x, d0 = blockIdx.y * daxes;
    const int nd = min(daxes, a.dim - d0);
    for (int k = threadIdx.x; k < nd * a.nb; k += blockDim.x) cl[k] = 0u;
    __syncthreads();
    const int64_t p0 = (int64_t)tile * kHistTile, n = npoints(a);
    for (int j = threadIdx.x; j < kHistTile; j += blockDim.x) {
        const int64_t i = p0 + j;
        if (i >= n) break;
        for (int e = 0; e < nd; ++e) {
            const int k = point_bin(a, i, d0 + e, a.ninc[d0 + e]);
            if (k >= 0) atomicAdd(&cl[e * a.nb + k], 1u);
        }
    }
    __syncthreads();
    for (int e = 0; e < nd; ++e) {
        uint32_t* out = a.cnt + ((int64_t)(d0 + e) * a.ntiles + tile) * a.nb;
        for (int k = threadIdx.x; k < a.nb; k += blockDim.x) out[k] = cl[e * a.nb + k];
    }
}

// Per-bin exclusive scan over the tiles (in place) and the bin totals.  One
// workgroup per axis and 64 bins: wave s takes the s-th of 16 runs of tiles
// (its sum first, then the scan from the runs before it), so 16 runs are read
// at once and a wave's loads are 256 contiguous bytes.  One workgroup per
// axis walking all tiles in turn took 49 us at 196 tiles of 5 x 400 bins.
constexpr int kScanBins = 64, kScanRuns = 16;

__global__ __launch_bounds__(kScanBins * kScanRuns) void hist_scan_kernel(HistArgs a) {
    __shared__ uint32_t part[kScanRuns][kScanBins];
    const int lane = threadIdx.x % kScanBins, run = threadIdx.x / kScanBins;
    const int d = blockIdx.y, k = blockIdx.x * kScanBins + lane;
    const int per = (a.ntiles + kScanRuns - 1) / kScanRuns;
    const int t0 = min(run * per, a.ntiles), t1 = min(t0 + per, a.ntiles);
    const bool live = k < a.nb;
    uint32_t* col = a.cnt + (int64_t)d * a.ntiles * a.nb + k;
    uint32_t s = 0;
    if (live) {
#pragma unroll 4
        for (int t = t0; t < t1; ++t) s += col[(int64_t)t * a.nb];
    }
    part[run][lane] = s;
    __syncthreads();
    uint32_t pre = 0;
    for (int r = 0; r < run; ++r) pre += part[r][lane];
    if (!live) return;
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
        const uint32_t v = col[(int64_t)t * a.nb];
        col[(int64_t)t * a.nb] = pre;
        pre += v;
    }
    if (run == kScanRuns - 1) a.total[d * a.nb + k] = pre;
}

// Exclusive scan of an axis's bin totals -> bin starts; one workgroup per axis.
// FEW: it scans the tiles itself, a bin per thread, instead of hist_scan.
// Up to kFewTiles tiles the launch costs more than the walk: a call of 10
// points, one axis of 100 bins, 29.7 us with it, 23.5 without (and with the
// short tile's empty groups left out); 4000 points of 1000 bins 38.8, 37.4;
// 8000 of 3000 the other way, 45.4, 46.1.
constexpr int kFewTiles = 4;
template <bool FEW>
__global__ __launch_bounds__(1024) void hist_start_kernel(HistArgs a) {
    __shared__ uint32_t wsum[16];
    const int d = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (int base = 0; base < a.nb; base += 1024) {
        const int k = base + threadIdx.x;
        uint32_t v = 0u;
        if (k < a.nb) {
            if constexpr (FEW) {
                uint32_t* col = a.cnt + (int64_t)d * a.ntiles * a.nb + k;
#pragma unroll 4
                for (int t = 0; t < a.ntiles; ++t) {
                    const uint32_t c = col[(int64_t)t * a.nb];
                    col[(int64_t)t * a.nb] = v;
                    v += c;
                }
                a.total[d * a.nb + k] = v;
            } else {
                v = a.total[d * a.nb + k];
            }
        }
        uint32_t incl = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wsum[w] = incl;
        __syncthreads();
        uint32_t pre = carry, tot = carry;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            if (q < w) pre += wsum[q];
            tot += wsum[q];
        }
        if (k < a.nb) a.start[d * a.nb + k] = pre + incl - v;
        carry = tot;
        __syncthreads();
    }
}

// One wave per (tile, axis).  Points of the tile are taken 64 at a time in
// order; equal keys within a group get consecutive ranks in lane order.  The
// lanes that share a lane's key are found from one ballot per key bit (a
// fixed number of instructions however many distinct keys the group has: a
// loop over the distinct keys took 251 us for 2e5 points and 5 axes of 400
// bins, this 20 us).  run[k]: the next position of bin k.
// FEW: few tiles, the last may be short (and its end is looked for).
template <bool FEW>
__global__ __launch_bounds__(64) void hist_scatter_kernel(HistArgs a, int keybits) {
    extern __shared__ uint32_t run[];
    const int tile = blockIdx.x, d = blockIdx.y;
    const int ni = a.ninc[d];
    const int lane = threadIdx.x;
    const uint32_t* tbase = a.cnt + ((int64_t)d * a.ntiles + tile) * a.nb;
    const uint32_t* bstart = a.start + d * a.nb;
    const int64_t p0 = (int64_t)tile * kHistTile, n = npoints(a);
    // the whole tile's loads in flight at once, with those of run[]
    constexpr int kGroups = kHistTile / 64;
    int key[kGroups];
    double fa[kGroups];
#pragma unroll
    for (int q = 0; q < kGroups; ++q) {
        const int64_t i = p0 + 64 * q + lane;
        key[q] = i < n ? point_bin(a, i, d, ni) : -1;
        fa[q] = i < n ? fabs(a.f[i]) : 0.0;
    }
#pragma unroll 4
    for (int k = lane; k < a.nb; k += 64) run[k] = bstart[k] + tbase[k];
    __syncthreads();
    double* out = a.sorted + (int64_t)d * a.n;
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int q = 0; q < kGroups; ++q) {
        if (FEW && p0 + 64 * q >= n) break;
        const bool on = key[q] >= 0;
        uint64_t m = __ballot(on);
        for (int b = 0; b < keybits; ++b) {
            const bool bit = (key[q] >> b) & 1;
            const uint64_t set = __ballot(bit);
            m &= bit ? set : ~set;
        }
        uint32_t base = 0;
        if (on) base = run[key[q]];
        __builtin_amdgcn_wave_barrier();
        if (on) {
            out[base + (uint32_t)__popcll(m & below)] = fa[q];
            if ((m & below) == 0) run[key[q]] = base + (uint32_t)__popcll(m);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// acc + lane 0's v + lane 1's v + ... + lane 15's v of each 16-lane row, in
// that order (every lane of the row alike): v_mov row_newbcast moves.
template <int L>
__device__ __forceinline__ void row_add(double& acc, double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)dpp0_i<0x150 + L>((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)dpp0_i<0x150 + L>((int)(uint32_t)(u >> 32));
    acc += __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
    if constexpr (L < 15) row_add<L + 1>(acc, v);
}

// The sums of a bin's values in point order: a 16-lane row per bin reads 16
// consecutive values at once (4 such loads in flight) and adds them one
// after the other from the row's lanes.  Past a bin's last value it adds
// +0.0 to a sum of absolute values, which leaves it as it is.  One thread
// per bin, each loading its own values, took 166 us for 2e5 points and 5 x
// 400 bins (the loads' latency per value), this 9 us.
__global__ __launch_bounds__(256) void hist_sum_kernel(HistArgs a) {
    const int d = blockIdx.y, row = threadIdx.x >> 4, l = threadIdx.x & 15;
    const int k = blockIdx.x * 16 + row;
    const bool live = k < a.ninc[d];
    const uint32_t s = live ? a.start[d * a.nb + k] : 0u, t = live ? a.total[d * a.nb + k] : 0u;
    const double* in = a.sorted + (int64_t)d * a.n + s;
    double acc = live ? a.sum_f[d * a.nb + k] : 0.0;
    constexpr int kAhead = 4;
    double cur[kAhead], nxt[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) cur[q] = (uint32_t)(16 * q + l) < t ? in[16 * q + l] : 0.0;
    for (uint64_t j = 0; __any(j < t); j += 16 * kAhead) {
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
            const uint64_t i = j + 16 * (kAhead + q) + l;
            nxt[q] = i < t ? in[i] : 0.0;
        }
        if (j < t) {
#pragma unroll
            for (int q = 0; q < kAhead; ++q) row_add<0>(acc, cur[q]);
        }
#pragma unroll
        for (int q = 0; q < kAhead; ++q) cur[q] = nxt[q];
    }
    if (live && l == 0) {
        a.sum_f[d * a.nb + k] = acc;
        a.n_f[d * a.nb + k] = a.n_f[d * a.nb + k] + (double)t;
    }
}

// The four passes on stream st; a's tables and counts are set.
static int launch_ordered(const HistArgs& a, hipStream_t st) {
    int maxn = 0, keybits = 1;
    for (int d = 0; d < a.dim; ++d) maxn = a.ninc[d] > maxn ? a.ninc[d] : maxn;
    while ((1 << keybits) < maxn) ++keybits;
    const size_t row = (size_t)a.nb * sizeof(uint32_t);
    // axes per hist_count workgroup: all that its LDS holds where the tiles
    // alone fill the chip (a tile's rows of y are then read once); fewer where
    // they do not (196 tiles of 5 axes: 5.0 us by axis, 9.7 us together)
    const int groups = std::min(a.dim, (1024 + a.ntiles - 1) / a.ntiles);
    const int fit = row >= kCountLds ? 1 : (int)(kCountLds / row);
    const int daxes = std::min(fit, (a.dim + groups - 1) / groups);
    hipLaunchKernelGGL(hist_count_kernel, dim3(a.ntiles, (a.dim + daxes - 1) / daxes), dim3(256), row * daxes, st, a,
                       daxes);
    if (a.ntiles <= kFewTiles) {
        hipLaunchKernelGGL(hist_start_kernel<true>, dim3(a.dim), dim3(1024), 0, st, a);
        hipLaunchKernelGGL(hist_scatter_kernel<true>, dim3(a.ntiles, a.dim), dim3(64), row, st, a, keybits);
    } else {
        hipLaunchKernelGGL(hist_scan_kernel, dim3((a.nb + kScanBins - 1) / kScanBins, a.dim),
                           dim3(kScanBins * kScanRuns), 0, st, a);
        hipLaunchKernelGGL(hist_start_kernel<false>, dim3(a.dim), dim3(1024), 0, st, a);
        hipLaunchKernelGGL(hist_scatter_kernel<false>, dim3(a.ntiles, a.dim), dim3(64), row, st, a, keybits);
    }
    hipLaunchKernelGGL(hist_sum_kernel, dim3((maxn + 15) / 16, a.dim), dim3(256), 0, st, a);
    return check_launch();
}

}  // namespace vgx

using namespace vgx;

extern "C" int vgx_train_hist(vgx_ctx* ctx, int dim, const int32_t* ninc, int ld, const double* y,
                              const double* f, int64_t n, double* sum_f, double* n_f, int ordered,
                              void* stream) {
    if (dim < 1 || dim > VGX_MAXDIM || ld < 2 || n < 0 || !ninc) return VGX_EINVAL;
    if (n == 0) return VGX_OK;
    if (n > 0xFFFFFFFFll) return VGX_ERANGE;
    hipStream_t st = (hipStream_t)stream;
    HistArgs a{};
    a.dim = dim;
    a.nb = ld - 1;
    a.y = y;
    a.f = f;
    a.n = n;
    a.sum_f = sum_f;
    a.n_f = n_f;
    for (int d = 0; d < dim; ++d) {
        if (ninc[d] < 1 || ninc[d] > a.nb) return VGX_EINVAL;
        a.ninc[d] = ninc[d];
    }
    if (!ordered) {
        size_t bytes = (size_t)dim * a.nb * (sizeof(double) + sizeof(uint32_t));
        a.use_lds = bytes <= 64 * 1024;
        int64_t b = (n + 255) / 256;
        if (b > 512) b = 512;
        hipLaunchKernelGGL(hist_fast_kernel, dim3((unsigned)b), dim3(256), a.use_lds ? bytes : 0,
                           st, a);
        return check_launch();
    }
    if (!ctx) return VGX_EINVAL;
    if ((size_t)a.nb * sizeof(uint32_t) > 64 * 1024) return VGX_ERANGE;
    a.ntiles = (int)((n + kHistTile - 1) / kHistTile);
    size_t ncnt = (size_t)dim * a.ntiles * a.nb;
    int rc = ctx->hist_cnt.ensure(ncnt * sizeof(uint32_t));
    if (rc) return rc;
    rc = ctx->hist_start.ensure(2 * (size_t)dim * a.nb * sizeof(uint32_t));
    if (rc) return rc;
    rc = ctx->hist_sorted.ensure((size_t)dim * n * sizeof(double));
    if (rc) return rc;
    a.cnt = (uint32_t*)ctx->hist_cnt.ptr;
    a.start = (uint32_t*)ctx->hist_start.ptr;
    a.total = a.start + (size_t)dim * a.nb;
    a.sorted = (double*)ctx->hist_sorted.ptr;
    return launch_ordered(a, st);
}

namespace vgx {

// The training histogram of a batch of the fused sampler, from its records,
// bit for bit the reference's add_training_data on the batch's points in
// order (pyx:457-463): the ordered mode above with the bins and values of
// the records.  cap bounds the batch's point count, which is read on the
// device from nrange.
int train_hist_records(vgx_ctx* ctx, int dim, const int32_t* ninc, int nb, const uint32_t* rbins,
                       int64_t rstride, const double* c2, const uint32_t* nrange, int64_t cap, double* sum_f,
                       double* n_f, hipStream_t st) {
    if (cap <= 0) return VGX_OK;
    if ((size_t)nb * sizeof(uint32_t) > 64 * 1024 || dim > VGX_MAXDIM) return VGX_ERANGE;
    HistArgs a{};
    a.dim = dim;
    a.nb = nb;
    a.n = cap;
    a.f = c2;
    a.sum_f = sum_f;
    a.n_f = n_f;
    a.rbins = rbins;
    a.rstride = rstride;
    a.nrange = nrange;
    for (int d = 0; d < dim; ++d) a.ninc[d] = ninc[d];
    a.ntiles = (int)((cap + kHistTile - 1) / kHistTile);
    int rc = ctx->hist_cnt.ensure((size_t)dim * a.ntiles * a.nb * sizeof(uint32_t));
    if (rc) return rc;
    if ((rc = ctx->hist_start.ensure(2 * (size_t)dim * a.nb * sizeof(uint32_t)))) return rc;
    if ((rc = ctx->hist_sorted.ensure((size_t)dim * cap * sizeof(double)))) return rc;
    a.cnt = (uint32_t*)ctx->hist_cnt.ptr;
    a.start = (uint32_t*)ctx->hist_start.ptr;
    a.total = a.start + (size_t)dim * a.nb;
    a.sorted = (double*)ctx->hist_sorted.ptr;
    return launch_ordered(a, st);
}

}  // namespace vgx

// ---- the ordered histogram without allocation -----------------------------
// For callers that cannot allocate device memory (code under HIP graph
// capture, tight serving loops): the ordered mode of vgx_train_hist with its
// temporaries (per-tile counts, bin starts and totals, the grouped values)
// in this file-scope array, one copy per GPU, held until the process ends.
// Its device address is looked up once per device (kernels take that
// address, never the array's host-side name).
namespace vgx {
constexpr size_t kNoAllocScratch = (size_t)128 << 20;  // bytes per device
static __device__ __align__(256) unsigned char scratch[kNoAllocScratch];

constexpr int kNoAllocDevices = 64;
static void* g_scratch_dev[kNoAllocDevices] = {};
static std::mutex g_scratch_mu;

// The current device's copy of `scratch` (its device address).
static int scratch_for_current_device(unsigned char** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return VGX_EHIP;
    if (dev < 0 || dev >= kNoAllocDevices) return VGX_ERANGE;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return VGX_EHIP;
        g_scratch_dev[dev] = p;
    }
    *out = (unsigned char*)g_scratch_dev[dev];
    return VGX_OK;
}

// Bytes of scratch the ordered histogram of n points needs, laid out as
// per-tile counts | bin starts and totals | grouped values (256-B aligned).
static size_t noalloc_layout(int dim, int nb, int64_t n, size_t* o_start, size_t* o_sorted) {
    const int64_t ntiles = (n + kHistTile - 1) / kHistTile;
    const size_t cnt = (((size_t)dim * ntiles * nb * sizeof(uint32_t)) + 255) & ~(size_t)255;
    const size_t st = ((2 * (size_t)dim * nb * sizeof(uint32_t)) + 255) & ~(size_t)255;
    *o_start = cnt;
    *o_sorted = cnt + st;
    return cnt + st + (size_t)dim * n * sizeof(double);
}
}  // namespace vgx

extern "C" int vgx_train_hist_noalloc(int dim, const int32_t* ninc, int ld, const double* y, const double* f,
                                      int64_t n, double* sum_f, double* n_f, void* stream) {
    if (dim < 1 || dim > VGX_MAXDIM || ld < 2 || n < 0 || !ninc) return VGX_EINVAL;
    if (n == 0) return VGX_OK;
    if (n > 0xFFFFFFFFll) return VGX_ERANGE;
    HistArgs a{};
    a.dim = dim;
    a.nb = ld - 1;
    a.y = y;
    a.f = f;
    a.n = n;
    a.sum_f = sum_f;
    a.n_f = n_f;
    for (int d = 0; d < dim; ++d) {
        if (ninc[d] < 1 || ninc[d] > a.nb) return VGX_EINVAL;
        a.ninc[d] = ninc[d];
    }
    if ((size_t)a.nb * sizeof(uint32_t) > 64 * 1024) return VGX_ERANGE;
    size_t o_start = 0, o_sorted = 0;
    if (noalloc_layout(dim, a.nb, n, &o_start, &o_sorted) > kNoAllocScratch) return VGX_ERANGE;
    unsigned char* base = nullptr;
    int rc = scratch_for_current_device(&base);
    if (rc) return rc;
    a.ntiles = (int)((n + kHistTile - 1) / kHistTile);
    a.cnt = (uint32_t*)base;
    a.start = (uint32_t*)(base + o_start);
    a.total = a.start + (size_t)dim * a.nb;
    a.sorted = (double*)(base + o_sorted);
    return launch_ordered(a, (hipStream_t)stream);
}
