// vgx_map.hip -- AdaptiveMap.map / invmap / jac1d on gfx950.
//
// Workgroups map whole tiles of points element by element: thread t of a
// workgroup takes elements t, t + T, ... of the tile's contiguous rows, so
// that every load and store of y and x is a contiguous run of lanes (a lane
// per point read one 64-byte row per load at 8 axes: 64 lines per wave
// instruction, 66 us for 1e6 points where the bytes take 27; this 28 us, and
// invmap 51 us against 94).  The axis
// Jacobians go through LDS and one thread per point multiplies them in axis
// order, as the reference does.  The FP64 grid (dim x ld) is staged in LDS
// once per workgroup where it fits (one persistent workgroup of 1024 lanes
// per CU), so its gathers never leave the CU.  Increments are formed
// as grid[k+1]-grid[k], the very subtraction the reference stores in `inc`
// (src/vegas/_vegas.pyx:130-131, 236-237, 589-592), so they are bit-equal.
#include <algorithm>

#include "vgx_internal.h"

namespace vgx {

constexpr int kMapThreads = 1024;
constexpr int kMapEl = 4;                   // elements per thread and tile, at most
constexpr size_t kMapLds = 156 * 1024;      // LDS of a workgroup
constexpr size_t kMapTileMax = 56 * 1024;   // of it, a tile's Jacobian factors, at most
constexpr size_t kMapGridMax = 136 * 1024;  // a larger grid is read from global memory
constexpr int kMapCells = 512;              // cells per axis of invmap's table, at most
// points from which the table saves more probes than it costs (1e6 points of 8
// axes of 1000: 50 us with it, 65 without; 5e4: no gain; with 10 increments
// it gains from 1e6 elements on and costs up to 1 us below, where 65,536 points
// of 24 axes cost 80 us with a table filled axis by axis)
constexpr int64_t kMapLutMin = 1 << 16;

struct MapArgs {
    int dim;
    int ld;
    int use_lds;
    int pts;      // points per tile
    int pad;      // LDS row of a point's factors (odd: no bank conflicts)
    int cells;    // invmap: cells per axis of the search table, 0: none
    DivMagic dm;  // of dim
    int32_t ninc[VGX_MAXDIM];
    const double* grid;
    int64_t n;
};

// LDS: grid (when staged) | Jacobian factors [pts][pad] | ninc | invmap's
// cell scales and table [dim][cells + 1]
// One axis of AdaptiveMap.map (pyx:347-359).  Returns x, multiplies J.
__device__ inline double map_axis(const double* g, int ni, double yv, double& J) {
    double t = yv * (double)ni;
    t = fmin(t, (double)ni);  // y > 1 takes the k >= ninc branch, as in the reference
    int k = (int)floor(t);
    k = k < 0 ? 0 : k;        // y < 0 is never produced; keep the read in bounds
    const double dl = t - (double)k;
    // (k = ninc: x is the last node, with the last increment)
    const bool in = k < ni;
    const double g0 = g[in ? k : ni - 1], g1 = g[in ? k + 1 : ni];
    const double inc = g1 - g0;
    J *= inc * (double)ni;
    return in ? g0 + inc * dl : g1;
}

// The cell of x on an axis from g0: a non-decreasing function of x (NaN: 0).
__device__ inline int map_cell(double xv, double g0, double scale, int cells) {
    const double c = (xv - g0) * scale;
    return c >= (double)(cells - 1) ? cells - 1 : c > 0.0 ? (int)c : 0;
}

// Row d of lut, [c]: the first node of axis d whose cell is c or more (ni + 1
// past the last), so that the nodes before [c] are below every x of cell c and
// those from [c + 1] on are above: the search of all nodes ends in between.
// All axes at once (one after the other, each with its division and few busy
// lanes, 24 axes of 10 increments took 64 us of the call's 81, now 17 in all).
__device__ inline void fill_lut(const MapArgs& a, const double* G, const int32_t* ninc, double* sc, uint16_t* lut) {
    for (int d = threadIdx.x; d < a.dim; d += kMapThreads)
        sc[d] = (double)a.cells / (G[d * a.ld + ninc[d]] - G[d * a.ld]);
    __syncthreads();
    const int row = a.ld + 1;
    for (int e = threadIdx.x; e < a.dim * row; e += kMapThreads) {
        const int d = e / row, i = e - d * row, ni = ninc[d];
        if (i > ni + 1) continue;
        const double* g = G + d * a.ld;
        const int c0 = i > 0 ? map_cell(g[i - 1], g[0], sc[d], a.cells) : -1;
        const int c1 = i <= ni ? map_cell(g[i], g[0], sc[d], a.cells) : a.cells;
        for (int c = c0 + 1; c <= c1; ++c) lut[d * (a.cells + 1) + c] = (uint16_t)i;
    }
    __syncthreads();
}

// AdaptiveMap.invmap (pyx:362-416) of a thread's elements together: for
// each, searchsorted(side='right') over the axis's live nodes, then the three
// branches of the reference.  The searches advance side by side, one probe
// of each at a time (all, or the first nq of a small tile), so that a wave has four LDS reads in flight instead of
// one; LDS reads and the FP64 divisions bound it.  x in v, y out; J the axis Jacobians.
template <bool FULL, typename T>
__device__ inline void invmap_elements(const MapArgs& a, const double* G, const int32_t* ninc, const double* sc,
                                       const uint16_t* lut, const uint32_t (&ax)[kMapEl], int nq, T (&v)[kMapEl],
                                       double (&J)[kMapEl]) {
    int lo[kMapEl], len[kMapEl];
#pragma unroll
    for (int q = 0; q < kMapEl; ++q) {
        lo[q] = len[q] = 0;
        if (!FULL && q >= nq) continue;
        len[q] = ninc[ax[q]] + 1;
        if (a.cells) {
            const uint16_t* c = lut + ax[q] * (a.cells + 1) + map_cell((double)v[q], G[ax[q] * a.ld], sc[ax[q]], a.cells);
            lo[q] = c[0];
            len[q] = (int)c[1] - lo[q];
        }
    }
    for (;;) {
        int left = 0;
#pragma unroll
        for (int q = 0; q < kMapEl; ++q) left |= len[q];
        if (!__any(left)) break;
#pragma unroll
        for (int q = 0; q < kMapEl; ++q) {
            if (!FULL && q >= nq) continue;
            const int half = len[q] >> 1;
            // (a finished search rereads its node, at most node ninc)
            const int mid = min(lo[q] + half, (int)ninc[ax[q]]);
            const bool up = len[q] > 0 && G[ax[q] * a.ld + mid] <= (double)v[q];
            lo[q] = up ? mid + 1 : lo[q];
            len[q] = up ? len[q] - half - 1 : half;
        }
    }
#pragma unroll
    for (int q = 0; q < kMapEl; ++q) {
        if (!FULL && q >= nq) continue;
        const int ni = ninc[ax[q]], k = min(max(lo[q] - 1, 0), ni - 1);
        const double* g = G + ax[q] * a.ld + k;
        const double g0 = g[0], inc = g[1] - g0;
        J[q] = inc * (double)ni;
        const double y = ((double)k + ((double)v[q] - g0) / inc) / (double)ni;
        v[q] = (T)(lo[q] <= 0 ? 0. : lo[q] > ni ? 1.0 : y);
    }
}

// OP: 0 map, 1 invmap, 2 jac1d.  in [n][dim]; out [n][dim] (x, y, or the
// axis Jacobians); jac [n] (not for jac1d).
// LDS: the grid is staged (its reads are then ds_*; one pointer for both would
// make them flat loads, which wait for the global accesses as well).
template <int OP, bool LDS, typename T>
__global__ __launch_bounds__(kMapThreads) void map_kernel(MapArgs a, const T* __restrict__ in,
                                                          T* __restrict__ out, T* __restrict__ jac) {
    extern __shared__ double lds[];
    const double* const G = LDS ? lds : a.grid;
    double* F = lds;
    if constexpr (LDS) {
        const int tot = a.dim * a.ld;
        for (int i = threadIdx.x; i < tot; i += kMapThreads) lds[i] = a.grid[i];
        F += tot;
    }
    int32_t* ni = reinterpret_cast<int32_t*>(F + (OP == 2 ? 0 : a.pts * a.pad));
    for (int d = threadIdx.x; d < a.dim; d += kMapThreads) ni[d] = a.ninc[d];
    const int dim = a.dim, tile = a.pts * dim;
    double* sc = reinterpret_cast<double*>(ni + VGX_MAXDIM);
    uint16_t* lut = reinterpret_cast<uint16_t*>(sc + VGX_MAXDIM);
    // this thread's elements: point and axis are the same in every tile
    uint32_t pt[kMapEl], ax[kMapEl];
#pragma unroll
    for (int q = 0; q < kMapEl; ++q) {
        const uint32_t e = threadIdx.x + q * kMapThreads;
        pt[q] = divq(e, a.dm);
        ax[q] = e - pt[q] * (uint32_t)dim;
    }
    const int64_t ntiles = (a.n + a.pts - 1) / a.pts;
    T cur[kMapEl], nxt[kMapEl];
    auto load = [&](int64_t t, T (&v)[kMapEl]) {
        const int64_t e0 = t * tile, left = a.n * dim - e0;
#pragma unroll
        for (int q = 0; q < kMapEl; ++q) {
            const int e = threadIdx.x + q * kMapThreads;
            v[q] = (e < tile && e < left) ? in[e0 + e] : (T)0;
        }
    };
    if ((int64_t)blockIdx.x < ntiles) load(blockIdx.x, cur);
    __syncthreads();
    if (OP == 1 && a.cells) fill_lut(a, G, ni, sc, lut);
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        // the next tile's loads are in flight while this one is mapped
        if (t + gridDim.x < ntiles) load(t + gridDim.x, nxt);
        const int64_t e0 = t * tile, left = a.n * dim - e0;
        double Ji[kMapEl];
        if constexpr (OP == 1) {
            const int nq = (int)(((left < tile ? left : tile) + kMapThreads - 1) / kMapThreads);
            if (nq == kMapEl) invmap_elements<true>(a, G, ni, sc, lut, ax, nq, cur, Ji);
            else invmap_elements<false>(a, G, ni, sc, lut, ax, nq, cur, Ji);
        }
#pragma unroll
        for (int q = 0; q < kMapEl; ++q) {
            const int e = threadIdx.x + q * kMapThreads;
            if (e < tile && e < left) {
                double J = 1.0, v;
                if constexpr (OP == 1) {
                    J = Ji[q];
                    v = (double)cur[q];
                } else {
                    v = map_axis(G + ax[q] * a.ld, ni[ax[q]], (double)cur[q], J);
                }
                out[e0 + e] = (T)(OP == 2 ? J : v);
                if constexpr (OP != 2) {
                    if (dim == 1) jac[e0 + e] = (T)J;
                    else F[pt[q] * a.pad + ax[q]] = J;
                }
            }
        }
        if (OP != 2 && dim > 1) {
            __syncthreads();
            const int64_t i0 = t * a.pts;
            for (int p = threadIdx.x; p < a.pts && i0 + p < a.n; p += kMapThreads) {
                double J = 1.0;
                for (int d = 0; d < dim; ++d) J *= F[p * a.pad + d];
                jac[i0 + p] = (T)J;
            }
            __syncthreads();
        }
#pragma unroll
        for (int q = 0; q < kMapEl; ++q) cur[q] = nxt[q];
    }
}

static int fill_map_args(MapArgs& a, int dim, const int32_t* ninc, const double* grid, int ld,
                         int64_t n) {
    if (dim < 1 || dim > VGX_MAXDIM || n < 0 || !ninc || !grid) return VGX_EINVAL;
    a.dim = dim;
    a.ld = ld;
    a.grid = grid;
    a.n = n;
    for (int d = 0; d < dim; ++d) {
        if (ninc[d] < 1 || ninc[d] + 1 > ld) return VGX_EINVAL;
        a.ninc[d] = ninc[d];
    }
    a.dm = make_divmagic((uint32_t)dim);
    a.use_lds = (size_t)dim * ld * sizeof(double) <= kMapGridMax;
    return VGX_OK;
}

template <int OP, typename T>
static int launch_map(MapArgs a, const T* in, T* out, T* jac, void* stream) {
    if (a.n == 0) return VGX_OK;
    const size_t gbytes = a.use_lds ? (size_t)a.dim * a.ld * sizeof(double) : 0;
    size_t lds = gbytes + VGX_MAXDIM * (sizeof(int32_t) + sizeof(double));
    a.cells = 0;
    if (OP == 1 && a.use_lds && a.n >= kMapLutMin) {
        // the largest table that leaves a tile of two elements per thread
        for (int c = kMapCells; c >= 64 && !a.cells; c /= 2)
            if (lds + (size_t)a.dim * (c + 1) * sizeof(uint16_t) + 20 * 1024 <= kMapLds) a.cells = c;
        lds += (size_t)a.dim * (a.cells ? a.cells + 1 : 0) * sizeof(uint16_t);
    }
    // Points per tile: at most kMapEl elements per thread, and the factors in
    // the LDS left.  invmap wants full tiles (its searches run side by side);
    // the others four tiles per workgroup, as long as a tile fills its
    // threads (the next tile's loads run ahead of the mapping).
    a.pad = a.dim | 1;
    const size_t room = std::min(kMapTileMax, kMapLds - lds - 16);
    const int64_t most = std::min<int64_t>(kMapEl * kMapThreads / a.dim, room / (8 * (size_t)a.pad));
    const int64_t split = 256 * (OP == 1 ? 1 : 4);
    const int64_t share = std::max<int64_t>((a.n + split - 1) / split, kMapThreads / a.dim);
    a.pts = (int)std::max<int64_t>(1, std::min(most, (share + 63) & ~(int64_t)63));
    if (OP == 1 && share > most) {
        // as many points in each of a workgroup's tiles (300,000 points of 5
        // axes: 1.4 tiles of 819 a workgroup 14.0 us, 2 of 592 13.2)
        const int64_t rounds = (share + most - 1) / most;
        a.pts = (int)std::min(most, ((share + rounds - 1) / rounds + 7) & ~(int64_t)7);
    }
    if (OP != 2) lds += (size_t)a.pts * a.pad * sizeof(double);
    lds = (lds + 15) & ~(size_t)15;
    auto kern = a.use_lds ? map_kernel<OP, true, T> : map_kernel<OP, false, T>;
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMapLds) != hipSuccess)
        return VGX_EHIP;
    // persistent workgroups: two per CU where its LDS and registers (64 of
    // map and jac1d) hold two, else one
    const int64_t tiles = (a.n + a.pts - 1) / a.pts, blocks = OP != 1 && lds <= kMapLds / 2 ? 512 : 256;
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min(tiles, blocks)), dim3(kMapThreads), lds,
                       (hipStream_t)stream, a, in, out, jac);
    return check_launch();
}

}  // namespace vgx

using namespace vgx;

extern "C" int vgx_map_f64(int dim, const int32_t* ninc, const double* grid, int ld,
                           const double* y, double* x, double* jac, int64_t n, void* stream) {
    MapArgs a;
    const int rc = fill_map_args(a, dim, ninc, grid, ld, n);
    return rc ? rc : launch_map<0>(a, y, x, jac, stream);
}

extern "C" int vgx_map_f32(int dim, const int32_t* ninc, const double* grid, int ld,
                           const float* y, float* x, float* jac, int64_t n, void* stream) {
    MapArgs a;
    const int rc = fill_map_args(a, dim, ninc, grid, ld, n);
    return rc ? rc : launch_map<0>(a, y, x, jac, stream);
}

extern "C" int vgx_invmap_f64(int dim, const int32_t* ninc, const double* grid, int ld,
                              const double* x, double* y, double* jac, int64_t n, void* stream) {
    MapArgs a;
    const int rc = fill_map_args(a, dim, ninc, grid, ld, n);
    return rc ? rc : launch_map<1>(a, x, y, jac, stream);
}

extern "C" int vgx_jac1d_f64(int dim, const int32_t* ninc, const double* grid, int ld,
                             const double* y, double* jac, int64_t n, void* stream) {
    MapArgs a;
    const int rc = fill_map_args(a, dim, ninc, grid, ld, n);
    return rc ? rc : launch_map<2>(a, y, jac, (double*)nullptr, stream);
}
