// vgx_flow.hip -- the learned map: an affine-coupling normalizing flow on
// [0,1]^D (D <= 15) with hand-written BF16 MFMA kernels (gfx950
// v_mfma_f32_16x16x16_bf16, FP32 accumulation, FP32 log-det).
//
// Map (the same arithmetic as oracle/flow_oracle.py): z -> u0 = logit(z) ->
// L couplings -> x = sigmoid(uL).  Coupling k conditions on the set A_k:
//   a = (u_d, d in A_k; 0 else; a_15 = 1),  h1 = relu(W1 a),
//   h2 = relu(W2 h1 + b2),  o = W3 h2 + b3,  s = 4 tanh(o_0..15 / 4),  t = o_16..31
//   u_B <- u_B e^s + t (forward),  u_B <- (u_B - t) e^-s (inverse).
//
// MFMA orientation.  Every GEMM is computed transposed, C[out][sample] =
// W[out][in] X[in][sample], on tiles of 16 samples.  With the 16x16x16
// instruction, lane l holds C[(l/16)*4 + i][l%16] (i < 4) and the B operand
// X[(l/16)*4 + j][l%16]: one layer's output tile mt, after bias, ReLU and the
// bf16 rounding, is the next layer's k-step mt in registers, with no data
// movement.  The coupling state u (dims (l/16)*4 + i of sample l%16) sits in
// the same lanes as s (output tile 0) and t (output tile 1), so the update is
// lane-local; per-sample sums reduce across the four lane groups.
//
// Kernels:
//   flow_sample   z (Philox) -> x, log J, f(x), sums of f J and (f J)^2: the
//                 estimator; layers streamed through LDS, samples in registers
//   flow_inverse  x -> z, log q(x), each layer's input saved (training)
//   flow_lossw    variance-loss weights c_i ~ w_i f_i^2 / q(x_i), normalised
//   flow_backward one layer: recompute, backprop, and the weight gradients
//                 (MFMA over the sample axis, operands staged in LDS)
//   flow_wgrad_reduce  the workgroups' weight-gradient sums, in a fixed order
//   flow_adam     Adam on the FP32 master weights, bf16 copies refreshed
#include <math.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "vgx_internal.h"

namespace vgx {

typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kFH = 128;             // hidden width
constexpr int kFI = 16;              // padded input width, column 15 = layer-1 bias
constexpr int kFO = 32;              // output rows: s 0..15, t 16..31
constexpr int kFMaxL = 8;            // layers
constexpr float kSMax = 4.0f;
// FP32 master parameters of one layer: W1 | W2 | b2 | W3 | b3
constexpr int kPW1 = 0, kPW2 = kPW1 + kFH * kFI, kPB2 = kPW2 + kFH * kFH, kPW3 = kPB2 + kFH,
              kPB3 = kPW3 + kFO * kFH, kPLayer = kPB3 + kFO;
// bf16 weights of one layer, W1 | W2 | W3, and the transposes W1t [16][128] |
// W2t [128][128] | W3t [128][32], in MFMA fragment order: blocks of 64 lanes
// by 8 values, so that an A operand is one 16-byte LDS read per lane whose
// lanes are consecutive (a row-major layout, whatever its padding, took two
// 8-byte reads with every second bank shared).  Value j of lane l of block
//   W2, W3, W1t, W2t (mt, kp): row 16 mt + l%16, column 32 kp + 16 (j/4) +
//                              4 (l/16) + j%4 (k-steps 2 kp and 2 kp + 1)
//   W3t: the same with its one kp; W1 (p): row 16 (2 p + j/4) + l%16, column
//                              4 (l/16) + j%4 (output tiles 2 p and 2 p + 1)
constexpr int kFrag = 64 * 8;
constexpr int kHW1 = 0, kHW2 = kHW1 + kFH * kFI, kHW3 = kHW2 + kFH * kFH, kHLayer = kHW3 + kFO * kFH;
constexpr int kTW1 = 0, kTW2 = kTW1 + kFI * kFH, kTW3 = kTW2 + kFH * kFH;

// Where element (row, col) of a matrix of nkp column blocks of 32 lies.
__host__ __device__ constexpr int frag_pos(int row, int col, int nkp) {
    return ((row >> 4) * nkp + (col >> 5)) * kFrag + (16 * ((col >> 2) & 3) + (row & 15)) * 8 + 4 * ((col >> 4) & 1) +
           (col & 3);
}
// The same of W1 [128][16].
__host__ __device__ constexpr int frag_pos1(int row, int col) {
    return (row >> 5) * kFrag + (16 * (col >> 2) + (row & 15)) * 8 + 4 * ((row >> 4) & 1) + (col & 3);
}

// FP32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
__device__ inline uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ inline bf16x4_t pack_bf(const f32x4_t v) {
    bf16x4_t r;
    r[0] = __builtin_bit_cast(short, (__bf16)v[0]);
    r[1] = __builtin_bit_cast(short, (__bf16)v[1]);
    r[2] = __builtin_bit_cast(short, (__bf16)v[2]);
    r[3] = __builtin_bit_cast(short, (__bf16)v[3]);
    return r;
}

__device__ inline f32x4_t mfma16(bf16x4_t a, bf16x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Two k-steps in one gfx950 v_mfma_f32_16x16x32_bf16: lane group g supplies
// 8 of the 32 products' operands for A and B alike, so any assignment of
// k to those 8 slots that A and B share gives the same sum.  Here slots
// 0..3 are k-step kt's k = 4g..4g+3 and slots 4..7 k-step kt+1's: the B
// operand is two C-layout tiles side by side (no data movement), the A
// operand one 16-byte read of weights in fragment order.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
__device__ inline bf16x8_t cat8(bf16x4_t lo, bf16x4_t hi) {
    typedef short s16x8_t __attribute__((ext_vector_type(8)));
    const s16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8_t, v);
}
__device__ inline f32x4_t mfma32(bf16x8_t a, bf16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Block b of weights in fragment order: this lane's 8 values.
__device__ inline bf16x8_t frag_w(const uint16_t* W, int b, int lane) {
    return *reinterpret_cast<const bf16x8_t*>(W + b * kFrag + lane * 8);
}
__device__ inline bf16x4_t half8(bf16x8_t v, int hi) {
    typedef short s16x8_t __attribute__((ext_vector_type(8)));
    const s16x8_t w = __builtin_bit_cast(s16x8_t, v);
    return hi ? __builtin_shufflevector(w, w, 4, 5, 6, 7) : __builtin_shufflevector(w, w, 0, 1, 2, 3);
}

// max(v, 0), 0 for a NaN: the median with 0 and infinity (relu_top) in one
// instruction (fmaxf takes a second to quiet its operand, 64 more a tile and
// layer; so does the median with a known infinity, which becomes fmaxf).
__device__ inline float relu_top() {
    float top = INFINITY;
    asm("" : "+s"(top));
    return top;
}
__device__ inline float relu(float v, float top) { return __builtin_amdgcn_fmed3f(v, 0.0f, top); }

__device__ inline float logsigp(float u) {
    const float au = fabsf(u);
    return -au - 2.0f * __logf(1.0f + __expf(-au));
}

// tanh(x / kSMax) = (1 - e)/(1 + e), e = exp(-2 |x| / kSMax) in [0, 1]: the
// quotient by the reciprocal, refined, and one correction of the quotient
// (the steps of a division without its scaling, which 1 <= 1 + e <= 2 does
// not need).
__device__ inline float tanh_s(float x) {
    const float e = __expf(fabsf(x) * (-2.0f / kSMax));
    const float n = 1.0f - e, d = 1.0f + e;
    float r = __builtin_amdgcn_rcpf(d);
    r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
    const float q = n * r;
    return copysignf(__builtin_fmaf(__builtin_fmaf(-d, q, n), r, q), x);
}

// The sum over a sample's four lanes (l, l ^ 16, l ^ 32, l ^ 48), in each of
// them, by swaps of rows and halves.  (By LDS permutes, whose latency a
// mixture's loop waits for at every component, 700,000 samples, 5 axes, 600
// Gaussians: 2930 us, so 2447.)
__device__ inline float group_sum(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

struct FlowArgs {
    int D, L;
    uint32_t amask[kFMaxL];       // conditioning set of each layer (bit d)
    const float* P;               // FP32 master parameters [L][kPLayer]
    const uint16_t* H;            // bf16 weights [L][kHLayer]
    const uint16_t* HT;           // bf16 transposes [L][kHLayer]
};

// One layer's weights and biases in LDS.
struct LayerLds {
    alignas(16) uint16_t W[kHLayer];
    alignas(16) float b2[kFH], b3[kFO];
};

__device__ inline void load_layer(const FlowArgs& f, int k, LayerLds* s, bool transposed, uint16_t* Wt) {
    const uint4* src = reinterpret_cast<const uint4*>(f.H + (size_t)k * kHLayer);
    uint4* dst = reinterpret_cast<uint4*>(s->W);
    for (int i = threadIdx.x; i < kHLayer / 8; i += blockDim.x) dst[i] = src[i];
    if (transposed) {
        const uint4* st = reinterpret_cast<const uint4*>(f.HT + (size_t)k * kHLayer);
        uint4* dt = reinterpret_cast<uint4*>(Wt);
        for (int i = threadIdx.x; i < kHLayer / 8; i += blockDim.x) dt[i] = st[i];
    }
    const float* p = f.P + (size_t)k * kPLayer;
    for (int i = threadIdx.x; i < kFH; i += blockDim.x) s->b2[i] = p[kPB2 + i];
    for (int i = threadIdx.x; i < kFO; i += blockDim.x) s->b3[i] = p[kPB3 + i];
}

// The conditioning input a of one tile as the B operand (dims (l/16)*4 + j).
__device__ inline bf16x4_t cond_input(const f32x4_t u, uint32_t amask, int D, int lane) {
    f32x4_t a;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int d = (lane >> 4) * 4 + j;
        a[j] = (d < D && ((amask >> d) & 1u)) ? u[j] : (d == kFI - 1 ? 1.0f : 0.0f);
    }
    return pack_bf(a);
}

// Layer 1 of the conditioner MLP for NT sample tiles: h1 = relu(W1 a) (bf16
// fragments, output tile mt = k-step mt of layer 2).
template <int NT>
__device__ inline void layer1(const LayerLds* s, const bf16x4_t (&a)[NT], int lane, bf16x4_t (&h1)[NT][8]) {
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const float top = relu_top();
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
        const bf16x4_t w = half8(frag_w(s->W + kHW1, mt / 2, lane), mt & 1);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            f32x4_t c = mfma16(w, a[t], zero);
#pragma unroll
            for (int i = 0; i < 4; ++i) c[i] = relu(c[i], top);
            h1[t][mt] = pack_bf(c);
        }
    }
}

// The conditioner MLP of NT tiles: o[t][0] = raw s, o[t][1] = t rows
// (l/16)*4+i, and h2 as bf16 fragments.  Each weight fragment read serves
// every tile.
template <int NT>
__device__ inline void mlp(const LayerLds* s, const bf16x4_t (&a)[NT], int lane, f32x4_t (&o)[NT][2],
                           bf16x4_t (&h2)[NT][8]) {
    // layer 2's output tiles accumulate MB at a time side by side
    // (independent MFMA chains), k-step by k-step
    constexpr int MB = NT == 1 ? 8 : 4;
    bf16x4_t h1[NT][8];
    const float top = relu_top();
    layer1<NT>(s, a, lane, h1);
#pragma unroll
    for (int mb = 0; mb < 8; mb += MB) {
        f32x4_t acc[NT][MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const f32x4_t b = *reinterpret_cast<const f32x4_t*>(s->b2 + 16 * (mb + m) + (lane >> 4) * 4);
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t][m] = b;
        }
        // a wave in its products goes first: the SIMD's waves, together after
        // the barrier, drift apart and their vector work fills the matrix
        // cores' gaps
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kp = 0; kp < 4; ++kp) {
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const bf16x8_t w = frag_w(s->W + kHW2, (mb + m) * 4 + kp, lane);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t][m] = mfma32(w, cat8(h1[t][2 * kp], h1[t][2 * kp + 1]), acc[t][m]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][m][i] = relu(acc[t][m][i], top);
                h2[t][mb + m] = pack_bf(acc[t][m]);
            }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(s->b3 + 16 * q + (lane >> 4) * 4);
#pragma unroll
        for (int t = 0; t < NT; ++t) o[t][q] = b;
    }
#pragma unroll
    for (int kp = 0; kp < 4; ++kp)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const bf16x8_t w = frag_w(s->W + kHW3, q * 4 + kp, lane);
#pragma unroll
            for (int t = 0; t < NT; ++t) o[t][q] = mfma32(w, cat8(h2[t][2 * kp], h2[t][2 * kp + 1]), o[t][q]);
        }
}

// ------------------------------------------------------------- sampling ----
constexpr int kFlowThreads = 768;
constexpr int kFlowTiles = 6;        // sample tiles (16 samples) per wave per pass
constexpr int kFlowNT = 2;           // of which the MLP takes this many at once
constexpr int kFlowWaves = kFlowThreads / 64;


struct FlowFcn {
    int kind;            // VGX_FCN_GAUSSMIX or VGX_FCN_DIAGRIDGE
    int ncomp;
    const double* A;
    const double* B;
    const double* c;     // GAUSSMIX: [ncomp][D]; DIAGRIDGE: [ncomp]
};

// The parameters A | B | c as FP32 in LDS.
__device__ inline void load_fcn(const FlowFcn& F, int D, float* Lc) {
    const int ncp = F.kind == VGX_FCN_DIAGRIDGE ? 3 * F.ncomp : F.ncomp * (2 + D);
    for (int i = threadIdx.x; i < ncp; i += blockDim.x)
        Lc[i] = (float)(i < F.ncomp ? F.A[i] : i < 2 * F.ncomp ? F.B[i - F.ncomp] : F.c[i - 2 * F.ncomp]);
}

// A copy of them that a kernel can read after the caller's arrays are gone:
// out = A [na] | B [na] | c [nc].
__global__ __launch_bounds__(256) void flow_hold_kernel(FlowFcn F, int na, int nc, double* out) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 2 * na + nc; i += gridDim.x * blockDim.x)
        out[i] = i < na ? F.A[i] : i < 2 * na ? F.B[i - na] : F.c[i - 2 * na];
}

struct SampleArgs {
    uint64_t n;          // samples
    uint64_t base;       // first sample index (Philox counter)
    uint32_t seed_lo, seed_hi, iteration;
    int tiles;           // sample tiles per wave and pass (even, up to kFlowTiles)
    double* part;        // [gridDim.x][4]: DD sum f J, DD sum (f J)^2
    float* xout;         // optional [n][16] x, and fout [n] = f J
    float* fout;
    int32_t* status;
};

// f at x of NT samples of this lane (dims (l/16)*4 + i), all four lanes of a
// sample cooperating; every lane of the sample returns f.  One LDS read of
// the parameters serves the NT samples.
template <int NT>
__device__ inline void flow_fcn(const FlowFcn& F, const float* Lc, const f32x4_t (&x)[NT], int D, int lane,
                                float (&fv)[NT]) {
    const int g = lane >> 4;
    float acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = 0.f;
    if (F.kind == VGX_FCN_DIAGRIDGE) {
        const float fd = (float)D;
        float xbar[NT], P[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float s1 = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * g + i < D) s1 += x[t][i];
            xbar[t] = group_sum(s1) / fd;
            float p = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * g + i < D) p += (x[t][i] - xbar[t]) * (x[t][i] - xbar[t]);
            P[t] = group_sum(p);
        }
        const float* A = Lc + g;
        const float* B = A + F.ncomp;
        const float* C = B + F.ncomp;
        auto term = [&](int k) {
            const float Ak = A[k], Bk = B[k], Ck = C[k];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const float dt = xbar[t] - Ck;
                acc[t] = __builtin_fmaf(Ak, __expf(-Bk * __builtin_fmaf(fd * dt, dt, P[t])), acc[t]);
            }
        };
        // four terms a step: their reads share the addresses and one wait
        // (a term a step spent more on addresses and waits than on the term)
        int k = 0;
        for (; k + 16 <= F.ncomp; k += 16) {
            term(k);
            term(k + 4);
            term(k + 8);
            term(k + 12);
        }
        for (; k + g < F.ncomp; k += 4) term(k);
#pragma unroll
        for (int t = 0; t < NT; ++t) fv[t] = group_sum(acc[t]);
        return;
    }
    for (int k = 0; k < F.ncomp; ++k) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float r = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * g + i < D) {
                    const float dt = x[t][i] - Lc[2 * F.ncomp + k * D + 4 * g + i];
                    r = __builtin_fmaf(dt, dt, r);
                }
            r = group_sum(r);
            acc[t] = __builtin_fmaf(Lc[k], __expf(-Lc[F.ncomp + k] * r), acc[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) fv[t] = acc[t];
}

// Per-wave tile state in LDS (kFlowTiles tiles: u as float4 per lane, and
// the log-Jacobian), so that tiles are indexed at run time without scratch.
struct TileState {
    f32x4_t u[kFlowTiles][64];
    float l[kFlowTiles][64];
};
constexpr size_t kLdsLayer = (sizeof(LayerLds) + 15) & ~(size_t)15;
constexpr size_t kStateLds = kFlowWaves * sizeof(TileState);
// What they leave of a CU's LDS for an integrand's parameters (1 KiB: the sums).
constexpr size_t kFlowFcnLds = 160 * 1024 - 1024 - kLdsLayer - kStateLds;
static_assert(160 * 1024 - 1024 - kLdsLayer - 8 * sizeof(TileState) >= 48 * 1024, "8 waves fit any mixture");

// A workgroup's waves and tiles of 16 samples per wave and pass: the smallest
// of these shapes whose workgroups, one per CU, cover the n samples in one
// pass; the last is full.  (At the full shape alone 20,000 samples would keep
// 18 of the CUs busy: a sample call of 2000 to 20,000 took 258-276 us, now
// 110-130, the copies above included.)
struct FlowShape {
    int waves, tiles, blocks;
};
static FlowShape flow_shape(int64_t n, int cus, int full_blocks, size_t fcn_lds) {
    static const int shapes[4][2] = {{4, 2}, {8, 2}, {12, 2}, {kFlowWaves, kFlowTiles}};
    const int64_t nt = (n + 15) / 16;
    for (const auto& s : shapes) {
        const int64_t blocks = (nt + s[0] * s[1] - 1) / (s[0] * s[1]);
        if (blocks <= cus && (s[0] <= 8 || fcn_lds <= kFlowFcnLds)) return {s[0], s[1], (int)blocks};
    }
    // A long mixture leaves LDS for the state of fewer waves' tiles, 8 or more:
    // the fewest that cover the samples in one pass, else as many as fit
    // (700,000 samples, 9 axes, 600 Gaussians: 8 waves 3103 us, 11 waves 2451).
    int waves = kFlowWaves;
    if (fcn_lds > kFlowFcnLds) {
        const int fit = (int)((kFlowFcnLds + kStateLds - fcn_lds) / sizeof(TileState));
        for (waves = 8; waves < std::min(kFlowWaves, fit) && nt > (int64_t)cus * waves * kFlowTiles;) ++waves;
    }
    const int64_t blocks = (nt + waves * kFlowTiles - 1) / (waves * kFlowTiles);
    return {waves, kFlowTiles, (int)std::min<int64_t>(full_blocks, blocks)};
}


// A call, or its constants would take registers from the layers' loop.
__device__ __noinline__ double exp_jac(double x) { return exp(x); }

// Bound by vector instructions (relu, conversions, the couplings' tanh and
// exp, the integrand) with the matrix cores 40-50 % busy.  4e6 samples, 9
// axes, 6 layers, 500 components: 2450 us with row-major weights and a tile
// at a time, 2480 -> 2175 with one-instruction relu and four ridge terms a
// step, 1940 with the products' priority and the couplings' short quotient,
// 1570 a call, calls back to back, with the parameters read in place (before:
// three copies to the host and one back, each waited for).  12 waves hold all of a layer in
// registers; with 16 the kernels spill 35 and are no faster, with 8 and four
// tiles at once 2012 where 12 took 1945.
__global__ __launch_bounds__(kFlowThreads) void flow_sample_kernel(FlowArgs f, FlowFcn F, SampleArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    LayerLds* L = reinterpret_cast<LayerLds*>(smem);
    TileState* TS = reinterpret_cast<TileState*>(smem + kLdsLayer) +
                    (threadIdx.x >> 6);
    float* Lc = reinterpret_cast<float*>(smem + kLdsLayer +
                                         (blockDim.x >> 6) * sizeof(TileState));
    __shared__ double red[kFlowWaves * 4];
    const int wave = threadIdx.x >> 6;
    int lane = threadIdx.x & 63;
    load_fcn(F, f.D, Lc);
    DD s1{0, 0}, s2{0, 0};
    const uint64_t pass = (blockDim.x >> 6) * a.tiles * 16;  // samples per pass of the workgroup
    for (uint64_t pb = blockIdx.x * pass; pb < a.n; pb += gridDim.x * pass) {
        asm volatile("" : "+v"(lane));  // addresses are formed when used, not held over the passes
        const int g = lane >> 4;
#pragma unroll 1
        for (int q = 0; q < a.tiles; ++q) {
            const uint64_t sidx = a.base + pb + (uint64_t)(wave * a.tiles + q) * 16 + (lane & 15);
            const U4 w = philox4x32_10_dev(U4{(uint32_t)sidx, (uint32_t)(sidx >> 32), a.iteration, (uint32_t)g},
                                       a.seed_lo, a.seed_hi);
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
            float l = 0.f;
            f32x4_t uq;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float z = (float)(ws[i] >> 8) * (1.0f / 16777216.0f) + (1.0f / 33554432.0f);
                const float l0 = __logf(z), l1 = __logf(1.0f - z);
                uq[i] = l0 - l1;
                if (4 * g + i < f.D) l -= l0 + l1;  // dz/du = z (1 - z)
            }
            TS->u[q][lane] = uq;
            TS->l[q][lane] = l;
        }
        for (int k = 0; k < f.L; ++k) {
            asm volatile("" : "+v"(lane));
            const int g = lane >> 4;
            __syncthreads();
            load_layer(f, k, L, false, nullptr);
            __syncthreads();
            const uint32_t am = f.amask[k];
#pragma unroll 1
            for (int q = 0; q < a.tiles; q += kFlowNT) {
                bf16x4_t a[kFlowNT];
                f32x4_t o[kFlowNT][2];
                bf16x4_t h2[kFlowNT][8];
#pragma unroll
                for (int t = 0; t < kFlowNT; ++t) a[t] = cond_input(TS->u[q + t][lane], am, f.D, lane);
                mlp<kFlowNT>(L, a, lane, o, h2);
#pragma unroll
                for (int t = 0; t < kFlowNT; ++t) {
                    f32x4_t uq = TS->u[q + t][lane];
                    float l = TS->l[q + t][lane];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int d = 4 * g + i;
                        if (d < f.D && !((am >> d) & 1u)) {
                            const float sv = kSMax * tanh_s(o[t][0][i]);
                            uq[i] = uq[i] * __expf(sv) + o[t][1][i];
                            l += sv;
                        }
                    }
                    TS->u[q + t][lane] = uq;
                    TS->l[q + t][lane] = l;
                }
            }
        }
#pragma unroll 1
        for (int q = 0; q < a.tiles; q += kFlowNT) {
            f32x4_t x[kFlowNT];
            float LJ[kFlowNT], fv[kFlowNT];
#pragma unroll
            for (int t = 0; t < kFlowNT; ++t) {
                const f32x4_t uq = TS->u[q + t][lane];
                float l = TS->l[q + t][lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    x[t][i] = 1.0f / (1.0f + __expf(-uq[i]));
                    if (4 * g + i < f.D) l += logsigp(uq[i]);
                }
                LJ[t] = group_sum(l);
            }
            flow_fcn<kFlowNT>(F, Lc, x, f.D, lane, fv);
#pragma unroll
            for (int t = 0; t < kFlowNT; ++t) {
                const uint64_t sl = pb + (uint64_t)(wave * a.tiles + q + t) * 16 + (lane & 15);
                const bool live = sl < a.n;
                if (fv[t] != fv[t] && live && a.status) atomicOr(a.status, (int32_t)VGX_ENAN);
                if (a.xout && live) *reinterpret_cast<f32x4_t*>(a.xout + sl * 16 + 4 * g) = x[t];
                if (g == 0) {
                    TS->l[q + t][lane] = fv[t];
                    TS->l[q + t][16 + lane] = LJ[t];
                }
            }
        }
        // the sums, a sample per lane, from what other lanes stored
        wave_lds_fence();
        for (int r = 0; r < a.tiles; r += 4) {
            const int q = r + (lane >> 4);
            const uint64_t sl = pb + (uint64_t)(wave * a.tiles + q) * 16 + (lane & 15);
            if (q < a.tiles && sl < a.n) {
                const float fl = TS->l[q][lane & 15], lj = TS->l[q][16 + (lane & 15)];
                // f = 0 where the map stretches enough for J to overflow is 0,
                // and so is a sample at the end of the unit interval: the last
                // of the 2^24 values of a z rounds to 1, whose u is infinite and
                // whose log J is a NaN where f is none
                const bool in = fl != 0.f && (lj == lj || fl != fl);
                const double fj = in ? (double)fl * exp_jac((double)lj) : 0.0;
                dd_add(s1, fj);
                dd_add(s2, fj * fj);
                if (a.xout) a.fout[sl] = (float)fj;
            }
        }
        wave_lds_fence();  // read before the next pass stores
    }
    s1 = wave_sum_dd(s1);
    s2 = wave_sum_dd(s2);
    if (lane == 0) {
        red[4 * wave] = s1.hi;
        red[4 * wave + 1] = s1.lo;
        red[4 * wave + 2] = s2.hi;
        red[4 * wave + 3] = s2.lo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        DD t1{0, 0}, t2{0, 0};
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            t1 = dd_sum(t1, DD{red[4 * w], red[4 * w + 1]});
            t2 = dd_sum(t2, DD{red[4 * w + 2], red[4 * w + 3]});
        }
        double* o = a.part + 4 * (size_t)blockIdx.x;
        o[0] = t1.hi; o[1] = t1.lo; o[2] = t2.hi; o[3] = t2.lo;
    }
}

// The integrand at given points x [n][16] (training data): f [n].
__global__ __launch_bounds__(256) void flow_eval_kernel(FlowFcn F, int D, const float* x, uint64_t n, float* fout) {
    extern __shared__ __align__(16) unsigned char smem[];
    float* Lc = reinterpret_cast<float*>(smem);
    load_fcn(F, D, Lc);
    __syncthreads();
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const uint64_t ntiles = (n + 15) / 16;
    for (uint64_t t = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); t < ntiles;
         t += (uint64_t)gridDim.x * (blockDim.x >> 6)) {
        const uint64_t sl = t * 16 + (lane & 15);
        f32x4_t xv[1] = {{0.5f, 0.5f, 0.5f, 0.5f}};
        if (sl < n) xv[0] = *reinterpret_cast<const f32x4_t*>(x + sl * 16 + 4 * g);
        float fv[1];
        flow_fcn<1>(F, Lc, xv, D, lane, fv);
        if (g == 0 && sl < n) fout[sl] = fv[0];
    }
}

// -------------------------------------------------------------- inverse ----
struct InvArgs {
    uint64_t n;
    const float* x;      // [n][16]
    float* saved;        // [L][n][16]: input of each layer
    float* u0;           // [n][16]
    float* logq;         // [n]
    int tiles;           // sample tiles per wave and pass (even, up to kFlowTiles)
};

__global__ __launch_bounds__(kFlowThreads) void flow_inverse_kernel(FlowArgs f, InvArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    LayerLds* L = reinterpret_cast<LayerLds*>(smem);
    TileState* TS = reinterpret_cast<TileState*>(smem + kLdsLayer) +
                    (threadIdx.x >> 6);
    const int wave = threadIdx.x >> 6;
    int lane = threadIdx.x & 63;
    const uint64_t pass = (blockDim.x >> 6) * a.tiles * 16;  // samples per pass of the workgroup
    for (uint64_t pb = blockIdx.x * pass; pb < a.n; pb += gridDim.x * pass) {
        asm volatile("" : "+v"(lane));  // addresses are formed when used, not held over the passes
        const int g = lane >> 4;
#pragma unroll 1
        for (int q = 0; q < a.tiles; ++q) {
            const uint64_t sl = pb + (uint64_t)(wave * a.tiles + q) * 16 + (lane & 15);
            f32x4_t xv = {0.5f, 0.5f, 0.5f, 0.5f};
            if (sl < a.n) xv = *reinterpret_cast<const f32x4_t*>(a.x + sl * 16 + 4 * g);
            float l = 0.f;
            f32x4_t uq;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float xc = fminf(fmaxf(xv[i], 1e-7f), 1.0f - 1e-7f);
                const float l0 = __logf(xc), l1 = __logf(1.0f - xc);
                uq[i] = (4 * g + i < f.D) ? l0 - l1 : 0.f;
                if (4 * g + i < f.D) l -= l0 + l1;
            }
            TS->u[q][lane] = uq;
            TS->l[q][lane] = l;
        }
        for (int k = f.L - 1; k >= 0; --k) {
            asm volatile("" : "+v"(lane));
            const int g = lane >> 4;
            __syncthreads();
            load_layer(f, k, L, false, nullptr);
            __syncthreads();
            const uint32_t am = f.amask[k];
#pragma unroll 1
            for (int q = 0; q < a.tiles; q += kFlowNT) {
                bf16x4_t ain[kFlowNT];
                f32x4_t o[kFlowNT][2];
                bf16x4_t h2[kFlowNT][8];
#pragma unroll
                for (int t = 0; t < kFlowNT; ++t) {
                    const uint64_t sl = pb + (uint64_t)(wave * a.tiles + q + t) * 16 + (lane & 15);
                    const f32x4_t uq = TS->u[q + t][lane];
                    if (sl < a.n) *reinterpret_cast<f32x4_t*>(a.saved + ((size_t)k * a.n + sl) * 16 + 4 * g) = uq;
                    ain[t] = cond_input(uq, am, f.D, lane);
                }
                mlp<kFlowNT>(L, ain, lane, o, h2);
#pragma unroll
                for (int t = 0; t < kFlowNT; ++t) {
                    f32x4_t uq = TS->u[q + t][lane];
                    float l = TS->l[q + t][lane];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int d = 4 * g + i;
                        if (d < f.D && !((am >> d) & 1u)) {
                            const float sv = kSMax * tanh_s(o[t][0][i]);
                            uq[i] = (uq[i] - o[t][1][i]) * __expf(-sv);
                            l -= sv;
                        }
                    }
                    TS->u[q + t][lane] = uq;
                    TS->l[q + t][lane] = l;
                }
            }
        }
#pragma unroll 1
        for (int q = 0; q < a.tiles; ++q) {
            const uint64_t sl = pb + (uint64_t)(wave * a.tiles + q) * 16 + (lane & 15);
            const f32x4_t uq = TS->u[q][lane];
            float l = TS->l[q][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * g + i < f.D) l += logsigp(uq[i]);
            const float LQ = group_sum(l);
            if (sl < a.n) {
                *reinterpret_cast<f32x4_t*>(a.u0 + sl * 16 + 4 * g) = uq;
                if (g == 0) a.logq[sl] = LQ;
            }
        }
    }
}

// ---------------------------------------------------------- loss weights ----
// log c_i = log w_i + 2 log|f_i| - log q_i (w given by its logarithm, so
// weights 1/(n q) of the flow's own samples cannot overflow); c normalised
// to sum 1 (two launches: the maximum, then the sum of exp(log c - max)).
// Terms that are not finite count as 0.
// pf, pq: exponents of |f| and q -- (2, 1) the variance loss, (1, 0) the
// forward KL divergence (maximum likelihood of the density |f|/I).
__device__ inline float lossw_log(const float* lw, const float* fv, const float* logq, uint64_t i, float pf,
                                  float pq) {
    const float fa = fabsf(fv[i]);
    if (!(fa > 0.f)) return -INFINITY;
    const float v = lw[i] + pf * __logf(fa) - pq * logq[i];
    return (v == v && fabsf(v) < INFINITY) ? v : -INFINITY;
}

__device__ inline uint32_t ord_f(float v) {
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ inline float unord_f(uint32_t o) {
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}

// One atomic per workgroup (the maximum is exact in any order).
__global__ __launch_bounds__(256) void flow_lossw_max_kernel(const float* w, const float* fv, const float* logq,
                                                             uint64_t n, float pf, float pq, uint32_t* mx) {
    __shared__ float red[4];
    float m = -INFINITY;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        m = fmaxf(m, lossw_log(w, fv, logq, i, pf, pq));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        if (m > -INFINITY) atomicMax(mx, ord_f(m));
    }
}

__global__ void flow_lossw_sum_kernel(const float* w, const float* fv, const float* logq, uint64_t n,
                                      float pf, float pq, const uint32_t* mx, float* c, double* part) {
    __shared__ double red[16];
    const bool none = *mx == 0u;  // no sample with f != 0
    const float m = none ? 0.f : unord_f(*mx);
    double s = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const float v = none ? 0.f : __expf(lossw_log(w, fv, logq, i, pf, pq) - m);
        c[i] = v;
        s += v;
    }
    s = wave_sum_fixed(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) t += red[k];
        part[blockIdx.x] = t;
    }
}

// The sum of the loss weights' partial sums, in a fixed order (thread t
// adds parts t, t + 256, ... in order; then the threads' sums in order).
__global__ __launch_bounds__(256) void flow_csum_kernel(const double* part, int nparts, double* out) {
    __shared__ double red[256];
    double t = 0.0;
    for (int i = threadIdx.x; i < nparts; i += 256) t += part[i];
    red[threadIdx.x] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        double u = 0.0;
        for (int i = 0; i < 256; ++i) u += red[i];
        *out = u;
    }
}

// ------------------------------------------------------------- backward ----
struct BwdArgs {
    uint64_t n;
    int k;                    // layer
    const float* saved;       // [L][n][16]
    const float* u0;          // [n][16]
    const float* c;           // [n] unnormalised weights
    const double* csum;       // the sum of c (flow_csum_kernel)
    float* G;                 // [n][16] dL/du (in: layer output; out: layer input)
    float* part;              // [gridDim.x][kPLayer] each workgroup's weight-gradient sums
};

// Backward of one layer together with its weight gradients.  Per round each
// wave takes one 16-sample tile (tile (round * gridDim.x + block) * 8 +
// wave), recomputes the layer's MLP, backpropagates through the coupling and
// the MLP, and the eight waves stage their GEMM operands in LDS in three
// phases:
//   1: dout (32 rows) | h2 (128)   -> dW3, b3
//   2: dh2 (128) | h1 (128)        -> dW2, b2 (h1 recomputed from a: 8 small MFMAs
//                                     instead of 16 registers held through the
//                                     backward GEMMs)
//   3: dh1 (128) | a (16)          -> dW1
// After each staging every wave adds its share of dW over the eight staged
// tiles, two tiles per v_mfma_f32_16x16x32_bf16 (k = the samples of both);
// an all-ones operand gives the bias sums.  The sums stay in registers over
// the rounds and are written once per workgroup: the operands never leave
// the CU.  The tile -> workgroup assignment is static, so the sums are
// reproducible.  Tiles past the end run on zero inputs: their dout is 0, so
// they add nothing.
// Two waves per SIMD (the registers of the sums) that meet at every phase:
// vector work, products and LDS reads mostly add up.  250,000 samples, 9
// axes: 95 us a layer with operands transposed in registers before staging
// (eight instructions a fragment, now transposed by the read) and a compare, a
// select and a bit per relu mask (now two packed instructions per two
// values), 69 us so; 13 us of it load the weights and write the sums.
// (Weight fragments read a step ahead, or 32 by 64 blocks of dW2 a wave,
// which need a third fewer operand reads: no change.)
constexpr int kBwdThreads = 512;
constexpr int kBwdWaves = kBwdThreads / 64;
constexpr int kSlotRows = 2 * kFH;         // the largest phase: dh2 | h1
// A slot is [sample][row], its row stride such that the 16 samples of a write
// and the 32-byte runs of a transposing read spread over the banks.
constexpr int kSlotLd = kSlotRows + 16;
constexpr int kSlot = kSlotLd * 16;        // bf16 elements per wave slot
constexpr int kNo3 = 2 * 9;                // dW3 output tiles: 2 row tiles x (8 column tiles + bias)

// The C-layout tile v (rows row0 + (l/16)*4 + i, sample l%16) into a slot, as
// it lies in the registers: one 8-byte write.
__device__ inline void stage(uint16_t* slot, int row0, const bf16x4_t v, int lane) {
    *reinterpret_cast<bf16x4_t*>(slot + (lane & 15) * kSlotLd + row0 + 4 * (lane >> 4)) = v;
}
// Operand fragment of slot rows row0.. (A and B alike: row row0 + l%16,
// samples (l/16)*4 .. +3), transposed by the read: in 16 lanes, lane 4 k + q
// reads rows 4 q .. +3 of sample k, and lane m receives row m of samples
// 0..3.
__device__ inline bf16x4_t frag_op(const uint16_t* slot, int row0, int lane) {
    typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4_t;
    const uint16_t* q = slot + (4 * (lane >> 4) + ((lane >> 2) & 3)) * kSlotLd + row0 + 4 * (lane & 3);
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4_t*)q);
}
// v where h > 0 (bf16 values, h not negative), 0 elsewhere: two values an
// instruction (the empty asm keeps the compiler from making a compare and a
// select of each).
__device__ inline bf16x4_t where_positive(const bf16x4_t v, const bf16x4_t h) {
    typedef short s16x2_t __attribute__((ext_vector_type(2)));
    typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
    const u32x2_t hv = __builtin_bit_cast(u32x2_t, h), vv = __builtin_bit_cast(u32x2_t, v);
    u32x2_t r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t hw = hv[i];
        const s16x2_t hs = __builtin_bit_cast(s16x2_t, hw);
        uint32_t m = __builtin_bit_cast(uint32_t, (s16x2_t)(-hs));
        asm("" : "+v"(m));
        m = __builtin_bit_cast(uint32_t, (s16x2_t)(__builtin_bit_cast(s16x2_t, m) >> 15));
        asm("" : "+v"(m));
        r[i] = vv[i] & m;
    }
    return __builtin_bit_cast(bf16x4_t, r);
}

// Rows row0.. of staged tiles j and j+1 as one k = 32 operand (A and B
// alike: slots 0..3 tile j's samples (l/16)*4.., slots 4..7 tile j+1's).
__device__ inline bf16x8_t frag_pair(const uint16_t* S, int j, int row0, int lane) {
    const uint16_t* s0 = S + j * kSlot;
    return cat8(frag_op(s0, row0, lane), frag_op(s0 + kSlot, row0, lane));
}

constexpr size_t kLdsBwd = kLdsLayer + sizeof(uint16_t) * kHLayer + sizeof(uint16_t) * (size_t)kBwdWaves * kSlot;
static_assert(kLdsBwd <= 160 * 1024, "backward LDS plan fits a CU");

__global__ __launch_bounds__(kBwdThreads) void flow_backward_kernel(FlowArgs f, BwdArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    LayerLds* L = reinterpret_cast<LayerLds*>(smem);
    uint16_t* Wt = reinterpret_cast<uint16_t*>(smem + kLdsLayer);
    uint16_t* S = Wt + kHLayer;
    // the wave index as a wave-uniform (SGPR) value: the output tiles a wave
    // owns and its slot address are then scalar
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4;
    uint16_t* my = S + w * kSlot;
    const int k = a.k;
    load_layer(f, k, L, true, Wt);
    __syncthreads();
    const double csum = *a.csum;
    const float inv_c = csum > 0 ? (float)(1.0 / csum) : 0.f;
    const uint32_t am = f.amask[k];
    const uint64_t ntiles = (a.n + 15) / 16;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t acc3[3], acc2[9], acc1 = zero;
#pragma unroll
    for (int q = 0; q < 9; ++q) acc2[q] = zero;
#pragma unroll
    for (int q = 0; q < 3; ++q) acc3[q] = zero;
    // all-ones operand (1 in column 0): row sums, the bias gradients
    bf16x4_t ones;
#pragma unroll
    for (int j = 0; j < 4; ++j) ones[j] = (lane & 15) == 0 ? (short)0x3F80 : (short)0;
    const bf16x8_t ones8 = cat8(ones, ones);
    // The inputs of a wave's next tile (saved u, c, and G or u0) are loaded
    // while the current tile computes.
    auto fetch = [&](uint64_t tl, f32x4_t& u, f32x4_t& gr, float& c) {
        const uint64_t s2 = tl * 16 + (lane & 15);
        u = zero;
        gr = zero;
        c = 0.f;
        if (tl < ntiles && s2 < a.n) {
            u = *reinterpret_cast<const f32x4_t*>(a.saved + ((size_t)k * a.n + s2) * 16 + 4 * g);
            c = a.c[s2];
            gr = *reinterpret_cast<const f32x4_t*>((k == 0 ? a.u0 : a.G) + s2 * 16 + 4 * g);
        }
    };
    const uint64_t per_round = (uint64_t)gridDim.x * kBwdWaves;
    const uint64_t rounds = (ntiles + per_round - 1) / per_round;
    uint64_t tile = (uint64_t)blockIdx.x * kBwdWaves + w;
    f32x4_t nx_u, nx_g;
    float nx_c;
    fetch(tile, nx_u, nx_g, nx_c);
    for (uint64_t rd = 0; rd < rounds; ++rd, tile += per_round) {
        const uint64_t sl = tile * 16 + (lane & 15);
        const bool live = sl < a.n;
        const f32x4_t uin = nx_u, graw = nx_g;
        const float cw = nx_c * inv_c;
        fetch(tile + per_round, nx_u, nx_g, nx_c);
        f32x4_t G = graw;
        if (k == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                G[i] = (live && 4 * g + i < f.D) ? -cw * (1.0f - 2.0f / (1.0f + __expf(-graw[i]))) : 0.f;
        }
        const bf16x4_t ain = cond_input(uin, am, f.D, lane);
        const bf16x4_t a1[1] = {ain};
        f32x4_t o1[1][2];
        bf16x4_t h2[1][8];
        mlp<1>(L, a1, lane, o1, h2);
        const f32x4_t (&o)[2] = o1[0];
        // coupling backward (inverse direction)
        f32x4_t dout0, dout1, Gin;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 4 * g + i;
            dout0[i] = 0.f;
            dout1[i] = 0.f;
            Gin[i] = G[i];
            if (d < f.D && !((am >> d) & 1u)) {
                const float th = tanh_s(o[0][i]);
                const float sv = kSMax * th;
                const float es = __expf(-sv);
                const float uout = (uin[i] - o[1][i]) * es;
                const float ds = -G[i] * uout + cw;
                dout0[i] = live ? ds * (1.0f - th * th) : 0.f;
                dout1[i] = live ? -G[i] * es : 0.f;
                Gin[i] = G[i] * es;
            }
        }
        const bf16x4_t do0 = pack_bf(dout0), do1 = pack_bf(dout1);
        // The staging and operand addresses of the phases below are formed
        // from this copy of the lane index when used (immediate offsets of the
        // LDS instructions): held from round to round they would take about
        // forty registers.
        int ln = lane;
        asm volatile("" : "+v"(ln));
        // ---- phase 1: dout | h2 -> dW3, b3 (output tile o = wave + 8 j)
        stage(my, 0, do0, ln);
        stage(my, 16, do1, ln);
#pragma unroll
        for (int q = 0; q < 8; ++q) stage(my, 32 + 16 * q, h2[0][q], ln);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBwdWaves; j += 2) {
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const int ot = w + kBwdWaves * e;
                if (ot < kNo3) {
                    const int q = ot % 9;
                    acc3[e] = mfma32(frag_pair(S, j, 16 * (ot / 9), ln),
                                     q < 8 ? frag_pair(S, j, 32 + 16 * q, ln) : ones8, acc3[e]);
                }
            }
        }
        // dh2 = W3^T dout (relu mask h2); dh1 = W2^T dh2 (mask h1); da = W1^T dh1
        bf16x4_t dh2[8];
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) {
            dh2[mt] = where_positive(pack_bf(mfma32(frag_w(Wt + kTW3, mt, lane), cat8(do0, do1), zero)), h2[0][mt]);
        }
        f32x4_t acc[8];
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) acc[mt] = zero;
#pragma unroll
        for (int kp2 = 0; kp2 < 4; ++kp2) {
            const bf16x8_t b = cat8(dh2[2 * kp2], dh2[2 * kp2 + 1]);
#pragma unroll
            for (int mt = 0; mt < 8; ++mt) acc[mt] = mfma32(frag_w(Wt + kTW2, mt * 4 + kp2, lane), b, acc[mt]);
            __builtin_amdgcn_sched_barrier(0);
        }
        bf16x4_t h1[1][8], dh1[8];
        layer1<1>(L, a1, lane, h1);
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) dh1[mt] = where_positive(pack_bf(acc[mt]), h1[0][mt]);
        f32x4_t da = zero;
#pragma unroll
        for (int kt = 0; kt < 8; kt += 2) da = mfma32(frag_w(Wt + kTW1, kt / 2, lane), cat8(dh1[kt], dh1[kt + 1]), da);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 4 * g + i;
            if (d < f.D && ((am >> d) & 1u)) Gin[i] += da[i];
        }
        if (live) *reinterpret_cast<f32x4_t*>(a.G + sl * 16 + 4 * g) = Gin;
        __syncthreads();
        // ---- phase 2: dh2 | h1 -> dW2, b2
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            stage(my, 16 * q, dh2[q], ln);
            stage(my, kFH + 16 * q, h1[0][q], ln);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBwdWaves; j += 2) {
            const bf16x8_t av = frag_pair(S, j, 16 * w, ln);
#pragma unroll
            for (int q = 0; q < 8; ++q) acc2[q] = mfma32(av, frag_pair(S, j, kFH + 16 * q, ln), acc2[q]);
            acc2[8] = mfma32(av, ones8, acc2[8]);
        }
        __syncthreads();
        // ---- phase 3: dh1 | a -> dW1
#pragma unroll
        for (int q = 0; q < 8; ++q) stage(my, 16 * q, dh1[q], ln);
        stage(my, kFH, ain, ln);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBwdWaves; j += 2) acc1 = mfma32(frag_pair(S, j, 16 * w, ln), frag_pair(S, j, kFH, ln), acc1);
        __syncthreads();
    }
    // C layout: lane l, i -> dW[16 r + (l/16)*4 + i][16 q + l%16]
    float* o = a.part + (size_t)blockIdx.x * kPLayer;
    const int cc = lane & 15;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int rr = 4 * g + i, r2 = 16 * w + rr;
#pragma unroll
        for (int q = 0; q < 8; ++q) o[kPW2 + r2 * kFH + 16 * q + cc] = acc2[q][i];
        if (cc == 0) o[kPB2 + r2] = acc2[8][i];
        o[kPW1 + r2 * kFI + cc] = acc1[i];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int ot = w + kBwdWaves * j;
            if (ot < kNo3) {
                const int q = ot % 9, row = 16 * (ot / 9) + rr;
                if (q < 8)
                    o[kPW3 + row * kFH + 16 * q + cc] = acc3[j][i];
                else if (cc == 0)
                    o[kPB3 + row] = acc3[j][i];
            }
        }
    }
}

// Sum of the workgroup partials into grad [kPLayer], in a fixed order: a
// workgroup takes 32 consecutive entries; its 8 part groups (thread j sums
// parts j, j + 8, ... in order) are added in group order.  Each wave reads
// 2 x 128 contiguous bytes per load, and 709 workgroups keep the loads of
// the whole device in flight.
constexpr int kRedCols = 32, kRedGroups = 8;

__global__ __launch_bounds__(kRedCols * kRedGroups) void flow_wgrad_reduce_kernel(const float* part, int nparts,
                                                                                  float* grad) {
    __shared__ double red[kRedGroups][kRedCols];
    const int il = threadIdx.x % kRedCols, j = threadIdx.x / kRedCols;
    const int i = blockIdx.x * kRedCols + il;
    double s = 0.0;
    if (i < kPLayer) {
        int p = j;
        for (; p + 3 * kRedGroups < nparts; p += 4 * kRedGroups) {
            const float v0 = part[(size_t)p * kPLayer + i];
            const float v1 = part[(size_t)(p + kRedGroups) * kPLayer + i];
            const float v2 = part[(size_t)(p + 2 * kRedGroups) * kPLayer + i];
            const float v3 = part[(size_t)(p + 3 * kRedGroups) * kPLayer + i];
            s += v0;
            s += v1;
            s += v2;
            s += v3;
        }
        for (; p < nparts; p += kRedGroups) s += part[(size_t)p * kPLayer + i];
    }
    red[j][il] = s;
    __syncthreads();
    if (j == 0 && i < kPLayer) {
        double t = 0.0;
        for (int q = 0; q < kRedGroups; ++q) t += red[q][il];
        grad[i] = (float)t;
    }
}

// ------------------------------------------------------------------ adam ----
struct AdamArgs {
    float* P;
    const float* grad;
    float* m;
    float* v;
    uint16_t* H;
    uint16_t* HT;
    int L;
    float lr, b1, b2, eps, c1, c2;   // c1 = 1 - b1^t, c2 = 1 - b2^t
    float clip;                       // gradient clip (max abs), 0 = none
};

__global__ void flow_adam_kernel(AdamArgs a) {
    const int total = a.L * kPLayer;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        float gr = a.grad[i];
        if (!(fabsf(gr) < INFINITY)) gr = 0.f;  // a non-finite component is skipped
        if (a.clip > 0) gr = fminf(fmaxf(gr, -a.clip), a.clip);
        const float m = a.b1 * a.m[i] + (1.f - a.b1) * gr;
        const float v = a.b2 * a.v[i] + (1.f - a.b2) * gr * gr;
        a.m[i] = m;
        a.v[i] = v;
        a.P[i] = a.P[i] - a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
    }
}

// bf16 copies (and transposes) of the weights after an update, in fragment
// order.
__global__ void flow_cast_kernel(const float* P, uint16_t* H, uint16_t* HT, int L) {
    constexpr int nlog = kFH * kFI + kFH * kFH + kFO * kFH;
    const int total = L * nlog;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int k = i / nlog, r = i % nlog;
        const float* p = P + (size_t)k * kPLayer;
        float v;
        int rh, rt;
        if (r < kFH * kFI) {                 // W1 [128][16] -> W1t [16][128]
            const int o = r / kFI, c = r % kFI;
            v = p[kPW1 + r];
            rh = kHW1 + frag_pos1(o, c);
            rt = kTW1 + frag_pos(c, o, 4);
        } else if (r < kFH * kFI + kFH * kFH) {  // W2 [128][128]
            const int q = r - kFH * kFI, o = q / kFH, c = q % kFH;
            v = p[kPW2 + q];
            rh = kHW2 + frag_pos(o, c, 4);
            rt = kTW2 + frag_pos(c, o, 4);
        } else {                             // W3 [32][128] -> W3t [128][32]
            const int q = r - kFH * kFI - kFH * kFH, o = q / kFH, c = q % kFH;
            v = p[kPW3 + q];
            rh = kHW3 + frag_pos(o, c, 4);
            rt = kTW3 + frag_pos(c, o, 1);
        }
        const uint16_t h = f2bf(v);
        H[(size_t)k * kHLayer + rh] = h;
        HT[(size_t)k * kHLayer + rt] = h;
    }
}

__global__ void flow_zero_u32_kernel(uint32_t* p, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0u;
}

// MFMA lane-layout probe: D = A B for 16x16 bf16 A, B given row-major.
__global__ void flow_mfma_probe_kernel(const uint16_t* A, const uint16_t* B, float* D) {
    const int lane = threadIdx.x & 63;
    bf16x4_t a, b;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        a[j] = (short)A[(lane & 15) * 16 + (lane >> 4) * 4 + j];
        b[j] = (short)B[((lane >> 4) * 4 + j) * 16 + (lane & 15)];
    }
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const f32x4_t c = mfma16(a, b, zero);
#pragma unroll
    for (int i = 0; i < 4; ++i) D[((lane >> 4) * 4 + i) * 16 + (lane & 15)] = c[i];
}

}  // namespace vgx

// ------------------------------------------------------------ host side ----
using namespace vgx;

struct vgx_flow {
    int D = 0, L = 0;
    uint32_t amask[kFMaxL] = {};
    float* P = nullptr;      // FP32 master [L][kPLayer]
    float* m = nullptr;
    float* v = nullptr;
    float* grad = nullptr;
    uint16_t* H = nullptr;
    uint16_t* HT = nullptr;
    // per-batch scratch (grown on demand)
    Scratch saved, u0, logq, c, G, wpart, cpart, spart, misc;
    hipEvent_t held = nullptr;  // an integrand's parameters have been copied
    hipEvent_t used = nullptr;  // and the copy read
    std::mutex hold_mu;         // from the one's record to the other's
    int step = 0;
};

static FlowArgs flow_args(const vgx_flow* fl) {
    FlowArgs f{};
    f.D = fl->D;
    f.L = fl->L;
    for (int k = 0; k < fl->L; ++k) f.amask[k] = fl->amask[k];
    f.P = fl->P;
    f.H = fl->H;
    f.HT = fl->HT;
    return f;
}

static size_t lds_layer() { return kLdsLayer; }
// backward: the layer, the transposed weights, the operand slots of the waves
static size_t lds_bwd() { return kLdsBwd; }

static int flow_cast(vgx_flow* fl, hipStream_t s) {
    hipLaunchKernelGGL(flow_cast_kernel, dim3(256), dim3(256), 0, s, (const float*)fl->P, fl->H, fl->HT, fl->L);
    return check_launch();
}

extern "C" int vgx_flow_destroy(vgx_flow* fl);

extern "C" int vgx_flow_create(int dim, int nlayers, const uint32_t* amask, vgx_flow** out) {
    if (!out || !amask || dim < 1 || dim > kFI - 1 || nlayers < 1 || nlayers > kFMaxL) return VGX_EINVAL;
    vgx_flow* fl = new vgx_flow();
    fl->D = dim;
    fl->L = nlayers;
    for (int k = 0; k < nlayers; ++k) fl->amask[k] = amask[k] & ((1u << dim) - 1u);
    const size_t np = (size_t)nlayers * kPLayer, nh = (size_t)nlayers * kHLayer;
    if (hipMalloc(&fl->P, np * 4) != hipSuccess || hipMalloc(&fl->m, np * 4) != hipSuccess ||
        hipMalloc(&fl->v, np * 4) != hipSuccess || hipMalloc(&fl->grad, np * 4) != hipSuccess ||
        hipMalloc(&fl->H, nh * 2) != hipSuccess || hipMalloc(&fl->HT, nh * 2) != hipSuccess) {
        delete fl;
        return VGX_ENOMEM;
    }
    if (hipMemset(fl->P, 0, np * 4) != hipSuccess || hipMemset(fl->m, 0, np * 4) != hipSuccess ||
        hipMemset(fl->v, 0, np * 4) != hipSuccess || hipMemset(fl->grad, 0, np * 4) != hipSuccess ||
        hipMemset(fl->H, 0, nh * 2) != hipSuccess || hipMemset(fl->HT, 0, nh * 2) != hipSuccess) {
        vgx_flow_destroy(fl);
        return VGX_EHIP;
    }
    if (hipFuncSetAttribute((const void*)flow_backward_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds_bwd()) != hipSuccess ||
        hipFuncSetAttribute((const void*)flow_inverse_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)(lds_layer() + kStateLds)) != hipSuccess ||
        hipEventCreateWithFlags(&fl->held, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&fl->used, hipEventDisableTiming) != hipSuccess) {
        vgx_flow_destroy(fl);
        return VGX_EHIP;
    }
    *out = fl;
    return VGX_OK;
}

extern "C" int vgx_flow_destroy(vgx_flow* fl) {
    if (!fl) return VGX_OK;
    (void)hipDeviceSynchronize();
    void* ps[] = {fl->P, fl->m, fl->v, fl->grad, fl->H, fl->HT};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    Scratch* ss[] = {&fl->saved, &fl->u0, &fl->logq, &fl->c, &fl->G, &fl->wpart, &fl->cpart, &fl->spart,
                     &fl->misc};
    for (Scratch* q : ss) q->release();
    for (hipEvent_t e : {fl->held, fl->used})
        if (e) (void)hipEventDestroy(e);
    delete fl;
    return VGX_OK;
}

extern "C" int vgx_flow_nparams(const vgx_flow* fl, int64_t* n) {
    if (!fl || !n) return VGX_EINVAL;
    *n = (int64_t)fl->L * kPLayer;
    return VGX_OK;
}

extern "C" int vgx_flow_set_params(vgx_flow* fl, const float* host, void* stream) {
    if (!fl || !host) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const size_t np = (size_t)fl->L * kPLayer;
    VGX_HIP(hipMemcpyAsync(fl->P, host, np * 4, hipMemcpyHostToDevice, s));
    VGX_HIP(hipMemsetAsync(fl->m, 0, np * 4, s));
    VGX_HIP(hipMemsetAsync(fl->v, 0, np * 4, s));
    fl->step = 0;
    int rc = flow_cast(fl, s);
    if (rc) return rc;
    VGX_HIP(hipStreamSynchronize(s));
    return VGX_OK;
}

extern "C" int vgx_flow_get_params(const vgx_flow* fl, float* host, float* grad_host, void* stream) {
    if (!fl) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const size_t np = (size_t)fl->L * kPLayer;
    if (host) VGX_HIP(hipMemcpyAsync(host, fl->P, np * 4, hipMemcpyDeviceToHost, s));
    if (grad_host) VGX_HIP(hipMemcpyAsync(grad_host, fl->grad, np * 4, hipMemcpyDeviceToHost, s));
    VGX_HIP(hipStreamSynchronize(s));
    return VGX_OK;
}

// Sampling scratch: a workgroup's sums (one workgroup per CU) | a copy of an
// integrand's FP64 parameters (kFlowFcnMax bytes as FP32).
constexpr size_t kFlowFcnMax = 48 * 1024;
static int flow_spart(vgx_flow* fl, const DeviceInfo& info) {
    return fl->spart.ensure((size_t)info.cus * 4 * 8 + 2 * kFlowFcnMax);
}

// The integrand as the kernels read it (its arrays are the caller's), and its
// LDS bytes.
static int flow_fcn_params(const vgx_flow* fl, const vgx_integrand* fcn, FlowFcn* F, size_t* lds) {
    if (!fcn || (fcn->kind != VGX_FCN_GAUSSMIX && fcn->kind != VGX_FCN_DIAGRIDGE) || fcn->ncomp < 1)
        return VGX_EINVAL;
    if (!fcn->A || !fcn->B || !fcn->c) return VGX_EINVAL;
    const size_t nc = (size_t)fcn->ncomp;
    *lds = (2 * nc + (fcn->kind == VGX_FCN_GAUSSMIX ? nc * fl->D : nc)) * 4;
    if (*lds > kFlowFcnMax) return VGX_ERANGE;  // staged in LDS with the layer
    *F = FlowFcn{fcn->kind, fcn->ncomp, fcn->A, fcn->B, fcn->c};
    return VGX_OK;
}

// For a call that returns before its kernel has run: the kernel reads a copy of
// the arrays, and flow_params_held, after its launch, waits until that has been
// taken, so that the caller may reuse or free them.  (The kernel is then
// already in the queue: waiting for the copy before the launch would leave
// the GPU idle for the launch.)  A second stream's copy waits for the first's
// reader; lk (of hold_mu) is held from one to the other, so that a second
// thread's call sees that reader.
static int flow_hold_params(vgx_flow* fl, FlowFcn* F, size_t lds, hipStream_t s) {
    const int na = F->ncomp, nc = (int)(lds / 4) - 2 * na;
    DeviceInfo info;
    int rc = device_info(&info);
    if (rc || (rc = flow_spart(fl, info))) return rc;
    double* d = (double*)fl->spart.ptr + 4 * (size_t)info.cus;
    VGX_HIP(hipStreamWaitEvent(s, fl->used, 0));
    hipLaunchKernelGGL(flow_hold_kernel, dim3((2 * na + nc + 1023) / 1024), dim3(256), 0, s, *F, na, nc, d);
    if ((rc = check_launch())) return rc;
    VGX_HIP(hipEventRecord(fl->held, s));
    F->A = d;
    F->B = d + na;
    F->c = d + 2 * na;
    return VGX_OK;
}
static int flow_params_held(vgx_flow* fl, hipStream_t s, std::unique_lock<std::mutex>& lk) {
    VGX_HIP(hipEventRecord(fl->used, s));
    lk.unlock();
    VGX_HIP(hipEventSynchronize(fl->held));
    return VGX_OK;
}

// Whether a call on s returns before its kernel has run.  (Not so a captured
// one, whose kernel runs when the graph does and reads the arrays then.)
static int flow_holds(hipStream_t s, bool* hold) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    VGX_HIP(hipStreamIsCapturing(s, &st));
    *hold = st == hipStreamCaptureStatusNone;
    return VGX_OK;
}

extern "C" int vgx_flow_sample(vgx_flow* fl, const vgx_integrand* fcn, int64_t n, uint64_t base, uint64_t seed,
                               uint32_t iteration, double* sums, float* xout, float* fout, int32_t* status,
                               void* stream) {
    if (!fl || n < 1 || (!sums && (!xout || !fout))) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    FlowFcn F{};
    size_t fcn_lds;
    int rc = flow_fcn_params(fl, fcn, &F, &fcn_lds);
    if (rc) return rc;
    bool hold = false;
    if (!sums && (rc = flow_holds(s, &hold))) return rc;
    std::unique_lock<std::mutex> lk(fl->hold_mu, std::defer_lock);
    if (hold) lk.lock();
    if (hold && (rc = flow_hold_params(fl, &F, fcn_lds, s))) return rc;
    DeviceInfo info;
    if ((rc = device_info(&info))) return rc;
    const FlowShape sh = flow_shape(n, info.cus, info.cus, fcn_lds);
    const int blocks = sh.blocks;
    if ((rc = flow_spart(fl, info))) return rc;
    SampleArgs a{};
    a.n = (uint64_t)n;
    a.base = base;
    a.seed_lo = (uint32_t)seed;
    a.seed_hi = (uint32_t)(seed >> 32);
    a.iteration = iteration;
    a.tiles = sh.tiles;
    a.part = (double*)fl->spart.ptr;
    a.xout = xout;
    a.fout = fout;
    a.status = status;
    const size_t lds = lds_layer() + sh.waves * sizeof(TileState) + fcn_lds;
    if (hipFuncSetAttribute((const void*)flow_sample_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
        return VGX_EHIP;
    hipEvent_t e0, e1;
    if (timed_slot(g_timing_ctx, kTimedFlowSample, &e0, &e1))
        hipExtLaunchKernelGGL(flow_sample_kernel, dim3(blocks), dim3(64 * sh.waves), (uint32_t)lds, s, e0, e1, 0,
                              flow_args(fl), F, a);
    else
        hipLaunchKernelGGL(flow_sample_kernel, dim3(blocks), dim3(64 * sh.waves), lds, s, flow_args(fl), F, a);
    if ((rc = check_launch())) return rc;
    if (!sums) return hold ? flow_params_held(fl, s, lk) : VGX_OK;
    std::vector<double> h((size_t)blocks * 4);
    VGX_HIP(hipMemcpyAsync(h.data(), a.part, h.size() * 8, hipMemcpyDeviceToHost, s));
    VGX_HIP(hipStreamSynchronize(s));
    DD t1{0, 0}, t2{0, 0};
    for (int b = 0; b < blocks; ++b) {
        t1 = dd_sum(t1, DD{h[4 * b], h[4 * b + 1]});
        t2 = dd_sum(t2, DD{h[4 * b + 2], h[4 * b + 3]});
    }
    sums[0] = t1.hi + t1.lo;
    sums[1] = t2.hi + t2.lo;
    return VGX_OK;
}

static int flow_inverse(vgx_flow* fl, const float* x, int64_t n, hipStream_t s) {
    int rc;
    const size_t nn = (size_t)n;
    if ((rc = fl->saved.ensure((size_t)fl->L * nn * 64))) return rc;
    if ((rc = fl->u0.ensure(nn * 64))) return rc;
    if ((rc = fl->logq.ensure(nn * 4))) return rc;
    DeviceInfo info;
    if ((rc = device_info(&info))) return rc;
    const FlowShape sh = flow_shape(n, info.cus, 2 * info.cus, 0);
    InvArgs a{(uint64_t)n, x, (float*)fl->saved.ptr, (float*)fl->u0.ptr, (float*)fl->logq.ptr, sh.tiles};
    hipLaunchKernelGGL(flow_inverse_kernel, dim3(sh.blocks), dim3(64 * sh.waves), lds_layer() + kStateLds, s,
                       flow_args(fl), a);
    return check_launch();
}

extern "C" int vgx_flow_logq(vgx_flow* fl, const float* x, int64_t n, float* logq, float* u0, void* stream) {
    if (!fl || !x || !logq || n < 1) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    int rc = flow_inverse(fl, x, n, s);
    if (rc) return rc;
    VGX_HIP(hipMemcpyAsync(logq, fl->logq.ptr, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    if (u0) VGX_HIP(hipMemcpyAsync(u0, fl->u0.ptr, (size_t)n * 64, hipMemcpyDeviceToDevice, s));
    return VGX_OK;
}

extern "C" int vgx_flow_grad(vgx_flow* fl, const float* x, const float* f, const float* logw, int64_t n,
                             int loss, void* stream) {
    if (!fl || !x || !f || !logw || n < 1) return VGX_EINVAL;
    if (loss != VGX_FLOW_LOSS_VARIANCE && loss != VGX_FLOW_LOSS_KL && loss != VGX_FLOW_LOSS_SQUARED) return VGX_EINVAL;
    const float* w = logw;
    hipStream_t s = (hipStream_t)stream;
    int rc = flow_inverse(fl, x, n, s);
    if (rc) return rc;
    const size_t nn = (size_t)n;
    const uint64_t ntiles = (nn + 15) / 16;
    const int nc = 1024;
    if ((rc = fl->c.ensure(nn * 4))) return rc;
    if ((rc = fl->G.ensure(nn * 64))) return rc;
    if ((rc = fl->cpart.ensure(nc * 8))) return rc;
    if ((rc = fl->misc.ensure(256))) return rc;
    DeviceInfo info;
    if ((rc = device_info(&info))) return rc;
    // one workgroup per CU (the layer's weights and the operand slots fill
    // the LDS), each writing its own weight-gradient sums
    const int nparts = (int)std::min<uint64_t>((uint64_t)info.cus, (ntiles + kBwdWaves - 1) / kBwdWaves);
    if ((rc = fl->wpart.ensure((size_t)nparts * kPLayer * 4))) return rc;
    uint32_t* mx = (uint32_t*)fl->misc.ptr;
    hipLaunchKernelGGL(flow_zero_u32_kernel, dim3(1), dim3(64), 0, s, mx, 1);
    const float pf = loss == VGX_FLOW_LOSS_KL ? 1.f : 2.f, pq = loss == VGX_FLOW_LOSS_VARIANCE ? 1.f : 0.f;
    hipLaunchKernelGGL(flow_lossw_max_kernel, dim3(256), dim3(256), 0, s, w, f, (const float*)fl->logq.ptr,
                       (uint64_t)n, pf, pq, mx);
    hipLaunchKernelGGL(flow_lossw_sum_kernel, dim3(nc), dim3(256), 0, s, w, f, (const float*)fl->logq.ptr,
                       (uint64_t)n, pf, pq, (const uint32_t*)mx, (float*)fl->c.ptr, (double*)fl->cpart.ptr);
    hipLaunchKernelGGL(flow_csum_kernel, dim3(1), dim3(256), 0, s, (const double*)fl->cpart.ptr, nc,
                       (double*)fl->misc.ptr + 1);
    if ((rc = check_launch())) return rc;
    const size_t blds = lds_bwd();
    for (int k = 0; k < fl->L; ++k) {
        BwdArgs b{};
        b.n = (uint64_t)n;
        b.k = k;
        b.saved = (const float*)fl->saved.ptr;
        b.u0 = (const float*)fl->u0.ptr;
        b.c = (const float*)fl->c.ptr;
        b.csum = (const double*)fl->misc.ptr + 1;
        b.G = (float*)fl->G.ptr;
        b.part = (float*)fl->wpart.ptr;
        hipEvent_t e0, e1;
        if (timed_slot(g_timing_ctx, kTimedFlowBwd, &e0, &e1))
            hipExtLaunchKernelGGL(flow_backward_kernel, dim3(nparts), dim3(kBwdThreads), (uint32_t)blds, s, e0, e1, 0,
                                  flow_args(fl), b);
        else
            hipLaunchKernelGGL(flow_backward_kernel, dim3(nparts), dim3(kBwdThreads), blds, s, flow_args(fl), b);
        hipLaunchKernelGGL(flow_wgrad_reduce_kernel, dim3((kPLayer + kRedCols - 1) / kRedCols),
                           dim3(kRedCols * kRedGroups), 0, s,
                           (const float*)fl->wpart.ptr, nparts,
                           fl->grad + (size_t)k * kPLayer);
        if ((rc = check_launch())) return rc;
    }
    return VGX_OK;
}

extern "C" int vgx_flow_adam(vgx_flow* fl, float lr, float b1, float b2, float eps, float clip, void* stream) {
    if (!fl) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    fl->step += 1;
    AdamArgs a{};
    a.P = fl->P;
    a.grad = fl->grad;
    a.m = fl->m;
    a.v = fl->v;
    a.H = fl->H;
    a.HT = fl->HT;
    a.L = fl->L;
    a.lr = lr;
    a.b1 = b1;
    a.b2 = b2;
    a.eps = eps;
    a.c1 = 1.f - powf(b1, (float)fl->step);
    a.c2 = 1.f - powf(b2, (float)fl->step);
    a.clip = clip;
    hipLaunchKernelGGL(flow_adam_kernel, dim3(256), dim3(256), 0, s, a);
    int rc = check_launch();
    if (rc) return rc;
    return flow_cast(fl, s);
}

extern "C" int vgx_flow_eval(vgx_flow* fl, const vgx_integrand* fcn, const float* x, int64_t n, float* f,
                             void* stream) {
    if (!fl || !x || !f || n < 1) return VGX_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    FlowFcn F{};
    size_t fcn_lds;
    int rc = flow_fcn_params(fl, fcn, &F, &fcn_lds);
    if (rc) return rc;
    const uint64_t ntiles = ((uint64_t)n + 15) / 16;
    const unsigned blocks = (unsigned)std::min<uint64_t>(4096, (ntiles + 3) / 4);
    if (hipFuncSetAttribute((const void*)flow_eval_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)(fcn_lds + 16)) != hipSuccess)
        return VGX_EHIP;
    bool hold = false;
    if ((rc = flow_holds(s, &hold))) return rc;
    std::unique_lock<std::mutex> lk(fl->hold_mu, std::defer_lock);
    if (hold) lk.lock();
    if (hold && (rc = flow_hold_params(fl, &F, fcn_lds, s))) return rc;
    hipLaunchKernelGGL(flow_eval_kernel, dim3(blocks), dim3(256), fcn_lds + 16, s, F, fl->D, x, (uint64_t)n, f);
    if ((rc = check_launch())) return rc;
    return hold ? flow_params_held(fl, s, lk) : VGX_OK;
}

extern "C" int vgx_flow_mfma_probe(const uint16_t* A, const uint16_t* B, float* D, void* stream) {
    if (!A || !B || !D) return VGX_EINVAL;
    hipLaunchKernelGGL(flow_mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, A, B, D);
    return check_launch();
}
