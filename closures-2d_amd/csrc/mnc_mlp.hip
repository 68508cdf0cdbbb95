// mnc_mlp.hip -- the learned warm start: an MLP 15 -> 128 -> 128 -> 128 -> 15
// with GELU, mapping the scaled moments u/u0 of an M4 closure to its scaled
// multipliers (alpha of the u0 = 1 problem), trained and evaluated with
// hand-written gfx950 kernels.  The reference has no counterpart (it starts
// every Newton solve from the previous step's alpha, momopt_update.cpp:236-238).
//
// Arithmetic: GEMM operands are rounded to bf16 (weights and activations) and
// multiplied on the matrix cores (v_mfma_f32_16x16x32_bf16) with FP32 sums; the
// master weights, biases, Adam moments and every elementwise step are FP32.
// Inputs and targets are standardised per component with statistics kept
// beside the weights.
//
// A training step is two launches: net_kernel (gather, forward, loss, backward) and
// update_kernel (weight gradients, Adam).  Measured at 4,096
// rows: 618 us before, in thirteen launches a step that read operands in 4-byte strides; now 28 us (17 + 11).
//
// Layouts (row-major FP32): a layer's weight is W[in][out] (y = x W + b).  The
// parameter vector is
//   W1[15][128] b1[128] W2[128][128] b2[128] W3[128][128] b3[128] W4[128][15] b4[15]
// (37,007 values), followed by in_mean[15] in_std[15] out_mean[15] out_std[15].
#include <algorithm>

#include "mnc_internal.h"

namespace mnc {
namespace {

typedef float mf32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 mbf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short mu16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ unsigned short to_bf16(float x) {
    const unsigned u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16);   // inf/NaN kept
    return (unsigned short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// GELU(x) = x Phi(x) and its derivative Phi(x) + x phi(x) (the exact, erf form).
// Both from one erf: the training pass keeps the derivative, not the argument.
__device__ __forceinline__ float gelu(float x, float e) { return 0.5f * x * (1.0f + e); }
__device__ __forceinline__ float gelu_grad(float x, float e) {
    const float cdf = 0.5f * (1.0f + e);
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

constexpr int kIn = 15, kH = 128, kOut = 15;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + kIn * kH, OFF_W2 = OFF_B1 + kH, OFF_B2 = OFF_W2 + kH * kH,
              OFF_W3 = OFF_B2 + kH, OFF_B3 = OFF_W3 + kH * kH, OFF_W4 = OFF_B3 + kH, OFF_B4 = OFF_W4 + kH * kOut,
              NPARAM = OFF_B4 + kOut;
static_assert(NPARAM == 37007, "parameter count");

// The weights as bf16 matrix operands, kept beside the FP32 masters: T = [out][in]
// for the forward products (a lane's eight k are 16 consecutive bytes), W = [in][out]
// for the backward ones; the 15-wide dimensions are padded with zeros.
constexpr int PK_T1 = 0, PK_T2 = PK_T1 + kH * 32, PK_T3 = PK_T2 + kH * kH, PK_T4 = PK_T3 + kH * kH,
              PK_W2 = PK_T4 + 16 * kH, PK_W3 = PK_W2 + kH * kH, PK_W4 = PK_W3 + kH * kH, PK_N = PK_W4 + kH * 32;

// The operands of the weight gradients, stored by the training pass: per block of
// 16 rows, [column][16 rows] in bf16, so that eight rows of a column are 16
// consecutive bytes and a wave's stores and loads are contiguous.
constexpr int CX = 0, CDY = 16, CA1 = 32, CA2 = CA1 + kH, CA3 = CA2 + kH, CZ1 = CA3 + kH, CZ2 = CZ1 + kH,
              CZ3 = CZ2 + kH, kCols = CZ3 + kH;
// dZ1 dZ2 dZ3 dY in FP32 for the bias sums, [column][row] over whole row blocks
constexpr int kBiasCols = 3 * kH + kOut;

__device__ __forceinline__ void pack_weight(unsigned short *pk, int i, float w) {
    const unsigned short h = to_bf16(w);
    if (i < OFF_B1) {
        pk[PK_T1 + (i % kH) * 32 + i / kH] = h;
    } else if (i >= OFF_W2 && i < OFF_B2) {
        const int k = (i - OFF_W2) / kH, j = (i - OFF_W2) % kH;
        pk[PK_T2 + j * kH + k] = h;
        pk[PK_W2 + k * kH + j] = h;
    } else if (i >= OFF_W3 && i < OFF_B3) {
        const int k = (i - OFF_W3) / kH, j = (i - OFF_W3) % kH;
        pk[PK_T3 + j * kH + k] = h;
        pk[PK_W3 + k * kH + j] = h;
    } else if (i >= OFF_W4 && i < OFF_B4) {
        const int k = (i - OFF_W4) / kOut, j = (i - OFF_W4) % kOut;
        pk[PK_T4 + j * kH + k] = h;
        pk[PK_W4 + k * 32 + j] = h;
    }
}

// The whole operand buffer from the masters (its padding included).
__global__ __launch_bounds__(256) void pack_kernel(const float *w, unsigned short *pk) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < NPARAM) pack_weight(pk, i, w[i]);
    if (i < kH * 17) {                                    // k = 15 .. 31 of T1 and W4
        const int r = i / 17, k = 15 + i % 17;
        pk[PK_T1 + r * 32 + k] = 0;
        pk[PK_W4 + r * 32 + k] = 0;
    }
    if (i < kH) pk[PK_T4 + 15 * kH + i] = 0;
}

// SplitMix64 (Steele, Lea & Flood 2014): the sample index of row i at step s.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}


// Rows of the network: drawn with replacement (seed != 0), list[i] of the
// unscaled moments u (list != null), or i0 + i.
struct NetArgs {
    const float *w;              // masters and standardisation
    const unsigned short *pk;
    const double *us, *as;
    const int *list, *count;     // count: if set, rows = *count, read on the device
    long long npairs, i0;
    unsigned long long seed;
    int rows;
    double *alpha;               // predictions, alpha[list ? list[i] : i][15]
    unsigned short *ops;         // training: [row block][kCols][16]
    float *dz;                   // training: [kBiasCols][16 ceil(rows / 16)]
    float *loss;                 // training: [row block]
};

__device__ __forceinline__ mf32x4 mma(mu16x8 a, mu16x8 b, mf32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mbf16x8, a), __builtin_bit_cast(mbf16x8, b), c, 0, 0, 0);
}

// B operands of 16 columns from rows of `ld` values: lane l takes row j0 + l%16,
// values 32 ks + 8 (l/16) .. + 7.
template <int KS>
__device__ __forceinline__ void load_ops(mu16x8 (&b)[KS], const unsigned short *p, int ld, int j0, int lane) {
#pragma unroll
    for (int k = 0; k < KS; ++k) b[k] = *(const mu16x8 *)(p + (j0 + (lane & 15)) * ld + 32 * k + 8 * (lane >> 4));
}

constexpr int kActStride = kH + 8;      // 272 B: the 16 rows' 16-byte reads fall on different banks
constexpr int kInStride = 40;

template <int KS, int STRIDE>
__device__ __forceinline__ mf32x4 mul(const unsigned short *act, const mu16x8 (&b)[KS], int lane) {
    mf32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k)
        acc = mma(*(const mu16x8 *)(act + (lane & 15) * STRIDE + 32 * k + 8 * (lane >> 4)), b[k], acc);
    return acc;
}

constexpr int kNetThreads = 512;

// One block of eight waves per 16 rows; wave v owns columns 16 v .. 16 v + 15 of
// every hidden layer.  What bounds it is latency: 16 rows need 3.5 MFLOP (0.4 us
// of a CU's matrix rate) and 6,144 GELUs behind a chain of 4 (predicting) or 7
// (training) dependent products, each closed by an LDS exchange.  So all weight
// operands (64 or 150 KB a block, out of L2) are loaded into registers before the
// first product, where the sample gather's latency covers them; activations pass
// from layer to layer in LDS and GELU' stays in registers.  16 rows a block
// because a minibatch of 4,096 is then one block per CU; eight waves so that two
// share a SIMD.  Predicting, a block walks over row blocks with its weights kept.
// TRAIN stores the weight gradients' operands, dZ and its rows' loss.
template <bool TRAIN>
__global__ __launch_bounds__(kNetThreads) void net_kernel(NetArgs g) {
    __shared__ __attribute__((aligned(16))) unsigned short xs[16 * kInStride];
    __shared__ __attribute__((aligned(16))) unsigned short ys[16 * kInStride];
    __shared__ __attribute__((aligned(16))) unsigned short act[2][16 * kActStride];
    __shared__ float ts[16][16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int jl = lane & 15, j = 16 * wv + jl, rq = 4 * (lane >> 4);
    const int rows = g.count ? min(g.rows, *g.count) : g.rows;
    const int nrb = (rows + 15) >> 4;
    if (int(blockIdx.x) >= nrb) return;
    const float *W = g.w, *stats = g.w + NPARAM;

    mu16x8 t1[1], t2[4], t3[4], t4[4], w4[1], w3[4], w2[4];
    load_ops<1>(t1, g.pk + PK_T1, 32, 16 * wv, lane);
    load_ops<4>(t2, g.pk + PK_T2, kH, 16 * wv, lane);
    load_ops<4>(t3, g.pk + PK_T3, kH, 16 * wv, lane);
    load_ops<4>(t4, g.pk + PK_T4, kH, 0, lane);
    if constexpr (TRAIN) {
        load_ops<1>(w4, g.pk + PK_W4, 32, 16 * wv, lane);
        load_ops<4>(w3, g.pk + PK_W3, kH, 16 * wv, lane);
        load_ops<4>(w2, g.pk + PK_W2, kH, 16 * wv, lane);
    }
    const float b1 = W[OFF_B1 + j], b2 = W[OFF_B2 + j], b3 = W[OFF_B3 + j], b4 = jl < kOut ? W[OFF_B4 + jl] : 0.f;
    const int gr = (tid >> 4) & 15, gk = tid & 15;    // the gathered element of this thread: input, or (TRAIN) target
    const bool target = tid >= 256;
    const float mean = gk < kIn ? stats[(target ? 30 : 0) + gk] : 0.f, std = gk < kIn ? stats[(target ? 45 : 15) + gk] : 1.f;
    if (!target) {                                    // k = 16 .. 31 of the 15-wide operands
        xs[gr * kInStride + 16 + gk] = 0;
        if (TRAIN) ys[gr * kInStride + 16 + gk] = 0;
    }

    for (int rb = blockIdx.x; rb < nrb; rb += gridDim.x) {
        const int i = rb * 16 + gr;
        float x = 0.f;
        if (i < rows && gk < kIn && (TRAIN || !target)) {
            if (g.list) {
                const double *uc = g.us + size_t(g.list[i]) * kIn;
                const double r = uc[0] > 0.0 ? 1.0 / uc[0] : 0.0;
                x = float((uc[gk] * r - mean) / std);
            } else {
                long long idx = g.seed ? (long long)(splitmix64(g.seed ^ (unsigned long long)i * 0xd1b54a32d192ed03ull) %
                                                     (unsigned long long)g.npairs)
                                       : (g.i0 + i);
                if (idx >= g.npairs) idx = g.npairs - 1;
                x = float(((target ? g.as : g.us)[idx * kIn + gk] - mean) / std);
            }
        }
        if (target) {
            if (TRAIN) ts[gr][gk] = x;
        } else {
            xs[gr * kInStride + gk] = to_bf16(x);
            if (TRAIN) g.ops[(size_t(rb) * kCols + CX + gk) * 16 + gr] = to_bf16(x);
        }
        __syncthreads();

        const int left = rows - rb * 16 - rq;            // of this lane's four rows, how many exist
        auto store_ops = [&](int col, const unsigned short (&h)[4]) {
            ushort4 v;
            v.x = left > 0 ? h[0] : 0;
            v.y = left > 1 ? h[1] : 0;
            v.z = left > 2 ? h[2] : 0;
            v.w = left > 3 ? h[3] : 0;
            *(ushort4 *)(g.ops + (size_t(rb) * kCols + col) * 16 + rq) = v;
        };
        float dg[3][4];
        auto forward = [&](int layer, mf32x4 z, float b, unsigned short *out, int col) {
            unsigned short h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = z[r] + b, e = erff(v * 0.70710678118654752f);
                if (TRAIN) dg[layer][r] = gelu_grad(v, e);
                h[r] = to_bf16(gelu(v, e));
                out[(rq + r) * kActStride + j] = h[r];
            }
            if (TRAIN) store_ops(col + j, h);
        };
        forward(0, mul<1, kInStride>(xs, t1, lane), b1, act[0], CA1);
        __syncthreads();
        forward(1, mul<4, kActStride>(act[0], t2, lane), b2, act[1], CA2);
        __syncthreads();
        forward(2, mul<4, kActStride>(act[1], t3, lane), b3, act[0], CA3);
        __syncthreads();
        if (wv == 0) {                                    // the 15 outputs: one tile
            const mf32x4 y = mul<4, kActStride>(act[0], t4, lane);
            if constexpr (TRAIN) {
                const float inv = 1.0f / float(rows * kOut);
                float loss = 0.f;
                unsigned short h[4];
                float dy[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float d = y[r] + b4 - ts[rq + r][jl];
                    const bool in = r < left && jl < kOut;
                    dy[r] = in ? 2.0f * d * inv : 0.f;
                    h[r] = to_bf16(dy[r]);
                    ys[(rq + r) * kInStride + jl] = h[r];
                    loss += in ? d * d * inv : 0.f;
                }
                store_ops(CDY + jl, h);
                if (jl < kOut)
                    *(float4 *)(g.dz + (size_t(3 * kH + jl) * nrb + rb) * 16 + rq) = make_float4(dy[0], dy[1], dy[2], dy[3]);
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) loss += __shfl_xor(loss, o);
                if (lane == 0) g.loss[rb] = loss;
            } else if (jl < kOut) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < left) {
                        const int ir = rb * 16 + rq + r;
                        const size_t o = size_t(g.list ? g.list[ir] : ir) * kOut + jl;
                        g.alpha[o] = double(y[r] + b4) * double(stats[45 + jl]) + double(stats[30 + jl]);
                    }
            }
        }
        if constexpr (TRAIN) {
            auto backward = [&](int layer, mf32x4 d, unsigned short *out, int col) {
                unsigned short h[4];
                float dz[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    dz[r] = r < left ? d[r] * dg[layer][r] : 0.f;
                    h[r] = to_bf16(dz[r]);
                    if (out) out[(rq + r) * kActStride + j] = h[r];
                }
                store_ops(col + j, h);
                *(float4 *)(g.dz + (size_t(layer * kH + j) * nrb + rb) * 16 + rq) = make_float4(dz[0], dz[1], dz[2], dz[3]);
            };
            __syncthreads();
            backward(2, mul<1, kInStride>(ys, w4, lane), act[1], CZ3);
            __syncthreads();
            backward(1, mul<4, kActStride>(act[1], w3, lane), act[0], CZ2);
            __syncthreads();
            backward(0, mul<4, kActStride>(act[0], w2, lane), nullptr, CZ1);
        }
        __syncthreads();
    }
}

struct UpdateArgs {
    const unsigned short *ops;
    const float *dz, *losses;
    int nrb;
    float *w;
    unsigned short *pk;
    float *grad, *m, *v, *loss;      // grad: if set, the gradient goes there and nothing is updated
    float lr, b1, b2, eps, c1, c2;
};

// Adam (Kingma & Ba 2015) for parameter i, and the new weight's matrix operands.
__device__ __forceinline__ void update(const UpdateArgs &g, int i, float gi) {
    if (g.grad) {
        g.grad[i] = gi;
        return;
    }
    const float mi = g.b1 * g.m[i] + (1.0f - g.b1) * gi;
    const float vi = g.b2 * g.v[i] + (1.0f - g.b2) * gi * gi;
    g.m[i] = mi;
    g.v[i] = vi;
    float wi = g.w[i];
    wi -= g.lr * (mi / g.c1) / (sqrtf(vi / g.c2) + g.eps);
    g.w[i] = wi;
    pack_weight(g.pk, i, wi);
}

constexpr int kTiles = 8 + 64 + 64 + 8;      // 16 x 16 blocks of dW1 dW2 dW3 dW4
constexpr int kSteps = 16;                   // matrix steps (32 rows) whose loads are in flight together

// dW = A^T dZ and the update: one wave per 16 x 16 block of a layer's weights, the
// rows in order, 32 to a matrix step.  The rows are not split over waves, so the
// sums keep one order whatever the batch is; what bounds the kernel is then a
// wave's own loads (256 KB for 4,096 rows, 2 us of matrix steps), hence 16 steps'
// operands (32 KB) on their way while the 16 before are multiplied.  Blocks past
// the tiles: a bias's column each, lane l summing rows l + 64 k + 256 m over m
// before the four k and the lanes are added; the last one adds up the losses.
__global__ __launch_bounds__(64, 1) void update_kernel(UpdateArgs g) {
    const int lane = threadIdx.x, b = blockIdx.x;
    if (b >= kTiles) {
        const int c = b - kTiles;
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        if (c < kBiasCols) {
            const int rows = 16 * g.nrb;
            const float *col = g.dz + size_t(c) * rows;
#pragma unroll 4
            for (int i = lane; i < rows; i += 256)
#pragma unroll
                for (int k = 0; k < 4; ++k) s[k] += i + 64 * k < rows ? col[i + 64 * k] : 0.f;
        } else {
            for (int i = lane; i < g.nrb; i += 64) s[0] += g.losses[i];
        }
        float t = (s[0] + s[2]) + (s[1] + s[3]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
        if (lane == 0) {
            if (c == kBiasCols) *g.loss = t;
            else update(g, c < kH ? OFF_B1 + c : c < 2 * kH ? OFF_B2 + c - kH : c < 3 * kH ? OFF_B3 + c - 2 * kH : OFF_B4 + c - 3 * kH, t);
        }
        return;
    }
    int ca, cz, off, ld, mi = 16, ni = 16;    // operand columns, where the block goes, its valid rows and columns
    if (b < 128) {
        const int i0 = 16 * ((b >> 3) & 7), k0 = 16 * (b & 7);
        ca = (b < 64 ? CA1 : CA2) + i0;
        cz = (b < 64 ? CZ2 : CZ3) + k0;
        off = (b < 64 ? OFF_W2 : OFF_W3) + i0 * kH + k0;
        ld = kH;
    } else if (b < 136) {
        const int k0 = 16 * (b - 128);
        ca = CX, cz = CZ1 + k0, off = OFF_W1 + k0, ld = kH, mi = kIn;
    } else {
        const int i0 = 16 * (b - 136);
        ca = CA3 + i0, cz = CDY, off = OFF_W4 + i0 * kOut, ld = kOut, ni = kOut;
    }
    // lane l supplies rows 8 (l/16) .. + 7 of a step: half a row block of column l%16
    const unsigned short *o = g.ops + size_t(lane >> 5) * kCols * 16 + (lane & 15) * 16 + 8 * ((lane >> 4) & 1);
    const unsigned short *oa = o + size_t(ca) * 16, *oz = o + size_t(cz) * 16;
    constexpr size_t kStep = size_t(2) * kCols * 16;
    const int nsteps = (g.nrb + 1) / 2;
    auto load = [&](mu16x8 (&a)[kSteps], mu16x8 (&z)[kSteps], int s0) {
        if (2 * (s0 + kSteps) <= g.nrb) {
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                a[u] = *(const mu16x8 *)(oa + (s0 + u) * kStep);
                z[u] = *(const mu16x8 *)(oz + (s0 + u) * kStep);
            }
        } else {
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                a[u] = z[u] = mu16x8{};
                if (2 * (s0 + u) + (lane >> 5) < g.nrb) {
                    a[u] = *(const mu16x8 *)(oa + (s0 + u) * kStep);
                    z[u] = *(const mu16x8 *)(oz + (s0 + u) * kStep);
                }
            }
        }
    };
    mf32x4 acc = {0.f, 0.f, 0.f, 0.f};
    mu16x8 a0[kSteps], z0[kSteps], a1[kSteps], z1[kSteps];
    load(a0, z0, 0);
    for (int s0 = 0; s0 < nsteps; s0 += 2 * kSteps) {
        load(a1, z1, s0 + kSteps);
#pragma unroll
        for (int u = 0; u < kSteps; ++u) acc = mma(a0[u], z0[u], acc);
        load(a0, z0, s0 + 2 * kSteps);
#pragma unroll
        for (int u = 0; u < kSteps; ++u) acc = mma(a1[u], z1[u], acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 4 * (lane >> 4) + r, j = lane & 15;
        if (i < mi && j < ni) update(g, off + i * ld + j, acc[r]);
    }
}

}  // namespace

// ---- host side ---------------------------------------------------------------

int mlp_param_count() { return NPARAM; }
size_t mlp_operand_floats() { return PK_N / 2; }

namespace {
int row_blocks(int rows) { return (rows + 15) / 16; }
size_t ops_floats(int rows) { return size_t(row_blocks(rows)) * kCols * 8; }

void launch_backprop(const MlpBuffers &b, const double *us, const double *as, long long npairs, int rows,
                     unsigned long long seed, bool adam, float lr, int step, hipStream_t s) {
    const int nrb = row_blocks(rows);
    unsigned short *ops = (unsigned short *)b.scratch;
    float *dz = b.scratch + ops_floats(rows), *losses = dz + size_t(kBiasCols) * 16 * nrb;
    NetArgs g{b.w, b.pk, us, as, nullptr, nullptr, npairs, 0, seed, rows, nullptr, ops, dz, losses};
    hipLaunchKernelGGL(net_kernel<true>, dim3(nrb), dim3(kNetThreads), 0, s, g);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.0f - powf(b1, float(step)), c2 = 1.0f - powf(b2, float(step));
    UpdateArgs u{ops, dz, losses, nrb, b.w, b.pk, adam ? nullptr : b.grad, b.m, b.v, b.loss, lr, b1, b2, eps, c1, c2};
    hipLaunchKernelGGL(update_kernel, dim3(kTiles + kBiasCols + 1), dim3(64), 0, s, u);
}

void launch_predict(NetArgs g, hipStream_t s) {
    const int blocks = std::min(row_blocks(g.rows), 512);   // two per CU, each walking over row blocks
    hipLaunchKernelGGL(net_kernel<false>, dim3(blocks), dim3(kNetThreads), 0, s, g);
}
}  // namespace

size_t mlp_scratch_floats(int rows) {
    return ops_floats(rows) + size_t(row_blocks(rows)) * (16 * kBiasCols + 1);
}

void mlp_pack(const MlpBuffers &b, hipStream_t s) {
    hipLaunchKernelGGL(pack_kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, s, b.w, b.pk);
}

void mlp_train_step(const MlpBuffers &b, const double *us, const double *as, long long npairs, int rows,
                    unsigned long long seed, float lr, int step, hipStream_t s) {
    launch_backprop(b, us, as, npairs, rows, seed, true, lr, step, s);
}

void mlp_gradient(const MlpBuffers &b, const double *us, const double *as, int rows, hipStream_t s) {
    launch_backprop(b, us, as, rows, rows, 0, false, 0.f, 1, s);
}

void mlp_predict(const MlpBuffers &b, const double *us, int rows, double *alpha, hipStream_t s) {
    launch_predict(NetArgs{b.w, b.pk, us, nullptr, nullptr, nullptr, rows, 0, 0, rows, alpha, nullptr, nullptr, nullptr}, s);
}

void mlp_predict_listed(const MlpBuffers &b, const double *u, const int *list, const int *count, int max_rows,
                        double *alpha, hipStream_t s) {
    launch_predict(NetArgs{b.w, b.pk, u, nullptr, list, count, max_rows, 0, 0, max_rows, alpha, nullptr, nullptr, nullptr}, s);
}

}  // namespace mnc
