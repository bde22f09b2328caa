// wc_mlp.hip -- the learned closure's network on gfx950 matrix cores.
//
// MLP 195 -> 128 -> 128 -> 128 -> 3 with SiLU, bf16 weights and activations, fp32 accumulation,
// all products on v_mfma_f32_32x32x16_bf16.  The input is padded to 208 features and the output
// to 32 columns (zero weights), so every product is a whole number of 32x32x16 MFMA tiles.
//
// Training (forward with stored activations, backward, Adam) is nine launches of one MFMA GEMM tile
// with strided operands, whose epilogues hold the elementwise work.  Inference is one fused
// kernel: a workgroup of four waves takes 128 particles, each wave 32 of them through all four
// layers, activations staying in LDS between layers.
//
// MFMA 32x32x16 bf16 lane layout (wave64, lane l): A operand = A[l % 32][8 (l / 32) + 0..7],
// B operand = B[8 (l / 32) + 0..7][l % 32], accumulator element r = C[8 (r / 4) + 4 (l / 32) +
// r % 4][l % 32].
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "wc_mlp.hpp"

namespace wc {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// float -> bf16, round to nearest even (one v_cvt_pk_bf16_f32 on gfx950; NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// SiLU with the hardware reciprocal (about 1 ulp): the network computes in bf16, so the correctly
// rounded division the rest of the library is built with would only cost time here.
__device__ __forceinline__ float silu(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

__device__ __forceinline__ f32x16 mfma(uint4 a, uint4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// ------------------------------------------------------------------------------------------
// GEMM tile: sum_k A(m,k) B(k,n), A(m,k) = A[m*sam + k*sak], B(k,n) = B[k*sbk + n*sbn] (bf16), fp32
// sums.  64x64 tile per workgroup (2x2 waves of 32x32 on v_mfma_f32_32x32x16_bf16); K in stages of 64
// staged through LDS as [row][k] (k contiguous, rows padded by 8), the next stage's global loads in
// flight while the current one is multiplied.
//
// Each operand tile (64 rows x 64 k) loads as 512 runs of 8 values along the operand's contiguous
// dimension -- k, or the row (m for A, n for B) when ROW_CONTIG -- two runs per thread, as one
// 16-byte load where the run lies inside the matrix and the addresses are aligned (`vec`), value
// by value (zeros outside) elsewhere.  Row-contiguous runs are transposed as they go into LDS.
//
// A step on 8,192 rows is a chain of kernels of 2-10 us each, none of which fills the chip: what it
// costs is their number.  The bias, the activation, its derivative and the output's error are therefore
// done on the accumulators (EPI), a layer's weight and bias gradients run beside the delta of the layer
// below, and k_finish adds the partial sums, steps Adam and writes the bf16 weights: nine launches where
// there were thirty, 181 us -> 96 us a step on 8,192 rows, 391 -> 260 us for a gradient on 51,207.
// ------------------------------------------------------------------------------------------
constexpr int kGemmTile = 64;
constexpr int kGemmKStage = 64;
constexpr int kGemmLdk = kGemmKStage + 8;

template <bool ROW_CONTIG>
__device__ __forceinline__ void gemm_load(uint4 (&v)[2], const uint16_t* __restrict__ X, long s_row, long s_k, int row0,
                                          int nrows, int k0, int kend, bool vec, int tid) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int q = tid * 2 + i;
        const int a = q >> 3, b = (q & 7) * 8;
        const int gr = row0 + (ROW_CONTIG ? b : a), gk = k0 + (ROW_CONTIG ? a : b);
        const bool full = ROW_CONTIG ? (gr + 8 <= nrows && gk < kend) : (gr < nrows && gk + 8 <= kend);
        if (vec && full) {
            v[i] = *reinterpret_cast<const uint4*>(&X[(long)gr * s_row + (long)gk * s_k]);
        } else {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                uint32_t e[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int rr = ROW_CONTIG ? gr + j + h : gr, kk = ROW_CONTIG ? gk : gk + j + h;
                    e[h] = (rr < nrows && kk < kend) ? X[(long)rr * s_row + (long)kk * s_k] : 0u;
                }
                w[j / 2] = e[0] | (e[1] << 16);
            }
            v[i] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

template <bool ROW_CONTIG>
__device__ __forceinline__ void gemm_store(const uint4 (&v)[2], uint16_t* tile, int tid) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int q = tid * 2 + i;
        const int a = q >> 3, b = (q & 7) * 8;
        if (!ROW_CONTIG) {
            *reinterpret_cast<uint4*>(&tile[a * kGemmLdk + b]) = v[i];
        } else {
            const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int j = 0; j < 8; ++j) tile[(b + j) * kGemmLdk + a] = (uint16_t)(w[j / 2] >> (16 * (j & 1)));
        }
    }
}

enum Epilogue {
    kSilu,     // z = acc + bias kept in Z, H = bf16(silu(z))
    kOutput,   // y = acc + bias to Y (rows of 4); with targets H = bf16(scale (y - t)) and the loss
    kBackward, // H = bf16(acc * silu'(Z)), silu'(z) = s (1 + z (1 - s)), s = sigmoid(z)
    kPartial,  // C of this split of K
};
struct GemmArgs {
    const uint16_t *A, *B;
    long sam, sak, sbk, sbn;
    int M, N, K, k_split;
    int nx, ny;        // tiles
    int vec_a, vec_b;
    float* C;          // kPartial: splits of M x N
    const float* bias;
    float* Z;          // M x N
    uint16_t* H;       // M x N
    const float* T;    // targets, rows of 4 (may be NULL)
    float* Y;          // may be NULL
    float scale;
    float* loss;       // kOutput: += sum (y - t)^2; kSilu: set to 0
};

template <bool A_ROWS, bool B_ROWS, int EPI>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, int block, uint16_t* As, uint16_t* Bs) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int by = block / g.nx % g.ny, bz = block / (g.nx * g.ny);
    const int m0 = by * kGemmTile, n0 = block % g.nx * kGemmTile;
    const int kbeg = bz * g.k_split;
    const int kend = min(g.K, kbeg + g.k_split);
    f32x16 acc = {};
    uint4 ra[2], rb[2];
    if (kbeg < kend) {
        gemm_load<A_ROWS>(ra, g.A, g.sam, g.sak, m0, g.M, kbeg, kend, g.vec_a != 0, tid);
        gemm_load<B_ROWS>(rb, g.B, g.sbn, g.sbk, n0, g.N, kbeg, kend, g.vec_b != 0, tid);
    }
    for (int k0 = kbeg; k0 < kend; k0 += kGemmKStage) {
        __syncthreads();  // the previous stage's operand reads are done
        gemm_store<A_ROWS>(ra, As, tid);
        gemm_store<B_ROWS>(rb, Bs, tid);
        __syncthreads();
        if (k0 + kGemmKStage < kend) {
            gemm_load<A_ROWS>(ra, g.A, g.sam, g.sak, m0, g.M, k0 + kGemmKStage, kend, g.vec_a != 0, tid);
            gemm_load<B_ROWS>(rb, g.B, g.sbn, g.sbk, n0, g.N, k0 + kGemmKStage, kend, g.vec_b != 0, tid);
        }
#pragma unroll
        for (int ks = 0; ks < kGemmKStage / 16; ++ks) {
            const int kq = ks * 16 + (lane >> 5) * 8;
            const uint4 a = *reinterpret_cast<const uint4*>(&As[(wm * 32 + (lane & 31)) * kGemmLdk + kq]);
            const uint4 b = *reinterpret_cast<const uint4*>(&Bs[(wn * 32 + (lane & 31)) * kGemmLdk + kq]);
            acc = mfma(a, b, acc);
        }
    }
    const int col = n0 + wn * 32 + (lane & 31);
    auto row_of = [&](int r) { return m0 + wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); };
    if constexpr (EPI == kPartial) {
        float* const C = g.C + (size_t)bz * g.M * g.N;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (row_of(r) < g.M && col < g.N) C[(long)row_of(r) * g.N + col] = acc[r];
    } else if constexpr (EPI == kSilu) {
        if (g.loss && block == 0 && tid == 0) *g.loss = 0.0f;
        const float bias = col < g.N ? g.bias[col] : 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const long at = (long)row_of(r) * g.N + col;
            if (row_of(r) < g.M && col < g.N) {
                const float z = acc[r] + bias;
                g.Z[at] = z;
                g.H[at] = f2bf(silu(z));
            }
        }
    } else {
        float err = 0.0f;
        const float bias = EPI == kOutput && col < kMlpOut ? g.bias[col] : 0.0f;
        float z[16];
        if constexpr (EPI == kBackward) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                z[r] = row_of(r) < g.M && col < g.N ? g.Z[(long)row_of(r) * g.N + col] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = row_of(r);
            if (row >= g.M || col >= g.N) continue;
            uint16_t h;
            if constexpr (EPI == kBackward) {
                const float s = 1.0f / (1.0f + __expf(-z[r]));
                h = f2bf(acc[r] * (s * (1.0f + z[r] * (1.0f - s))));
            } else {
                const float y = acc[r] + bias;
                if (g.Y && col < 4) g.Y[(long)row * 4 + col] = col < kMlpOut ? y : 0.0f;
                if (!g.T) continue;
                const float d = col < kMlpOut ? y - g.T[(long)row * 4 + col] : 0.0f;
                err += d * d;
                h = f2bf(g.scale * d);
            }
            g.H[(long)row * g.N + col] = h;
        }
        if constexpr (EPI == kOutput) {
            if (!g.T) return;
            for (int d = 32; d >= 1; d >>= 1) err += __shfl_xor(err, d);
            if (lane == 0 && wn == 0) atomicAdd(g.loss, err);
        }
    }
}

// Bias gradients, first part: sums of D's columns (M x N, bf16) over chunks of kColsumRows rows, 64 columns
// and 4 row groups a workgroup, in a fixed order.
__device__ __forceinline__ void column_sums(const uint16_t* __restrict__ D, float* __restrict__ part, int M, int N,
                                            int block, float* red) {
    const int l = threadIdx.x & 63, g = threadIdx.x >> 6, nx = (N + 63) / 64;
    const int c = block % nx * 64 + l, chunk = block / nx, r0 = chunk * kColsumRows;
    const int r1 = min(M, r0 + kColsumRows);
    float s = 0.0f;
    if (c < N) {
#pragma unroll 32
        for (int r = r0 + g; r < r1; r += 4) s += bf2f(D[(long)r * N + c]);
    }
    red[g * 64 + l] = s;
    __syncthreads();
    if (g == 0 && c < N) part[(long)chunk * N + c] = ((red[l] + red[64 + l]) + red[128 + l]) + red[192 + l];
}

template <bool A_ROWS, bool B_ROWS, int EPI>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
    __shared__ __attribute__((aligned(16))) uint16_t As[kGemmTile * kGemmLdk];  // [m][k]
    __shared__ __attribute__((aligned(16))) uint16_t Bs[kGemmTile * kGemmLdk];  // [n][k]
    gemm_tile<A_ROWS, B_ROWS, EPI>(g, (int)blockIdx.x, As, Bs);
}

// A layer's weight gradient H^T D, split over the rows of the batch, its bias gradient's partial sums and the
// layer below's delta, all from D.
__global__ __launch_bounds__(256) void k_gemm_backward(GemmArgs weights, int weight_blocks, GemmArgs delta,
                                                       int delta_blocks, float* colpart) {
    __shared__ __attribute__((aligned(16))) uint16_t As[kGemmTile * kGemmLdk];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[kGemmTile * kGemmLdk];
    const int block = (int)blockIdx.x;
    if (block < weight_blocks)
        gemm_tile<true, true, kPartial>(weights, block, As, Bs);
    else if (block < weight_blocks + delta_blocks)
        gemm_tile<false, false, kBackward>(delta, block - weight_blocks, As, Bs);
    else
        column_sums(weights.B, colpart, weights.K, weights.N, block - weight_blocks - delta_blocks,
                    reinterpret_cast<float*>(As));
}

// Gradients from the partial sums, in a fixed order, and with ADAM the update and the weights' bf16 copies
// (row-major [k][n] for the GEMMs, transposed [n][k] for the fused inference kernel).  A workgroup takes 256
// weights or a layer's biases.
struct FinishArgs {
    struct {
        const float *wpart, *bpart;
        uint16_t *rowmajor, *transposed;
        int w_off, b_off, K, N, splits, first;  // first: workgroup
    } layer[4];
    int chunks;      // of the bias sums
    float *w, *grad, *m, *v;
    float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__global__ __launch_bounds__(256) void k_finish(FinishArgs f) {
    int l = 3;
    while (l > 0 && (int)blockIdx.x < f.layer[l].first) --l;
    const auto& a = f.layer[l];
    const int block = (int)blockIdx.x - a.first, nw = a.K * a.N, wblocks = (nw + 255) / 256, tid = threadIdx.x;
    auto apply = [&](int i, float g) {
        f.grad[i] = g;
        if constexpr (ADAM) {
            const float mi = f.b1 * f.m[i] + (1.0f - f.b1) * g;
            const float vi = f.b2 * f.v[i] + (1.0f - f.b2) * g * g;
            f.m[i] = mi;
            f.v[i] = vi;
            f.w[i] -= f.lr * (mi / f.c1) / (sqrtf(vi / f.c2) + f.eps);
        }
    };
    if (block < wblocks) {
        const int i = block * 256 + tid;
        if (i >= nw) return;
        float s = 0.0f;
#pragma unroll 16
        for (int k = 0; k < a.splits; ++k) s += a.wpart[(size_t)k * nw + i];
        apply(a.w_off + i, s);
        if constexpr (ADAM) {
            const uint16_t h = f2bf(f.w[a.w_off + i]);
            const int k = i / a.N, n = i % a.N;
            a.rowmajor[i] = h;
            a.transposed[(long)n * a.K + k] = h;
        }
    } else {
        if (tid >= a.N) return;
        float s = 0.0f;
#pragma unroll 8
        for (int k = 0; k < f.chunks; ++k) s += a.bpart[(size_t)k * a.N + tid];
        apply(a.b_off + tid, s);
    }
}

// bf16 copies of the master weights, as k_finish writes them.
__global__ void k_cast(const float* __restrict__ w, uint16_t* __restrict__ rowmajor, uint16_t* __restrict__ transposed,
                       int K, int N) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= K * N) return;
    const int k = i / N, n = i % N;
    const uint16_t h = f2bf(w[i]);
    rowmajor[i] = h;
    transposed[(long)n * K + k] = h;
}

// ------------------------------------------------------------------------------------------
// Fused inference: Y[n x 4] = MLP(X[n x 208]).  Persistent: one workgroup of eight waves per CU
// copies all four layers' weights and biases into LDS once (bf16, transposed [out][in], each row
// padded so that the 16 rows an MFMA operand read touches spread over the banks)
// and then walks tiles of 128 rows; each wave takes 16 rows of a tile through the four layers on
// v_mfma_f32_16x16x32_bf16.
//
// MFMA 16x16x32 bf16 lane layout (wave64, lane l, c = l % 16, q = l / 16): A operand =
// A[c][8 q + 0..7], B operand = B[8 q + 0..7][c], accumulator element r = D[4 q + r][c].
//
// Each layer computes the transposed product Z^T = W^T H^T: the weights are the A operand (rows
// of W^T from LDS) and the activations the B operand, so lane (q, c) works on row c.  Output tile
// j leaves hidden neuron 16 j + 4 q + r of row c in lane (q, c); the next layer's B operand wants
// 8 values of row c at input positions 32 s + 8 q + t.  Defining position p = 32 s + 8 q + t to
// hold neuron 32 s + 16 (t / 4) + 4 q + t % 4 -- the lane's own accumulators acc[2 s + t / 4][t % 4]
// -- makes every activation stay in the lane that produced it: the input columns of layers 2-4 are
// stored in that order in LDS, and activations never leave registers.
// ------------------------------------------------------------------------------------------
struct InferWeights {
    const uint16_t* w1t;  // [128][208]
    const uint16_t* w2t;  // [128][128]
    const uint16_t* w3t;  // [128][128]
    const uint16_t* w4t;  // [32][128]
    const float *b1, *b2, *b3, *b4;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

constexpr int kLd1 = kMlpInPad + 8;   // LDS row length of layer 1's weights (208 used, 8 zero)
// LDS row length of layers 2-4's weights: 72 dwords.  Measured on gfx950 (SQ_LDS_BANK_CONFLICT
// over the kernel's operand reads): rows of 68, 76, 80, 84 or 92 dwords spend 45 % of the LDS's
// active cycles in bank conflicts, 96 dwords 63 %, and 72 or 88 dwords 27 %.
constexpr int kLdH = kMlpHidden + 16;
constexpr int kInferWaves = 8;
constexpr int kInferRows = 16;                         // rows per wave and tile
constexpr int kInferTile = kInferWaves * kInferRows;   // rows per tile
constexpr int kKSteps1 = (kMlpInPad + 31) / 32;        // layer 1's k steps of 32 (the last half used)
constexpr int kKStepsH = kMlpHidden / 32;              // k steps of layers 2-4
constexpr int kW4Rows = 16;                            // the output layer's A operand rows (3 used)
constexpr int kInferLdsHalves = kMlpHidden * kLd1 + 2 * kMlpHidden * kLdH + kW4Rows * kLdH;
constexpr int kInferBias = 3 * kMlpHidden + 4;         // b1 | b2 | b3 | b4[0..3], floats
static_assert(kInferLdsHalves % 8 == 0, "the biases follow the weights 16-byte aligned");
static_assert(kInferLdsHalves * 2 + kInferBias * 4 <= 160 * 1024, "weights must fit one CU's LDS");
static_assert(32 * kKSteps1 <= kLd1 + 8, "layer 1's last k step reads at most 8 values past a row");

struct InferLds {
    uint16_t *w1, *w2, *w3, *w4;  // [128][kLd1], [128][kLdH] x 2, [16][kLdH]
    float* bias;                  // [kInferBias]
};

__device__ __forceinline__ InferLds infer_lds(uint16_t* s_mem) {
    InferLds L;
    L.w1 = s_mem;
    L.w2 = L.w1 + kMlpHidden * kLd1;
    L.w3 = L.w2 + kMlpHidden * kLdH;
    L.w4 = L.w3 + kMlpHidden * kLdH;
    L.bias = reinterpret_cast<float*>(s_mem + kInferLdsHalves);
    return L;
}

__device__ __forceinline__ uint32_t pack2bf(float lo, float hi) {
    typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Layer 1's input order.  Its first six k steps (192 positions) hold the 32 neighbours' values:
// lane quarter q takes neighbours 8q .. 8q + 7, whose 48 values are features 48q .. 48q + 47, as
// 8 consecutive features per k step: position p = 32 s + 8 q + t holds feature 48 q + 8 s + t.
// Every lane then starts step s at the same offset, (8 s) mod 6, into its first neighbour of the
// step, a constant.  Step 6 holds features 192 .. 223 in order (the three scalars, then zeros).
__device__ __forceinline__ int layer1_chunk(int p8) {  // source chunk of 8 features for chunk p8
    return p8 < 24 ? 6 * (p8 & 3) + (p8 >> 2) : p8;
}

// Weights and biases into LDS, 8 values per copy.  Layer 1's input columns are stored in the
// order above, and its row padding is zeroed (its last k step multiplies it, and the first 8
// values of the next row, by zero inputs).  Layers 2-4 store input position p = 32 s + 8 q + t of
// each row from neuron 32 s + 16 (t / 4) + 4 q + t % 4: the 8 positions of one copy are two runs
// of 4 neurons, 16 apart.
__device__ __forceinline__ void stage_weights(const InferWeights& W, const InferLds& L, int tid, int nthreads) {
    for (int i = tid; i < kMlpHidden * (kLd1 / 8); i += nthreads) {
        const int r = i / (kLd1 / 8), q = i % (kLd1 / 8);
        const int src = layer1_chunk(q);
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (src < kMlpInPad / 8) v = reinterpret_cast<const uint4*>(W.w1t)[r * (kMlpInPad / 8) + src];
        *reinterpret_cast<uint4*>(&L.w1[r * kLd1 + q * 8]) = v;
    }
    constexpr int kChunks = kMlpHidden / 8;
    for (int i = tid; i < (2 * kMlpHidden + kW4Rows) * kChunks; i += nthreads) {
        const int r = i / kChunks, p8 = i % kChunks;
        const uint16_t* src;
        uint16_t* dst;
        if (r < kMlpHidden) {
            src = W.w2t + (size_t)r * kMlpHidden;
            dst = L.w2 + r * kLdH;
        } else if (r < 2 * kMlpHidden) {
            src = W.w3t + (size_t)(r - kMlpHidden) * kMlpHidden;
            dst = L.w3 + (r - kMlpHidden) * kLdH;
        } else {
            src = W.w4t + (size_t)(r - 2 * kMlpHidden) * kMlpHidden;
            dst = L.w4 + (r - 2 * kMlpHidden) * kLdH;
        }
        const int s = p8 >> 2, q = p8 & 3;
        const uint2 lo = *reinterpret_cast<const uint2*>(src + 32 * s + 4 * q);
        const uint2 hi = *reinterpret_cast<const uint2*>(src + 32 * s + 16 + 4 * q);
        *reinterpret_cast<uint4*>(dst + 8 * p8) = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
    for (int i = tid; i < kInferBias; i += nthreads)
        L.bias[i] = i < kMlpHidden       ? W.b1[i]
                    : i < 2 * kMlpHidden ? W.b2[i - kMlpHidden]
                    : i < 3 * kMlpHidden ? W.b3[i - 2 * kMlpHidden]
                                         : W.b4[i - 3 * kMlpHidden];
}

// Layer 1's B operand for a wave's 16 rows from row0, in layer 1's input order (rows at or past
// n, and features at or past 208, read as zeros).
__device__ __forceinline__ void load_rows(uint4 (&a)[kKSteps1], const uint16_t* __restrict__ X, long row0, uint32_t n,
                                          int lane) {
    const int row = lane & 15, q4 = lane >> 4;
    const bool live = row0 + row < (long)n;
#pragma unroll
    for (int s = 0; s < kKSteps1; ++s) a[s] = make_uint4(0u, 0u, 0u, 0u);
    if (live) {
        const uint16_t* src = X + (row0 + row) * kMlpInPad;
#pragma unroll
        for (int s = 0; s < kKSteps1; ++s) {
            const int chunk = layer1_chunk(4 * s + q4);
            if (chunk < kMlpInPad / 8) a[s] = *reinterpret_cast<const uint4*>(src + 8 * chunk);
        }
    }
}

// hout = bf16(silu(W^T hin + b)) for a wave's 16 rows: W^T rows from LDS with stride LDW, the
// input in registers (KSTEPS B operands), the output in the next layer's B operand order.
template <int KSTEPS, int LDW, int GROUP = 8>
__device__ __forceinline__ void infer_layer(const uint4 (&hin)[KSTEPS], const uint16_t* wt, const float* bias,
                                            uint4 (&hout)[kKStepsH], int lane) {
    const int c = lane & 15, q4 = lane >> 4;
    // accumulators start at the bias: element r of tile j is neuron 16 j + 4 q + r
    f32x4 acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = *reinterpret_cast<const f32x4*>(&bias[16 * j + 4 * q4]);
    // the weights of one group of GROUP output tiles in flight while the previous group's
    // products run; the scheduling barriers keep the compiler from hoisting every group's loads
    // (and their registers) up front
    static_assert(8 % GROUP == 0, "groups split a k step's 8 output tiles");
    constexpr int kGroups = KSTEPS * (8 / GROUP);
    const uint16_t* wrow = wt + c * LDW + 8 * q4;
    uint4 w[2][GROUP];
#pragma unroll
    for (int g = 0; g < GROUP; ++g) w[0][g] = *reinterpret_cast<const uint4*>(&wrow[16 * g * LDW]);
#pragma unroll
    for (int i = 0; i < kGroups; ++i) {
        const int s = i / (8 / GROUP), j0 = (i % (8 / GROUP)) * GROUP;
        if (i + 1 < kGroups) {
            const int s1 = (i + 1) / (8 / GROUP), j1 = ((i + 1) % (8 / GROUP)) * GROUP;
#pragma unroll
            for (int g = 0; g < GROUP; ++g)
                w[(i + 1) & 1][g] = *reinterpret_cast<const uint4*>(&wrow[16 * (j1 + g) * LDW + 32 * s1]);
        }
#pragma unroll
        for (int g = 0; g < GROUP; ++g) acc[j0 + g] = mfma16(w[i & 1][g], hin[s], acc[j0 + g]);
        __builtin_amdgcn_sched_barrier(0);
    }
    // every write below depends on every read above, so hout may be hin
#pragma unroll
    for (int s = 0; s < kKStepsH; ++s) {
        const f32x4 a = acc[2 * s], b = acc[2 * s + 1];
        hout[s] = make_uint4(pack2bf(silu(a[0]), silu(a[1])), pack2bf(silu(a[2]), silu(a[3])),
                             pack2bf(silu(b[0]), silu(b[1])), pack2bf(silu(b[2]), silu(b[3])));
    }
}

// Output layer: one 16-row A operand tile (rows 0..2 used); lanes 0..15 hold outputs 0..3 of
// row c and write Y's 4 columns (column 3 zero).
__device__ __forceinline__ void infer_output(const uint4 (&h)[kKStepsH], const InferLds& L, float* __restrict__ Y,
                                             long row0, int rows_left, int lane) {
    const int c = lane & 15, q4 = lane >> 4;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < kKStepsH; ++s)
        acc = mfma16(*reinterpret_cast<const uint4*>(&L.w4[c * kLdH + 32 * s + 8 * q4]), h[s], acc);
    if (q4 == 0 && c < rows_left) {
        const float* b4 = L.bias + 3 * kMlpHidden;
        float* y = Y + (row0 + c) * 4;
        y[0] = acc[0] + b4[0];
        y[1] = acc[1] + b4[1];
        y[2] = acc[2] + b4[2];
        y[3] = 0.0f;
    }
}

__global__ __launch_bounds__(kInferWaves * 64) void k_mlp_infer(const uint16_t* __restrict__ X, InferWeights W,
                                                                 float* __restrict__ Y, uint32_t n) {
    __shared__ __attribute__((aligned(16))) uint16_t s_mem[kInferLdsHalves + 2 * kInferBias];
    const InferLds L = infer_lds(s_mem);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    const uint32_t tiles = (n + kInferTile - 1) / kInferTile;
    uint4 xa[kKSteps1];
    if (blockIdx.x < tiles) load_rows(xa, X, (long)blockIdx.x * kInferTile + wave * kInferRows, n, lane);
    stage_weights(W, L, tid, kInferWaves * 64);
    __syncthreads();

    // From here on LDS is read-only and the waves are independent; the next tile's input rows
    // load while the current tile is computed.
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const long row0 = (long)tile * kInferTile + wave * kInferRows;
        const int rows_left = (int)max(0L, min((long)kInferRows, (long)n - row0));
        uint4 h[kKStepsH];
        infer_layer<kKSteps1, kLd1>(xa, L.w1, L.bias, h, lane);
        const uint32_t next = tile + gridDim.x;
        if (next < tiles) load_rows(xa, X, (long)next * kInferTile + wave * kInferRows, n, lane);
        infer_layer<kKStepsH, kLdH>(h, L.w2, L.bias + kMlpHidden, h, lane);
        infer_layer<kKStepsH, kLdH>(h, L.w3, L.bias + 2 * kMlpHidden, h, lane);
        infer_output(h, L, Y, row0, rows_left, lane);
    }
}

// ------------------------------------------------------------------------------------------
// Inference on the closure's inputs without the feature matrix: each lane forms its own layer-1
// operand from the neighbour lists.  Lane l (row l % 16, quarter q = l / 16) holds, in layer 1's
// input order, the values of neighbours 8q .. 8q + 7 of its row: k step s < 6 takes neighbours
// a_s = floor(8 s / 6) and a_s + 1 of the eight, from value (8 s) mod 6 of the first.  The next
// tile's rows are fetched in phases between the current tile's layers (the row counts a tile
// earlier still, then the list entries, the records, and last the values), so the loads land
// while the matrix cores work.
// ------------------------------------------------------------------------------------------
constexpr int kFeatSteps = 6;  // k-steps of neighbour values (192 columns)
constexpr int kLaneNeighbours = 8;

struct RowFetch {
    uint32_t row, listed;
    bool live;
    uint32_t listed_next;  // the count of the row one tile further on, loaded a tile early
    float4 p;              // own position and density
    float3 pv;             // own velocity
    uint32_t e[kLaneNeighbours];                          // phase 1: list entries (or selected slots)
    float3 q[kLaneNeighbours], qv[kLaneNeighbours];       // phase 2: the neighbours' records
};

__device__ __forceinline__ float3 load3(const float4* a, uint32_t i) {
    const float* f = reinterpret_cast<const float*>(a) + 4 * (size_t)i;
    return float3{f[0], f[1], f[2]};
}

__device__ __forceinline__ uint32_t row_count(const ClosureRows& cr, long row0, uint32_t n, int lane) {
    const long row = row0 + (lane & 15);
    return row < (long)n ? cr.ncount[row] : 0u;
}

// phase 1: the row's list entries and own record; `listed` arrived a tile earlier, so the loads
// go to the list itself or, past 32 neighbours, to the 32 slots its selection wrote (cr.sel)
__device__ __forceinline__ void fetch_entries(RowFetch& f, const ClosureRows& cr, long row0, uint32_t n, int lane) {
    const int r16 = lane & 15, q4 = lane >> 4;
    f.live = row0 + r16 < (long)n;
    f.row = f.live ? (uint32_t)(row0 + r16) : 0u;
    f.listed = f.listed_next;
    f.p = cr.posrho[f.row];
    f.pv = load3(cr.velp, f.row);
    // entry k of the row at base + k * step: the selection's row (step 1) or the list's column
    // (step stride), one selected address advanced per entry rather than a branch per source
    const bool sel = f.listed > 32u;
    const size_t step = sel ? (size_t)1 : cr.stride;
    const uint32_t* src =
        (sel ? cr.sel + (size_t)f.row * kSelRow : cr.nlist + f.row) + (size_t)(kLaneNeighbours * q4) * step;
#pragma unroll
    for (int i = 0; i < kLaneNeighbours; ++i) {
        f.e[i] = *src;
        src += step;
    }
}

// phase 2: the neighbours' records (entries past a list may be stale: a slot out of range is
// replaced by the row's own, so every load stays inside the buffers)
__device__ __forceinline__ void fetch_records(RowFetch& f, const ClosureRows& cr, uint32_t n, int lane) {
    // a scalar base plus one 32-bit byte offset for both records (slots are below 2^28)
#pragma unroll
    for (int i = 0; i < kLaneNeighbours; ++i) {
        const uint32_t off = (f.e[i] < n ? f.e[i] : f.row) << 4;
        const float* a = reinterpret_cast<const float*>(reinterpret_cast<const char*>(cr.posrho) + off);
        const float* b = reinterpret_cast<const float*>(reinterpret_cast<const char*>(cr.velp) + off);
        f.q[i] = float3{a[0], a[1], a[2]};
        f.qv[i] = float3{b[0], b[1], b[2]};
    }
}

// phase 3: the layer-1 operand, formed as the feature kernel forms its rows (same operations, so
// the same bf16 values)
__device__ __forceinline__ void form_rows(uint4 (&a)[kKSteps1], const RowFetch& f, const ClosureRows& cr, int lane) {
    const int q4 = lane >> 4;
    if (!f.live) {
#pragma unroll
        for (int s = 0; s < kKSteps1; ++s) a[s] = make_uint4(0u, 0u, 0u, 0u);
        return;
    }
    const uint32_t cnt = f.listed > 32u ? 32u : f.listed;  // longer lists keep their 32 nearest
    const float inv_h = 1.0f / cr.h;
    float v[kLaneNeighbours][6];
    uint32_t mask[kLaneNeighbours];
#pragma unroll
    for (int i = 0; i < kLaneNeighbours; ++i) {
        // zeros past the list by masking the bits (an opaque mask keeps the loads unconditional)
        mask[i] = (uint32_t)(kLaneNeighbours * q4 + i) < cnt ? ~0u : 0u;
        asm("" : "+v"(mask[i]));
        v[i][0] = (f.q[i].x - f.p.x) * inv_h;
        v[i][1] = (f.q[i].y - f.p.y) * inv_h;
        v[i][2] = (f.q[i].z - f.p.z) * inv_h;
        v[i][3] = f.qv[i].x - f.pv.x;
        v[i][4] = f.qv[i].y - f.pv.y;
        v[i][5] = f.qv[i].z - f.pv.z;
    }
    // each packed pair belongs to one neighbour (6 values each, pairs start at even positions), so
    // its mask applies to the pair: bf16 pairs of masked values, with half the masking
#pragma unroll
    for (int s = 0; s < kFeatSteps; ++s) {
        const int first = (8 * s) / 6, o = (8 * s) % 6;  // compile-time
        static_assert((8 * kFeatSteps) % 2 == 0 && 6 % 2 == 0, "pairs within a neighbour");
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const int i = o + e < 6 ? first : first + 1, k = o + e < 6 ? o + e : o + e - 6;
            w[e / 2] = pack2bf(v[i][k], v[i][k + 1]) & mask[i];
        }
        a[s] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    // columns 192..207: the density deviation, the step multiplier and the filled fraction
    const float rho_rel = (f.p.w / cr.rho0 - 1.0f) * 10.0f;
    a[kFeatSteps] = q4 == 0 ? make_uint4(pack2bf(rho_rel, cr.dt_mult * 0.25f),
                                         pack2bf((float)cnt * (1.0f / 32.0f), 0.0f), 0u, 0u)
                            : make_uint4(0u, 0u, 0u, 0u);
}

__global__ __launch_bounds__(kInferWaves * 64) void k_mlp_infer_closure(ClosureRows cr, InferWeights W,
                                                                         float* __restrict__ Y, uint32_t n) {
    __shared__ __attribute__((aligned(16))) uint16_t s_mem[kInferLdsHalves + 2 * kInferBias];
    const InferLds L = infer_lds(s_mem);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    const uint32_t tiles = (n + kInferTile - 1) / kInferTile;
    uint4 xa[kKSteps1];
    RowFetch f;
    if (blockIdx.x < tiles) {
        f.listed_next = row_count(cr, (long)blockIdx.x * kInferTile + wave * kInferRows, n, lane);
        fetch_entries(f, cr, (long)blockIdx.x * kInferTile + wave * kInferRows, n, lane);
        const uint32_t second = blockIdx.x + gridDim.x;
        f.listed_next = second < tiles ? row_count(cr, (long)second * kInferTile + wave * kInferRows, n, lane) : 0u;
        fetch_records(f, cr, n, lane);
        form_rows(xa, f, cr, lane);
    }
    stage_weights(W, L, tid, kInferWaves * 64);
    __syncthreads();

    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const long row0 = (long)tile * kInferTile + wave * kInferRows;
        const int rows_left = (int)max(0L, min((long)kInferRows, (long)n - row0));
        const uint32_t next = tile + gridDim.x;
        const bool more = next < tiles;
        uint4 h[kKStepsH];
        infer_layer<kKSteps1, kLd1, 4>(xa, L.w1, L.bias, h, lane);
        if (more) {
            fetch_entries(f, cr, (long)next * kInferTile + wave * kInferRows, n, lane);
            const uint32_t after = next + gridDim.x;
            f.listed_next = after < tiles ? row_count(cr, (long)after * kInferTile + wave * kInferRows, n, lane) : 0u;
        }
        infer_layer<kKStepsH, kLdH, 4>(h, L.w2, L.bias + kMlpHidden, h, lane);
        if (more) fetch_records(f, cr, n, lane);
        infer_layer<kKStepsH, kLdH, 4>(h, L.w3, L.bias + 2 * kMlpHidden, h, lane);
        infer_output(h, L, Y, row0, rows_left, lane);
        if (more) form_rows(xa, f, cr, lane);
    }
}

inline unsigned nblk(long n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

// ------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------
// M x N product with K in `splits`; the caller fills in the epilogue's operands.
static GemmArgs gemm_args(const uint16_t* A, long sam, long sak, const uint16_t* B, long sbk, long sbn, int M, int N,
                          int K, int splits) {
    GemmArgs g{};
    g.A = A, g.B = B;
    g.sam = sam, g.sak = sak, g.sbk = sbk, g.sbn = sbn;
    g.M = M, g.N = N, g.K = K;
    g.k_split = ((K + splits - 1) / splits + kGemmKStage - 1) / kGemmKStage * kGemmKStage;
    g.nx = (N + kGemmTile - 1) / kGemmTile;
    g.ny = (M + kGemmTile - 1) / kGemmTile;
    // may runs of 8 along the contiguous dimension load as one 16-byte access (aligned base, the other stride
    // a multiple of 8)?
    auto aligned = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    g.vec_a = aligned(A) && (sam == 1 ? sak % 8 == 0 : (sak == 1 && sam % 8 == 0));
    g.vec_b = aligned(B) && (sbn == 1 ? sbk % 8 == 0 : (sbk == 1 && sbn % 8 == 0));
    return g;
}

// Splits of a weight gradient's sum over M rows: at least 256 rows each, up to about 512 workgroups and
// kMlpSplits (k_finish reads them all).
static int weight_splits(int kin, int n, int M) {
    const int tiles = ((kin + kGemmTile - 1) / kGemmTile) * ((n + kGemmTile - 1) / kGemmTile);
    if (M < 1024) return 1;
    const int want = std::min(std::min((M + 255) / 256, (512 + tiles - 1) / tiles), kMlpSplits);
    const int k_split = ((M + want - 1) / want + kGemmKStage - 1) / kGemmKStage * kGemmKStage;
    return (M + k_split - 1) / k_split;
}

MlpLayout mlp_layout() {
    MlpLayout L;
    size_t o = 0;
    L.w1 = o; o += (size_t)kMlpInPad * kMlpHidden;
    L.b1 = o; o += kMlpHidden;
    L.w2 = o; o += (size_t)kMlpHidden * kMlpHidden;
    L.b2 = o; o += kMlpHidden;
    L.w3 = o; o += (size_t)kMlpHidden * kMlpHidden;
    L.b3 = o; o += kMlpHidden;
    L.w4 = o; o += (size_t)kMlpHidden * kMlpOutPad;
    L.b4 = o; o += kMlpOutPad;
    L.total = o;
    return L;
}

hipError_t mlp_refresh_bf16(Mlp& m, hipStream_t s) {
    const MlpLayout L = mlp_layout();
    struct {
        size_t off;
        int K, N;
        uint16_t *rm, *tr;
    } mats[4] = {{L.w1, kMlpInPad, kMlpHidden, m.w1, m.w1t},
                 {L.w2, kMlpHidden, kMlpHidden, m.w2, m.w2t},
                 {L.w3, kMlpHidden, kMlpHidden, m.w3, m.w3t},
                 {L.w4, kMlpHidden, kMlpOutPad, m.w4, m.w4t}};
    for (auto& x : mats) {
        hipLaunchKernelGGL(k_cast, dim3(nblk((long)x.K * x.N, 256)), dim3(256), 0, s, m.master + x.off, x.rm, x.tr, x.K,
                           x.N);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t mlp_infer(const Mlp& m, const uint16_t* X, float* Y, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const MlpLayout L = mlp_layout();
    InferWeights W{m.w1t, m.w2t, m.w3t, m.w4t, m.master + L.b1, m.master + L.b2, m.master + L.b3, m.master + L.b4};
    // one workgroup per CU (the kernel holds most of a CU's LDS), each walking several tiles
    const unsigned tiles = nblk(n, kInferTile);
    hipLaunchKernelGGL(k_mlp_infer, dim3(tiles < 256u ? tiles : 256u), dim3(kInferWaves * 64), 0, s, X, W, Y, n);
    return hipGetLastError();
}

hipError_t mlp_infer_closure(const Mlp& m, const ClosureRows& rows, float* Y, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const MlpLayout L = mlp_layout();
    InferWeights W{m.w1t, m.w2t, m.w3t, m.w4t, m.master + L.b1, m.master + L.b2, m.master + L.b3, m.master + L.b4};
    const unsigned tiles = nblk(n, kInferTile);
    hipLaunchKernelGGL(k_mlp_infer_closure, dim3(tiles < 256u ? tiles : 256u), dim3(kInferWaves * 64), 0, s, rows, W,
                       Y, n);
    return hipGetLastError();
}

// Forward through the GEMM path, keeping what the backward pass needs.  With T, also the loss
// and the output-layer delta.
hipError_t mlp_forward_train(Mlp& m, const uint16_t* X, const float* T, float* Y, uint32_t M, hipStream_t s) {
    const MlpLayout L = mlp_layout();
    const float* bias[4] = {m.master + L.b1, m.master + L.b2, m.master + L.b3, m.master + L.b4};
    const uint16_t* w[4] = {m.w1, m.w2, m.w3, m.w4};
    for (int l = 0; l < 4; ++l) {
        const int kin = l == 0 ? kMlpInPad : kMlpHidden, n = l == 3 ? kMlpOutPad : kMlpHidden;
        GemmArgs g = gemm_args(l == 0 ? X : m.h[l - 1], kin, 1, w[l], n, 1, (int)M, n, kin, 1);
        g.bias = bias[l];
        if (l < 3) {
            g.Z = m.z[l];
            g.H = m.h[l];
            g.loss = l == 0 && T ? m.loss : nullptr;
            hipLaunchKernelGGL((k_gemm<false, true, kSilu>), dim3(g.nx * g.ny), dim3(256), 0, s, g);
        } else {
            g.H = m.d4;
            g.T = T;
            g.Y = Y;
            g.scale = 2.0f / (3.0f * (float)M);
            g.loss = m.loss;
            hipLaunchKernelGGL((k_gemm<false, true, kOutput>), dim3(g.nx * g.ny), dim3(256), 0, s, g);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Gradients of the mean squared error into m.grad (after mlp_forward_train with targets); with adam, also one
// step of Adam.
hipError_t mlp_backward(Mlp& m, const uint16_t* X, uint32_t M, bool adam, float lr, hipStream_t s) {
    const MlpLayout L = mlp_layout();
    const size_t w_off[4] = {L.w1, L.w2, L.w3, L.w4}, b_off[4] = {L.b1, L.b2, L.b3, L.b4};
    uint16_t* const w[4] = {m.w1, m.w2, m.w3, m.w4};
    uint16_t* const wt[4] = {m.w1t, m.w2t, m.w3t, m.w4t};
    uint16_t* const delta[4] = {m.d[0], m.d[1], m.d[0], m.d4};  // D_l; D_{l-1} is written while D_l is read
    FinishArgs f{};
    f.chunks = (int)((M + kColsumRows - 1) / kColsumRows);
    int blocks = 0;
    for (int l = 0; l < 4; ++l) {
        const int kin = l == 0 ? kMlpInPad : kMlpHidden, n = l == 3 ? kMlpOutPad : kMlpHidden;
        auto& a = f.layer[l];
        a.wpart = m.wpart + kMlpSplits * (w_off[l] - (l > 0 ? (size_t)l * kMlpHidden : 0u));  // biases lie between
        a.bpart = m.colpart[l];
        a.rowmajor = w[l], a.transposed = wt[l];
        a.w_off = (int)w_off[l], a.b_off = (int)b_off[l];
        a.K = kin, a.N = n;
        a.splits = weight_splits(kin, n, (int)M);
        a.first = blocks;
        blocks += (kin * n + 255) / 256 + 1;
    }
    for (int l = 3; l >= 0; --l) {
        // dW_l = H_{l-1}^T D_l (H_{-1} = X)
        const auto& a = f.layer[l];
        GemmArgs g = gemm_args(l == 0 ? X : m.h[l - 1], 1, a.K, delta[l], a.N, 1, a.K, a.N, (int)M, a.splits);
        g.C = const_cast<float*>(a.wpart);
        const int wblocks = g.nx * g.ny * a.splits, cblocks = (a.N + 63) / 64 * f.chunks;
        // D_{l-1} = (D_l W_l^T) * silu'(Z_{l-1})
        GemmArgs d{};
        if (l > 0) {
            d = gemm_args(delta[l], a.N, 1, w[l], 1, a.N, (int)M, kMlpHidden, a.N, 1);
            d.Z = m.z[l - 1];
            d.H = delta[l - 1];
        }
        const int dblocks = d.nx * d.ny;
        hipLaunchKernelGGL(k_gemm_backward, dim3(wblocks + dblocks + cblocks), dim3(256), 0, s, g, wblocks, d, dblocks,
                           m.colpart[l]);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    f.w = m.master, f.grad = m.grad, f.m = m.adam_m, f.v = m.adam_v;
    if (adam) {
        m.adam_t += 1;
        f.lr = lr, f.b1 = 0.9f, f.b2 = 0.999f, f.eps = 1e-8f;
        f.c1 = 1.0f - powf(f.b1, (float)m.adam_t), f.c2 = 1.0f - powf(f.b2, (float)m.adam_t);
        hipLaunchKernelGGL(k_finish<true>, dim3(blocks), dim3(256), 0, s, f);
    } else {
        hipLaunchKernelGGL(k_finish<false>, dim3(blocks), dim3(256), 0, s, f);
    }
    return hipGetLastError();
}

}  // namespace wc
