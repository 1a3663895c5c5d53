// Learned warm start: a small ReLU MLP trained and evaluated on the GPU (gfx950).
//
// No counterpart in the reference: this is the network that predicts a correction
// to SolverSAP's plain initial velocity.  bfloat16 operands with float32
// accumulation; bfloat16 rounding points: normalised inputs, weights, hidden
// activations and back-propagated gradients; biases, the output and all
// accumulations are float32.
//
// Every layer of a row depends on that row alone, so a network whose activations
// fit in LDS (net_fits) runs whole on row blocks:
//   forward     one launch: a workgroup normalises its rows into LDS and takes them
//               through all layers, streaming the weights from L2
//   gradients   two launches: the same forward pass, then the loss gradient and the
//               back-propagation through all layers in place of the activations, writing
//               each activation and gradient transposed; then every layer's weight
//               gradient (K = batch), the bias gradients and the loss in one launch
// All matrix operands in memory are packed in 16 x 32 tiles in the order of the
// lanes of v_mfma_f32_16x16x32_bf16 (packed_index), so that each operand load of a
// wave is one contiguous kilobyte.
//
// Wider networks use one GEMM per product, C[M x N] = A[M x K] . B[N x K]^T with
// both operands row-major and contiguous along K, one wave per 64 x 64 tile:
//   forward      h_{l+1} = relu(h_l W_l^T + b_l)        A = h_l,        B = W_l
//   input grad   dz_l    = (dz_{l+1} W_l) * [h_l > 0]    A = dz_{l+1},   B = W_l^T
//   weight grad  dW_l    = dz_{l+1}^T h_l                A = dz_{l+1}^T, B = h_l^T
// and the epilogues write each activation / gradient both row-major and transposed.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/sapx.h"

namespace sapx {
namespace mlp {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kMaxLayers = 8;

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN
    u += 0x7fffu + ((u >> 16) & 1u);                     // round to nearest, ties to even
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

enum Epilogue : int {
    EPI_F32 = 0,         // Cf = acc (+ bias)
    EPI_RELU_BF16 = 1,   // Cb = bf16(relu(acc + bias)), optional transposed copy Ct
    EPI_MASK_BF16 = 2,   // Cb = bf16(acc * [H > 0]), transposed copy Ct, column sums of acc * [H > 0] into colsum
};

struct GemmArgs {
    const uint16_t* A;
    const uint16_t* B;
    int lda, ldb;
    int K;
    const float* bias;
    float* Cf;
    uint16_t* Cb;
    uint16_t* Ct;
    int ldc, ldt;
    const uint16_t* H;
    int ldh;
    float* colsum;
};

// one wave: a 64 x 64 tile of C at (blockIdx.y, blockIdx.x); M, N multiples of 64,
// K a multiple of 16, operand rows 8-byte aligned
template <int EPI>
__global__ __launch_bounds__(64) void gemm_nt_kernel(GemmArgs g) {
    const int lane = threadIdx.x;
    const int r = lane & 15, kq = lane >> 4;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    f4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* Ap = g.A + (size_t)(m0 + r) * g.lda + 4 * kq;
    const uint16_t* Bp = g.B + (size_t)(n0 + r) * g.ldb + 4 * kq;
    const size_t as = (size_t)16 * g.lda, bs = (size_t)16 * g.ldb;
    for (int k0 = 0; k0 < g.K; k0 += 16) {
        s4 a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const s4*>(Ap + i * as + k0);
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const s4*>(Bp + j * bs + k0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    // D layout: acc[i][j][e] = C[m0 + 16 i + 4 kq + e][n0 + 16 j + r]
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n0 + 16 * j + r;
        const float bn = g.bias ? g.bias[n] : 0.0f;
        float csum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int mb = m0 + 16 * i + 4 * kq;
            uint16_t tb[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = mb + e;
                float v = acc[i][j][e];
                if (EPI == EPI_F32) {
                    g.Cf[(size_t)m * g.ldc + n] = v + bn;
                } else if (EPI == EPI_RELU_BF16) {
                    v = fmaxf(v + bn, 0.0f);
                    const uint16_t h = f2bf(v);
                    g.Cb[(size_t)m * g.ldc + n] = h;
                    tb[e] = h;
                } else {
                    v = bf2f(g.H[(size_t)m * g.ldh + n]) > 0.0f ? v : 0.0f;
                    const uint16_t h = f2bf(v);
                    g.Cb[(size_t)m * g.ldc + n] = h;
                    tb[e] = h;
                    csum += v;
                }
            }
            if (EPI != EPI_F32 && g.Ct) {
                // four consecutive rows of column n: one 8-byte store into the transposed copy
                const uint64_t packed = (uint64_t)tb[0] | ((uint64_t)tb[1] << 16) | ((uint64_t)tb[2] << 32) |
                                        ((uint64_t)tb[3] << 48);
                *reinterpret_cast<uint64_t*>(g.Ct + (size_t)n * g.ldt + mb) = packed;
            }
        }
        if (EPI == EPI_MASK_BF16) {
            // lanes r, r + 16, r + 32, r + 48 hold the same column
            csum += __shfl_xor(csum, 16, 64);
            csum += __shfl_xor(csum, 32, 64);
            if (kq == 0) atomicAdd(g.colsum + n, csum);
        }
    }
}

// x_raw [B x F] float32 -> normalised bfloat16 rows [Bp x d0] and the transposed copy
// [d0 x Bp]; rows >= B and columns >= F are zero
__global__ void normalize_input_kernel(const float* x, int B, int F, int Bp, int d0, const float* mean, const float* stdv,
                                       uint16_t* xb, uint16_t* xt) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)Bp * d0) return;
    const int b = (int)(t / d0), f = (int)(t % d0);
    float v = 0.0f;
    if (b < B && f < F) v = (x[(size_t)b * F + f] - mean[f]) / stdv[f];
    const uint16_t h = f2bf(v);
    xb[t] = h;
    xt[(size_t)f * Bp + b] = h;
}

// normalised output y [Bp x dL] -> y_raw [B x O] = y * std + mean
__global__ void unnormalize_output_kernel(const float* y, int B, int O, int dL, const float* mean, const float* stdv,
                                          float* out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= B * O) return;
    const int b = t / O, o = t % O;
    out[t] = y[(size_t)b * dL + o] * stdv[o] + mean[o];
}

// mean squared error over the real outputs in normalised units, its gradient dz
// (bfloat16, row-major and transposed) and the output bias gradient (column sums);
// blocks of 256 threads = 4 row lanes x 64 columns, 64 rows per block
__global__ __launch_bounds__(256) void loss_grad_kernel(const float* y, const float* target, int B, int O, int Bp,
                                                        int dL, const float* mean, const float* stdv, uint16_t* dz,
                                                        uint16_t* dzt, float* dbias, float* loss) {
    __shared__ float part[4][64];
    __shared__ float lpart[256];
    const int c = threadIdx.x & 63, rl = threadIdx.x >> 6;
    const float scale = 2.0f / ((float)B * (float)O);
    float cs = 0.0f, ls = 0.0f;
    for (int cc = c; cc < dL; cc += 64) {
        float csc = 0.0f;
        for (int k = 0; k < 16; ++k) {
            const int b = blockIdx.x * 64 + rl * 16 + k;
            if (b >= Bp) break;
            float d = 0.0f;
            if (b < B && cc < O) {
                const float t = (target[(size_t)b * O + cc] - mean[cc]) / stdv[cc];
                d = y[(size_t)b * dL + cc] - t;
                ls += d * d;
            }
            const float gz = scale * d;
            const uint16_t h = f2bf(gz);
            dz[(size_t)b * dL + cc] = h;
            dzt[(size_t)cc * Bp + b] = h;
            csc += gz;
        }
        if (cc == c) cs = csc;
        else atomicAdd(dbias + cc, csc);  // only when dL > 64
    }
    part[rl][c] = cs;
    lpart[threadIdx.x] = ls;
    __syncthreads();
    if (rl == 0 && c < dL) atomicAdd(dbias + c, part[0][c] + part[1][c] + part[2][c] + part[3][c]);
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) lpart[threadIdx.x] += lpart[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, lpart[0] / ((float)B * (float)O));
}

__global__ void fill_kernel(float* p, size_t n, float v) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

struct LayerOffsets {
    int L;
    int dims[kMaxLayers + 1];
    long long w_off[kMaxLayers];   // flat float offset of W_l (b_l follows it)
    long long wb_off[kMaxLayers];  // offset of W_l inside the bfloat16 weight arrays
    long long total;
};

// ---------------------------------------------------------------------------
// networks whose activations fit in LDS
// ---------------------------------------------------------------------------
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8;               // waves of a row-block workgroup
constexpr int kRowPad = 8;              // bfloat16 padding of an LDS row: the 16 rows of a fragment
                                        // start four banks apart
constexpr size_t kMaxLds = 160 * 1024;

// element (r, k) of an operand with K columns: tiles of 16 rows x 32 columns, inside a tile the
// eight consecutive columns of lane (r % 16) + 16 * ((k % 32) / 8)
__host__ __device__ __forceinline__ size_t packed_index(int r, int k, int K) {
    return ((size_t)(r >> 4) * (K >> 5) + (k >> 5)) * 512 + (((r & 15) + 16 * ((k & 31) >> 3)) << 3) + (k & 7);
}

// LDS offset (elements) of layer l's activations for `rows` rows
__host__ __device__ __forceinline__ int act_offset(const LayerOffsets& lo, int l, int rows) {
    int off = 0;
    for (int i = 0; i < l; ++i) off += rows * (lo.dims[i] + kRowPad);
    return off;
}
// inference keeps two layers at a time: the even ones share one buffer, the odd ones the other behind
// it, so the two never take more than all layers together (one wide layer among narrow ones: two
// buffers of the widest would)
__host__ __device__ __forceinline__ int widest(const LayerOffsets& lo, int parity) {
    int w = 0;
    for (int l = parity; l <= lo.L; l += 2) w = lo.dims[l] > w ? lo.dims[l] : w;
    return w;
}

// CT tiles of 16 columns starting at tile t0, MT tiles of 16 rows: acc = act . W^T over `steps` pairs
// of MFMA column groups (act: LDS rows of stride ls; Wp: packed weights).  The weights of U steps are
// loaded while the U before them multiply; `ready` runs after the first loads are under way and
// before the first read of act.
template <int MT, int CT, int U, typename Ready>
__device__ __forceinline__ void tile_product(const uint16_t* act, int ls, const uint16_t* Wp, int steps, int t0, Ready&& ready,
                                             f4 (&acc)[MT][CT]) {
    const int lane = threadIdx.x & 63;
    const uint16_t* ap = act + (lane & 15) * ls + 8 * (lane >> 4);
    const uint16_t* bp = Wp + (size_t)t0 * steps * 512 + lane * 8;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    b8 b0[U][CT], b1[U][CT];
    auto load = [&](b8 (&b)[U][CT], int c) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < CT; ++j) b[u][j] = *reinterpret_cast<const b8*>(bp + ((size_t)j * steps + c * U + u) * 512);
        __builtin_amdgcn_sched_barrier(0);  // issued here: left alone they sink to their first use
    };
    auto multiply = [&](const b8 (&b)[U][CT], int c) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            b8 a[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) a[i] = *reinterpret_cast<const b8*>(ap + i * 16 * ls + (c * U + u) * 32);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[u][j], acc[i][j], 0, 0, 0);
        }
    };
    const int chunks = steps / U;
    load(b0, 0);
    ready();
    int c = 0;
    for (; c + 2 <= chunks; c += 2) {
        load(b1, c + 1);
        multiply(b0, c);
        if (c + 2 < chunks) load(b0, c + 2);
        multiply(b1, c + 1);
    }
    if (c < chunks) multiply(b0, c);
}

__device__ __forceinline__ uint64_t pack4(const uint16_t* h) {
    return (uint64_t)h[0] | ((uint64_t)h[1] << 16) | ((uint64_t)h[2] << 32) | ((uint64_t)h[3] << 48);
}

struct RowBlockArgs {
    LayerOffsets lo;
    const float* params;
    const uint16_t* wb;    // packed W_l [dims[l+1] x dims[l]]
    const uint16_t* wt;    // packed W_l^T [dims[l] x dims[l+1]] (gradients only)
    const float* norm;     // x_mean [F], x_std [F], y_mean [O], y_std [O]
    const float* x;
    int B, Bp, F, O;
    float* y;              // forward: the output rows
    // gradients
    const float* target;
    uint16_t* ht[kMaxLayers];   // packed h_l^T [dims[l] x Bp]
    uint16_t* dzt[kMaxLayers];  // packed dz_{l+1}^T [dims[l+1] x Bp]
    float* bias_part;      // workgroups x bias columns of all layers
    int bias_cols;
    float* loss_part;      // one per workgroup
};

// the layer's column tiles, shared out over the waves; starts with the workgroup's barrier after the
// writes of `act`.  pre(n) loads what the epilogue epi(n, pre(n), acc, j) of column n needs, ahead of
// the product.
template <int MT, int CT, int U, typename Pre, typename Epi>
__device__ __forceinline__ void layer_tiles(const uint16_t* act, int ls, const uint16_t* Wp, int K, int N, Pre&& pre, Epi&& epi) {
    const int wave = threadIdx.x >> 6, tiles = N >> 4;
    bool first = true;
    auto ready = [&] {
        if (first) __syncthreads();
        first = false;
    };
    for (int t0 = wave * CT; t0 < tiles; t0 += kWaves * CT) {
        f4 acc[MT][CT];
        float3 col[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) col[j] = pre(16 * (t0 + j) + (threadIdx.x & 15));
        tile_product<MT, CT, U>(act, ls, Wp, K >> 5, t0, ready, acc);
#pragma unroll
        for (int j = 0; j < CT; ++j) epi(16 * (t0 + j) + (threadIdx.x & 15), col[j], acc, j);
    }
    ready();
}
// four column tiles a wave where every wave gets them, fewer in narrow layers (their waves would
// idle); K is a multiple of 64: chunks of four steps where they divide it, else of two
template <int MT, typename Pre, typename Epi>
__device__ __forceinline__ void layer(const uint16_t* act, int ls, const uint16_t* Wp, int K, int N, Pre&& pre, Epi&& epi) {
    const int tiles = N >> 4;
    const bool four = K % 128 == 0;
    if (tiles % (4 * kWaves) == 0) {
        if (four) layer_tiles<MT, 4, 4>(act, ls, Wp, K, N, pre, epi);
        else layer_tiles<MT, 4, 2>(act, ls, Wp, K, N, pre, epi);
    } else if (tiles % (2 * kWaves) == 0) {
        if (four) layer_tiles<MT, 2, 4>(act, ls, Wp, K, N, pre, epi);
        else layer_tiles<MT, 2, 2>(act, ls, Wp, K, N, pre, epi);
    } else {
        if (four) layer_tiles<MT, 1, 4>(act, ls, Wp, K, N, pre, epi);
        else layer_tiles<MT, 1, 2>(act, ls, Wp, K, N, pre, epi);
    }
}

// One workgroup: 16 MT rows through the whole network (TRAIN: and back).  Bound by streaming the
// weights (1.4 MB at 311-512-512-512-35) from L2 into each CU, so the next weights are always under
// way: within a layer U steps ahead, and a layer's first ones before the barrier that ends the layer
// before it.  4096 rows of that network: 21 us (six launches of one GEMM per layer took 89); forward
// and back-propagation of a training step 44 us (was 680 for the whole step, now 44 + 17 + 8).
template <int MT, bool TRAIN>
__global__ __launch_bounds__(kWaves * 64) void row_block_kernel(RowBlockArgs g) {
    extern __shared__ __attribute__((aligned(16))) uint16_t sm[];
    constexpr int R = 16 * MT;
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4;
    const int r0 = blockIdx.x * R;
    const int L = g.lo.L;
    // inference needs two layers' activations at a time, training keeps them all
    const int odd = TRAIN ? 0 : R * (widest(g.lo, 0) + kRowPad);
    auto act = [&](int l) { return sm + (TRAIN ? act_offset(g.lo, l, R) : (l & 1) * odd); };
    {
        const int d0 = g.lo.dims[0], ls = d0 + kRowPad;
        const float* mean = g.norm;
        const float* stdv = g.norm + g.F;
        uint16_t* X = act(0);
        // a wave takes R / 8 rows, eight features a lane: all their loads are in flight together
        constexpr int RW = R / kWaves, FU = 8;
        const int row = (tid >> 6) * RW;
        for (int f0 = 0; f0 < d0; f0 += 64 * FU) {
            float mu[FU], sd[FU], xv[RW][FU];
#pragma unroll
            for (int u = 0; u < FU; ++u) {
                const int f = f0 + 64 * u + lane;
                mu[u] = f < g.F ? mean[f] : 0.0f;
                sd[u] = f < g.F ? stdv[f] : 1.0f;
#pragma unroll
                for (int r = 0; r < RW; ++r)
                    xv[r][u] = f < g.F && r0 + row + r < g.B ? g.x[(size_t)(r0 + row + r) * g.F + f] : mu[u];
            }
#pragma unroll
            for (int u = 0; u < FU; ++u) {
                const int f = f0 + 64 * u + lane;
                if (f < d0) {
#pragma unroll
                    for (int r = 0; r < RW; ++r) X[(row + r) * ls + f] = f2bf((xv[r][u] - mu[u]) / sd[u]);
                }
            }
        }
        if (TRAIN) {
            __syncthreads();
            for (int e = tid; e < d0 * (R / 8); e += kWaves * 64) {
                const int f = e % d0, r = 8 * (e / d0);
                uint16_t h[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) h[u] = X[(r + u) * ls + f];
                uint64_t* o = reinterpret_cast<uint64_t*>(g.ht[0] + packed_index(f, r0 + r, g.Bp));
                o[0] = pack4(h);
                o[1] = pack4(h + 4);
            }
        }
    }
    const float* ymean = g.norm + 2 * g.F;
    const float* ystd = ymean + g.O;
    float lsum = 0.0f;
    int bcol = 0;  // first bias column of layer l
    for (int l = 0; l < L; ++l) {
        const int K = g.lo.dims[l], N = g.lo.dims[l + 1];
        const float* bias = g.params + g.lo.w_off[l] + (long long)K * N;
        const uint16_t* Wp = g.wb + g.lo.wb_off[l];
        const auto out_pre = [&](int n) {
            const bool real = n < g.O;
            return float3{bias[n], real ? ystd[n] : 1.0f, real ? ymean[n] : 0.0f};
        };
        if (l < L - 1) {
            uint16_t* H = act(l + 1);
            const int hs = N + kRowPad;
            const auto pre = [&](int n) { return float3{bias[n], 0.0f, 0.0f}; };
            layer<MT>(act(l), K + kRowPad, Wp, K, N, pre, [&](int n, float3 c, auto& acc, int j) {
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    uint16_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        h[e] = f2bf(fmaxf(acc[i][j][e] + c.x, 0.0f));
                        H[(16 * i + 4 * kq + e) * hs + n] = h[e];
                    }
                    if (TRAIN) *reinterpret_cast<uint64_t*>(g.ht[l + 1] + packed_index(n, r0 + 16 * i + 4 * kq, g.Bp)) = pack4(h);
                }
            });
            bcol += N;
        } else if (!TRAIN) {
            layer<MT>(act(l), K + kRowPad, Wp, K, N, out_pre, [&](int n, float3 c, auto& acc, int j) {
                if (n >= g.O) return;
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int b = r0 + 16 * i + 4 * kq + e;
                        if (b < g.B) g.y[(size_t)b * g.O + n] = (acc[i][j][e] + c.x) * c.y + c.z;
                    }
            });
        } else {
            // mean squared error over the real outputs in normalised units, and its gradient
            const float scale = 2.0f / ((float)g.B * (float)g.O);
            uint16_t* H = act(L);
            const int hs = N + kRowPad;
            float* bp = g.bias_part + (size_t)blockIdx.x * g.bias_cols + bcol;
            layer<MT>(act(l), K + kRowPad, Wp, K, N, out_pre, [&](int n, float3 c, auto& acc, int j) {
                const bool real = n < g.O;
                float cs = 0.0f;
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    uint16_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int b = r0 + 16 * i + 4 * kq + e;
                        float d = 0.0f;
                        if (real && b < g.B) {
                            d = acc[i][j][e] + c.x - (g.target[(size_t)b * g.O + n] - c.z) / c.y;
                            lsum += d * d;
                        }
                        const float gz = scale * d;
                        cs += gz;
                        h[e] = f2bf(gz);
                        H[(16 * i + 4 * kq + e) * hs + n] = h[e];
                    }
                    *reinterpret_cast<uint64_t*>(g.dzt[L - 1] + packed_index(n, r0 + 16 * i + 4 * kq, g.Bp)) = pack4(h);
                }
                cs += __shfl_xor(cs, 16, 64);
                cs += __shfl_xor(cs, 32, 64);
                if (kq == 0) bp[n] = cs;
            });
        }
    }
    if (!TRAIN) return;
    // back-propagation: dz_l = (dz_{l+1} W_l) * [h_l > 0], in the place of h_l
    for (int l = L - 1; l > 0; --l) {
        const int K = g.lo.dims[l + 1], N = g.lo.dims[l];
        bcol -= N;  // bias columns of layer l - 1
        uint16_t* H = act(l);
        const int hs = N + kRowPad;
        float* bp = g.bias_part + (size_t)blockIdx.x * g.bias_cols + bcol;
        const auto pre = [](int) { return float3{0.0f, 0.0f, 0.0f}; };
        layer<MT>(act(l + 1), K + kRowPad, g.wt + g.lo.wb_off[l], K, N, pre, [&](int n, float3, auto& acc, int j) {
            float cs = 0.0f;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                uint16_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint16_t* p = H + (16 * i + 4 * kq + e) * hs + n;
                    const float v = bf2f(*p) > 0.0f ? acc[i][j][e] : 0.0f;
                    cs += v;
                    h[e] = f2bf(v);
                    *p = h[e];
                }
                *reinterpret_cast<uint64_t*>(g.dzt[l - 1] + packed_index(n, r0 + 16 * i + 4 * kq, g.Bp)) = pack4(h);
            }
            cs += __shfl_xor(cs, 16, 64);
            cs += __shfl_xor(cs, 32, 64);
            if (kq == 0) bp[n] = cs;
        });
    }
    __syncthreads();
    // this block's share of the loss
    float* red = reinterpret_cast<float*>(sm);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
    if (lane == 0) red[tid >> 6] = lsum;
    __syncthreads();
    if (tid == 0) {
        float s = 0.0f;
        for (int w = 0; w < kWaves; ++w) s += red[w];
        g.loss_part[blockIdx.x] = s;
    }
}

struct WeightGradArgs {
    LayerOffsets lo;
    const uint16_t* ht[kMaxLayers];
    const uint16_t* dzt[kMaxLayers];
    int Bp;
    float* grads;
    int tile0[kMaxLayers + 1];  // first 64 x 64 weight tile of each layer
    const float* bias_part;
    const float* loss_part;
    int blocks, bias_cols;      // row blocks, bias columns of all layers
    float inv_count;            // 1 / (B O)
    float* loss;
};

// Every layer's weight gradient dW_l = dz_{l+1}^T h_l in one launch (a single layer's 64 x 64 tiles
// would leave most CUs idle: 98 us each for one of 64 tiles of 4096 rows, all of them now 17 us): a
// workgroup owns a tile, its waves split the batch and add up in LDS; the last workgroups add the row
// blocks' bias gradients (64 columns each) and the loss, in a fixed order.
__global__ __launch_bounds__(kWaves * 64) void weight_grad_kernel(WeightGradArgs g) {
    __shared__ float red[kWaves / 2][64 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // blocks go round the eight XCDs: each XCD takes consecutive tiles, whose operands share its L2
    // (in plain order every XCD would read nearly all of them)
    const int ntile = g.tile0[g.lo.L], share = (ntile + 7) >> 3;
    int t = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
    if ((int)blockIdx.x >= 8 * share) {
        t = (int)blockIdx.x - 8 * share;
        float s = 0.0f;
        if (64 * t < g.bias_cols) {
            const int c = 64 * t + lane;
            for (int b = wave; b < g.blocks; b += kWaves) s += g.bias_part[(size_t)b * g.bias_cols + c];
        } else {
            for (int b = tid; b < g.blocks; b += kWaves * 64) s += g.loss_part[b];
        }
        red[0][tid] = s;
        __syncthreads();
        if (wave > 0) return;
        for (int w = 1; w < kWaves; ++w) s += red[0][64 * w + lane];
        if (64 * t < g.bias_cols) {
            int c = 64 * t + lane, l = 0;
            while (c >= g.lo.dims[l + 1]) c -= g.lo.dims[++l];
            g.grads[g.lo.w_off[l] + (long long)g.lo.dims[l] * g.lo.dims[l + 1] + c] = s;
        } else {
            for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
            if (lane == 0 && g.loss) g.loss[0] = s * g.inv_count;
        }
        return;
    }
    if (t >= ntile || t >= ((int)(blockIdx.x & 7) + 1) * share) return;
    int l = 0;
    while (t >= g.tile0[l + 1]) ++l;
    t -= g.tile0[l];
    const int din = g.lo.dims[l], nt = din >> 6;
    const int m0 = 64 * (t / nt), n0 = 64 * (t % nt);
    const int steps = g.Bp >> 5;
    const uint16_t* Ap = g.dzt[l] + (size_t)(m0 >> 4) * steps * 512 + lane * 8;
    const uint16_t* Bq = g.ht[l] + (size_t)(n0 >> 4) * steps * 512 + lane * 8;
    f4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    // wave w takes steps w, w + 8, ...; the operands of two steps are loaded together
    auto group = [&](auto width, int s) {
        constexpr int V = decltype(width)::value;
        b8 a[V][4], b[V][4];
#pragma unroll
        for (int u = 0; u < V; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[u][i] = *reinterpret_cast<const b8*>(Ap + ((size_t)i * steps + s + u * kWaves) * 512);
                b[u][i] = *reinterpret_cast<const b8*>(Bq + ((size_t)i * steps + s + u * kWaves) * 512);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < V; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i], b[u][j], acc[i][j], 0, 0, 0);
    };
    int s = wave;
    for (; s + kWaves < steps; s += 2 * kWaves) group(std::integral_constant<int, 2>{}, s);
    if (s < steps) group(std::integral_constant<int, 1>{}, s);
    // halve the waves' partial tiles until one is left (fixed order)
#pragma unroll
    for (int half = kWaves / 2; half > 0; half >>= 1) {
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<f4*>(&red[wave - half][((4 * i + j) * 64 + lane) * 4]) = acc[i][j];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += *reinterpret_cast<const f4*>(&red[wave][((4 * i + j) * 64 + lane) * 4]);
        }
        __syncthreads();
    }
    // the tile goes out over all waves, 16 lanes per row
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) red[0][(16 * i + 4 * (lane >> 4) + e) * 64 + 16 * j + (lane & 15)] = acc[i][j][e];
    }
    __syncthreads();
    float* out = g.grads + g.lo.w_off[l] + (long long)m0 * din + n0;
    for (int e = tid; e < 64 * 64; e += kWaves * 64) out[(long long)(e >> 6) * din + (e & 63)] = red[0][e];
}

// Adam (bias-corrected moments) and the packed bfloat16 weights: a workgroup takes a 64 x 64 tile of
// one layer's W_l, updates it and writes the tile of W_l and of W_l^T through LDS; the last
// workgroups take the biases.
__global__ __launch_bounds__(256) void adam_packed_kernel(float* p, const float* grad, float* m, float* v, LayerOffsets lo,
                                                          WeightGradArgs tiles, float lr, float b1, float b2, float eps,
                                                          float c1, float c2, uint16_t* wb, uint16_t* wt, int update) {
    __shared__ uint16_t sw[64][64 + 8];
    auto adam = [&](float& x, float g, float& mm, float& vv) {
        mm = b1 * mm + (1.0f - b1) * g;
        vv = b2 * vv + (1.0f - b2) * g * g;
        x -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    };
    int t = blockIdx.x;
    if (t >= tiles.tile0[lo.L]) {
        int c = 256 * (t - tiles.tile0[lo.L]) + threadIdx.x, l = 0;
        while (l < lo.L && c >= lo.dims[l + 1]) c -= lo.dims[++l];
        if (l < lo.L && update) {
            const long long t = lo.w_off[l] + (long long)lo.dims[l] * lo.dims[l + 1] + c;
            adam(p[t], grad[t], m[t], v[t]);
        }
        return;
    }
    int l = 0;
    while (t >= tiles.tile0[l + 1]) ++l;
    t -= tiles.tile0[l];
    const int nin = lo.dims[l], nout = lo.dims[l + 1], nt = nin >> 6;
    const int o0 = 64 * (t / nt), i0 = 64 * (t % nt);
    // rows of W_l start at multiples of 64 floats: four parameters a load
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int o = 16 * k + (threadIdx.x >> 4), i = 4 * (threadIdx.x & 15);
        const long long t = lo.w_off[l] + (long long)(o0 + o) * nin + i0 + i;
        float4 x = *reinterpret_cast<const float4*>(p + t);
        if (update) {
            const float4 gr = *reinterpret_cast<const float4*>(grad + t);
            float4 mm = *reinterpret_cast<const float4*>(m + t), vv = *reinterpret_cast<const float4*>(v + t);
            adam(x.x, gr.x, mm.x, vv.x);
            adam(x.y, gr.y, mm.y, vv.y);
            adam(x.z, gr.z, mm.z, vv.z);
            adam(x.w, gr.w, mm.w, vv.w);
            *reinterpret_cast<float4*>(p + t) = x;
            *reinterpret_cast<float4*>(m + t) = mm;
            *reinterpret_cast<float4*>(v + t) = vv;
        }
        const uint16_t h[4] = {f2bf(x.x), f2bf(x.y), f2bf(x.z), f2bf(x.w)};
        *reinterpret_cast<uint64_t*>(&sw[o][i]) = pack4(h);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * 8; e += 256) {
        // eight columns of one row of the tile: of W_l, then of W_l^T
        const int r = e & 63, k = 8 * (e >> 6);
        uint16_t h[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) h[u] = sw[r][k + u];
        uint64_t* o = reinterpret_cast<uint64_t*>(wb + lo.wb_off[l] + packed_index(o0 + r, i0 + k, nin));
        o[0] = pack4(h);
        o[1] = pack4(h + 4);
#pragma unroll
        for (int u = 0; u < 8; ++u) h[u] = sw[k + u][r];
        o = reinterpret_cast<uint64_t*>(wt + lo.wb_off[l] + packed_index(i0 + r, o0 + k, nout));
        o[0] = pack4(h);
        o[1] = pack4(h + 4);
    }
}

// Adam over the flat parameters (bias-corrected moments), then the bfloat16 weight
// copies W_l and W_l^T are refreshed from the float32 master values
__global__ void adam_kernel(float* p, const float* grad, float* m, float* v, LayerOffsets lo, float lr, float b1,
                            float b2, float eps, float c1, float c2, uint16_t* wb, uint16_t* wt, int update) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= lo.total) return;
    float x = p[t];
    if (update) {
        const float g = grad[t];
        const float mm = b1 * m[t] + (1.0f - b1) * g;
        const float vv = b2 * v[t] + (1.0f - b2) * g * g;
        m[t] = mm;
        v[t] = vv;
        x -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
        p[t] = x;
    }
    for (int l = 0; l < lo.L; ++l) {
        const long long nin = lo.dims[l], nout = lo.dims[l + 1];
        const long long rel = t - lo.w_off[l];
        if (rel >= 0 && rel < nin * nout) {
            const long long o = rel / nin, i = rel % nin;
            const uint16_t h = f2bf(x);
            wb[lo.wb_off[l] + o * nin + i] = h;
            wt[lo.wb_off[l] + i * nout + o] = h;
        }
    }
}

}  // namespace mlp
}  // namespace sapx

using namespace sapx::mlp;

namespace sapx {
void set_last_error(const char* msg);
}

namespace {
int32_t mfail(int32_t code, const std::string& msg) {
    sapx::set_last_error(msg.c_str());
    return code;
}
}  // namespace

#define MLP_HIP(expr)                                                                        \
    do {                                                                                     \
        hipError_t _e = (expr);                                                              \
        if (_e != hipSuccess) return mfail(SAPX_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

struct SapxMlp {
    LayerOffsets lo{};
    int in_features = 0, out_features = 0;
    long long wb_total = 0;
    float* params = nullptr;
    float* grads = nullptr;
    float* m = nullptr;
    float* v = nullptr;
    uint16_t* wb = nullptr;
    uint16_t* wt = nullptr;
    float* norm = nullptr;  // x_mean [F], x_std [F], y_mean [O], y_std [O]
    float* loss = nullptr;
    int adam_t = 0;
    // workspace for batches up to cap rows
    int cap = 0;
    uint16_t* xb = nullptr;
    uint16_t* xt = nullptr;
    uint16_t* h[kMaxLayers] = {nullptr};
    uint16_t* ht[kMaxLayers] = {nullptr};
    float* y = nullptr;
    uint16_t* dz[2] = {nullptr, nullptr};
    uint16_t* dzt[2] = {nullptr, nullptr};
    // a network that runs on row blocks: packed transposed activations (ht) and gradients, the row
    // blocks' bias gradients and losses, and y for outputs that overlap their input (other forward
    // passes need no workspace)
    bool row_blocks = false;
    uint16_t* dzp[kMaxLayers] = {nullptr};
    float* bias_part = nullptr;
    float* loss_part = nullptr;
    void free_ws() {
        void* ps[] = {xb, xt, y, dz[0], dz[1], dzt[0], dzt[1], bias_part, loss_part};
        for (void* p : ps)
            if (p) (void)hipFree(p);
        for (int l = 0; l < kMaxLayers; ++l) {
            if (h[l]) (void)hipFree(h[l]);
            if (ht[l]) (void)hipFree(ht[l]);
            if (dzp[l]) (void)hipFree(dzp[l]);
            h[l] = ht[l] = dzp[l] = nullptr;
        }
        xb = xt = nullptr;
        y = bias_part = loss_part = nullptr;
        dz[0] = dz[1] = dzt[0] = dzt[1] = nullptr;
        cap = 0;
    }
    ~SapxMlp() {
        free_ws();
        void* ps[] = {params, grads, m, v, wb, wt, norm, loss};
        for (void* p : ps)
            if (p) (void)hipFree(p);
    }
    int maxw() const {
        int w = 0;
        for (int l = 0; l <= lo.L; ++l) w = lo.dims[l] > w ? lo.dims[l] : w;
        return w;
    }
    int bias_cols() const {
        int c = 0;
        for (int l = 1; l <= lo.L; ++l) c += lo.dims[l];
        return c;
    }
    size_t train_lds(int mt) const { return (size_t)act_offset(lo, lo.L + 1, 16 * mt) * 2; }
    size_t forward_lds(int mt) const { return (size_t)16 * mt * (widest(lo, 0) + widest(lo, 1) + 2 * kRowPad) * 2; }
};

// all layers' activations of 16 rows fit in the LDS of a workgroup (then two buffers of the forward pass do)
static bool net_fits(const SapxMlp* M) { return M->train_lds(1) <= kMaxLds; }

static int32_t reserve(SapxMlp* M, int batch) {
    const int Bp = (batch + 63) / 64 * 64;
    if (Bp <= M->cap) return SAPX_OK;
    M->free_ws();
    const int L = M->lo.L;
    const size_t mw = (size_t)M->maxw();
    if (M->row_blocks) {
        for (int l = 0; l < L; ++l) {
            MLP_HIP(hipMalloc(&M->ht[l], (size_t)Bp * M->lo.dims[l] * 2));
            MLP_HIP(hipMalloc(&M->dzp[l], (size_t)Bp * M->lo.dims[l + 1] * 2));
        }
        MLP_HIP(hipMalloc(&M->bias_part, (size_t)(Bp / 16) * M->bias_cols() * 4));
        MLP_HIP(hipMalloc(&M->loss_part, (size_t)(Bp / 16) * 4));
        MLP_HIP(hipMalloc(&M->y, (size_t)Bp * M->out_features * 4));
        M->cap = Bp;
        return SAPX_OK;
    }
    MLP_HIP(hipMalloc(&M->xb, (size_t)Bp * M->lo.dims[0] * 2));
    MLP_HIP(hipMalloc(&M->xt, (size_t)Bp * M->lo.dims[0] * 2));
    for (int l = 1; l < L; ++l) {
        MLP_HIP(hipMalloc(&M->h[l], (size_t)Bp * M->lo.dims[l] * 2));
        MLP_HIP(hipMalloc(&M->ht[l], (size_t)Bp * M->lo.dims[l] * 2));
    }
    MLP_HIP(hipMalloc(&M->y, (size_t)Bp * M->lo.dims[L] * 4));
    for (int k = 0; k < 2; ++k) {
        MLP_HIP(hipMalloc(&M->dz[k], (size_t)Bp * mw * 2));
        MLP_HIP(hipMalloc(&M->dzt[k], (size_t)Bp * mw * 2));
    }
    M->cap = Bp;
    return SAPX_OK;
}

static hipError_t gemm(int epi, const GemmArgs& g, int M, int N, hipStream_t st) {
    const dim3 grid(N / 64, M / 64), block(64);
    switch (epi) {
        case EPI_F32: hipLaunchKernelGGL(gemm_nt_kernel<EPI_F32>, grid, block, 0, st, g); break;
        case EPI_RELU_BF16: hipLaunchKernelGGL(gemm_nt_kernel<EPI_RELU_BF16>, grid, block, 0, st, g); break;
        default: hipLaunchKernelGGL(gemm_nt_kernel<EPI_MASK_BF16>, grid, block, 0, st, g); break;
    }
    return hipGetLastError();
}

static void weight_tiles(const SapxMlp* M, WeightGradArgs* a) {
    a->lo = M->lo;
    a->tile0[0] = 0;
    for (int l = 0; l < M->lo.L; ++l) a->tile0[l + 1] = a->tile0[l] + (M->lo.dims[l] / 64) * (M->lo.dims[l + 1] / 64);
}

template <int MT, bool TRAIN>
static hipError_t launch_row_blocks(const RowBlockArgs& a, size_t lds, hipStream_t st) {
    // idempotent, and cheap next to the launch: no flag that threads would share
    const hipError_t e = hipFuncSetAttribute((const void*)row_block_kernel<MT, TRAIN>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((row_block_kernel<MT, TRAIN>), dim3((a.Bp + 16 * MT - 1) / (16 * MT)), dim3(kWaves * 64), lds, st, a);
    return hipGetLastError();
}

static RowBlockArgs row_block_args(const SapxMlp* M, const float* x, int batch) {
    RowBlockArgs a{};
    a.lo = M->lo;
    a.params = M->params;
    a.wb = M->wb;
    a.wt = M->wt;
    a.norm = M->norm;
    a.x = x;
    a.B = batch;
    a.F = M->in_features;
    a.O = M->out_features;
    a.bias_cols = M->bias_cols();
    return a;
}

static hipError_t refresh_bf16(SapxMlp* M, hipStream_t st, int update, float lr, float b1, float b2, float eps) {
    float c1 = 1.0f, c2 = 1.0f;
    if (update) {
        c1 = 1.0f - powf(b1, (float)M->adam_t);
        c2 = 1.0f - powf(b2, (float)M->adam_t);
    }
    const int threads = 256;
    if (M->row_blocks) {
        WeightGradArgs tiles{};
        weight_tiles(M, &tiles);
        const int blocks = tiles.tile0[M->lo.L] + (M->bias_cols() + threads - 1) / threads;
        hipLaunchKernelGGL(adam_packed_kernel, dim3(blocks), dim3(threads), 0, st, M->params, M->grads, M->m, M->v, M->lo,
                           tiles, lr, b1, b2, eps, c1, c2, M->wb, M->wt, update);
        return hipGetLastError();
    }
    const unsigned blocks = (unsigned)((M->lo.total + threads - 1) / threads);
    hipLaunchKernelGGL(adam_kernel, dim3(blocks), dim3(threads), 0, st, M->params, M->grads, M->m, M->v, M->lo, lr, b1,
                       b2, eps, c1, c2, M->wb, M->wt, update);
    return hipGetLastError();
}

// forward pass of `batch` rows already normalised into M->xb / M->xt; output (normalised) in M->y
static int32_t forward_normalised(SapxMlp* M, int Bp, hipStream_t st) {
    const int L = M->lo.L;
    for (int l = 0; l < L; ++l) {
        GemmArgs g{};
        g.A = l == 0 ? M->xb : M->h[l];
        g.lda = M->lo.dims[l];
        g.B = M->wb + M->lo.wb_off[l];
        g.ldb = M->lo.dims[l];
        g.K = M->lo.dims[l];
        g.bias = M->params + M->lo.w_off[l] + (long long)M->lo.dims[l] * M->lo.dims[l + 1];
        if (l < L - 1) {
            g.Cb = M->h[l + 1];
            g.Ct = M->ht[l + 1];
            g.ldc = M->lo.dims[l + 1];
            g.ldt = Bp;
            MLP_HIP(gemm(EPI_RELU_BF16, g, Bp, M->lo.dims[l + 1], st));
        } else {
            g.Cf = M->y;
            g.ldc = M->lo.dims[L];
            MLP_HIP(gemm(EPI_F32, g, Bp, M->lo.dims[L], st));
        }
    }
    return SAPX_OK;
}

static int32_t normalise(SapxMlp* M, const float* x, int batch, int Bp, hipStream_t st) {
    const int d0 = M->lo.dims[0];
    const size_t tot = (size_t)Bp * d0;
    hipLaunchKernelGGL(normalize_input_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, x, batch,
                       M->in_features, Bp, d0, M->norm, M->norm + M->in_features, M->xb, M->xt);
    MLP_HIP(hipGetLastError());
    return SAPX_OK;
}

extern "C" {

int32_t sapx_mlp_create(int32_t layers, const int32_t* dims, int32_t in_features, int32_t out_features,
                        SapxMlp** out) {
    if (!out || !dims || layers < 1 || layers > kMaxLayers) return mfail(SAPX_ERR_INVALID, "sapx_mlp_create: bad layer count");
    for (int l = 0; l <= layers; ++l)
        if (dims[l] <= 0 || dims[l] % 64 != 0) return mfail(SAPX_ERR_INVALID, "sapx_mlp_create: widths must be positive multiples of 64");
    if (in_features <= 0 || in_features > dims[0] || out_features <= 0 || out_features > dims[layers])
        return mfail(SAPX_ERR_INVALID, "sapx_mlp_create: real widths exceed the padded widths");
    SapxMlp* M = new SapxMlp();
    M->lo.L = layers;
    long long off = 0, woff = 0;
    for (int l = 0; l <= layers; ++l) M->lo.dims[l] = dims[l];
    for (int l = 0; l < layers; ++l) {
        M->lo.w_off[l] = off;
        M->lo.wb_off[l] = woff;
        off += (long long)dims[l] * dims[l + 1] + dims[l + 1];
        woff += (long long)dims[l] * dims[l + 1];
    }
    M->lo.total = off;
    M->wb_total = woff;
    M->in_features = in_features;
    M->out_features = out_features;
    M->row_blocks = net_fits(M);
    const size_t pb = (size_t)off * 4;
    if (hipMalloc(&M->params, pb) != hipSuccess || hipMalloc(&M->grads, pb) != hipSuccess ||
        hipMalloc(&M->m, pb) != hipSuccess || hipMalloc(&M->v, pb) != hipSuccess ||
        hipMalloc(&M->wb, (size_t)woff * 2) != hipSuccess || hipMalloc(&M->wt, (size_t)woff * 2) != hipSuccess ||
        hipMalloc(&M->norm, (size_t)(2 * in_features + 2 * out_features) * 4) != hipSuccess ||
        hipMalloc(&M->loss, 4) != hipSuccess) {
        delete M;
        return mfail(SAPX_ERR_HIP, "sapx_mlp_create: hipMalloc failed");
    }
    (void)hipMemset(M->params, 0, pb);
    (void)hipMemset(M->grads, 0, pb);
    (void)hipMemset(M->m, 0, pb);
    (void)hipMemset(M->v, 0, pb);
    (void)hipMemset(M->wb, 0, (size_t)woff * 2);
    (void)hipMemset(M->wt, 0, (size_t)woff * 2);
    std::vector<float> nrm(2 * in_features + 2 * out_features, 0.0f);
    for (int f = 0; f < in_features; ++f) nrm[in_features + f] = 1.0f;
    for (int o = 0; o < out_features; ++o) nrm[2 * in_features + out_features + o] = 1.0f;
    (void)hipMemcpy(M->norm, nrm.data(), nrm.size() * 4, hipMemcpyHostToDevice);
    *out = M;
    return SAPX_OK;
}

void sapx_mlp_destroy(SapxMlp* mlp) { delete mlp; }

int64_t sapx_mlp_param_count(const SapxMlp* mlp) { return mlp ? (int64_t)mlp->lo.total : 0; }

int32_t sapx_mlp_write(SapxMlp* M, int32_t which, const float* host, int64_t count) {
    if (!M || !host) return mfail(SAPX_ERR_INVALID, "sapx_mlp_write: null argument");
    const int F = M->in_features, O = M->out_features;
    if (which == SAPX_MLP_PARAMS) {
        if (count != M->lo.total) return mfail(SAPX_ERR_INVALID, "sapx_mlp_write: parameter count mismatch");
        MLP_HIP(hipMemcpy(M->params, host, (size_t)count * 4, hipMemcpyHostToDevice));
        MLP_HIP(hipMemset(M->m, 0, (size_t)count * 4));
        MLP_HIP(hipMemset(M->v, 0, (size_t)count * 4));
        M->adam_t = 0;
        MLP_HIP(refresh_bf16(M, nullptr, 0, 0.0f, 0.0f, 0.0f, 0.0f));
        MLP_HIP(hipDeviceSynchronize());
        return SAPX_OK;
    }
    const int off[4] = {0, F, 2 * F, 2 * F + O};
    const int len[4] = {F, F, O, O};
    if (which < SAPX_MLP_X_MEAN || which > SAPX_MLP_Y_STD) return mfail(SAPX_ERR_INVALID, "sapx_mlp_write: bad buffer id");
    const int k = which - SAPX_MLP_X_MEAN;
    if (count != len[k]) return mfail(SAPX_ERR_INVALID, "sapx_mlp_write: normalisation length mismatch");
    MLP_HIP(hipMemcpy(M->norm + off[k], host, (size_t)count * 4, hipMemcpyHostToDevice));
    return SAPX_OK;
}

int32_t sapx_mlp_read(const SapxMlp* M, int32_t which, float* host, int64_t count) {
    if (!M || !host) return mfail(SAPX_ERR_INVALID, "sapx_mlp_read: null argument");
    const float* src = which == SAPX_MLP_PARAMS ? M->params : which == SAPX_MLP_GRADS ? M->grads : nullptr;
    if (!src) return mfail(SAPX_ERR_INVALID, "sapx_mlp_read: bad buffer id");
    if (count != M->lo.total) return mfail(SAPX_ERR_INVALID, "sapx_mlp_read: parameter count mismatch");
    MLP_HIP(hipDeviceSynchronize());
    MLP_HIP(hipMemcpy(host, src, (size_t)count * 4, hipMemcpyDeviceToHost));
    return SAPX_OK;
}

int32_t sapx_mlp_reserve(SapxMlp* M, int32_t batch) {
    if (!M || batch <= 0) return mfail(SAPX_ERR_INVALID, "sapx_mlp_reserve: bad batch");
    return reserve(M, batch);
}

int32_t sapx_mlp_forward(SapxMlp* M, const float* x, int32_t batch, float* y, void* stream) {
    if (!M || !x || !y || batch <= 0) return mfail(SAPX_ERR_INVALID, "sapx_mlp_forward: bad argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (M->row_blocks) {
        RowBlockArgs a = row_block_args(M, x, batch);
        a.Bp = (batch + 15) / 16 * 16;
        // an output that overlaps the input goes through the workspace: a block writes its rows of y while
        // others still read theirs of x
        const size_t out_bytes = (size_t)batch * M->out_features * 4;
        const uintptr_t xa = (uintptr_t)x, ya = (uintptr_t)y;
        const bool overlap = ya < xa + (size_t)batch * M->in_features * 4 && xa < ya + out_bytes;
        if (overlap) {
            const int32_t rc = reserve(M, batch);
            if (rc != SAPX_OK) return rc;
        }
        a.y = overlap ? M->y : y;
        // Blocks of 16 rows while that gives each of the 256 CUs at most one (4096 rows: 21 us; 20 us
        // at 16 rows, the time one CU takes to read the weights at about 37 bytes a cycle), else 32
        // rows, which read the weights half as often (8192 rows: 26 us against 30 us in blocks of
        // 16; 64 rows a block lose the second workgroup of a CU: 58 against 53 us at 16384).
        if (batch > 4096 && M->forward_lds(2) <= kMaxLds) MLP_HIP((launch_row_blocks<2, false>(a, M->forward_lds(2), st)));
        else MLP_HIP((launch_row_blocks<1, false>(a, M->forward_lds(1), st)));
        if (overlap) MLP_HIP(hipMemcpyAsync(y, M->y, out_bytes, hipMemcpyDeviceToDevice, st));
        return SAPX_OK;
    }
    const int32_t rc = reserve(M, batch);
    if (rc != SAPX_OK) return rc;
    const int Bp = (batch + 63) / 64 * 64;
    int32_t r = normalise(M, x, batch, Bp, st);
    if (r != SAPX_OK) return r;
    r = forward_normalised(M, Bp, st);
    if (r != SAPX_OK) return r;
    const int O = M->out_features, F = M->in_features;
    hipLaunchKernelGGL(unnormalize_output_kernel, dim3((batch * O + 255) / 256), dim3(256), 0, st, M->y, batch, O,
                       M->lo.dims[M->lo.L], M->norm + 2 * F, M->norm + 2 * F + O, y);
    MLP_HIP(hipGetLastError());
    return SAPX_OK;
}

int32_t sapx_mlp_gradients(SapxMlp* M, const float* x, const float* target, int32_t batch, float* loss, void* stream) {
    if (!M || !x || !target || batch <= 0) return mfail(SAPX_ERR_INVALID, "sapx_mlp_gradients: bad argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int32_t r = reserve(M, batch);
    if (r != SAPX_OK) return r;
    const int Bp = (batch + 63) / 64 * 64;
    const int L = M->lo.L, F = M->in_features, O = M->out_features;
    if (M->row_blocks) {
        RowBlockArgs a = row_block_args(M, x, batch);
        a.Bp = Bp;
        a.target = target;
        a.bias_part = M->bias_part;
        a.loss_part = M->loss_part;
        WeightGradArgs w{};
        weight_tiles(M, &w);
        for (int l = 0; l < L; ++l) {
            a.ht[l] = M->ht[l];
            a.dzt[l] = M->dzp[l];
            w.ht[l] = M->ht[l];
            w.dzt[l] = M->dzp[l];
        }
        // blocks of 32 rows beyond one 16-row block a CU (8192 rows: 90 us against 113 us for a gradient)
        const bool two = batch > 4096 && M->train_lds(2) <= kMaxLds;
        if (two) MLP_HIP((launch_row_blocks<2, true>(a, M->train_lds(2), st)));
        else MLP_HIP((launch_row_blocks<1, true>(a, M->train_lds(1), st)));
        w.Bp = Bp;
        w.grads = M->grads;
        w.bias_part = M->bias_part;
        w.loss_part = M->loss_part;
        w.blocks = Bp / (two ? 32 : 16);
        w.bias_cols = a.bias_cols;
        w.inv_count = 1.0f / ((float)batch * (float)O);
        w.loss = loss;
        hipLaunchKernelGGL(weight_grad_kernel, dim3((w.tile0[L] + 7) / 8 * 8 + a.bias_cols / 64 + 1), dim3(kWaves * 64), 0, st, w);
        MLP_HIP(hipGetLastError());
        return SAPX_OK;
    }
    r = normalise(M, x, batch, Bp, st);
    if (r != SAPX_OK) return r;
    r = forward_normalised(M, Bp, st);
    if (r != SAPX_OK) return r;
    // bias gradients and the loss accumulate atomically: clear them with a fill kernel
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((M->lo.total + 255) / 256)), dim3(256), 0, st, M->grads,
                       (size_t)M->lo.total, 0.0f);
    hipLaunchKernelGGL(fill_kernel, dim3(1), dim3(64), 0, st, M->loss, (size_t)1, 0.0f);
    MLP_HIP(hipGetLastError());
    const int dL = M->lo.dims[L];
    hipLaunchKernelGGL(loss_grad_kernel, dim3(Bp / 64), dim3(256), 0, st, M->y, target, batch, O, Bp, dL,
                       M->norm + 2 * F, M->norm + 2 * F + O, M->dz[0], M->dzt[0],
                       M->grads + M->lo.w_off[L - 1] + (long long)M->lo.dims[L - 1] * dL, M->loss);
    MLP_HIP(hipGetLastError());
    int cur = 0;
    for (int l = L - 1; l >= 0; --l) {
        const int din = M->lo.dims[l], dout = M->lo.dims[l + 1];
        // dW_l = dz_{l+1}^T h_l
        GemmArgs gw{};
        gw.A = M->dzt[cur];
        gw.lda = Bp;
        gw.B = l == 0 ? M->xt : M->ht[l];
        gw.ldb = Bp;
        gw.K = Bp;
        gw.Cf = M->grads + M->lo.w_off[l];
        gw.ldc = din;
        MLP_HIP(gemm(EPI_F32, gw, dout, din, st));
        if (l > 0) {
            // dz_l = (dz_{l+1} W_l) * [h_l > 0]; the bias gradient of layer l-1 is its column sum
            GemmArgs gx{};
            gx.A = M->dz[cur];
            gx.lda = dout;
            gx.B = M->wt + M->lo.wb_off[l];
            gx.ldb = dout;
            gx.K = dout;
            gx.Cb = M->dz[cur ^ 1];
            gx.Ct = M->dzt[cur ^ 1];
            gx.ldc = din;
            gx.ldt = Bp;
            gx.H = M->h[l];
            gx.ldh = din;
            gx.colsum = M->grads + M->lo.w_off[l - 1] + (long long)M->lo.dims[l - 1] * din;
            MLP_HIP(gemm(EPI_MASK_BF16, gx, Bp, din, st));
            cur ^= 1;
        }
    }
    if (loss) MLP_HIP(hipMemcpyAsync(loss, M->loss, 4, hipMemcpyDeviceToDevice, st));
    return SAPX_OK;
}

int32_t sapx_mlp_adam(SapxMlp* M, float lr, float beta1, float beta2, float eps, void* stream) {
    if (!M) return mfail(SAPX_ERR_INVALID, "sapx_mlp_adam: null model");
    M->adam_t += 1;
    MLP_HIP(refresh_bf16(M, reinterpret_cast<hipStream_t>(stream), 1, lr, beta1, beta2, eps));
    return SAPX_OK;
}

}  // extern "C"
