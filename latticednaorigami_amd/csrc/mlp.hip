// mlp.hip - training kernels of the learned proposal's network (ldo_mlp.h).
//
// One sample is a 7x7x7 one-hot box (13 channels per site) around a staple
// end domain's anchor plus the domain's identity; the network is
//   z1 = b1 + sum over sites of W1[site*13 + channel] + emb[id] . W1e
//   h1 = relu(z1); z2 = h1 W2 + b2; h2 = relu(z2); z3 = h2 W3 + b3;
//   h3 = relu(z3); z4 = h3 W4 + b4 (36 logits), masked softmax.
//
// A batch is some hundred samples: the products with W2, W3 and W4 are 10 to
// 30 MFLOP each and far below what fills the card, so what counts is the
// number of launches and of dependent round trips.  A training step is four
// launches:
//   mlp_layer1    the first layer (a gather: its input is one-hot)
//   mlp_tile      16 samples per workgroup through every other layer, the
//                 softmax and back to dz1, activations in LDS
//   mlp_grads     all parameter gradients, one kind of block for each
//   mlp_adam      the update, and the bf16 copies of W2, W3, W4 that
//                 mlp_tile multiplies by, laid out as MFMA operands
// Products run on gfx950's 16x16x32 bf16 MFMA with FP32 accumulation.
// Measured on an MI355X against a GEMM, bias pass or reduction per launch (27
// launches and four pageable copies a step): 16 steps of batch 256 11.1 ->
// 2.3 ms, scoring 1000 samples 285 -> 87 us.  At batch 128 the kernels take
// 14.6 (layer1), 17.9 (tile), 26.0 (grads) and 9.4 us (adam), 72 us a step
// where the launches of one thing each took 440.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/ldo.h"
#include "../../include/ldo_mlp.h"
#include "plan.h"

namespace {

constexpr int H = LDO_MLP_HIDDEN;
constexpr int NO = LDO_MLP_OUT;
constexpr int NS = LDO_MLP_SITES;
constexpr int NE = LDO_MLP_EMBED;

typedef float v4f __attribute__((ext_vector_type(4)));

// float -> bf16 bits, round to nearest even (finite inputs)
__device__ inline short to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// v_mfma_f32_16x16x32_bf16 operands: A(i, k) in lane i + 16*(k/8), element
// k%8; B(k, j) in lane j + 16*(k/8), element k%8; D(i, j) in lane j + 16*(i/4),
// element i%4.  (Only the row and column mappings matter: A and B share the k
// mapping, so any order of k inside the instruction gives the same products.)
// A packed matrix holds B's elements in that order, 512 per (16 columns, 32
// rows): a lane's operand is one 16-byte load, a wavefront's 1 KB in a row.
__device__ inline int packed_at(int k, int n, int k_steps) {
    int lane = (n & 15) + 16 * ((k & 31) >> 3);
    return (((n >> 4) * k_steps + (k >> 5)) * 64 + lane) * 8 + (k & 7);
}
// element offsets of the packed matrices (rows x columns, padded to 32 x 16)
constexpr int NP = 48;                   // outputs padded to whole tiles
constexpr int KP = 64;                   // and to whole k steps
constexpr int PK_W2 = 0;                 // W2  [H][H]
constexpr int PK_W2T = PK_W2 + H * H;    // W2' [H][H]
constexpr int PK_W3 = PK_W2T + H * H;
constexpr int PK_W3T = PK_W3 + H * H;
constexpr int PK_W4 = PK_W3T + H * H;    // W4  [H][NP]
constexpr int PK_W4T = PK_W4 + H * NP;   // W4' [KP][H]
constexpr int PK_TOTAL = PK_W4T + KP * H;

// writes parameter i of the flat vector to the packed copies it is in
__device__ inline void pack_param(const ldo_mlp_layout& L, int64_t i, float v, short* pk) {
    if (i < L.w2) {
        return;
    }
    short q = to_bf16(v);
    if (i >= L.w4) {
        int o = (int)(i - L.w4);
        if (o < H * NO) {
            int k = o / NO, n = o % NO;
            pk[PK_W4 + packed_at(k, n, H / 32)] = q;
            pk[PK_W4T + packed_at(n, k, KP / 32)] = q;
        }
        return;
    }
    int o = (int)(i - (i >= L.w3 ? L.w3 : L.w2));
    if (o < H * H) {
        int base = i >= L.w3 ? PK_W3 : PK_W2;
        int k = o / H, n = o % H;
        pk[base + packed_at(k, n, H / 32)] = q;
        pk[base + H * H + packed_at(n, k, H / 32)] = q;
    }
}

__global__ void mlp_pack(const float* p, ldo_mlp_layout L, short* pk) {
    int64_t i = L.w2 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < L.total) {
        pack_param(L, i, p[i], pk);
    }
}

// h1 of one sample per workgroup, one hidden unit per lane: 343 rows of 1 KB
// from L2, added in site order.  Two sets of 24 loads alternate, so that a set
// is on its way while the other is added.  Also clears the embedding gradients.
constexpr int L1_SET = 24;
__global__ void __launch_bounds__(H)
    mlp_layer1(const float* P, ldo_mlp_layout L, const uint8_t* ch, const int32_t* id, int batch,
               unsigned short* h1, float* g_emb, int n_emb) {
    constexpr int PAD = (NS + 2 * L1_SET - 1) / (2 * L1_SET) * (2 * L1_SET);
    __shared__ int row[PAD];
    int b = blockIdx.x, j = threadIdx.x;
    for (int i = blockIdx.x * H + j; i < n_emb; i += gridDim.x * H) {
        g_emb[i] = 0.f;
    }
    for (int s = j; s < PAD; s += H) {
        row[s] = s < NS ? s * LDO_MLP_CHANNELS + ch[(size_t)b * NS + s] : 0;
    }
    __syncthreads();
    const float* W = P + L.w1 + j;
    const float* e = P + L.emb + (int64_t)id[b] * NE;
    float s = P[L.b1 + j];
    float w0[L1_SET], w1[L1_SET];
#pragma unroll
    for (int q = 0; q < L1_SET; q++) {
        w0[q] = W[(int64_t)row[q] * H];
    }
#pragma unroll 1
    for (int site = 0; site < PAD; site += 2 * L1_SET) {
#pragma unroll
        for (int q = 0; q < L1_SET; q++) {
            w1[q] = W[(int64_t)row[site + L1_SET + q] * H];
        }
#pragma unroll
        for (int q = 0; q < L1_SET; q++) {
            s += site + q < NS ? w0[q] : 0.f;
        }
        int nx = site + 2 * L1_SET < PAD ? site + 2 * L1_SET : 0;
#pragma unroll
        for (int q = 0; q < L1_SET; q++) {
            w0[q] = W[(int64_t)row[nx + q] * H];
        }
#pragma unroll
        for (int q = 0; q < L1_SET; q++) {
            s += site + L1_SET + q < NS ? w1[q] : 0.f;
        }
    }
    for (int k = 0; k < NE; k++) {
        s = fmaf(e[k], P[L.w1e + k * H + j], s);
    }
    h1[(size_t)b * H + j] = (unsigned short)to_bf16(fmaxf(s, 0.f));
}

// One tile of 16 samples through layers 2 to 4 and, when training, back to
// dz1.  Eight wavefronts: each owns two 16-column tiles of a hidden layer.
// Activations stay in LDS as bf16 (rows padded by 16 bytes against bank
// conflicts), where the products read them; gradients leave as FP32 (dz1 to
// dz4) and, with the activations, transposed as bf16 operands of the weight
// gradients ([unit][sample], samples padded to 32).
constexpr int TB = 16;         // samples per tile
constexpr int TW = 8;          // wavefronts
constexpr int TR = H + 8;      // LDS row of a hidden layer
constexpr int TO = KP + 8;     // LDS row of dz4
struct TileArgs {
    const float* P;
    ldo_mlp_layout L;
    const short* pk;
    const unsigned short* h1;
    const uint8_t* legal;
    const int32_t* tgt;
    int batch, cols; // cols: padded samples of the transposed operands
    float *dz1, *dz2, *dz3, *dz4, *logp;
    double* loss;
    unsigned short *h1t, *h2t, *h3t, *dz2t, *dz3t, *dz4t;
};

// acc = rows of `act` (LDS, 16 x 32 k_steps) times the packed tile at `w`
__device__ inline v4f tile_product(const unsigned short* act, int stride, const short* w,
                                   int k_steps, int lane) {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const unsigned short* a = act + (lane & 15) * stride + (lane >> 4) * 8;
    const short* b = w + lane * 8;
#pragma unroll 8
    for (int k = 0; k < k_steps; k++) {
        v8bf x, y;
        __builtin_memcpy(&x, a + 32 * k, sizeof x);
        __builtin_memcpy(&y, b + 512 * k, sizeof y);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
    }
    return acc;
}

// the tile's 16 samples of unit `c` to column block s0 of the transposed copy
__device__ inline void store_transposed(const unsigned short* act, int stride, int units, int s0,
                                        int cols, unsigned short* out) {
    for (int u = threadIdx.x; u < 2 * units; u += 64 * TW) {
        int c = u >> 1, half = (u & 1) * 8;
        unsigned short v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = act[(half + i) * stride + c];
        }
        __builtin_memcpy(out + (size_t)c * cols + s0 + half, v, sizeof v);
    }
}

template <bool TRAIN>
__global__ void __launch_bounds__(64 * TW) mlp_tile(TileArgs g) {
    __shared__ __attribute__((aligned(16))) unsigned short act[3][TB * TR]; // h1, h2, h3
    __shared__ __attribute__((aligned(16))) unsigned short grad[2][TB * TR];
    __shared__ __attribute__((aligned(16))) unsigned short out[TB * TO];
    __shared__ float z4[TB][NP];
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int s0 = blockIdx.x * TB;
    int col = lane & 15, row = (lane >> 4) * 4;
    for (int i = tid; i < TB * H / 8; i += 64 * TW) {
        int r = i / (H / 8), c = i % (H / 8) * 8;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (s0 + r < g.batch) {
            __builtin_memcpy(&v, __builtin_assume_aligned(g.h1 + (size_t)(s0 + r) * H + c, 16),
                             sizeof v);
        }
        __builtin_memcpy(__builtin_assume_aligned(&act[0][r * TR + c], 16), &v, sizeof v);
    }
    __syncthreads();
    for (int layer = 0; layer < 2; layer++) {
        const short* w = g.pk + (layer == 0 ? PK_W2 : PK_W3);
        const float* bias = g.P + (layer == 0 ? g.L.b2 : g.L.b3);
        for (int q = 0; q < 2; q++) {
            int nt = wave + TW * q;
            v4f acc = tile_product(act[layer], TR, w + (size_t)nt * (H / 32) * 512, H / 32, lane);
            float bv = bias[nt * 16 + col];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float h = s0 + row + t < g.batch ? fmaxf(acc[t] + bv, 0.f) : 0.f;
                act[layer + 1][(row + t) * TR + nt * 16 + col] = (unsigned short)to_bf16(h);
            }
        }
        __syncthreads();
    }
    if (wave < NP / 16) {
        v4f acc = tile_product(act[2], TR, g.pk + PK_W4 + (size_t)wave * (H / 32) * 512, H / 32,
                               lane);
        int n = wave * 16 + col;
        float bv = n < NO ? g.P[g.L.b4 + n] : 0.f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            z4[row + t][n] = acc[t] + bv;
        }
    }
    __syncthreads();
    // masked log-softmax, loss and d(mean loss)/dz4: a wavefront per sample
    for (int r = wave; r < TB; r += TW) {
        int b = s0 + r;
        bool real = b < g.batch;
        bool lg = real && lane < NO && g.legal[(size_t)b * NO + lane] != 0;
        float z = lane < NO ? z4[r][lane] : 0.f;
        float m = lg ? z : -INFINITY;
        for (int w = 32; w > 0; w /= 2) {
            m = fmaxf(m, __shfl_xor(m, w));
        }
        double sum = lg ? exp((double)(z - m)) : 0.0;
        for (int w = 32; w > 0; w /= 2) {
            sum += __shfl_xor(sum, w);
        }
        double lse = (double)m + log(sum);
        if (!TRAIN) {
            if (real && lane < NO) {
                g.logp[(size_t)b * NO + lane] = lg ? (float)((double)z - lse) : -INFINITY;
            }
            continue;
        }
        float d = 0.f;
        if (real) {
            int t = g.tgt[b];
            double p = lg ? exp((double)z - lse) : 0.0;
            d = lane < NO ? (float)((p - (lane == t ? 1.0 : 0.0)) / g.batch) : 0.f;
            if (lane == t) {
                g.loss[b] = lse - (double)z;
            }
            if (lane < NO) {
                g.dz4[(size_t)b * NO + lane] = d;
            }
        }
        out[r * TO + lane] = (unsigned short)to_bf16(d);
    }
    if (!TRAIN) {
        return;
    }
    __syncthreads();
    store_transposed(act[0], TR, H, s0, g.cols, g.h1t);
    store_transposed(act[1], TR, H, s0, g.cols, g.h2t);
    store_transposed(act[2], TR, H, s0, g.cols, g.h3t);
    store_transposed(out, TO, NP, s0, g.cols, g.dz4t);
    for (int layer = 2; layer >= 0; layer--) {
        const unsigned short* d = layer == 2 ? out : grad[layer & 1];
        int stride = layer == 2 ? TO : TR, ks = layer == 2 ? KP / 32 : H / 32;
        const short* w = g.pk + (layer == 2 ? PK_W4T : (layer == 1 ? PK_W3T : PK_W2T));
        float* dz = layer == 2 ? g.dz3 : (layer == 1 ? g.dz2 : g.dz1);
        unsigned short* dn = grad[(layer + 1) & 1];
        for (int q = 0; q < 2; q++) {
            int nt = wave + TW * q;
            v4f acc = tile_product(d, stride, w + (size_t)nt * ks * 512, ks, lane);
            int n = nt * 16 + col;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float v = (short)act[layer][(row + t) * TR + n] > 0 ? acc[t] : 0.f;
                if (s0 + row + t < g.batch) {
                    dz[(size_t)(s0 + row + t) * H + n] = v;
                }
                else {
                    v = 0.f;
                }
                dn[(row + t) * TR + n] = (unsigned short)to_bf16(v);
            }
        }
        __syncthreads();
        if (layer > 0) {
            store_transposed(dn, TR, H, s0, g.cols, layer == 2 ? g.dz3t : g.dz2t);
        }
    }
}

// Every parameter gradient, in blocks of 256 lanes of one kind each:
//   W1    one site per block: a sample adds its dz1 row to the row of its
//         channel there, 13 sums in registers picked by a scalar branch.  No
//         atomics and no clearing: the 22 M atomic adds of a batch of 256 took
//         most of the step.
//   W1e   one embedding dimension per block
//   bias  one layer per block
//   emb   one sample per wavefront
//   W2-W4 one 16 x 16 tile per wavefront, K = samples
struct GradArgs {
    const float* P;
    ldo_mlp_layout L;
    const uint8_t* ch;
    const int32_t* id;
    int batch, cols;
    const float *dz1, *dz2, *dz3, *dz4;
    const unsigned short *h1t, *h2t, *h3t, *dz2t, *dz3t, *dz4t;
    float* G;
};
constexpr int GB_W1 = NS, GB_W1E = NE, GB_BIAS = 4;
constexpr int GB_MM = (H / 16) * (H / 16) / 4;        // blocks of a hidden matrix
constexpr int GB_M4 = (H / 16) * (NP / 16) / 4;
inline int grad_blocks(int batch) {
    return GB_W1 + GB_W1E + GB_BIAS + 2 * GB_MM + GB_M4 + (batch + 3) / 4;
}

__device__ inline void grad_w1(const GradArgs& g, int site, int j) {
    __shared__ uint8_t chs[1024];
    float acc[LDO_MLP_CHANNELS];
#pragma unroll
    for (int c = 0; c < LDO_MLP_CHANNELS; c++) {
        acc[c] = 0.f;
    }
    for (int b0 = 0; b0 < g.batch; b0 += 1024) {
        int nb = g.batch - b0 < 1024 ? g.batch - b0 : 1024;
        __syncthreads();
        for (int b = j; b < nb; b += 256) {
            chs[b] = g.ch[(size_t)(b0 + b) * NS + site];
        }
        __syncthreads();
        for (int b = 0; b < nb; b += 8) {
            float d[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                d[q] = b + q < nb ? g.dz1[(size_t)(b0 + b + q) * H + j] : 0.f;
            }
#pragma unroll
            for (int q = 0; q < 8; q++) {
                int c = __builtin_amdgcn_readfirstlane((int)chs[(b + q) & 1023]);
                c = b + q < nb ? c : 0;
#pragma unroll
                for (int k = 0; k < LDO_MLP_CHANNELS; k++) {
                    if (c == k) {
                        acc[k] += d[q];
                    }
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < LDO_MLP_CHANNELS; c++) {
        g.G[g.L.w1 + (int64_t)(site * LDO_MLP_CHANNELS + c) * H + j] = acc[c];
    }
}

// rows 16 i0.. of A' (transposed activations) times dz' rows 16 j0..
__device__ inline void grad_tile(const unsigned short* at, const unsigned short* dt, int cols,
                                 int i0, int j0, int n, float* out, int lane) {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const unsigned short* a = at + (size_t)(i0 * 16 + (lane & 15)) * cols + (lane >> 4) * 8;
    const unsigned short* d = dt + (size_t)(j0 * 16 + (lane & 15)) * cols + (lane >> 4) * 8;
#pragma unroll 4
    for (int k = 0; k < cols; k += 32) {
        v8bf x, y;
        __builtin_memcpy(&x, a + k, sizeof x);
        __builtin_memcpy(&y, d + k, sizeof y);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
    }
    int j = j0 * 16 + (lane & 15);
    if (j < n) {
        for (int t = 0; t < 4; t++) {
            out[(size_t)(i0 * 16 + (lane >> 4) * 4 + t) * n + j] = acc[t];
        }
    }
}

__global__ void __launch_bounds__(256) mlp_grads(GradArgs g) {
    int b = blockIdx.x, j = threadIdx.x, lane = j & 63, wave = j >> 6;
    if (b < GB_W1) {
        grad_w1(g, b, j);
        return;
    }
    b -= GB_W1;
    if (b < GB_W1E) {
        float s = 0.f;
#pragma unroll 8
        for (int r = 0; r < g.batch; r++) {
            s = fmaf(g.P[g.L.emb + (int64_t)g.id[r] * NE + b], g.dz1[(size_t)r * H + j], s);
        }
        g.G[g.L.w1e + b * H + j] = s;
        return;
    }
    b -= GB_W1E;
    if (b < GB_BIAS) {
        const float* dz = b == 0 ? g.dz1 : (b == 1 ? g.dz2 : (b == 2 ? g.dz3 : g.dz4));
        int64_t o = b == 0 ? g.L.b1 : (b == 1 ? g.L.b2 : (b == 2 ? g.L.b3 : g.L.b4));
        int n = b == 3 ? NO : H;
        if (j < n) {
            // in sample order, sixteen loads in flight
            float s = 0.f;
#pragma unroll 16
            for (int r = 0; r < g.batch; r++) {
                s += dz[(size_t)r * n + j];
            }
            g.G[o + j] = s;
        }
        return;
    }
    b -= GB_BIAS;
    if (b < 2 * GB_MM) {
        bool third = b >= GB_MM;
        int t = (third ? b - GB_MM : b) * 4 + wave;
        grad_tile(third ? g.h2t : g.h1t, third ? g.dz3t : g.dz2t, g.cols, t / (H / 16),
                  t % (H / 16), H, g.G + (third ? g.L.w3 : g.L.w2), lane);
        return;
    }
    b -= 2 * GB_MM;
    if (b < GB_M4) {
        int t = b * 4 + wave;
        grad_tile(g.h3t, g.dz4t, g.cols, t / (NP / 16), t % (NP / 16), NO, g.G + g.L.w4, lane);
        return;
    }
    b -= GB_M4;
    int r = b * 4 + wave;
    if (r >= g.batch) {
        return;
    }
    // the sample's share of its identity's embedding gradient: lane l holds
    // units l, l + 64, ... of all 16 sums
    float s[NE];
#pragma unroll
    for (int k = 0; k < NE; k++) {
        s[k] = 0.f;
    }
    for (int c = lane; c < H; c += 64) {
        float d = g.dz1[(size_t)r * H + c];
#pragma unroll
        for (int k = 0; k < NE; k++) {
            s[k] = fmaf(g.P[g.L.w1e + k * H + c], d, s[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < NE; k++) {
        for (int w = 32; w > 0; w /= 2) {
            s[k] += __shfl_xor(s[k], w);
        }
    }
    if (lane == 0) {
        for (int k = 0; k < NE; k++) {
            atomicAdd(&g.G[g.L.emb + (int64_t)g.id[r] * NE + k], s[k]);
        }
    }
}

__global__ void mlp_fill(float* x, int64_t n, float v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        x[i] = v;
    }
}

__global__ void mlp_adam(float* p, const float* g, float* m, float* v, ldo_mlp_layout L, short* pk,
                         float lr, float b1, float b2, float eps, float c1, float c2) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= L.total) {
        return;
    }
    float gi = g[i];
    float mi = b1 * m[i] + (1.f - b1) * gi;
    float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    pack_param(L, i, pi, pk);
}

struct MlpError {
    int code;
    std::string msg;
};

void hcheck(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        throw MlpError {LDO_E_HIP, std::string(what) + ": " + hipGetErrorString(e)};
    }
}

// Host memory that transfers go through: pinned, or ordinary memory (which the
// runtime stages itself) where none can be had.
struct HostBuf {
    void* mem = nullptr;
    bool pinned = false;
    void alloc(size_t bytes) {
        pinned = hipHostMalloc(&mem, bytes, hipHostMallocDefault) == hipSuccess;
        if (!pinned) {
            (void)hipGetLastError();
            mem = std::malloc(bytes);
            if (mem == nullptr) {
                throw MlpError {LDO_E_HIP, "host memory for a batch"};
            }
        }
    }
    ~HostBuf() {
        if (pinned) {
            (void)hipHostFree(mem);
        }
        else {
            std::free(mem);
        }
    }
};

struct MlpCtx {
    int n_ident = 0;
    int cap = 0;
    ldo_mlp_layout L {};
    int64_t adam_t = 0;
    float* d_p = nullptr;
    float* d_g = nullptr;
    float* d_m = nullptr;
    float* d_v = nullptr;
    // one batch of samples as one transfer: channels | ident | legal | target,
    // each part at a multiple of 16 bytes (upload_batch), and the same on the
    // host
    uint8_t* d_in = nullptr;
    HostBuf h_in;
    size_t in_bytes = 0;
    uint8_t* d_ch = nullptr;
    int32_t* d_id = nullptr;
    uint8_t* d_legal = nullptr;
    int32_t* d_tgt = nullptr;
    short* d_pk = nullptr; // packed bf16 copies of W2, W3, W4
    unsigned short* h1 = nullptr;
    unsigned short* tr = nullptr; // transposed operands of the weight gradients
    float *dz1 = nullptr, *dz2 = nullptr, *dz3 = nullptr, *dz4 = nullptr, *logp = nullptr;
    double* d_loss = nullptr;
    HostBuf h_out; // losses or log-probabilities
    hipStream_t stream = nullptr;
    std::string err;
};

std::string g_mlp_create_error;

// Runs f; after an error nothing of the call stays on its way to or from the
// caller's memory and the batch's.
template <class F>
int mguarded(MlpCtx* c, F f) {
    std::string& err = c ? c->err : g_mlp_create_error;
    int code = LDO_E_HIP;
    try {
        f();
        err.clear();
        return LDO_OK;
    } catch (MlpError& e) {
        err = e.msg;
        code = e.code;
    } catch (std::exception& e) {
        err = e.what();
    }
    if (c && c->stream) {
        (void)hipStreamSynchronize(c->stream);
    }
    return code;
}

template <class T>
void dalloc(T*& p, size_t n, const char* what) {
    hcheck(hipMalloc(&p, std::max<size_t>(1, n) * sizeof(T)), what);
}

void free_mlp(MlpCtx* c) {
    if (c->stream) {
        (void)hipStreamSynchronize(c->stream);
    }
    void* ptrs[] = {c->d_p, c->d_g, c->d_m, c->d_v, c->d_in, c->d_pk, c->h1, c->tr,
                    c->dz1, c->dz2, c->dz3, c->dz4, c->logp, c->d_loss};
    for (void* p: ptrs) {
        if (p) {
            (void)hipFree(p);
        }
    }
    if (c->stream) {
        (void)hipStreamDestroy(c->stream);
    }
    delete c;
}

void fill(MlpCtx& c, float* x, int64_t n, float v) {
    hipLaunchKernelGGL(mlp_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream, x, n,
                       v);
}

// the packed copies after a change of the parameters from outside
void pack(MlpCtx& c) {
    int64_t n = c.L.total - c.L.w2;
    hipLaunchKernelGGL(mlp_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream, c.d_p,
                       c.L, c.d_pk);
}

size_t part_bytes(size_t n) {
    return (n + 15) / 16 * 16;
}

// validates a batch and copies it to the device
void upload_batch(MlpCtx& c, int batch, const uint8_t* ch, const int32_t* id, const uint8_t* legal,
                  const int32_t* tgt) {
    if (batch < 1 || batch > c.cap || !ch || !id || !legal) {
        throw MlpError {LDO_E_ARG, "batch must be 1..max_batch with channels, ident and legal"};
    }
    uint8_t top = 0; // one pass without a branch, which the compiler vectorises
    for (int64_t i = 0; i < (int64_t)batch * NS; i++) {
        top = ch[i] > top ? ch[i] : top;
    }
    if (top >= LDO_MLP_CHANNELS) {
        throw MlpError {LDO_E_ARG, "channel out of range"};
    }
    for (int b = 0; b < batch; b++) {
        if (id[b] < 0 || id[b] >= c.n_ident) {
            throw MlpError {LDO_E_ARG, "identity index out of range"};
        }
        int n_legal = 0;
        for (int k = 0; k < NO; k++) {
            n_legal += legal[b * NO + k] != 0;
        }
        if (n_legal == 0) {
            throw MlpError {LDO_E_ARG, "a sample has no legal output"};
        }
        if (tgt && (tgt[b] < 0 || tgt[b] >= NO || !legal[b * NO + tgt[b]])) {
            throw MlpError {LDO_E_ARG, "target is not a legal output"};
        }
    }
    // every call that reads these buffers ends with its stream idle, after an
    // error too (mguarded), so they are free here
    size_t o_id = part_bytes((size_t)batch * NS), o_lg = o_id + part_bytes((size_t)batch * 4),
           o_tg = o_lg + part_bytes((size_t)batch * NO), n = o_tg + (size_t)batch * 4;
    uint8_t* h = (uint8_t*)c.h_in.mem;
    std::memcpy(h, ch, (size_t)batch * NS);
    std::memcpy(h + o_id, id, (size_t)batch * 4);
    std::memcpy(h + o_lg, legal, (size_t)batch * NO);
    if (tgt) {
        std::memcpy(h + o_tg, tgt, (size_t)batch * 4);
    }
    c.d_ch = c.d_in;
    c.d_id = (int32_t*)(c.d_in + o_id);
    c.d_legal = c.d_in + o_lg;
    c.d_tgt = (int32_t*)(c.d_in + o_tg);
    hcheck(hipMemcpyAsync(c.d_in, h, n, hipMemcpyHostToDevice, c.stream), "copy batch");
}

// the transposed operands of a batch: h1, h2, h3, dz2, dz3 ([H][cols]), dz4 ([NP][cols])
int padded(int batch) {
    return (batch + 31) / 32 * 32;
}

void network(MlpCtx& c, int batch, bool train) {
    int cols = padded(batch);
    size_t hc = (size_t)H * cols;
    hipLaunchKernelGGL(mlp_layer1, dim3(batch), dim3(H), 0, c.stream, c.d_p, c.L,
                       c.d_ch, c.d_id, batch, c.h1, c.d_g + c.L.emb, train ? c.n_ident * NE : 0);
    TileArgs t {c.d_p, c.L, c.d_pk, c.h1, c.d_legal, c.d_tgt, batch, cols, c.dz1, c.dz2, c.dz3,
                c.dz4, c.logp, c.d_loss, c.tr, c.tr + hc, c.tr + 2 * hc, c.tr + 3 * hc,
                c.tr + 4 * hc, c.tr + 5 * hc};
    if (!train) {
        hipLaunchKernelGGL(mlp_tile<false>, dim3((batch + TB - 1) / TB), dim3(64 * TW), 0, c.stream,
                           t);
        return;
    }
    // both tiles of every 32 columns, so that the padding is written
    hipLaunchKernelGGL(mlp_tile<true>, dim3(cols / TB), dim3(64 * TW), 0, c.stream, t);
    GradArgs g {c.d_p, c.L, c.d_ch, c.d_id, batch, cols, c.dz1, c.dz2, c.dz3, c.dz4, t.h1t, t.h2t,
                t.h3t, t.dz2t, t.dz3t, t.dz4t, c.d_g};
    hipLaunchKernelGGL(mlp_grads, dim3(grad_blocks(batch)), dim3(256), 0, c.stream, g);
}

} // namespace

extern "C" {

int ldo_mlp_layout_of(int32_t n_ident, ldo_mlp_layout* out) {
    if (n_ident < 1 || !out) {
        return LDO_E_ARG;
    }
    ldo::mlp_layout(n_ident, *out);
    return LDO_OK;
}

int ldo_mlp_create(int32_t n_ident, int32_t max_batch, const float* params, uint64_t seed,
                   void** out) {
    MlpCtx* c = new MlpCtx;
    int rc = mguarded(nullptr, [&] {
        if (n_ident < 1 || max_batch < 1 || max_batch > 65536 || !out) {
            throw MlpError {LDO_E_ARG, "n_ident >= 1, 1 <= max_batch <= 65536 and out required"};
        }
        c->n_ident = n_ident;
        c->cap = max_batch;
        ldo::mlp_layout(n_ident, c->L);
        hcheck(hipStreamCreate(&c->stream), "stream");
        int64_t n = c->L.total;
        dalloc(c->d_p, n, "params");
        dalloc(c->d_g, n, "grads");
        dalloc(c->d_m, n, "adam m");
        dalloc(c->d_v, n, "adam v");
        size_t cols = padded(max_batch), bh = cols * H, bo = (size_t)max_batch * NO;
        c->in_bytes = part_bytes((size_t)max_batch * NS) + 2 * part_bytes((size_t)max_batch * 4) +
                      part_bytes(bo);
        dalloc(c->d_in, c->in_bytes, "batch");
        c->h_in.alloc(c->in_bytes);
        c->h_out.alloc(std::max(bo * sizeof(float), max_batch * sizeof(double)));
        dalloc(c->d_pk, PK_TOTAL, "packed weights");
        dalloc(c->h1, bh, "activations");
        dalloc(c->tr, (5 * H + NP) * cols, "transposed operands");
        for (float** p: {&c->dz1, &c->dz2, &c->dz3}) {
            dalloc(*p, bh, "gradients");
        }
        dalloc(c->dz4, bo, "logit grads");
        dalloc(c->logp, bo, "log-probs");
        dalloc(c->d_loss, max_batch, "loss");
        std::vector<float> h(n, 0.f);
        if (params) {
            std::memcpy(h.data(), params, n * sizeof(float));
        }
        else {
            std::mt19937_64 g(seed);
            auto uni = [&](int64_t off, int64_t cnt, float lim) {
                std::uniform_real_distribution<float> u(-lim, lim);
                for (int64_t i = 0; i < cnt; i++) {
                    h[off + i] = u(g);
                }
            };
            const ldo_mlp_layout& L = c->L;
            uni(L.w1, (int64_t)LDO_MLP_FEATURES * H, std::sqrt(6.f / NS));
            uni(L.emb, (int64_t)n_ident * NE, 1.f);
            uni(L.w1e, (int64_t)NE * H, std::sqrt(6.f / NE));
            uni(L.w2, (int64_t)H * H, std::sqrt(6.f / H));
            uni(L.w3, (int64_t)H * H, std::sqrt(6.f / H));
            uni(L.w4, (int64_t)H * NO, std::sqrt(6.f / H));
        }
        hcheck(hipMemcpy(c->d_p, h.data(), n * sizeof(float), hipMemcpyHostToDevice), "upload");
        fill(*c, c->d_m, n, 0.f);
        fill(*c, c->d_v, n, 0.f);
        fill(*c, c->d_g, n, 0.f);
        fill(*c, (float*)c->d_pk, PK_TOTAL / 2, 0.f); // the padding stays zero
        pack(*c);
        hcheck(hipGetLastError(), "init kernels");
        hcheck(hipStreamSynchronize(c->stream), "init sync");
    });
    if (rc != LDO_OK) {
        free_mlp(c);
        return rc;
    }
    *out = c;
    return LDO_OK;
}

void ldo_mlp_destroy(void* mlp) {
    if (mlp) {
        free_mlp(static_cast<MlpCtx*>(mlp));
    }
}

const char* ldo_mlp_last_error(void* mlp) {
    return mlp ? static_cast<MlpCtx*>(mlp)->err.c_str() : g_mlp_create_error.c_str();
}

int ldo_mlp_get_params(void* mlp, float* out) {
    MlpCtx* c = static_cast<MlpCtx*>(mlp);
    return mguarded(c, [&] {
        if (!out) {
            throw MlpError {LDO_E_ARG, "out required"};
        }
        hcheck(hipStreamSynchronize(c->stream), "sync");
        hcheck(hipMemcpy(out, c->d_p, c->L.total * sizeof(float), hipMemcpyDeviceToHost),
               "download params");
    });
}

int ldo_mlp_set_params(void* mlp, const float* in) {
    MlpCtx* c = static_cast<MlpCtx*>(mlp);
    return mguarded(c, [&] {
        if (!in) {
            throw MlpError {LDO_E_ARG, "in required"};
        }
        hcheck(hipStreamSynchronize(c->stream), "sync");
        hcheck(hipMemcpy(c->d_p, in, c->L.total * sizeof(float), hipMemcpyHostToDevice),
               "upload params");
        pack(*c);
        hcheck(hipGetLastError(), "pack");
        hcheck(hipStreamSynchronize(c->stream), "pack sync");
    });
}

int ldo_mlp_loss_grad(void* mlp, int32_t batch, const uint8_t* channels, const int32_t* ident,
                      const uint8_t* legal, const int32_t* target, double* loss, float* grads) {
    MlpCtx* c = static_cast<MlpCtx*>(mlp);
    return mguarded(c, [&] {
        if (!target || !loss) {
            throw MlpError {LDO_E_ARG, "target and loss required"};
        }
        upload_batch(*c, batch, channels, ident, legal, target);
        network(*c, batch, true);
        hcheck(hipGetLastError(), "loss/grad kernels");
        double* l = (double*)c->h_out.mem;
        hcheck(hipMemcpyAsync(l, c->d_loss, batch * sizeof(double), hipMemcpyDeviceToHost,
                              c->stream),
               "download loss");
        if (grads) {
            hcheck(hipMemcpyAsync(grads, c->d_g, c->L.total * sizeof(float),
                                  hipMemcpyDeviceToHost, c->stream),
                   "download grads");
        }
        hcheck(hipStreamSynchronize(c->stream), "loss/grad sync");
        double s = 0;
        for (int b = 0; b < batch; b++) {
            s += l[b];
        }
        *loss = s / batch;
    });
}

int ldo_mlp_adam_step(void* mlp, float lr, float beta1, float beta2, float eps) {
    MlpCtx* c = static_cast<MlpCtx*>(mlp);
    return mguarded(c, [&] {
        c->adam_t++;
        float c1 = 1.f - std::pow(beta1, (float)c->adam_t);
        float c2 = 1.f - std::pow(beta2, (float)c->adam_t);
        int64_t n = c->L.total;
        hipLaunchKernelGGL(mlp_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream,
                           c->d_p, c->d_g, c->d_m, c->d_v, c->L, c->d_pk, lr, beta1, beta2, eps, c1, c2);
        hcheck(hipGetLastError(), "adam");
        hcheck(hipStreamSynchronize(c->stream), "adam sync");
    });
}

int ldo_mlp_log_probs(void* mlp, int32_t batch, const uint8_t* channels, const int32_t* ident,
                      const uint8_t* legal, float* out) {
    MlpCtx* c = static_cast<MlpCtx*>(mlp);
    return mguarded(c, [&] {
        if (!out) {
            throw MlpError {LDO_E_ARG, "out required"};
        }
        upload_batch(*c, batch, channels, ident, legal, nullptr);
        network(*c, batch, false);
        hcheck(hipGetLastError(), "forward kernels");
        size_t bytes = (size_t)batch * NO * sizeof(float);
        hcheck(hipMemcpyAsync(c->h_out.mem, c->logp, bytes, hipMemcpyDeviceToHost, c->stream),
               "download log-probs");
        hcheck(hipStreamSynchronize(c->stream), "forward sync");
        std::memcpy(out, c->h_out.mem, bytes);
    });
}

} // extern "C"
