/*
 * The refinement-priority network on the matrix cores: a 4-layer MLP
 * (KP -> 64 -> 64 -> 64 -> 1, ReLU) with BF16 weights and activations and FP32
 * accumulation.  The three 64-wide layers run as v_mfma_f32_16x16x32_bf16 tiles out of
 * LDS; the 64 -> 1 output layer is a per-row dot product on the VALU (an MFMA tile
 * would be 1/16 used).
 *
 * MFMA 16x16x32 operand layout (wave64): lane l holds A[l%16][8(l/16) .. 8(l/16)+7]
 * and B[8(l/16) .. +7][l%16]; the accumulator's element i is D[4(l/16)+i][l%16].
 * Every operand here is therefore read as 8 consecutive BF16 of a row: activations
 * are stored sample-major, forward weights output-major (W^T) and the copies used to
 * back-propagate input-major (W).
 *
 * Rounding, which the CPU restatement of the network follows:
 *   weights and input features: BF16 (round to nearest even) of the FP32 values
 *   z = sum_k bf(x_k) bf(w_ko) in FP32, + bias (FP32)
 *   h = bf(relu(z)); ReLU derivative taken as [h > 0]
 *   output y = (s0 + s1) + (s2 + s3) + b3, s_q = sequential FP32 sum of 16 products
 *   back-propagated deltas: BF16 of the FP32 products / MFMA sums, masked by [h > 0]
 */
#ifndef VMX_REFINER_H
#define VMX_REFINER_H

#include <hip/hip_runtime.h>

#include "features.h"

namespace vmx {
namespace nn {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));

constexpr int WS = W + 8;  // LDS row stride of 64-wide activations (16-byte aligned rows)

__device__ inline bf16x8_t ld8(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(p));
}
__device__ inline bf16x8_t gather8(const uint16_t* p, int stride) {
    u16x8_t r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = p[i * stride];
    return __builtin_bit_cast(bf16x8_t, r);
}

/* One 16x16 tile: sum over K of A[16][K] (rows a, stride lda) times B[K][16] given as
   B^T rows (bt, stride ldb). */
__device__ inline f32x4_t mm_tile(const uint16_t* a, int lda, const uint16_t* bt, int ldb, int K, int lane) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    const int r = lane & 15, kq = (lane >> 4) * 8;
    for (int k0 = 0; k0 < K; k0 += 32)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ld8(a + r * lda + k0 + kq), ld8(bt + r * ldb + k0 + kq), acc, 0, 0,
                                                      0);
    return acc;
}

/* Forward weights in LDS. */
template <int KP>
struct alignas(16) NetW {  // size a multiple of 16 bytes (copied as 16-byte words)
    uint16_t w0t[W][KP + 8];
    uint16_t w1t[W][WS];
    uint16_t w2t[W][WS];
    float b0[W], b1[W], b2[W], w3[W];
    float b3, mu, sigma, pad;
};
/* NetW<KP> from w1t on, with the layout it has there: the part of the forward weights
   a kernel keeps in LDS when it reads the first layer from device memory. */
struct alignas(16) NetTail {
    uint16_t w1t[W][WS];
    uint16_t w2t[W][WS];
    float b0[W], b1[W], b2[W], w3[W];
    float b3, mu, sigma, pad;
};
template <int KP>
constexpr size_t net_tail_offset() {
    return sizeof(uint16_t) * W * (KP + 8);
}

static_assert(sizeof(NetW<288>) == net_tail_offset<288>() + sizeof(NetTail), "NetTail is the tail of NetW");
static_assert(sizeof(NetW<128>) == net_tail_offset<128>() + sizeof(NetTail), "NetTail is the tail of NetW");

/* Input-major copies for back-propagation. */
struct alignas(16) NetWN {
    uint16_t w1n[W][WS];
    uint16_t w2n[W][WS];
};

template <int KP>
__device__ inline void load_net(NetW<KP>& n, const float* __restrict__ p) {
    using L = Layout<KP>;
    for (int i = threadIdx.x; i < KP * W; i += blockDim.x) n.w0t[i % W][i / W] = f2bf(p[L::w0 + i]);
    for (int i = threadIdx.x; i < W * W; i += blockDim.x) {
        n.w1t[i % W][i / W] = f2bf(p[L::w1 + i]);
        n.w2t[i % W][i / W] = f2bf(p[L::w2 + i]);
    }
    for (int i = threadIdx.x; i < W; i += blockDim.x) {
        n.b0[i] = p[L::b0 + i];
        n.b1[i] = p[L::b1 + i];
        n.b2[i] = p[L::b2 + i];
        n.w3[i] = bf2f(f2bf(p[L::w3 + i]));
    }
    if (threadIdx.x == 0) {
        n.b3 = p[L::b3];
        n.mu = p[L::mu];
        n.sigma = p[L::sigma];
    }
}

/* The LDS image of a network (what load_net builds), written once to device memory so
   kernels that only run the forward pass copy it with 16-byte loads. */
template <int KP>
__global__ void k_pack_net(const float* __restrict__ p, NetW<KP>* out) {
    load_net<KP>(*out, p);
}

/* What a training step reads: the forward image and the input-major copies, kept in device
   memory beside the FP32 parameters and renewed by the optimizer (building them from the
   parameters in every block was most of a step). */
template <int KP>
struct TrainNet {
    NetW<KP> net;
    NetWN n;
};

template <int KP>
__device__ inline void load_net_n(NetWN& n, const float* __restrict__ p) {
    using L = Layout<KP>;
    for (int i = threadIdx.x; i < W * W; i += blockDim.x) {
        n.w1n[i / W][i % W] = f2bf(p[L::w1 + i]);
        n.w2n[i / W][i % W] = f2bf(p[L::w2 + i]);
    }
}

template <int KP>
__global__ void k_pack_train(const float* __restrict__ p, TrainNet<KP>* out) {
    load_net<KP>(out->net, p);
    load_net_n<KP>(out->n, p);
}

/* Parameter i of the flat array into the images. */
template <int KP>
__device__ inline void store_param(TrainNet<KP>& t, uint32_t i, float x) {
    using L = Layout<KP>;
    if (i < uint32_t(L::b0)) {
        t.net.w0t[i % W][i / W] = f2bf(x);
    } else if (i < uint32_t(L::w1)) {
        t.net.b0[i - L::b0] = x;
    } else if (i < uint32_t(L::b1)) {
        const uint32_t q = i - L::w1;
        t.net.w1t[q % W][q / W] = t.n.w1n[q / W][q % W] = f2bf(x);
    } else if (i < uint32_t(L::w2)) {
        t.net.b1[i - L::b1] = x;
    } else if (i < uint32_t(L::b2)) {
        const uint32_t q = i - L::w2;
        t.net.w2t[q % W][q / W] = t.n.w2n[q / W][q % W] = f2bf(x);
    } else if (i < uint32_t(L::w3)) {
        t.net.b2[i - L::b2] = x;
    } else if (i < uint32_t(L::b3)) {
        t.net.w3[i - L::w3] = bf2f(f2bf(x));
    } else {
        t.net.b3 = x;
    }
}

/* out[R][W] = bf(relu(x[R][K] W + b)); R a multiple of 16; all waves of the block. */
__device__ inline void dense_relu(const uint16_t* wt, int ldw, const float* bias, const uint16_t* x, int ldx, int K,
                                  int R, uint16_t* out) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int units = (R / 16) * (W / 16);
    for (int u = wave; u < units; u += nw) {
        const int rt = u / (W / 16), ct = u % (W / 16);
        const f32x4_t acc = mm_tile(x + rt * 16 * ldx, ldx, wt + ct * 16 * ldw, ldw, K, lane);
        const int col = ct * 16 + (lane & 15);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = rt * 16 + (lane >> 4) * 4 + i;
            const float z = acc[i] + bias[col];
            out[row * WS + col] = f2bf(z > 0.f ? z : 0.f);
        }
    }
}

/* y[r] = h[r] . w3 + b3 for r < R (R a multiple of 16); four lanes per row. */
__device__ inline void dense_out(const float* w3, float b3, const uint16_t* h, int R, float* y) {
    for (int q = threadIdx.x; q < R * 4; q += blockDim.x) {
        const int row = q >> 2, part = q & 3;
        const uint16_t* hr = h + row * WS + part * 16;
        float s = 0.f;
        for (int k = 0; k < 16; ++k) s += bf2f(hr[k]) * w3[part * 16 + k];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        if (part == 0) y[row] = s + b3;
    }
}

/* Forward pass of R rows of BF16 features xs[R][KP+8]: hidden activations into h0, h1,
   h2 ([R][WS] each; h2 may alias h0), raw outputs into y.  Contains __syncthreads. */
template <int KP, typename Net>
__device__ inline void forward_rows(const uint16_t* w0t, const Net& n, const uint16_t* xs, int R, uint16_t* h0,
                                    uint16_t* h1, uint16_t* h2, float* y) {
    dense_relu(w0t, KP + 8, n.b0, xs, KP + 8, KP, R, h0);
    __syncthreads();
    dense_relu(&n.w1t[0][0], WS, n.b1, h0, WS, W, R, h1);
    __syncthreads();
    dense_relu(&n.w2t[0][0], WS, n.b2, h1, WS, W, R, h2);
    __syncthreads();
    dense_out(n.w3, n.b3, h2, R, y);
    __syncthreads();
}
template <int KP>
__device__ inline void forward_block(const NetW<KP>& n, const uint16_t* xs, int R, uint16_t* h0, uint16_t* h1,
                                     uint16_t* h2, float* y) {
    forward_rows<KP>(&n.w0t[0][0], n, xs, R, h0, h1, h2, y);
}
/* The same with the first layer's weights w0t ([W][KP+8], BF16) read from device memory
   (the packed image of NetW<KP>) and the rest from LDS. */
template <int KP>
__device__ inline void forward_block_w0dev(const uint16_t* w0t, const NetTail& n, const uint16_t* xs, int R,
                                           uint16_t* h0, uint16_t* h1, uint16_t* h2, float* y) {
    forward_rows<KP>(w0t, n, xs, R, h0, h1, h2, y);
}

/* ---------------------------------------------------------------- inference
   Raw network outputs for n rows of BF16 features X[n][KP]; 64 rows per tile. */
template <int KP>
__global__ void __launch_bounds__(256) k_mlp_forward(const float* __restrict__ params, const uint16_t* __restrict__ X,
                                                     uint64_t n, float* __restrict__ y) {
    __shared__ NetW<KP> net;
    __shared__ __attribute__((aligned(16))) uint16_t xs[64][KP + 8];
    __shared__ __attribute__((aligned(16))) uint16_t h[2][64][WS];
    __shared__ float yo[64];
    load_net<KP>(net, params);
    for (uint64_t base = uint64_t(blockIdx.x) * 64; base < n; base += uint64_t(gridDim.x) * 64) {
        __syncthreads();
        for (int i = threadIdx.x; i < 64 * KP; i += blockDim.x) {
            const int r = i / KP, k = i % KP;
            xs[r][k] = base + r < n ? X[(base + r) * KP + k] : uint16_t(0);
        }
        __syncthreads();
        forward_block<KP>(net, &xs[0][0], 64, &h[0][0][0], &h[1][0][0], &h[0][0][0], yo);
        if (threadIdx.x < 64 && base + threadIdx.x < n) y[base + threadIdx.x] = yo[threadIdx.x];
    }
}

/* ---------------------------------------------------------------- training
   Gradient of 0.5 * sum_r c (y_r - (t_r - mu) / sigma)^2 over one 64-row tile per block
   (rows idx[blk*64 ..], c = inv_batch), written to part[blk][trained]; the block's loss
   sum goes to loss[blk] (want_grad = 0: the loss only).  Deterministic: no atomics.
   A minibatch of 1024 rows is 16 blocks, one per CU and most of the chip idle, so a step is
   its chain of layers: 16 waves take a 16x16 tile each (4 waves took four in turn), weights
   come as images, and activations and deltas are kept both row-major and transposed (each
   tile by two MFMAs, one per operand order, whose results a lane stores as 8 bytes), so
   that every operand of the next product is one 16-byte read.  KP = 32: 37 us a step, now
   10.5; KP = 288: 104, now 15.9.  Sums over the rows run in row order. */
constexpr int TRAIN_THREADS = 1024;
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

template <int KP>
struct TrainLds {
    // wide first layers (37 KB at KP = 288) are read from device memory
    static constexpr bool W0_DEV = KP >= 128;
    typename std::conditional<W0_DEV, NetTail, NetW<KP>>::type net;
    NetWN n;
    alignas(16) uint16_t xs[64][KP + 8];
    alignas(16) uint16_t h[3][64][WS];   // [row][feature]
    alignas(16) uint16_t ht[2][W][WS];   // [feature][row], layers 0 and 1
    alignas(16) uint16_t g[2][64][WS];
    alignas(16) uint16_t gt[2][W][WS];
    float y[64], dy[64];
};

template <int KP>
__global__ void __launch_bounds__(TRAIN_THREADS)
    k_mlp_grad(const TrainNet<KP>* __restrict__ tn, const uint16_t* __restrict__ X, const float* __restrict__ tgt,
               const uint32_t* __restrict__ idx, uint32_t count, float inv_batch, float* __restrict__ part,
               float* __restrict__ loss, int want_grad) {
    using L = Layout<KP>;
    using LD = TrainLds<KP>;
    __shared__ LD S;
    constexpr int NT = TRAIN_THREADS, NW = NT / 64;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r16 = lane & 15, q4 = (lane >> 4) * 4;
    const uint32_t base = blockIdx.x * 64u;
    float* out = part + size_t(blockIdx.x) * L::trained;
    {
        constexpr size_t skip = LD::W0_DEV ? net_tail_offset<KP>() : 0;
        const uint4* a = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(&tn->net) + skip);
        uint4* d = reinterpret_cast<uint4*>(&S.net);
        for (int i = tid; i < int(sizeof(S.net) / 16); i += NT) d[i] = a[i];
        const uint4* a2 = reinterpret_cast<const uint4*>(&tn->n);
        uint4* d2 = reinterpret_cast<uint4*>(&S.n);
        for (int i = tid; i < int(sizeof(S.n) / 16); i += NT) d2[i] = a2[i];
        constexpr int V = KP / 8;  // 16-byte pieces of a row (KP is a multiple of 32)
        for (int i = tid; i < 64 * V; i += NT) {
            const int r = i / V, k = i % V;
            const uint4 z = make_uint4(0u, 0u, 0u, 0u);
            *reinterpret_cast<uint4*>(&S.xs[r][8 * k]) =
                base + r < count ? reinterpret_cast<const uint4*>(X + size_t(idx[base + r]) * KP)[k] : z;
        }
    }
    float tg = 0.f;
    if (tid < 64 && base + tid < count) tg = tgt[idx[base + tid]];
    __syncthreads();
    const uint16_t* w0t;
    if constexpr (LD::W0_DEV)
        w0t = &tn->net.w0t[0][0];
    else
        w0t = &S.net.w0t[0][0];
    // forward: tile (rt, ct) of each layer to wave 4 rt + ct
    const int rt = wave >> 2, ct = wave & 3;
    auto layer = [&](const uint16_t* wt, int ldw, const float* bias, const uint16_t* x, int ldx, int K, uint16_t* h,
                     uint16_t* ht) {
        const uint16_t *xr = x + rt * 16 * ldx, *wr = wt + ct * 16 * ldw;
        {  // a lane's four results: features ct * 16 + q4 + i of row rt * 16 + r16
            const f32x4_t acc = mm_tile(wr, ldw, xr, ldx, K, lane);
            bf16x4_t v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float z = acc[i] + bias[ct * 16 + q4 + i];
                v[i] = __bf16(z > 0.f ? z : 0.f);
            }
            *reinterpret_cast<bf16x4_t*>(h + (rt * 16 + r16) * WS + ct * 16 + q4) = v;
        }
        if (ht) {  // rows rt * 16 + q4 + i of feature ct * 16 + r16
            const f32x4_t acc = mm_tile(xr, ldx, wr, ldw, K, lane);
            const float bv = bias[ct * 16 + r16];
            bf16x4_t v;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float z = acc[i] + bv;
                v[i] = __bf16(z > 0.f ? z : 0.f);
            }
            *reinterpret_cast<bf16x4_t*>(ht + (ct * 16 + r16) * WS + rt * 16 + q4) = v;
        }
        __syncthreads();
    };
    static_assert(NW == 16, "a wave per tile of a layer");
    layer(w0t, KP + 8, S.net.b0, &S.xs[0][0], KP + 8, KP, &S.h[0][0][0], &S.ht[0][0][0]);
    layer(&S.net.w1t[0][0], WS, S.net.b1, &S.h[0][0][0], WS, W, &S.h[1][0][0], &S.ht[1][0][0]);
    layer(&S.net.w2t[0][0], WS, S.net.b2, &S.h[1][0][0], WS, W, &S.h[2][0][0], nullptr);
    dense_out(S.net.w3, S.net.b3, &S.h[2][0][0], 64, S.y);
    __syncthreads();
    if (tid < 64) {
        float d = 0.f;
        if (base + tid < count) {
            const float t = (tg - S.net.mu) / S.net.sigma;
            d = S.y[tid] - t;
        }
        S.dy[tid] = d * inv_batch;
        S.y[tid] = 0.5f * d * d * inv_batch;
    }
    __syncthreads();
    if (wave == NW - 1) {  // the loss, and with it the output bias's gradient
        if (lane == 0) {
            float s = 0.f, ls = 0.f;
#pragma unroll 16
            for (int r = 0; r < 64; ++r) {
                s += S.dy[r];
                ls += S.y[r];
            }
            if (want_grad) out[L::b3] = s;
            loss[blockIdx.x] = ls;
        }
    }
    if (!want_grad) return;  // validation
    if (wave == NW - 2) {  // output layer
        float s = 0.f;
#pragma unroll 16
        for (int r = 0; r < 64; ++r) s += bf2f(S.h[2][r][lane]) * S.dy[r];
        out[L::w3 + lane] = s;
    }
    {
        const int r = tid >> 4, k0 = (tid & 15) * 4;  // four features of a row
        uint16_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = bf2f(S.h[2][r][k0 + i]) > 0.f ? f2bf(S.dy[r] * S.net.w3[k0 + i]) : uint16_t(0);
            S.g[0][r][k0 + i] = v[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) S.gt[0][k0 + i][r] = v[i];
    }
    __syncthreads();
    // sum over the rows, in row order, of feature `lane` of a transposed delta
    auto bias_grad = [&](const uint16_t* gt, float* o) {
        float s = 0.f;
#pragma unroll
        for (int r = 0; r < 64; r += 8) {
            const u16x8_t v = *reinterpret_cast<const u16x8_t*>(gt + lane * WS + r);
#pragma unroll
            for (int i = 0; i < 8; ++i) s += bf2f(v[i]);
        }
        o[lane] = s;
    };
    // tile (mt, nt) of A^T B over the rows, both transposed
    auto weight_grad = [&](const uint16_t* at, const uint16_t* bt, int mt, int nt, float* o) {
        const f32x4_t acc = mm_tile(at + mt * 16 * WS, WS, bt + nt * 16 * WS, WS, 64, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[(mt * 16 + q4 + i) * W + nt * 16 + r16] = acc[i];
    };
    // hidden layers 2 and 1: dW = h_in^T g, db = sum g, g_in = (g W^T) masked
#pragma unroll
    for (int l = 2; l >= 1; --l) {
        const int cur = l == 2 ? 0 : 1, nxt = cur ^ 1;
        const uint16_t *hin = &S.h[l - 1][0][0], *hint = &S.ht[l - 1][0][0];
        const uint16_t *gl = &S.g[cur][0][0], *glt = &S.gt[cur][0][0];
        const uint16_t* wn = l == 2 ? &S.n.w2n[0][0] : &S.n.w1n[0][0];
        {
            const uint16_t *gr = gl + rt * 16 * WS, *wr = wn + ct * 16 * WS;
            const f32x4_t a = mm_tile(wr, WS, gr, WS, W, lane);  // inputs ct * 16 + q4 + i of row rt * 16 + r16
            const f32x4_t b = mm_tile(gr, WS, wr, WS, W, lane);  // rows rt * 16 + q4 + i of input ct * 16 + r16
            uint16_t* ga = &S.g[nxt][rt * 16 + r16][ct * 16 + q4];
            uint16_t* gb = &S.gt[nxt][ct * 16 + r16][rt * 16 + q4];
            const uint16_t* ha = hin + (rt * 16 + r16) * WS + ct * 16 + q4;
            const uint16_t* hb = hint + (ct * 16 + r16) * WS + rt * 16 + q4;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ga[i] = bf2f(ha[i]) > 0.f ? f2bf(a[i]) : uint16_t(0);
                gb[i] = bf2f(hb[i]) > 0.f ? f2bf(b[i]) : uint16_t(0);
            }
        }
        weight_grad(hint, glt, rt, ct, out + (l == 2 ? L::w2 : L::w1));
        if (wave == l) bias_grad(glt, out + (l == 2 ? L::b2 : L::b1));
        __syncthreads();
    }
    // input layer: dW0 = x^T g0 (g0 is in g[0] and gt[0] after the loop)
    for (int u = wave; u < (KP / 16) * 4; u += NW) {
        const int mt = u / 4, nt = u % 4, kq = (lane >> 4) * 8;
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s0 = 0; s0 < 64; s0 += 32)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gather8(&S.xs[s0 + kq][mt * 16 + r16], KP + 8),
                                                          ld8(&S.gt[0][nt * 16 + r16][s0 + kq]), acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[L::w0 + (mt * 16 + q4 + i) * W + nt * 16 + r16] = acc[i];
    }
    if (wave == NW - 1) bias_grad(&S.gt[0][0][0], out + L::b0);
}

/* 64-bit FNV-1a over the 32-bit words of row i (kp BF16 features, then the target's
   bits): a content key whose sort gives the pairs one order whatever order the device
   wrote them in. */
static __global__ void k_row_hash(const uint16_t* __restrict__ X, const float* __restrict__ tgt, uint64_t n, int kp,
                           uint64_t* __restrict__ key, uint32_t* __restrict__ idx) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t* w = reinterpret_cast<const uint32_t*>(X + i * uint64_t(kp));
    uint64_t h = 0xcbf29ce484222325ull;
    for (int k = 0; k < kp / 2; ++k) {
        h ^= w[k];
        h *= 0x100000001b3ull;
    }
    h ^= __builtin_bit_cast(uint32_t, tgt[i]);
    h *= 0x100000001b3ull;
    key[i] = h;
    idx[i] = uint32_t(i);
}

/* Sum of the per-block partial gradients in block order. */
static __global__ void k_sum_parts(const float* __restrict__ part, uint32_t nblk, uint32_t P, float* __restrict__ grad) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    float s = 0.f;
    for (uint32_t b = 0; b < nblk; ++b) s += part[size_t(b) * P + i];
    grad[i] = s;
}

/* Adam (Kingma & Ba 2015) on the trained parameters; the gradient is the block-ordered
   sum of the partials, whose loads are all in flight at once.  c1, c2 are the bias
   corrections 1/(1-beta^t).  The new values go into the images too. */
template <int KP>
__global__ void __launch_bounds__(64) k_adam(float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                                             const float* __restrict__ part, TrainNet<KP>* __restrict__ tn, uint32_t nblk,
                                             uint32_t P, float lr, float b1, float b2, float eps, float c1, float c2) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    const float pi = p[i], m0 = m[i], v0 = v[i];
    float gsum = 0.f;
    for (uint32_t b0 = 0; b0 < nblk; b0 += 16) {
        float g[16];
#pragma unroll
        for (uint32_t u = 0; u < 16; ++u) g[u] = part[size_t(b0 + u < nblk ? b0 + u : 0u) * P + i];
#pragma unroll
        for (uint32_t u = 0; u < 16; ++u)
            if (b0 + u < nblk) gsum += g[u];
    }
    const float mi = b1 * m0 + (1.f - b1) * gsum;
    const float vi = b2 * v0 + (1.f - b2) * gsum * gsum;
    m[i] = mi;
    v[i] = vi;
    const float x = pi - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    p[i] = x;
    store_param<KP>(*tn, i, x);
}

}  // namespace nn
}  // namespace vmx

#endif
