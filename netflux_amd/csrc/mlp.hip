// Warm-start network: MLP 6 -> 128 -> 128 -> 128 -> 5 with GELU, BF16
// weights and activations as MFMA operands, FP32 accumulation, FP32 master
// weights and Adam state.  Inputs are per-cell features (Mach, bump height,
// centroid x, y, z, wall distance); outputs are the primitive variables,
// both normalised per component.
//
// All products run on BF16 MFMA (v_mfma_f32_16x16x32_bf16).  Inference is one
// kernel; a training step is three: the minibatch through the network and
// back (k_train), the weight gradients dW = dZ X^T over the batch with the
// bias and loss sums (k_wgrad), and the sum over batch splits with Adam
// (k_update).  Activations go between them as [16-sample tile][feature][16]:
// a block of k_train writes whole lines, and k_wgrad's operand fragments are
// 16-byte loads of adjacent rows.  Weight gradients
// reduce over the batch with a fixed split-K partition and a fixed-order sum
// (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/netflux.h"
#include "host_pipe.hpp"
#include "mlp.hpp"

using nf::mlp::HID;
using nf::mlp::IN;
using nf::mlp::OUT;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// flattened parameter layout: W1 [HID][IN], b1, W2 [HID][HID], b2, W3, b3,
// W4 [OUT][HID], b4 (row-major [out][in], as a linear layer stores them)
constexpr int64_t OFF_W1 = 0, OFF_B1 = OFF_W1 + HID * IN;
constexpr int64_t OFF_W2 = OFF_B1 + HID, OFF_B2 = OFF_W2 + HID * HID;
constexpr int64_t OFF_W3 = OFF_B2 + HID, OFF_B3 = OFF_W3 + HID * HID;
constexpr int64_t OFF_W4 = OFF_B3 + HID, OFF_B4 = OFF_W4 + OUT * HID;
constexpr int64_t NPARAM = OFF_B4 + OUT;

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

// ---------------------------------------------------------------------------
// Fused network: one block takes NC x 16 samples through every layer, so
// activations never leave the CU.  Each of its 8 / RT waves computes RT MFMA
// row tiles (16 RT features) of each hidden layer, keeps those rows of all
// weights in registers as MFMA operands for as long as it lives (the grid is
// persistent), and hands its activations to the other waves through LDS as
// [sample][feature] BF16, so that a lane's operand fragment of the next layer
// -- 8 consecutive features of one sample -- is one 16-byte read.  Every
// product is accumulated over k in steps of 32 in increasing order.
constexpr int LDH = HID + 8;  // row stride of the LDS activations: 16-byte aligned, 16 columns over all banks

// MFMA operand fragment of row r (R real rows), columns [k, k + 8) of a
// row-major [R][HID] BF16 matrix
__device__ __forceinline__ bf16x8 row_frag(const __bf16 *W, int r, int k, int R) {
    if (r < R) return *reinterpret_cast<const bf16x8 *>(W + r * HID + k);
    bf16x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = (__bf16)0.0f;
    return z;
}
// the same of the [HID][IN] input layer: columns IN.. are zero
__device__ __forceinline__ bf16x8 in_frag(const __bf16 *W, int r, int k) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = k + e < IN ? W[r * IN + k + e] : (__bf16)0.0f;
    return v;
}

struct Infer {
    const __bf16 *pb;   // BF16 parameters
    const float *p;     // FP32 parameters (biases)
    const float *norm;  // in_shift[6], in_scale[6], out_shift[5], out_scale[5]
    const float *x;     // x(f, j) = x[f * xf + j * xj]
    int64_t xf, xj;
    float *y;           // y(o, j) = y[o * yo + j * yj]
    int64_t yo, yj;
    int64_t n;
};

// Bound by the erf of the three GELUs (384 per sample, about 45 VALU
// instructions each), not by the products or by memory.  Layer by layer (11
// launches, 3.6 KB per sample through HBM) 700 samples took 38 us and
// 1,463,340 samples 2.4 ms; one launch that moves 44 bytes per sample takes
// 6.0 us and 0.44 ms.
template <int NC, int RT>
__global__ __launch_bounds__(512 / RT) void k_infer(Infer g) {
    __shared__ __attribute__((aligned(16))) __bf16 H[2][NC * 16][LDH];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, col = lane & 15, q4 = lane >> 4;
    const int64_t ntiles = (g.n + NC * 16 - 1) / (NC * 16);
    bf16x8 a1[RT], a2[RT][4], a3[RT][4], a4[4];
    f32x4 b1[RT], b2[RT], b3[RT];
    float b4[4], osh[4], osc[4];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int r = 16 * (RT * w + i);
        a1[i] = in_frag(g.pb + OFF_W1, r + col, 8 * q4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a2[i][q] = row_frag(g.pb + OFF_W2, r + col, 32 * q + 8 * q4, HID);
            a3[i][q] = row_frag(g.pb + OFF_W3, r + col, 32 * q + 8 * q4, HID);
        }
        b1[i] = *reinterpret_cast<const f32x4 *>(g.p + OFF_B1 + r + 4 * q4);
        b2[i] = *reinterpret_cast<const f32x4 *>(g.p + OFF_B2 + r + 4 * q4);
        b3[i] = *reinterpret_cast<const f32x4 *>(g.p + OFF_B3 + r + 4 * q4);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) a4[q] = row_frag(g.pb + OFF_W4, col, 32 * q + 8 * q4, OUT);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int o = 4 * q4 + r;
        b4[r] = o < OUT ? g.p[OFF_B4 + o] : 0.f;
        osh[r] = o < OUT ? g.norm[12 + o] : 0.f;
        osc[r] = o < OUT ? g.norm[17 + o] : 0.f;
    }
    // activations of one product, [2 row tiles][NC sample tiles], to LDS
    auto store = [&](const f32x4 (*acc)[NC], const f32x4 *b, __bf16 (*S)[LDH]) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) h[r] = (__bf16)gelu(acc[i][c][r] + b[i][r]);
                *reinterpret_cast<bf16x4 *>(&S[c * 16 + col][16 * (RT * w + i) + 4 * q4]) = h;
            }
    };
    auto layer = [&](const bf16x8 (*a)[4], const f32x4 *b, const __bf16 (*S)[LDH], __bf16 (*D)[LDH]) {
        f32x4 acc[RT][NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bf16x8 h = *reinterpret_cast<const bf16x8 *>(&S[c * 16 + col][32 * q + 8 * q4]);
#pragma unroll
                for (int i = 0; i < RT; ++i)
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][q], h, acc[i][c], 0, 0, 0);
            }
        }
        store(acc, b, D);
    };
    int p = 0;  // the buffer the input layer writes; it was last read two barriers ago
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x, p ^= 1) {
        const int64_t j0 = t * (NC * 16);
        f32x4 acc[RT][NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            // padding samples repeat the last one and are not stored
            const int64_t j = j0 + c * 16 + col < g.n ? j0 + c * 16 + col : g.n - 1;
            bf16x8 v;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = q4 == 0 && e < IN ? (__bf16)((g.x[(e < IN ? e : 0) * g.xf + j * g.xj] - g.norm[e < IN ? e : 0]) *
                                                    g.norm[6 + (e < IN ? e : 0)])
                                         : (__bf16)0.0f;
#pragma unroll
            for (int i = 0; i < RT; ++i)
                acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[i], v, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
        store(acc, b1, H[p]);
        __syncthreads();
        layer(a2, b2, H[p], H[p ^ 1]);
        __syncthreads();
        layer(a3, b3, H[p ^ 1], H[p]);
        __syncthreads();
        for (int c = w; c < NC; c += 8 / RT) {
            f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 4; ++q)
                y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a4[q], *reinterpret_cast<const bf16x8 *>(&H[p][c * 16 + col][32 * q + 8 * q4]), y, 0, 0, 0);
            const int64_t j = j0 + c * 16 + col;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * q4 + r < OUT && j < g.n) g.y[(4 * q4 + r) * g.yo + j * g.yj] = (y[r] + b4[r]) * osc[r] + osh[r];
        }
    }
}

// ---------------------------------------------------------------------------
// Training.  Transposed BF16 weights for the backward products (rows are the
// layer's inputs): W2^T, W3^T [HID][HID], W4^T [HID][8], its columns OUT.. zero
constexpr int64_t PT2 = 0, PT3 = PT2 + HID * HID, PT4 = PT3 + HID * HID, NPT = PT4 + HID * 8;

__device__ __forceinline__ size_t tix(int tile, int rows, int r, int col) { return ((size_t)tile * rows + r) * 16 + col; }

struct Train {
    const __bf16 *pb, *pt;  // BF16 parameters and their transposes
    const float *p;         // FP32 parameters (biases)
    const float *norm;      // in_shift[6], in_scale[6], out_shift[5], out_scale[5], out_iscale[5]
    const float *x, *y;     // raw samples [.][IN], targets [.][OUT]
    const int64_t *idx;     // minibatch: sample idx[first + j], or null: first + j
    int64_t first;
    int n, ld;              // samples, and rounded up to 64: samples n.. are stored as zeros
    float inv_count;
    __bf16 *X0, *A[3], *dZb[3], *dYb;  // [ld / 16][rows][16]
    float *dZ[3], *dY;                 // the same, for the bias sums
    float *se;                         // [ld] squared error of each sample
};

// The samples of a minibatch through the network and back, 16 per block tile,
// organised as k_infer; GELU and its derivative share one erf, and the
// pre-activations stay in registers.  Bound by the erf and exp of 3 x 128
// activations per sample in the few waves a minibatch has (2,048 samples:
// 128 blocks), not by the products.  A step of 2,048 samples took 33 launches
// and 157 us when every product, activation and sum was one; it takes 29 us
// (k_train 15, k_wgrad 6, k_update 3.6): eight waves of one row tile each
// (four of two: 34 us with [row][sample] activations, eight 31 us), the
// activations in 16-sample tiles (29 us).
__global__ __launch_bounds__(512) void k_train(Train g) {
    constexpr int RT = 1;  // row tiles per wave
    __shared__ __attribute__((aligned(16))) __bf16 H[2][16][LDH];
    __shared__ __attribute__((aligned(16))) __bf16 D[16][8];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, col = lane & 15, q4 = lane >> 4;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    bf16x8 none;
#pragma unroll
    for (int e = 0; e < 8; ++e) none[e] = (__bf16)0.0f;
    bf16x8 a1[RT], a2[RT][4], a3[RT][4], a4[4], t2[RT][4], t3[RT][4], t4[RT];
    f32x4 b1[RT], b2[RT], b3[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int r = 16 * (RT * w + i);
        a1[i] = in_frag(g.pb + OFF_W1, r + col, 8 * q4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a2[i][q] = row_frag(g.pb + OFF_W2, r + col, 32 * q + 8 * q4, HID);
            a3[i][q] = row_frag(g.pb + OFF_W3, r + col, 32 * q + 8 * q4, HID);
            t2[i][q] = row_frag(g.pt + PT2, r + col, 32 * q + 8 * q4, HID);
            t3[i][q] = row_frag(g.pt + PT3, r + col, 32 * q + 8 * q4, HID);
        }
        t4[i] = q4 == 0 ? *reinterpret_cast<const bf16x8 *>(g.pt + PT4 + (r + col) * 8) : none;
        b1[i] = *reinterpret_cast<const f32x4 *>(g.p + OFF_B1 + r + 4 * q4);
        b2[i] = *reinterpret_cast<const f32x4 *>(g.p + OFF_B2 + r + 4 * q4);
        b3[i] = *reinterpret_cast<const f32x4 *>(g.p + OFF_B3 + r + 4 * q4);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) a4[q] = row_frag(g.pb + OFF_W4, col, 32 * q + 8 * q4, OUT);
    int p = 0;
    for (int t = blockIdx.x; t < g.ld / 16; t += gridDim.x, p ^= 1) {
        const int j = t * 16 + col;
        const bool live = j < g.n;
        const int64_t src = g.idx ? g.idx[g.first + (live ? j : g.n - 1)] : g.first + (live ? j : g.n - 1);
        f32x4 gd[3][RT];  // gelu' of the three layers
        auto product = [&](const bf16x8 (*a)[4], const __bf16 (*S)[LDH], f32x4 *acc) {
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[i] = zero;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bf16x8 h = *reinterpret_cast<const bf16x8 *>(&S[col][32 * q + 8 * q4]);
#pragma unroll
                for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][q], h, acc[i], 0, 0, 0);
            }
        };
        auto activate = [&](int l, const f32x4 *acc, const f32x4 *b, __bf16 (*S)[LDH]) {
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int f = 16 * (RT * w + i) + 4 * q4;
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float z = acc[i][r] + b[i][r];
                    const float e = 1.0f + erff(z * 0.70710678118654752f);
                    h[r] = (__bf16)(0.5f * z * e);
                    gd[l][i][r] = 0.5f * e + z * 0.39894228040143268f * expf(-0.5f * z * z);
                    g.A[l][tix(t, HID, f + r, col)] = live ? h[r] : (__bf16)0.0f;
                }
                *reinterpret_cast<bf16x4 *>(&S[col][f]) = h;
            }
        };
        f32x4 acc[RT];
        {
            bf16x8 v = none;
            if (q4 == 0) {
#pragma unroll
                for (int e = 0; e < IN; ++e) {
                    v[e] = (__bf16)((g.x[src * IN + e] - g.norm[e]) * g.norm[6 + e]);
                    if (w == 0) g.X0[tix(t, IN, e, col)] = live ? v[e] : (__bf16)0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[i], v, zero, 0, 0, 0);
        }
        activate(0, acc, b1, H[p]);
        __syncthreads();
        product(a2, H[p], acc);
        activate(1, acc, b2, H[p ^ 1]);
        __syncthreads();
        product(a3, H[p ^ 1], acc);
        activate(2, acc, b3, H[p]);
        __syncthreads();
        if (w == 0) {
            // output layer: D = Y - T, dY = 2 D / (OUT n); rows OUT.. are zero
            f32x4 y = zero;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a4[q], *reinterpret_cast<const bf16x8 *>(&H[p][col][32 * q + 8 * q4]), y, 0, 0, 0);
            float d[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = 4 * q4 + r;
                d[r] = 0.f;
                if (o < OUT) {
                    const float T = (g.y[src * OUT + o] - g.norm[12 + o]) * g.norm[22 + o];
                    d[r] = (y[r] + g.p[OFF_B4 + o]) - T;
                    const float gy = 2.0f * d[r] * g.inv_count;
                    g.dY[tix(t, OUT, o, col)] = live ? gy : 0.f;
                    g.dYb[tix(t, OUT, o, col)] = live ? (__bf16)gy : (__bf16)0.0f;
                    D[col][o] = (__bf16)gy;
                } else if (o < 8) {
                    D[col][o] = (__bf16)0.0f;
                }
            }
            const float d4 = __shfl(d[0], (lane + 16) & 63, 64);
            if (q4 == 0) g.se[j] = live ? (((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]) + d[3] * d[3]) + d4 * d4 : 0.f;
        }
        __syncthreads();
        auto back = [&](int l, __bf16 (*S)[LDH]) {
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int f = 16 * (RT * w + i) + 4 * q4;
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float d = acc[i][r] * gd[l][i][r];
                    h[r] = (__bf16)d;
                    g.dZ[l][tix(t, HID, f + r, col)] = live ? d : 0.f;
                    g.dZb[l][tix(t, HID, f + r, col)] = live ? h[r] : (__bf16)0.0f;
                }
                if (S) *reinterpret_cast<bf16x4 *>(&S[col][f]) = h;
            }
        };
        {
            const bf16x8 v = q4 == 0 ? *reinterpret_cast<const bf16x8 *>(&D[col][0]) : none;
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t4[i], v, zero, 0, 0, 0);
        }
        back(2, H[p ^ 1]);
        __syncthreads();
        product(t3, H[p ^ 1], acc);
        back(1, H[p]);
        __syncthreads();
        product(t2, H[p], acc);
        back(0, nullptr);
    }
}

constexpr int KSPLIT = 512;  // batch samples per split of the weight-gradient sums

struct Wgrad {
    const __bf16 *X0, *A[3], *dZb[3], *dYb;
    const float *dZ[3], *dY, *se;
    int n, ld, splits;
    float *part;       // [splits][NPARAM] partial weight gradients
    float *g;          // [NPARAM] bias gradients
    float *loss_part;  // [n / 256] sums of squared errors
};

// 16 x (16 NT) tiles of a weight gradient dW = dZ X^T over one batch split
template <int NT>
__device__ __forceinline__ void wgrad_tile(const __bf16 *Z, int rows, int r0, const __bf16 *X, int cols, int c0,
                                           int k0, int k1, float *out) {
    const int lane = threadIdx.x & 63, col = lane & 15, q4 = lane >> 4;
    f32x4 acc[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows outside the matrix repeat its last one; their results are not stored
    // the lane's 8 samples k + 8 q4 .. are half a row of tile (k + 8 q4) / 16
    const __bf16 *zp = Z + tix(q4 >> 1, rows, min(r0 + col, rows - 1), 8 * (q4 & 1));
    const __bf16 *xp[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) xp[i] = X + tix(q4 >> 1, cols, min(c0 + 16 * i + col, cols - 1), 8 * (q4 & 1));
    auto step = [&](int k) {
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(zp + (size_t)k * rows);
#pragma unroll
        for (int i = 0; i < NT; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a, *reinterpret_cast<const bf16x8 *>(xp[i] + (size_t)k * cols), acc[i], 0, 0, 0);
    };
    if (k1 - k0 == KSPLIT) {  // a full split: every load in flight
#pragma unroll
        for (int k = 0; k < KSPLIT; k += 32) step(k0 + k);
    } else {
        for (int k = k0; k < k1; k += 32) step(k);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = r0 + 4 * q4 + r, c = c0 + 16 * i + col;
            if (m < rows && c < cols) out[m * cols + c] = acc[i][r];
        }
}

// sum over 256 threads in a fixed order; valid in thread 0
__device__ __forceinline__ float sum256(float s, float *sh) {
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

constexpr int WG_UNITS = 76;  // wave tiles of all weight gradients of one split
constexpr int wgrad_blocks(int splits) { return (WG_UNITS * splits + 3) / 4; }

// Every sum over the batch in one launch: the weight gradients (one wave per
// 16 x 32 tile and split; latency-bound, so as many waves as tiles), the bias
// gradients (one block per row) and the loss (one block per 256 samples).
__global__ __launch_bounds__(256) void k_wgrad(Wgrad g) {
    __shared__ float sh[4];
    int b = blockIdx.x;
    const int nw = wgrad_blocks(g.splits);
    if (b < nw) {
        const int q = b * 4 + (threadIdx.x >> 6);
        if (q >= WG_UNITS * g.splits) return;
        const int z = q / WG_UNITS, u = q % WG_UNITS;
        const int k0 = z * KSPLIT, k1 = min(g.ld, k0 + KSPLIT);
        float *out = g.part + (size_t)z * NPARAM;
        if (u < 32) wgrad_tile<2>(g.dZb[2], HID, 16 * (u >> 2), g.A[1], HID, 32 * (u & 3), k0, k1, out + OFF_W3);
        else if (u < 64) wgrad_tile<2>(g.dZb[1], HID, 16 * ((u - 32) >> 2), g.A[0], HID, 32 * (u & 3), k0, k1, out + OFF_W2);
        else if (u < 68) wgrad_tile<2>(g.dYb, OUT, 0, g.A[2], HID, 32 * (u & 3), k0, k1, out + OFF_W4);
        else wgrad_tile<1>(g.dZb[0], HID, 16 * (u - 68), g.X0, IN, 0, k0, k1, out + OFF_W1);
        return;
    }
    b -= nw;
    if (b < 3 * HID + OUT) {
        const int l = b / HID, r = b % HID;
        const float *X = l < 3 ? g.dZ[l] : g.dY;
        float s = 0.f;
#pragma unroll 4
        for (int j = threadIdx.x; j < g.n; j += 256) s += X[tix(j >> 4, l < 3 ? HID : OUT, r, j & 15)];
        s = sum256(s, sh);
        if (threadIdx.x == 0) g.g[(l == 0 ? OFF_B1 : (l == 1 ? OFF_B2 : (l == 2 ? OFF_B3 : OFF_B4))) + r] = s;
        return;
    }
    b -= 3 * HID + OUT;
    const int j = b * 256 + threadIdx.x;
    const float s = sum256(j < g.n ? g.se[j] : 0.f, sh);
    if (threadIdx.x == 0) g.loss_part[b] = s;
}

__device__ __forceinline__ bool is_bias(int64_t i) {
    return (i >= OFF_B1 && i < OFF_W2) || (i >= OFF_B2 && i < OFF_W3) || (i >= OFF_B3 && i < OFF_W4) || i >= OFF_B4;
}
// BF16 copies of parameter i
__device__ __forceinline__ void put_bf16(int64_t i, float v, __bf16 *pb, __bf16 *pt) {
    const __bf16 h = (__bf16)v;
    pb[i] = h;
    if (i >= OFF_W2 && i < OFF_B2) pt[PT2 + (i - OFF_W2) % HID * HID + (i - OFF_W2) / HID] = h;
    if (i >= OFF_W3 && i < OFF_B3) pt[PT3 + (i - OFF_W3) % HID * HID + (i - OFF_W3) / HID] = h;
    if (i >= OFF_W4 && i < OFF_B4) pt[PT4 + (i - OFF_W4) % HID * 8 + (i - OFF_W4) / HID] = h;
}

struct Update {
    const float *part;  // [splits][NPARAM]
    int splits;
    float *g, *p, *m, *v;
    __bf16 *pb, *pt;
    float lr_t, b1, b2, eps;
};

// gradient = sum over splits in order; with ADAM a step on the FP32 masters
// (bias-corrected step size lr_t) and their BF16 copies
template <bool ADAM>
__global__ __launch_bounds__(256) void k_update(Update a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= NPARAM) return;
    float gi = 0.f;
    if (is_bias(i)) gi = a.g[i];
    else {
#pragma unroll 4
        for (int q = 0; q < a.splits; ++q) gi += a.part[(size_t)q * NPARAM + i];
        a.g[i] = gi;
    }
    if (!ADAM) return;
    const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gi;
    const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    const float pi = a.p[i] - a.lr_t * mi / (sqrtf(vi) + a.eps);
    a.p[i] = pi;
    put_bf16(i, pi, a.pb, a.pt);
}

__global__ __launch_bounds__(256) void k_to_bf16(const float *p, __bf16 *pb, __bf16 *pt) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < NPARAM) put_bf16(i, p[i], pb, pt);
}

__global__ __launch_bounds__(256) void k_copy(const float *x, float *y, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = x[i];
}

}  // namespace

// ---------------------------------------------------------------------------
constexpr int64_t NOALLOC_MAX = 16384;  // samples per nf_mlp_predict_noalloc call

struct nf_mlp {
    std::string err;
    hipStream_t stream = nullptr;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // FP32 [NPARAM]
    __bf16 *pb = nullptr, *pt = nullptr;                           // BF16 copy, transposes (PT2..)
    float *xcopy = nullptr;  // inputs of a predict_noalloc call whose outputs lie over them, [NOALLOC_MAX][IN]
    float *norm = nullptr;  // device: in_shift[6], in_scale[6], out_shift[5], out_scale[5], out_iscale[5]
    float hnorm[27] = {};
    bool norm_set = false;  // false: training sets it from the data
    int64_t adam_t = 0;
    // workspace for batches of up to `cap` samples
    int cap = 0;
    __bf16 *X0 = nullptr, *A[3] = {nullptr, nullptr, nullptr}, *dZb[3] = {nullptr, nullptr, nullptr}, *dYb = nullptr;
    float *dZ[3] = {nullptr, nullptr, nullptr}, *dY = nullptr, *se = nullptr;
    float *part = nullptr, *loss_part = nullptr;
    std::vector<void *> ws;
    int device = 0;  // device current at nf_mlp_create, holding the parameters
    // device copies of the caller's host arrays (inputs [n][6], targets or
    // outputs [n][5]) and the minibatch order, kept and grown as needed
    float *dx = nullptr, *dy = nullptr;
    int64_t *didx = nullptr;
    int64_t data_cap = 0;
    nf::HostPipe pipe;  // large arrays across the boundary
};

namespace {

constexpr int64_t NC1_MAX = 12288;  // samples up to which inference takes 16 per block (infer)

int fail(nf_mlp *m, int code, const std::string &msg) {
    if (m) m->err = msg;
    return code;
}
#define HIPM(expr)                                                                          \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                             \
            (void)hipGetLastError(); /* reported here, not by the next call's launches */   \
            return fail(mm, NF_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));   \
        }                                                                                   \
    } while (0)

int ensure_ws(nf_mlp *mm, int n) {
    if (n <= mm->cap) return NF_OK;
    mm->cap = 0;  // (until every array is there)
    for (void *q : mm->ws) (void)hipFree(q);
    mm->ws.clear();
    const int cap = (n + 255) / 256 * 256;
    auto al = [&](auto **ptr, size_t count) -> int {
        void *q = nullptr;
        HIPM(hipMalloc(&q, count * sizeof(**ptr)));
        mm->ws.push_back(q);
        *ptr = static_cast<std::remove_reference_t<decltype(*ptr)>>(q);
        return NF_OK;
    };
    int rc;
    if ((rc = al(&mm->X0, (size_t)IN * cap))) return rc;
    for (int l = 0; l < 3; ++l) {
        if ((rc = al(&mm->A[l], (size_t)HID * cap))) return rc;
        if ((rc = al(&mm->dZb[l], (size_t)HID * cap))) return rc;
        if ((rc = al(&mm->dZ[l], (size_t)HID * cap))) return rc;
    }
    if ((rc = al(&mm->dY, (size_t)OUT * cap))) return rc;
    if ((rc = al(&mm->dYb, (size_t)OUT * cap))) return rc;
    if ((rc = al(&mm->se, (size_t)cap))) return rc;
    if ((rc = al(&mm->part, (size_t)((cap + KSPLIT - 1) / KSPLIT) * NPARAM))) return rc;
    if ((rc = al(&mm->loss_part, (size_t)cap / 256 + 1))) return rc;
    mm->cap = cap;
    return NF_OK;
}

// inference of n samples on the device: x(f, j) = x[f * xf + j * xj],
// y(o, j) = y[o * yo + j * yj]; one launch, no workspace
hipError_t infer(const nf_mlp *m, const float *x, int64_t xf, int64_t xj, float *y, int64_t yo, int64_t yj, int64_t n,
                 hipStream_t s) {
    if (n < 1) return hipSuccess;
    const Infer g{m->pb, m->p, m->norm, x, xf, xj, y, yo, yj, n};
    // 64 samples per block share one read of the weights and activations
    // (one block's latency 12.4 us up to 2 blocks per CU), 16 per block are
    // done in 6.0 us while at most about 3 of them share a CU: 9.2 against
    // 12.5 us at 8,192 samples, 16.5 against 12.5 us at 16,384
    if (n > NC1_MAX) hipLaunchKernelGGL((k_infer<4, 2>), dim3((unsigned)std::min<int64_t>((n + 63) / 64, 512)), dim3(256), 0, s, g);
    else hipLaunchKernelGGL((k_infer<1, 1>), dim3((unsigned)((n + 15) / 16)), dim3(512), 0, s, g);
    return hipGetLastError();
}

// loss partials and gradient partials of n samples: first + j, or idx[first + j]
hipError_t gradients(nf_mlp *m, const int64_t *idx, int64_t first, int n, hipStream_t s) {
    const int ld = (n + 63) / 64 * 64, splits = (n + KSPLIT - 1) / KSPLIT;
    Train t{m->pb, m->pt, m->p, m->norm, m->dx, m->dy, idx, first, n, ld, 1.0f / ((float)OUT * (float)n), m->X0,
            {}, {}, m->dYb, {}, m->dY, m->se};
    Wgrad g{m->X0, {}, {}, m->dYb, {}, m->dY, m->se, n, ld, splits, m->part, m->g, m->loss_part};
    for (int l = 0; l < 3; ++l) {
        g.A[l] = t.A[l] = m->A[l];
        g.dZb[l] = t.dZb[l] = m->dZb[l];
        g.dZ[l] = t.dZ[l] = m->dZ[l];
    }
    hipLaunchKernelGGL(k_train, dim3(std::min(ld / 16, 256)), dim3(512), 0, s, t);
    hipError_t e = hipGetLastError();
    if (e) return e;
    hipLaunchKernelGGL(k_wgrad, dim3(wgrad_blocks(splits) + 3 * HID + OUT + (n + 255) / 256), dim3(256), 0, s, g);
    return hipGetLastError();
}

// gradient from its partials; lr_t, o: an Adam step too
template <bool ADAM>
hipError_t update(nf_mlp *m, int n, hipStream_t s, float lr_t, const nf_train_opts *o) {
    Update u{m->part, (n + KSPLIT - 1) / KSPLIT, m->g, m->p, m->m, m->v, m->pb, m->pt, lr_t, 0.f, 0.f, 0.f};
    if (o) u.b1 = o->beta1, u.b2 = o->beta2, u.eps = o->eps;
    hipLaunchKernelGGL(k_update<ADAM>, dim3((NPARAM + 255) / 256), dim3(256), 0, s, u);
    return hipGetLastError();
}

float sum_loss(nf_mlp *m, int n) {
    const int nb = (n + 255) / 256;
    std::vector<float> h(nb);
    if (hipMemcpy(h.data(), m->loss_part, nb * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) return NAN;
    double s = 0;
    for (float x : h) s += x;
    return (float)(s / ((double)OUT * n));
}

int upload_norm(nf_mlp *mm) {
    float h[27];
    std::memcpy(h, mm->hnorm, 22 * sizeof(float));
    for (int o = 0; o < OUT; ++o) h[22 + o] = 1.0f / mm->hnorm[17 + o];
    HIPM(hipMemcpy(mm->norm, h, sizeof h, hipMemcpyHostToDevice));
    return NF_OK;
}

// room for n samples in the data buffers (allocates only when n grows)
int ensure_data(nf_mlp *mm, int64_t n) {
    if (n <= mm->data_cap) return NF_OK;
    HIPM(hipStreamSynchronize(mm->stream));
    for (void *q : {(void *)mm->dx, (void *)mm->dy, (void *)mm->didx})
        if (q) HIPM(hipFree(q));
    mm->dx = mm->dy = nullptr;
    mm->didx = nullptr;
    mm->data_cap = 0;
    const int64_t cap = (n + 255) / 256 * 256;
    HIPM(hipMalloc(&mm->dx, (size_t)IN * cap * sizeof(float)));
    HIPM(hipMalloc(&mm->dy, (size_t)OUT * cap * sizeof(float)));
    HIPM(hipMalloc(&mm->didx, (size_t)cap * sizeof(int64_t)));
    mm->data_cap = cap;
    return NF_OK;
}

// the caller's samples and targets, as they are
int upload_data(nf_mlp *mm, const float *x, const float *y, int64_t n) {
    HIPM(mm->pipe.up(mm->dx, x, (size_t)IN * n * sizeof(float), mm->stream));
    HIPM(mm->pipe.up(mm->dy, y, (size_t)OUT * n * sizeof(float), mm->stream));
    return NF_OK;
}

}  // namespace

namespace nf {
namespace mlp {

hipError_t predict_device(nf_mlp *m, const float *x, int64_t n, float *y, hipStream_t s) {
    return infer(m, x, n, 1, y, n, 1, n, s);
}

}  // namespace mlp
}  // namespace nf

// ============================================================================
extern "C" {

int64_t nf_mlp_n_params(void) { return NPARAM; }

int nf_mlp_predict_noalloc(nf_mlp *mm, const float *x, int64_t n, float *y, void *stream) {
    if (!mm || !x || !y || n < 0) return NF_E_ARG;
    if (n > NOALLOC_MAX)
        return fail(mm, NF_E_ARG,
                    "nf_mlp_predict_noalloc: " + std::to_string(n) + " samples exceed the maximum of " +
                        std::to_string(NOALLOC_MAX) + " per call");
    if (n == 0) return NF_OK;
    int dev = -1;
    HIPM(hipGetDevice(&dev));
    if (dev != mm->device)
        return fail(mm, NF_E_ARG, "nf_mlp_predict_noalloc: the network's device must be current");
    const hipStream_t s = stream ? static_cast<hipStream_t>(stream) : mm->stream;
    // y over x: a block's outputs would replace inputs that another block has
    // not read yet
    const uintptr_t xa = reinterpret_cast<uintptr_t>(x), ya = reinterpret_cast<uintptr_t>(y);
    if (xa < ya + OUT * n * sizeof(float) && ya < xa + IN * n * sizeof(float)) {
        hipLaunchKernelGGL(k_copy, dim3((unsigned)((IN * n + 255) / 256)), dim3(256), 0, s, x, mm->xcopy, (int)(IN * n));
        HIPM(hipGetLastError());
        x = mm->xcopy;
    }
    HIPM(infer(mm, x, 1, IN, y, 1, OUT, n, s));
    return NF_OK;
}

int nf_mlp_create(uint64_t seed, nf_mlp **out) {
    if (!out) return NF_E_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return NF_E_NOGPU;
    struct Destroy {  // (where the creation fails)
        void operator()(nf_mlp *m) const { (void)nf_mlp_destroy(m); }
    };
    std::unique_ptr<nf_mlp, Destroy> hold(new nf_mlp);
    nf_mlp *mm = hold.get();
    HIPM(hipGetDevice(&mm->device));
    HIPM(hipStreamCreateWithFlags(&mm->stream, hipStreamNonBlocking));
    // one allocation; the moments and pt, which start at zero, side by side
    constexpr size_t ROW = (NPARAM * sizeof(float) + 255) & ~(size_t)255, TR = (NPT * sizeof(__bf16) + 255) & ~(size_t)255;
    char *base = nullptr;
    HIPM(hipMalloc(&base, 5 * ROW + TR + (32 + IN * NOALLOC_MAX) * sizeof(float)));
    mm->p = reinterpret_cast<float *>(base);  // (the one that is freed)
    mm->g = reinterpret_cast<float *>(base + ROW);
    mm->m = reinterpret_cast<float *>(base + 2 * ROW);
    mm->v = reinterpret_cast<float *>(base + 3 * ROW);
    mm->pt = reinterpret_cast<__bf16 *>(base + 4 * ROW);
    mm->pb = reinterpret_cast<__bf16 *>(base + 4 * ROW + TR);
    mm->norm = reinterpret_cast<float *>(base + 5 * ROW + TR);
    mm->xcopy = mm->norm + 32;
    HIPM(hipMemset(mm->pt, 0, NPT * sizeof(__bf16)));
    // uniform(+-1/sqrt(fan_in)) weights and biases, a linear layer's default
    std::mt19937_64 rng(seed);
    std::vector<float> h(NPARAM);
    auto fill = [&](int64_t off, int64_t cnt, int fan_in) {
        std::uniform_real_distribution<float> U(-1.0f / std::sqrt((float)fan_in), 1.0f / std::sqrt((float)fan_in));
        for (int64_t i = 0; i < cnt; ++i) h[off + i] = U(rng);
    };
    fill(OFF_W1, HID * IN + HID, IN);
    fill(OFF_W2, HID * HID + HID, HID);
    fill(OFF_W3, HID * HID + HID, HID);
    fill(OFF_W4, OUT * HID + OUT, HID);
    int rc = nf_mlp_set_params(mm, h.data());
    if (rc) return rc;
    for (int f = 0; f < 6; ++f) mm->hnorm[6 + f] = 1.0f;
    for (int o = 0; o < 5; ++o) mm->hnorm[17 + o] = 1.0f;
    if ((rc = upload_norm(mm))) return rc;
    *out = hold.release();
    return NF_OK;
}

int nf_mlp_destroy(nf_mlp *mm) {
    if (!mm) return NF_OK;
    if (mm->stream) (void)hipStreamSynchronize(mm->stream);
    for (void *q : mm->ws) (void)hipFree(q);
    for (void *q : {(void *)mm->p, (void *)mm->dx, (void *)mm->dy, (void *)mm->didx})
        if (q) (void)hipFree(q);
    if (mm->stream) (void)hipStreamDestroy(mm->stream);
    delete mm;
    return NF_OK;
}

const char *nf_mlp_last_error(const nf_mlp *m) { return m ? m->err.c_str() : "null network"; }

int nf_mlp_get_params(nf_mlp *mm, float *params) {
    if (!mm || !params) return NF_E_ARG;
    HIPM(hipStreamSynchronize(mm->stream));
    HIPM(hipMemcpy(params, mm->p, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
    return NF_OK;
}

int nf_mlp_set_params(nf_mlp *mm, const float *params) {
    if (!mm || !params) return NF_E_ARG;
    HIPM(hipStreamSynchronize(mm->stream));
    HIPM(hipMemcpy(mm->p, params, NPARAM * sizeof(float), hipMemcpyHostToDevice));
    HIPM(hipMemset(mm->m, 0, (mm->v - mm->m + NPARAM) * sizeof(float)));  // both moments
    mm->adam_t = 0;
    hipLaunchKernelGGL(k_to_bf16, dim3((NPARAM + 255) / 256), dim3(256), 0, mm->stream, (const float *)mm->p, mm->pb,
                       mm->pt);
    HIPM(hipGetLastError());
    HIPM(hipStreamSynchronize(mm->stream));
    return NF_OK;
}

int nf_mlp_set_norm(nf_mlp *mm, const float *in_shift, const float *in_scale, const float *out_shift,
                    const float *out_scale) {
    if (!mm || !in_shift || !in_scale || !out_shift || !out_scale) return NF_E_ARG;
    for (int o = 0; o < OUT; ++o)
        if (!(out_scale[o] != 0.0f)) return NF_E_ARG;
    std::memcpy(mm->hnorm, in_shift, 6 * sizeof(float));
    std::memcpy(mm->hnorm + 6, in_scale, 6 * sizeof(float));
    std::memcpy(mm->hnorm + 12, out_shift, 5 * sizeof(float));
    std::memcpy(mm->hnorm + 17, out_scale, 5 * sizeof(float));
    mm->norm_set = true;
    return upload_norm(mm);
}

int nf_mlp_get_norm(nf_mlp *mm, float *in_shift, float *in_scale, float *out_shift, float *out_scale) {
    if (!mm || !in_shift || !in_scale || !out_shift || !out_scale) return NF_E_ARG;
    std::memcpy(in_shift, mm->hnorm, 6 * sizeof(float));
    std::memcpy(in_scale, mm->hnorm + 6, 6 * sizeof(float));
    std::memcpy(out_shift, mm->hnorm + 12, 5 * sizeof(float));
    std::memcpy(out_scale, mm->hnorm + 17, 5 * sizeof(float));
    return NF_OK;
}

int nf_mlp_predict(nf_mlp *mm, const float *x, int64_t n, float *y) {
    if (!mm || !x || !y || n < 0) return NF_E_ARG;
    if (n == 0) return NF_OK;
    int rc;
    // both arrays cross as they are ([n][6], [n][5]): the kernel reads samples
    if ((rc = ensure_data(mm, n))) return rc;
    HIPM(mm->pipe.up(mm->dx, x, (size_t)IN * n * sizeof(float), mm->stream));
    HIPM(infer(mm, mm->dx, 1, IN, mm->dy, 1, OUT, n, mm->stream));
    HIPM(mm->pipe.down(y, mm->dy, (size_t)OUT * n * sizeof(float), mm->stream));
    return NF_OK;
}

// loss and gradient of one batch; x [n][6], y [n][5] raw host arrays
int nf_mlp_loss_grad(nf_mlp *mm, const float *x, const float *y, int64_t n, float *loss, float *grad) {
    if (!mm || !x || !y || n < 1 || n > (1 << 20)) return NF_E_ARG;
    int rc;
    if ((rc = ensure_ws(mm, (int)n)) || (rc = ensure_data(mm, n))) return rc;
    if ((rc = upload_data(mm, x, y, n))) return rc;
    const int c = (int)n;
    hipError_t e = gradients(mm, nullptr, 0, c, mm->stream);
    if (!e) e = update<false>(mm, c, mm->stream, 0.f, nullptr);
    if (!e) e = hipStreamSynchronize(mm->stream);
    if (e != hipSuccess) return fail(mm, NF_E_HIP, std::string("loss_grad: ") + hipGetErrorString(e));
    if (loss) *loss = sum_loss(mm, c);
    if (grad) HIPM(hipMemcpy(grad, mm->g, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
    return NF_OK;
}

// Adam over shuffled minibatches of the whole set; x [n][6], y [n][5] raw
// host arrays.  Normalisation: if never set, mean/std of the data.
int nf_mlp_train(nf_mlp *mm, const float *x, const float *y, int64_t n, const nf_train_opts *o,
                 nf_train_stats *st) {
    if (!mm || !x || !y || !o || o->batch < 256 || o->batch % 256 || o->epochs < 0 || n < 256) return NF_E_ARG;
    int rc;
    const int B = (int)std::min<int64_t>(o->batch, n / 256 * 256);
    if ((rc = ensure_ws(mm, B))) return rc;
    if (!mm->norm_set) {
        // per-component mean and standard deviation of the training data
        for (int f = 0; f < IN + OUT; ++f) {
            double s = 0, s2 = 0;
            for (int64_t j = 0; j < n; ++j) {
                const double v = f < IN ? x[j * IN + f] : y[j * OUT + (f - IN)];
                s += v;
                s2 += v * v;
            }
            const double mean = s / n, sd = std::sqrt(std::max(0.0, s2 / n - mean * mean));
            if (f < IN) {
                mm->hnorm[f] = (float)mean;
                mm->hnorm[6 + f] = sd > 0 ? (float)(1.0 / sd) : 1.0f;
            } else {
                mm->hnorm[12 + f - IN] = (float)mean;
                mm->hnorm[17 + f - IN] = sd > 0 ? (float)sd : 1.0f;
            }
        }
        if ((rc = upload_norm(mm))) return rc;
        mm->norm_set = true;
    }
    if ((rc = ensure_data(mm, n))) return rc;
    if ((rc = upload_data(mm, x, y, n))) return rc;
    int64_t *didx = mm->didx;
    std::vector<int64_t> idx(n);
    for (int64_t j = 0; j < n; ++j) idx[j] = j;
    std::mt19937_64 rng(o->seed);
    hipEvent_t e0, e1;
    HIPM(hipEventCreate(&e0));
    HIPM(hipEventCreate(&e1));
    HIPM(hipEventRecord(e0, mm->stream));
    const int64_t per_epoch = n / B;
    float first = NAN, last = NAN;
    int64_t steps = 0;
    hipError_t e = hipSuccess;
    for (int ep = 0; ep < o->epochs && !e; ++ep) {
        std::shuffle(idx.begin(), idx.end(), rng);
        e = hipStreamSynchronize(mm->stream);  // the previous epoch still reads didx
        if (!e) e = hipMemcpy(didx, idx.data(), n * sizeof(int64_t), hipMemcpyHostToDevice);
        const float lr = o->lr * std::pow(o->lr_decay > 0 ? o->lr_decay : 1.0f, (float)ep);
        double ep_loss = 0;
        for (int64_t q = 0; q < per_epoch && !e; ++q) {
            e = gradients(mm, didx, q * B, B, mm->stream);
            if (e) break;
            ++mm->adam_t;
            const double bc1 = 1.0 - std::pow((double)o->beta1, (double)mm->adam_t);
            const double bc2 = 1.0 - std::pow((double)o->beta2, (double)mm->adam_t);
            e = update<true>(mm, B, mm->stream, (float)(lr * std::sqrt(bc2) / bc1), o);
            ++steps;
            if (q == 0 || q == per_epoch - 1) {
                if (!e) e = hipStreamSynchronize(mm->stream);
                const float l = e ? NAN : sum_loss(mm, B);
                if (ep == 0 && q == 0) first = l;
                ep_loss = l;
            }
        }
        last = (float)ep_loss;
    }
    if (!e) e = hipEventRecord(e1, mm->stream);
    if (!e) e = hipEventSynchronize(e1);
    float ms = 0;
    if (!e) (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (e != hipSuccess) return fail(mm, NF_E_HIP, std::string("train: ") + hipGetErrorString(e));
    if (st) {
        st->loss_first = first;
        st->loss_last = last;
        st->steps = steps;
        st->elapsed_ms = ms;
    }
    return NF_OK;
}

}  // extern "C"
