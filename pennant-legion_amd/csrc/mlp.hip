// The learned QCS closure's network on the device: parameters, BF16 MFMA
// kernels for training (forward, backward, Adam) and batched inference.
//
// Training step on a minibatch of B tuples (BF16 operands, FP32 accumulation;
// H1, H2 and the gradients fed to the next product are rounded to BF16 where
// the MFMA consumes them):
//   Z1 = X W1^T          H1 = relu(Z1)
//   Z2 = H1 W2^T + b2    H2 = relu(Z2)
//   Y  = H2 W3^T + b3    loss = sum_b sum_o (Y - T)^2 / B
//   dY = 2 (Y - T) / B
//   dW3 = dY^T H2   db3 = colsum dY    dZ2 = (dY W3) * [H2 > 0]
//   dW2 = dZ2^T H1  db2 = colsum dZ2   dZ1 = (dZ2 W2) * [H1 > 0]
//   dW1 = dZ1^T X   (column 10 of X is 1, so dW1[:,10] is the bias gradient)
// Three launches a step: k_rows (a wave takes 32 rows through forward and
// backward in registers), k_grads (the weight gradients over the batch, bias
// and loss sums), k_update (sums of the partials, Adam, the BF16 copies).
// Every reduction runs in a fixed order (split-K partials summed in order), so
// training is deterministic.
//
// What bounds a step at B = 8192 is latency: k_rows 9.0 us (the row list over
// PCIe, the gathered tuples, a chain of 26 products), k_grads 10.8 us (eight
// rounds of loads of what other XCDs have just written; loading twice or four
// times as far ahead changed nothing), k_update 5.4 us, and the host's draw of
// the next step's rows, 30 us, beside them: 32 us a step.  One kernel per
// product and elementwise step (22 launches, 112 us of kernels, drawing while
// the GPU waited) took 262 us.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "closure.h"
#include "common.h"

using namespace pn;

struct pennant_mlp {
    float* p = nullptr;        // FP32 master parameters (PN_MLP_NPARAM)
    float* g = nullptr;        // gradient
    float* m = nullptr;        // Adam moments
    float* v = nullptr;
    __bf16* w1b = nullptr;     // BF16 copies, row-major [out][in]
    __bf16* w2b = nullptr;
    __bf16* w2t = nullptr;     // W2 transposed, [in][out]
    __bf16* w3b = nullptr;
    ClosurePack* pack = nullptr;
    float lo[PN_MLP_NF], hi[PN_MLP_NF];
    int adam_t = 0;
    // batch buffers (capacity cap rows, a multiple of 32): per unit a row of
    // the batch's values
    int64_t cap = 0;
    int* idx_host[2] = {};     // pinned: the rows of a step, read by the kernel
    hipEvent_t read[2] = {};   // when they have been read
    __bf16 *xt = nullptr, *h1t = nullptr, *h2t = nullptr, *dyt = nullptr, *dz2t = nullptr, *dz1t = nullptr;
    float *lrow = nullptr, *lossp = nullptr;
    float* part = nullptr;     // split-K partials
    float* losses = nullptr;   // per step
    int loss_cap = 0;
    hipStream_t stream = nullptr;
    std::string err;
};

namespace {

#define MCK(x) do { const int e_ = (int)(x); if (e_ != 0) return e_; } while (0)

// ---------------------------------------------------------------------------
// A wave's rows through the network.
//
// The products are taken as C^T = W act^T, so that a lane's accumulator
// holds one batch row (lane % 32) and the units 8 (q / 4) + 4 (lane / 32) + q
// % 4 of register q.  The next product wants, per 16 units, units 0-7 in the
// low half of the wave and 8-15 in the high half: one swap of the halves per
// register pair, and no pass through LDS.  Within an MFMA the units stay in
// order, so a result does not depend on how the rows are spread over waves.

// Units 16 c .. 16 c + 15 of an accumulator pair (already rounded: packed
// pairs of registers), as the B operand of the next product.
__device__ __forceinline__ bf16x8 next_operand(const unsigned (&v)[2][8], int c) {
    const unsigned* a = &v[c >> 1][4 * (c & 1)];
    u32x4 o;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        const auto r = __builtin_amdgcn_permlane32_swap(a[d], a[2 + d], false, false);
        o[d] = r[0];
        o[2 + d] = r[1];
    }
    return as_bf16x8(o);
}
__device__ __forceinline__ float bf_lo(unsigned v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf_hi(unsigned v) { return __uint_as_float(v & 0xffff0000u); }

// relu(a), relu(b) as a BF16 pair.  max(z, 0) is the number where z is a NaN
// (relu_bf16, on the rounded bits, keeps a NaN whose sign bit is clear): a unit
// with a NaN bias or input is off in every row.
__device__ __forceinline__ unsigned relu_max(float a, float b) { return pack_bf16(fmaxf(a, 0.f), fmaxf(b, 0.f)); }

// Register pairs (2 d, 2 d + 1) of an accumulator to rows [unit][b] of dst.
__device__ __forceinline__ void store_units(const unsigned (&v)[2][8], __bf16* dst, int64_t ld, int64_t b, int h) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const int64_t u = 32 * mb + 8 * (d >> 1) + 4 * h + 2 * (d & 1);
            unsigned short* o = reinterpret_cast<unsigned short*>(dst) + u * ld + b;
            o[0] = (unsigned short)v[mb][d];
            o[ld] = (unsigned short)(v[mb][d] >> 16);
        }
}

typedef float f32x2a __attribute__((ext_vector_type(2), aligned(4)));

struct RowArgs {
    const float* p;
    const __bf16 *w1b, *w2b, *w2t, *w3b;
    int64_t n;                 // rows
    const float* x;            // rows of 10 features, or tuples
    const int* idx;            // training: the tuple of row b (NULL: tuple b)
    float* y;                  // inference: n x 2
    int64_t ld;                // training: row length of the buffers below
    __bf16 *xt, *h1t, *h2t, *dyt, *dz2t, *dz1t;
    float* lrow;
};

// 32 rows a wave: forward, and with TRAIN the loss of each row and its
// backward values; rows past n give zeros.
template <bool TRAIN>
__global__ void __launch_bounds__(64) k_rows(RowArgs a) {
    const int lane = threadIdx.x, h = lane >> 5, r = lane & 31;
    const int64_t b = (int64_t)blockIdx.x * 32 + r;
    const bool in = b < a.n;
    const int64_t bc = in ? b : a.n - 1;
    const float* row = TRAIN ? a.x + (a.idx ? (int64_t)a.idx[bc] : bc) * PN_MLP_TUPLE : a.x + bc * PN_MLP_NF;
    // the row's inputs 8 h .. 8 h + 7 (10: the bias slot, 11-15: zeros), and
    // its targets in the low half
    f32x2a f[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = *reinterpret_cast<const f32x2a*>(row + (h ? 8 : 2 * k));
    f32x2a t = {0.f, 0.f};
    if constexpr (TRAIN) t = *reinterpret_cast<const f32x2a*>(row + PN_MLP_NF);
    bf16x8 w1[2], w2[2][4];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        w1[mb] = *reinterpret_cast<const bf16x8*>(a.w1b + (32 * mb + r) * PN_MLP_K1 + 8 * h);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            w2[mb][c] = *reinterpret_cast<const bf16x8*>(a.w2b + (32 * mb + r) * PN_MLP_NH + 16 * c + 8 * h);
    }
    u32x4 xv;
    xv[0] = pack_bf16(f[0][0], f[0][1]);
    xv[1] = h ? pack_bf16(1.f, 0.f) : pack_bf16(f[1][0], f[1][1]);
    xv[2] = h ? 0u : pack_bf16(f[2][0], f[2][1]);
    xv[3] = h ? 0u : pack_bf16(f[3][0], f[3][1]);
    if (!in) xv = u32x4{0u, 0u, 0u, 0u};
    const bf16x8 x = as_bf16x8(xv);
    // layer 1
    unsigned h1[2][8], h2[2][8];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        const f32x16 zero = {};
        const f32x16 z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1[mb], x, zero, 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 8; ++d) h1[mb][d] = relu_max(z[2 * d], z[2 * d + 1]);
    }
    // layer 2
    bf16x8 act[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) act[c] = next_operand(h1, c);
    const float* b2 = a.p + PN_MLP_OFF_B2;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        f32x16 z = {};
#pragma unroll
        for (int c = 0; c < 4; ++c) z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w2[mb][c], act[c], z, 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const float* bu = b2 + 32 * mb + 8 * (d >> 1) + 4 * h + 2 * (d & 1);
            const unsigned v = relu_max(z[2 * d] + bu[0], z[2 * d + 1] + bu[1]);
            h2[mb][d] = in ? v : 0u;
        }
    }
    // output layer: rows 0 and 1 of W3, the others zero
    f32x16 z3 = {};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const bf16x8 zero8 = {};
        const bf16x8 w = r < PN_MLP_NO
                             ? *reinterpret_cast<const bf16x8*>(a.w3b + r * PN_MLP_NH + 16 * c + 8 * h)
                             : zero8;
        z3 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, next_operand(h2, c), z3, 0, 0, 0);
    }
    // the outputs of row r are in its low lane
    const float y0 = z3[0] + a.p[PN_MLP_OFF_B3], y1 = z3[1] + a.p[PN_MLP_OFF_B3 + 1];
    if constexpr (!TRAIN) {
        if (in && !h) {
            const f32x2a y = {y0, y1};
            *reinterpret_cast<f32x2a*>(a.y + 2 * b) = y;
        }
        return;
    }
    const float d0 = y0 - t[0], d1 = y1 - t[1];
    const float inv = 2.f / (float)a.n;
    const unsigned dy = (in && !h) ? pack_bf16(inv * d0, inv * d1) : 0u;
    if (!h) {
        a.lrow[b] = in ? d0 * d0 + d1 * d1 : 0.f;
        unsigned short* o = reinterpret_cast<unsigned short*>(a.dyt) + b;
        o[0] = (unsigned short)dy;
        o[a.ld] = (unsigned short)(dy >> 16);
    }
    {
        unsigned short* o = reinterpret_cast<unsigned short*>(a.xt) + (int64_t)(8 * h) * a.ld + b;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            o[(2 * k) * a.ld] = (unsigned short)xv[k];
            o[(2 * k + 1) * a.ld] = (unsigned short)(xv[k] >> 16);
        }
    }
    store_units(h1, a.h1t, a.ld, b, h);
    store_units(h2, a.h2t, a.ld, b, h);
    // dZ2 = (dY W3) [H2 > 0]: two of the product's 16 inputs
    u32x4 dyv = {dy, 0u, 0u, 0u};
    unsigned g2[2][8], g1[2][8];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        const unsigned short* w = reinterpret_cast<const unsigned short*>(a.w3b) + 32 * mb + r;
        const u32x4 wv = {h ? 0u : ((unsigned)w[0] | ((unsigned)w[PN_MLP_NH] << 16)), 0u, 0u, 0u};
        const f32x16 zero = {};
        const f32x16 z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(wv), as_bf16x8(dyv), zero, 0, 0, 0);
#pragma unroll
        for (int d = 0; d < 8; ++d)
            g2[mb][d] = pack_bf16(bf_lo(h2[mb][d]) > 0.f ? z[2 * d] : 0.f, bf_hi(h2[mb][d]) > 0.f ? z[2 * d + 1] : 0.f);
    }
    store_units(g2, a.dz2t, a.ld, b, h);
    // dZ1 = (dZ2 W2) [H1 > 0]
#pragma unroll
    for (int c = 0; c < 4; ++c) act[c] = next_operand(g2, c);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        f32x16 z = {};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bf16x8 w = *reinterpret_cast<const bf16x8*>(a.w2t + (32 * mb + r) * PN_MLP_NH + 16 * c + 8 * h);
            z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, act[c], z, 0, 0, 0);
        }
#pragma unroll
        for (int d = 0; d < 8; ++d)
            g1[mb][d] = pack_bf16(bf_lo(h1[mb][d]) > 0.f ? z[2 * d] : 0.f, bf_hi(h1[mb][d]) > 0.f ? z[2 * d + 1] : 0.f);
    }
    store_units(g1, a.dz1t, a.ld, b, h);
}

// ---------------------------------------------------------------------------
// The gradients over the batch.  Long reductions are split into ranges of kper
// rows (about 512, at most 64 ranges); a wave takes one 32 x 32 tile of one
// gradient and one range, and its partial goes to part[range] (in the flat
// parameter layout).  Blocks after those sum the columns of dY and dZ2 (the
// bias gradients) and the rows' losses, 256 at a time.
struct GradArgs {
    int64_t rows, ld;
    int kper, ksplit;
    const __bf16 *xt, *h1t, *h2t, *dyt, *dz2t, *dz1t;
    const float* lrow;
    float* part;               // ksplit x PN_MLP_NPARAM
    float* g;
    float* lossp;              // per 256 rows
};
#define PN_GTILES 8            // dW2: 2 x 2, dW1: 2 x 1, dW3: 1 x 2

// The block's sum of v in a fixed tree; thread 0 has it.
__device__ __forceinline__ float tree256(float v) {
    __shared__ float sh[256];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
        __syncthreads();
    }
    return sh[0];
}

__global__ void __launch_bounds__(256) k_grads(GradArgs a) {
    const int gblocks = a.ksplit * PN_GTILES / 4;
    int blk = blockIdx.x;
    if (blk < gblocks) {
        const int item = blk * 4 + (threadIdx.x >> 6);
        const int tile = item & (PN_GTILES - 1), range = item / PN_GTILES;
        const int lane = threadIdx.x & 63, h = lane >> 5, r = lane & 31;
        // gradient C[i][j] = sum_b A[i][b] B[j][b]
        const __bf16 *A, *B;
        int i0 = 0, j0 = 0, M = 64, N = 64, off;
        if (tile < 4) {
            A = a.dz2t; B = a.h1t; off = PN_MLP_OFF_W2; i0 = 32 * (tile >> 1); j0 = 32 * (tile & 1);
        } else if (tile < 6) {
            A = a.dz1t; B = a.xt; off = PN_MLP_OFF_W1; i0 = 32 * (tile & 1); N = PN_MLP_K1;
        } else {
            A = a.dyt; B = a.h2t; off = PN_MLP_OFF_W3; j0 = 32 * (tile & 1); M = PN_MLP_NO;
        }
        const bool ain = i0 + r < M, bin = j0 + r < N;
        const __bf16* pa = A + (int64_t)(ain ? i0 + r : 0) * a.ld + 8 * h;
        const __bf16* pb = B + (int64_t)(bin ? j0 + r : 0) * a.ld + 8 * h;
        const bf16x8 zero8 = {};
        const int64_t kb = (int64_t)range * a.kper;
        const int64_t ke = kb + a.kper < a.rows ? kb + a.kper : a.rows;
        f32x16 acc = {};
        // rows past the batch hold zeros up to the next multiple of 32; four
        // products' operands are loaded before the first is used
        constexpr int AHEAD = 4;
        for (int64_t k0 = kb; k0 < ke; k0 += 16 * AHEAD) {
            bf16x8 va[AHEAD], vb[AHEAD];
#pragma unroll
            for (int s = 0; s < AHEAD; ++s) {
                const int64_t k = k0 + 16 * s < ke ? k0 + 16 * s : kb;
                va[s] = *reinterpret_cast<const bf16x8*>(pa + k);
                vb[s] = *reinterpret_cast<const bf16x8*>(pb + k);
            }
#pragma unroll
            for (int s = 0; s < AHEAD; ++s)
                if (k0 + 16 * s < ke)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ain ? va[s] : zero8, bin ? vb[s] : zero8, acc, 0, 0, 0);
        }
        float* C = a.part + (int64_t)range * PN_MLP_NPARAM + off;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int ci = i0 + 8 * (q >> 2) + 4 * h + (q & 3), cj = j0 + r;
            if (ci < M && cj < N) C[ci * N + cj] = acc[q];
        }
        return;
    }
    blk -= gblocks;
    if (blk < PN_MLP_NO + PN_MLP_NH) {
        const __bf16* col = blk < PN_MLP_NO ? a.dyt + blk * a.ld : a.dz2t + (blk - PN_MLP_NO) * a.ld;
        float s = 0.f;
#pragma unroll 8
        for (int64_t b = threadIdx.x; b < a.rows; b += 256) s += (float)col[b];
        s = tree256(s);
        if (threadIdx.x == 0) a.g[blk < PN_MLP_NO ? PN_MLP_OFF_B3 + blk : PN_MLP_OFF_B2 + blk - PN_MLP_NO] = s;
        return;
    }
    blk -= PN_MLP_NO + PN_MLP_NH;
    const int64_t b = (int64_t)blk * 256 + threadIdx.x;
    const float s = tree256(b < a.rows ? a.lrow[b] : 0.f);
    if (threadIdx.x == 0) a.lossp[blk] = s;
}

// ---------------------------------------------------------------------------
// Where a parameter's BF16 copies live: the row-major ones and the A-operand
// pack of the fused inference (ClosurePack).
__device__ __forceinline__ void put_param(int i, float v, __bf16* w1b, __bf16* w2b, __bf16* w2t, __bf16* w3b,
                                          ClosurePack* pk) {
    const __bf16 e = (__bf16)v;
    __bf16* q = nullptr;
    if (i < PN_MLP_OFF_W2) {
        const int row = i / PN_MLP_K1, k = i % PN_MLP_K1;
        w1b[i] = e;
        q = reinterpret_cast<__bf16*>(&pk->w1[row >> 5][(row & 31) + 32 * (k >> 3)]) + (k & 7);
    } else if (i < PN_MLP_OFF_B2) {
        const int j = i - PN_MLP_OFF_W2, row = j / PN_MLP_NH, k = j % PN_MLP_NH, kk = k & 15;
        w2b[j] = e;
        w2t[k * PN_MLP_NH + row] = e;
        q = reinterpret_cast<__bf16*>(&pk->w2[row >> 5][k >> 4][(row & 31) + 32 * ((kk >> 2) & 1)]) + 4 * (kk >> 3) + (kk & 3);
    } else if (i < PN_MLP_OFF_W3) {
        const int u = i - PN_MLP_OFF_B2, w = u & 31;
        pk->b2c[u >> 5][(w >> 2) & 1][4 * (w >> 3) + (w & 3)] = v;
        return;
    } else if (i < PN_MLP_OFF_B3) {
        const int j = i - PN_MLP_OFF_W3, row = j / PN_MLP_NH, k = j % PN_MLP_NH, kk = k & 15;
        w3b[j] = e;
        q = reinterpret_cast<__bf16*>(&pk->w3[k >> 4][row + 32 * ((kk >> 2) & 1)]) + 4 * (kk >> 3) + (kk & 3);
    } else {
        pk->b3[i - PN_MLP_OFF_B3] = v;
        return;
    }
    *q = e;
}

struct UpdateArgs {
    int ksplit, nloss;
    const float* part;
    const float* lossp;
    float* g;
    float* loss;
    // Adam (ADAM)
    float *p, *m, *v;
    float lr, b1, b2, eps, c1, c2;
    __bf16 *w1b, *w2b, *w2t, *w3b;
    ClosurePack* pack;
};

// One thread a parameter: its gradient (the ranges' partials summed in order)
// and with ADAM its bias-corrected update and BF16 copies; one thread more
// sums the loss.
template <bool ADAM>
__global__ void __launch_bounds__(256) k_update(UpdateArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i == PN_MLP_NPARAM) {
        float s = 0.f;
        for (int k = 0; k < a.nloss; ++k) s += a.lossp[k];
        *a.loss = s;
    }
    if (i >= PN_MLP_NPARAM) return;
    float gi;
    if ((i >= PN_MLP_OFF_B2 && i < PN_MLP_OFF_W3) || i >= PN_MLP_OFF_B3) {
        gi = a.g[i];
    } else {
        gi = a.part[i];
#pragma unroll 16
        for (int z = 1; z < a.ksplit; ++z) gi += a.part[(int64_t)z * PN_MLP_NPARAM + i];
        a.g[i] = gi;
    }
    if constexpr (ADAM) {
        if (i < PN_MLP_OFF_W2 && (i % PN_MLP_K1) > PN_MLP_NF) return;   // these inputs are zero
        const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gi;
        const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gi * gi;
        a.m[i] = mi;
        a.v[i] = vi;
        const float pi = a.p[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
        a.p[i] = pi;
        put_param(i, pi, a.w1b, a.w2b, a.w2t, a.w3b, a.pack);
    }
}

// Every parameter's BF16 copies, and zeros where the output layer's pack has
// no row.
__global__ void __launch_bounds__(256) k_pack(const float* __restrict__ p, __bf16* w1b, __bf16* w2b, __bf16* w2t,
                                              __bf16* w3b, ClosurePack* pk) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < PN_MLP_NPARAM) put_param(i, p[i], w1b, w2b, w2t, w3b, pk);
    if (i < 4 * 64 && (i & 31) >= PN_MLP_NO) {
        const bf16x8 zero = {};
        pk->w3[i >> 6][i & 63] = zero;
    }
}

// Batched inference through the same wave routine the fused predictor uses:
// each lane packs one row of x (n x 10) and receives its two outputs.  Every
// lane of a wave takes part (rows past n are evaluated on zero features and
// discarded).
__global__ void __launch_bounds__(256) k_mlp_wave(const ClosurePack* __restrict__ pk, int64_t n,
                                                  const float* __restrict__ x, float* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool valid = i < n;
    float f[PN_MLP_NF];
#pragma unroll
    for (int k = 0; k < PN_MLP_NF; ++k) f[k] = valid ? x[i * PN_MLP_NF + k] : 0.f;
    u32x4 lo, hi;
    pack_features(f, lo, hi);
    const uint64_t need = __ballot(valid);
    float y0, y1;
    mlp_wave(pk, lo, hi, (uint32_t)need != 0u, (need >> 32) != 0u, y0, y1);
    if (valid) {
        y[2 * i] = y0;
        y[2 * i + 1] = y1;
    }
}

inline int nb(int64_t n) { return (int)((n + 255) / 256); }

// Buffers for batches of B rows; with `rows` also the host's lists of them.
int ensure_batch(pennant_mlp* m, int64_t B, bool rows) {
    const int64_t ld = (B + 31) / 32 * 32;
    if (ld > m->cap) {
        if (m->lrow) (void)hipFree(m->lrow);
        m->lrow = nullptr;
        m->cap = 0;
        // one allocation: two FP32 rows, then the BF16 ones (ld is a multiple
        // of 32, so each is 16-byte aligned)
        constexpr size_t HALF = PN_MLP_K1 + 4 * PN_MLP_NH + PN_MLP_NO;
        MCK(hipMalloc(&m->lrow, (size_t)ld * (2 * 4 + HALF * 2)));
        m->lossp = m->lrow + ld;
        m->xt = reinterpret_cast<__bf16*>(m->lossp + ld);
        m->h1t = m->xt + PN_MLP_K1 * ld;
        m->h2t = m->h1t + PN_MLP_NH * ld;
        m->dz2t = m->h2t + PN_MLP_NH * ld;
        m->dz1t = m->dz2t + PN_MLP_NH * ld;
        m->dyt = m->dz1t + PN_MLP_NH * ld;
        for (int*& h : m->idx_host) {
            if (h) (void)hipHostFree(h);
            h = nullptr;
        }
        if (!m->part) MCK(hipMalloc(&m->part, (size_t)64 * PN_MLP_NPARAM * 4));
        m->cap = ld;
    }
    for (int k = 0; k < 2 && rows; ++k) {
        if (!m->idx_host[k]) MCK(hipHostMalloc((void**)&m->idx_host[k], (size_t)m->cap * 4));
        if (!m->read[k]) MCK(hipEventCreateWithFlags(&m->read[k], hipEventDisableTiming));
    }
    return 0;
}

int repack(pennant_mlp* m) {
    hipLaunchKernelGGL(k_pack, dim3(nb(PN_MLP_NPARAM)), dim3(256), 0, m->stream, m->p, m->w1b, m->w2b, m->w2t, m->w3b,
                       m->pack);
    MCK(hipGetLastError());
    MCK(hipMemcpyAsync(m->pack->lo, m->lo, sizeof m->lo, hipMemcpyHostToDevice, m->stream));
    MCK(hipMemcpyAsync(m->pack->hi, m->hi, sizeof m->hi, hipMemcpyHostToDevice, m->stream));
    return 0;
}

RowArgs row_args(const pennant_mlp* m, int64_t n, const float* x) {
    RowArgs a = {};
    a.p = m->p;
    a.w1b = m->w1b; a.w2b = m->w2b; a.w2t = m->w2t; a.w3b = m->w3b;
    a.n = n;
    a.x = x;
    return a;
}

// Forward and backward of the B rows idx (NULL: 0 .. B - 1) of the tuples;
// `read` (may be NULL) is recorded once idx has been read.
int launch_batch(pennant_mlp* m, const float* tuples, const int* idx, int64_t B, hipEvent_t read) {
    hipStream_t s = m->stream;
    RowArgs a = row_args(m, B, tuples);
    a.idx = idx;
    a.ld = m->cap;
    a.xt = m->xt; a.h1t = m->h1t; a.h2t = m->h2t; a.dyt = m->dyt; a.dz2t = m->dz2t; a.dz1t = m->dz1t;
    a.lrow = m->lrow;
    hipLaunchKernelGGL(k_rows<true>, dim3((unsigned)((B + 31) / 32)), dim3(64), 0, s, a);
    if (read) MCK(hipEventRecord(read, s));
    GradArgs g;
    g.rows = B;
    g.ld = m->cap;
    int64_t ksplit = B > 1024 ? (B + 511) / 512 : 1;
    if (ksplit > 64) ksplit = 64;
    g.kper = (int)((B + ksplit - 1) / ksplit + 15) / 16 * 16;
    g.ksplit = (int)((B + g.kper - 1) / g.kper);
    g.xt = m->xt; g.h1t = m->h1t; g.h2t = m->h2t; g.dyt = m->dyt; g.dz2t = m->dz2t; g.dz1t = m->dz1t;
    g.lrow = m->lrow;
    g.part = m->part;
    g.g = m->g;
    g.lossp = m->lossp;
    hipLaunchKernelGGL(k_grads, dim3(g.ksplit * PN_GTILES / 4 + PN_MLP_NO + PN_MLP_NH + nb(B)), dim3(256), 0, s, g);
    return (int)hipGetLastError();
}
UpdateArgs update_args(pennant_mlp* m, int64_t B, float* loss) {
    UpdateArgs u = {};
    int64_t ksplit = B > 1024 ? (B + 511) / 512 : 1;
    if (ksplit > 64) ksplit = 64;
    const int kper = (int)((B + ksplit - 1) / ksplit + 15) / 16 * 16;
    u.ksplit = (int)((B + kper - 1) / kper);
    u.nloss = nb(B);
    u.part = m->part;
    u.lossp = m->lossp;
    u.g = m->g;
    u.loss = loss;
    return u;
}

}  // namespace

extern "C" {

int pennant_mlp_num_params(void) { return PN_MLP_NPARAM; }

pennant_mlp* pennant_mlp_create(uint64_t seed) {
    pennant_mlp* m = new pennant_mlp();
    bool ok = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) == hipSuccess;
    // one allocation: the pack, the FP32 vectors, the BF16 copies (each
    // 16-byte aligned)
    constexpr size_t NP = (PN_MLP_NPARAM + 3) / 4 * 4;
    ok = ok && hipMalloc(&m->pack, sizeof(ClosurePack) + 4 * NP * 4 +
                                       (PN_MLP_NH * (PN_MLP_K1 + 2 * PN_MLP_NH) + PN_MLP_NO * PN_MLP_NH) * 2) == hipSuccess;
    if (ok) {
        static_assert(sizeof(ClosurePack) % 16 == 0, "the FP32 vectors follow the pack");
        m->p = reinterpret_cast<float*>(m->pack + 1);
        m->g = m->p + NP;
        m->m = m->g + NP;
        m->v = m->m + NP;
        m->w1b = reinterpret_cast<__bf16*>(m->v + NP);
        m->w2b = m->w1b + PN_MLP_NH * PN_MLP_K1;
        m->w2t = m->w2b + PN_MLP_NH * PN_MLP_NH;
        m->w3b = m->w2t + PN_MLP_NH * PN_MLP_NH;
    }
    if (!ok) { pennant_mlp_destroy(m); return nullptr; }
    // He-uniform initial weights from a seeded generator; zero biases
    std::vector<float> h(PN_MLP_NPARAM, 0.f);
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    const double a1 = std::sqrt(6.0 / (PN_MLP_NF + 1)), a2 = std::sqrt(6.0 / PN_MLP_NH);
    for (int o = 0; o < PN_MLP_NH; ++o)
        for (int k = 0; k < PN_MLP_NF; ++k) h[PN_MLP_OFF_W1 + o * PN_MLP_K1 + k] = (float)(a1 * u(rng));
    for (int i = 0; i < PN_MLP_NH * PN_MLP_NH; ++i) h[PN_MLP_OFF_W2 + i] = (float)(a2 * u(rng));
    for (int i = 0; i < PN_MLP_NO * PN_MLP_NH; ++i) h[PN_MLP_OFF_W3 + i] = (float)(a2 * u(rng));
    for (int k = 0; k < PN_MLP_NF; ++k) { m->lo[k] = -INFINITY; m->hi[k] = INFINITY; }
    if (pennant_mlp_set_params(m, h.data(), PN_MLP_NPARAM) != 0) { pennant_mlp_destroy(m); return nullptr; }
    return m;
}

void pennant_mlp_destroy(pennant_mlp* m) {
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    void* bufs[] = {m->pack, m->lrow, m->part, m->losses};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    for (int* h : m->idx_host)
        if (h) (void)hipHostFree(h);
    for (hipEvent_t e : m->read)
        if (e) (void)hipEventDestroy(e);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

int pennant_mlp_set_params(pennant_mlp* m, const float* host, int n) {
    if (n != PN_MLP_NPARAM) return PENNANT_EINVAL;
    MCK(hipMemcpyAsync(m->p, host, PN_MLP_NPARAM * 4, hipMemcpyHostToDevice, m->stream));
    MCK(hipMemsetAsync(m->m, 0, PN_MLP_NPARAM * 4, m->stream));
    MCK(hipMemsetAsync(m->v, 0, PN_MLP_NPARAM * 4, m->stream));
    m->adam_t = 0;
    MCK(repack(m));
    return (int)hipStreamSynchronize(m->stream);
}

int pennant_mlp_get_params(pennant_mlp* m, float* host, int n) {
    if (n != PN_MLP_NPARAM) return PENNANT_EINVAL;
    MCK(hipMemcpyAsync(host, m->p, PN_MLP_NPARAM * 4, hipMemcpyDeviceToHost, m->stream));
    return (int)hipStreamSynchronize(m->stream);
}

int pennant_mlp_set_envelope(pennant_mlp* m, const float* lo, const float* hi) {
    for (int k = 0; k < PN_MLP_NF; ++k) { m->lo[k] = lo[k]; m->hi[k] = hi[k]; }
    MCK(repack(m));
    return (int)hipStreamSynchronize(m->stream);
}

int pennant_mlp_get_envelope(pennant_mlp* m, float* lo, float* hi) {
    for (int k = 0; k < PN_MLP_NF; ++k) { lo[k] = m->lo[k]; hi[k] = m->hi[k]; }
    return 0;
}

const void* pennant_mlp_device_pack(pennant_mlp* m) { return m->pack; }

int pennant_mlp_forward(pennant_mlp* m, const float* x, int64_t n, float* y, int path) {
    if (n < 0 || (path != 0 && path != 1)) return PENNANT_EINVAL;
    if (n == 0) return 0;
    if (path == 1) {
        hipLaunchKernelGGL(k_mlp_wave, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, m->pack,
                           n, x, y);
        MCK(hipGetLastError());
        return (int)hipStreamSynchronize(m->stream);
    }
    // a launch has fewer than 2^32 threads, two a row
    constexpr int64_t chunk = (int64_t)1 << 30;
    for (int64_t b0 = 0; b0 < n; b0 += chunk) {
        RowArgs a = row_args(m, n - b0 < chunk ? n - b0 : chunk, x + b0 * PN_MLP_NF);
        a.y = y + 2 * b0;
        hipLaunchKernelGGL(k_rows<false>, dim3((unsigned)((a.n + 31) / 32)), dim3(64), 0, m->stream, a);
    }
    MCK(hipGetLastError());
    return (int)hipStreamSynchronize(m->stream);
}

int pennant_mlp_loss_grad(pennant_mlp* m, const float* tuples, int64_t n, float* grad, float* loss) {
    if (n <= 0 || n > (1 << 30)) return PENNANT_EINVAL;
    MCK(ensure_batch(m, n, false));
    MCK(launch_batch(m, tuples, nullptr, n, nullptr));
    const UpdateArgs u = update_args(m, n, m->lossp + nb(n));
    hipLaunchKernelGGL(k_update<false>, dim3(nb(PN_MLP_NPARAM + 1)), dim3(256), 0, m->stream, u);
    MCK(hipGetLastError());
    MCK(hipMemcpyAsync(grad, m->g, PN_MLP_NPARAM * 4, hipMemcpyDeviceToHost, m->stream));
    MCK(hipMemcpyAsync(loss, u.loss, 4, hipMemcpyDeviceToHost, m->stream));
    MCK(hipStreamSynchronize(m->stream));
    *loss /= (float)n;
    return 0;
}

int pennant_mlp_train(pennant_mlp* m, const float* tuples, int64_t n, int steps, int batch, float lr,
                      uint64_t seed, float* loss_out) {
    if (n <= 0 || n > (1 << 30) || steps < 0 || batch <= 0 || batch > (1 << 22)) return PENNANT_EINVAL;
    MCK(hipGetLastError());      // what another call has left is reported before the first step
    MCK(ensure_batch(m, batch, true));
    if (steps > m->loss_cap) {
        if (m->losses) (void)hipFree(m->losses);
        m->losses = nullptr;
        m->loss_cap = 0;
        MCK(hipMalloc(&m->losses, (size_t)steps * 4));
        m->loss_cap = steps;
    }
    std::mt19937_64 rng(seed);
    std::uniform_int_distribution<int64_t> pick(0, n - 1);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    int rc = 0;
    for (int st = 0; st < steps && !rc; ++st) {
        // a step's rows are drawn while the steps before it run; the kernel
        // reads them from the host's list, which is free again two steps later
        int* idx = m->idx_host[st & 1];
        if (st >= 2 && (rc = (int)hipEventSynchronize(m->read[st & 1]))) break;
        for (int b = 0; b < batch; ++b) idx[b] = (int)pick(rng);
        if ((rc = launch_batch(m, tuples, idx, batch, m->read[st & 1]))) break;
        m->adam_t += 1;
        UpdateArgs u = update_args(m, batch, m->losses + st);
        u.c1 = 1.f - std::pow(b1, (float)m->adam_t);
        u.c2 = 1.f - std::pow(b2, (float)m->adam_t);
        // cosine decay from lr to lr/50 over the call's steps
        u.lr = lr * (0.02f + 0.98f * 0.5f * (1.f + std::cos(3.14159265f * (float)st / (float)steps)));
        u.b1 = b1; u.b2 = b2; u.eps = eps;
        u.p = m->p; u.m = m->m; u.v = m->v;
        u.w1b = m->w1b; u.w2b = m->w2b; u.w2t = m->w2t; u.w3b = m->w3b; u.pack = m->pack;
        hipLaunchKernelGGL(k_update<true>, dim3(nb(PN_MLP_NPARAM + 1)), dim3(256), 0, m->stream, u);
        rc = (int)hipGetLastError();
    }
    if (!rc && loss_out && steps > 0)
        rc = (int)hipMemcpyAsync(loss_out, m->losses, (size_t)steps * 4, hipMemcpyDeviceToHost, m->stream);
    // (also after an error: the kernels read the caller's tuples and the row lists)
    const int rc2 = (int)hipStreamSynchronize(m->stream);
    if (rc || rc2) return rc ? rc : rc2;
    if (loss_out)
        for (int st = 0; st < steps; ++st) loss_out[st] /= (float)batch;
    return 0;
}

}  // extern "C"
