// fg_mlp.hip -- per-pixel Monte-Carlo error model: features and a small MLP
// (16 inputs, 12 used -> 64 -> 64 -> 1, ReLU) with BF16 weights and FP32
// accumulation on the gfx950 matrix cores, forward and backward.
//
// No counterpart in the reference.  The model predicts log(s), s the
// per-sample standard deviation sqrt(p (1 - p)) of a pixel's coverage
// indicator, from local statistics of the intensity plane; the sample budget
// of the adaptive renderer is proportional to s.
//
// Layout.  Parameters are one f32 array (fg_mlp.h offsets): W1 [16][64]
// (rows 12..15 zero), b1 [64], W2 [64][64] (input-major), b2 [64], w3 [64],
// b3.  Features are BF16 [n][16].  A wave works on 16 rows at a time, with
// the weights as BF16 matrix operands in its registers:
//   layer 1: Z1 = X W1 + b1      4 x v_mfma_f32_16x16x16_bf16 (one per 16 outputs)
//   layer 2: Z2 = H1 W2 + b2     8 x v_mfma_f32_16x16x32_bf16, H1 = relu(Z1) in BF16
//   layer 3: y = H2 . w3 + b3    FP32 dot products (a 64-vector), H2 = relu(Z2)
// The forward pass adds a bias after its layer's sum, and layer 3's columns one
// after the other: its predictions decide integer budgets, so their bits are
// part of its result.  In the gradient the biases are the accumulators' initial
// values.
// Backward of the loss per row (fused, per tile), either the squared error to
// a target t, L = (y - t)^2, g = dL/dy = 2 (y - t), or the Gaussian negative
// log-likelihood of a residual t under the predicted log std y,
// L = y + t^2 e^(-2y) / 2, g = 1 - t^2 e^(-2y) (the exponent clamped to
// [-80, 80]); then with g scaled by 1 / n:
//   dZ2 = g w3 * [Z2 > 0], dZ1 = (dZ2 W2^T) * [Z1 > 0]
//   dW3 = H2^T g, dW2 = H1^T dZ2, dW1 = X^T dZ1 (MFMA over the 16 rows), biases
//   by sums.  Products feeding a matrix instruction use BF16 operands (dZ2,
//   dZ1, H1, X); their accumulations are FP32.  The CPU reference in the
//   tests rounds the same operands to BF16 at the same points.
// Matrix operand layouts (wave64): 16x16x16: lane l holds A[l%16][4(l/16)+0..3],
// B[4(l/16)+0..3][l%16]; 16x16x32: A[l%16][8(l/16)+0..7], B[8(l/16)+0..7][l%16];
// both: D[4(l/16)+0..3][l%16].
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fg_kernels.h"
#include "fg_mlp.h"

namespace fg {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf16_float(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

// relu and round to BF16 (v_cvt_pk_bf16_f32: nearest even).  The median with
// the largest finite value is one instruction where fmaxf takes two (it first
// quiets its operand); an infinity rounds to BF16 infinity from there as well,
// and a NaN gives 0 either way.
__device__ __forceinline__ v4bf relu_bf16(v4f c)
{
    v4f h;
    for (int i = 0; i < 4; ++i) h[i] = __builtin_amdgcn_fmed3f(c[i], 0.0f, 3.402823466e+38f);
    return __builtin_convertvector(h, v4bf);
}
__device__ __forceinline__ v8bf join(v4bf a, v4bf b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
__device__ __forceinline__ v4f mfma16(v4bf a, v4bf b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(v4s, a), __builtin_bit_cast(v4s, b), c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma32(v8bf a, v8bf b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Features 4g..4g+3 of a row: 8 bytes, in one load where the rows are so
// aligned (aligned: uniform).
__device__ __forceinline__ v4bf load_x(const uint16_t *X, long long row, int g, bool aligned)
{
    const uint16_t *p = X + row * 16 + 4 * g;
    if (aligned) return *reinterpret_cast<const v4bf *>(p);
    v4bf x;
    for (int t = 0; t < 4; ++t) x[t] = __builtin_bit_cast(__bf16, p[t]);
    return x;
}

// Feature r of rows row0 + 4g..+3 (0 past n).
__device__ __forceinline__ v4bf load_x_column(const uint16_t *X, long long row0, long long n, int r, int g)
{
    v4bf x = {};
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
        const long long row = row0 + 4 * g + i;
        if (row < n) x[i] = __builtin_bit_cast(__bf16, X[row * 16 + r]);
    }
    return x;
}

// Forward pass for inference, without LDS: the layers are computed
// transposed, Z1^T = W1^T X^T (16x16x16: A = a 16-output block of W1^T,
// B = X^T) and Z2^T = W2^T H1^T (16x16x32), so that a lane's accumulator
// holds row r = lane % 16 of the activations, columns cb*16 + 4g + i
// (g = lane / 16, i = 0..3).  Those are exactly the B operand layer 2 needs
// (row r, eight k per lane) under a fixed permutation of k within each
// 32-chunk: logical k = 8g + t is H1 column kc*32 + 4g + t (t < 4) or
// kc*32 + 16 + 4g + t - 4 (t >= 4); W2^T's operand is loaded in the same
// order, so the products are unchanged.  Weights, biases and w3 live in
// registers for the whole kernel; each lane reads its row's four features
// (8 bytes) from HBM.  Layer 3 sums the lane's 16 columns, then across the
// four lanes of the row.
__device__ __forceinline__ int mlp_h1_column(int kc, int g, int t)
{
    return kc * 32 + (t < 4 ? 4 * g + t : 16 + 4 * g + (t - 4));
}

// The layers' weights as matrix operands of lane (r, g), the same registers
// serving as A of the transposed product and as B of the plain one (the
// operand layouts mirror each other).
struct MlpWeights {
    v4bf w1[4];     // W1[4g + t][cb * 16 + r]
    v8bf w2[4][2];  // W2[mlp_h1_column(kc, g, t)][cb * 16 + r]
};
// The workgroup's copy of the operands, lane by lane.  It is filled by short
// loops over the parameters, coalesced (straight into registers they are 140
// gathers a lane).
struct MlpOperands {
    __bf16 w1[4][64][4];
    __bf16 w2[4][2][64][8];
};
// Where element (outer column, inner index) of a 64 x 64 operand lies: the
// inverse of mlp_h1_column.
__device__ __forceinline__ int mlp_operand_at(int outer, int inner)
{
    const int cb = outer >> 4, r = outer & 15, kc = inner >> 5, kk = inner & 31;
    const int g = (kk & 15) >> 2, t = (kk & 3) + ((kk >> 4) << 2);
    return ((cb * 2 + kc) * 64 + g * 16 + r) * 8 + t;
}
__device__ __forceinline__ void fill_operands(const float *P, MlpOperands &s)
{
#pragma unroll 1
    for (int i = threadIdx.x; i < 16 * 64; i += blockDim.x) {
        const int k = i >> 6, j = i & 63;
        s.w1[j >> 4][(k >> 2) * 16 + (j & 15)][k & 3] = (__bf16)P[kMlpW1 + i];
    }
#pragma unroll 2
    for (int i = threadIdx.x; i < 64 * 64; i += blockDim.x)
        (&s.w2[0][0][0][0])[mlp_operand_at(i & 63, i >> 6)] = (__bf16)P[kMlpW2 + i];
}
__device__ __forceinline__ void load_weights(const MlpOperands &s, MlpWeights &w, int lane)
{
    for (int cb = 0; cb < 4; ++cb) {
        w.w1[cb] = *reinterpret_cast<const v4bf *>(s.w1[cb][lane]);
        for (int kc = 0; kc < 2; ++kc) w.w2[cb][kc] = *reinterpret_cast<const v8bf *>(s.w2[cb][kc][lane]);
    }
}

// Bounded by instruction issue: 12 matrix instructions and about 130 VALU per
// 16 rows, which do not overlap fully.  2.07M rows (75 MB): 44 us with the
// conversions in hardware, 88 us with conversions in software.  (The biases as
// initial accumulators and layer 3 in four fused chains are 4 us less, and move
// one budget in about 1e5 by a sample.)  More rows in flight (two to eight tiles
// ahead, four at once) and two or four waves per SIMD instead of three: no
// difference.
constexpr int kTiles = 2;  // 16-row tiles a wave works on at once
__global__ __launch_bounds__(256, 3) void mlp_forward_kernel(const float *P, const uint16_t *X, long long n, float *out,
                                                          bool aligned)
{
    __shared__ __align__(16) MlpOperands s_op;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    fill_operands(P, s_op);
    __syncthreads();
    MlpWeights w;
    load_weights(s_op, w, lane);
    v4f b1[4], b2[4], w3[4];
    for (int cb = 0; cb < 4; ++cb)
        for (int i = 0; i < 4; ++i) {
            const int j = cb * 16 + 4 * g + i;
            b1[cb][i] = P[kMlpB1 + j];
            b2[cb][i] = P[kMlpB2 + j];
            w3[cb][i] = (float)(__bf16)P[kMlpW3 + j];
        }
    const float b3 = P[kMlpB3];
    const long long tiles = (n + 15) / 16;
    const long long stride = (long long)gridDim.x * 4 * kTiles;
    const v4bf zero = {};
    const v4f zero4 = {};
    long long tt = ((long long)blockIdx.x * 4 + wid) * kTiles;
    v4bf x[kTiles], xn[kTiles];  // this step's rows, and the next one's, in flight meanwhile
    auto fetch = [&](v4bf *v, long long at) {
        for (int u = 0; u < kTiles; ++u) {
            const long long row = (at + u) * 16 + r;
            v[u] = row < n ? load_x(X, row, g, aligned) : zero;
        }
    };
    fetch(x, tt);
    for (; tt < tiles; tt += stride) {
        fetch(xn, tt + stride);
        // layer 1 (transposed) and the B operand of layer 2
        v8bf h0[kTiles], h1[kTiles];
        for (int u = 0; u < kTiles; ++u) {
            v4bf h[4];
            for (int cb = 0; cb < 4; ++cb) h[cb] = relu_bf16(mfma16(w.w1[cb], x[u], zero4) + b1[cb]);
            h0[u] = join(h[0], h[1]);
            h1[u] = join(h[2], h[3]);
        }
        // layer 2 (transposed) and layer 3
        float y[kTiles];
        for (int u = 0; u < kTiles; ++u) {
            float acc = 0.0f;
            for (int cb = 0; cb < 4; ++cb) {
                const v4f c = mfma32(w.w2[cb][1], h1[u], mfma32(w.w2[cb][0], h0[u], zero4)) + b2[cb];
                for (int i = 0; i < 4; ++i) acc += fmaxf(c[i], 0.0f) * w3[cb][i];
            }
            y[u] = acc;
        }
        for (int u = 0; u < kTiles; ++u) {
            y[u] += __shfl_xor(y[u], 16, 64);
            y[u] += __shfl_xor(y[u], 32, 64);
            const long long row = (tt + u) * 16 + r;
            if (g == 0 && row < n) out[row] = y[u] + b3;
        }
        for (int u = 0; u < kTiles; ++u) x[u] = xn[u];
    }
}

// Fused forward + backward of the loss (loss_kind 0: squared error, 1:
// Gaussian negative log-likelihood of the residual) over rows [0, n) with
// loss scale 1 / n_total; gradients are added to grad (kMlpParams f32) and
// the unscaled loss sum to *loss.
//
// Every layer is computed in both layouts, plain (lane (r, g): rows 4g..4g+3, column r of a block of
// 16) and transposed (lane: row r, columns 4g..4g+3), by the same operands in
// swapped places: the plain form is what the products over rows (dW1, dW2)
// take as operands, the transposed form what the next product along the
// layers takes, so nothing crosses lanes but y and its gradient, and LDS
// holds only W2's backward operands and the T-layout vectors.  X in the plain
// layout is X times the identity; a NaN or an infinity makes its whole row NaN
// there (it meets the identity's zeros), and such a tile is read from memory
// instead (every tile read so: 51 us for 46 at 400003 rows, 185 for 162 at 2M).
// Bounded by instruction issue at many rows (2M rows: 0.17 ms, 650 us before);
// at few by the set-up and the atomics on grad, kMlpParams a workgroup: one
// workgroup per 256 rows up to one per CU (per 1024 rows: 34 us instead of 27
// at 65536 rows).  65536 rows: 195 us with a workgroup per 64 rows, the
// transposes through LDS and the reduction by LDS float atomics.
constexpr int kGradBlock = 512;
__global__ __launch_bounds__(kGradBlock, 2) void mlp_grad_kernel(const float *P, const uint16_t *X,
                                                                 const float *target, long long n, float inv_total,
                                                                 int loss_kind, float *grad, float *loss, bool aligned)
{
    constexpr int NW = kGradBlock / 64;
    __shared__ __align__(16) MlpOperands s_op;
    __shared__ v8bf s_w2[4][2][64];   // lane (r, g): W2[cb * 16 + r][mlp_h1_column(kc, g, t)]
    __shared__ v4f s_b1[16], s_b2[16], s_w3[16];
    __shared__ v4f s_part[4][20][64];  // the final reduction
    __shared__ float s_vec[NW][194];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    fill_operands(P, s_op);
#pragma unroll 2
    for (int i = threadIdx.x; i < 64 * 64; i += kGradBlock)
        reinterpret_cast<__bf16 *>(&s_w2[0][0][0])[mlp_operand_at(i >> 6, i & 63)] = (__bf16)P[kMlpW2 + i];
    if (threadIdx.x < 64) {
        const int j = threadIdx.x;
        s_b1[j >> 2][j & 3] = P[kMlpB1 + j];
        s_b2[j >> 2][j & 3] = P[kMlpB2 + j];
        s_w3[j >> 2][j & 3] = (float)(__bf16)P[kMlpW3 + j];
    }
    __syncthreads();
    MlpWeights w;
    load_weights(s_op, w, lane);
    float b1n[4], b2n[4], w3n[4];
    for (int cb = 0; cb < 4; ++cb) {
        b1n[cb] = P[kMlpB1 + cb * 16 + r];
        b2n[cb] = P[kMlpB2 + cb * 16 + r];
        w3n[cb] = (float)(__bf16)P[kMlpW3 + cb * 16 + r];
    }
    const float b3 = P[kMlpB3];
    v4bf ident;
    for (int t = 0; t < 4; ++t) ident[t] = (__bf16)(4 * g + t == r ? 1.0f : 0.0f);
    const v4f zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    v4f dw2[4][4], dw1[4];
    for (int a = 0; a < 4; ++a) {
        dw1[a] = zero4;
        for (int b = 0; b < 4; ++b) dw2[a][b] = zero4;
    }
    float db1[4] = {0, 0, 0, 0}, db2[4] = {0, 0, 0, 0}, dw3[4] = {0, 0, 0, 0}, db3 = 0.0f, lsum = 0.0f;
    const long long tiles = (n + 15) / 16, stride = (long long)gridDim.x * NW;
    long long tt = (long long)blockIdx.x * NW + wid;
    v4bf x = {};
    float t = 0.0f;
    if (tt < tiles && tt * 16 + r < n) {
        x = load_x(X, tt * 16 + r, g, aligned);
        t = target[tt * 16 + r];
    }
    for (; tt < tiles; tt += stride) {
        // keeps the LDS operands from being held in registers all loop long,
        // where they spilled
        asm volatile("" ::: "memory");
        const long long row = tt * 16 + r, next = row + stride * 16;
        v4bf xnext = {};
        float tnext = 0.0f;
        if (next < n) {  // the next tile's, in flight meanwhile
            xnext = load_x(X, next, g, aligned);
            tnext = target[next];
        }
        const v4f xf = mfma16(x, ident, zero4);
        v4bf xn = __builtin_convertvector(xf, v4bf);
        const float xs = (xf[0] + xf[1]) + (xf[2] + xf[3]);
        if (__builtin_expect(__any(xs != xs), 0)) xn = load_x_column(X, tt * 16, n, r, g);
        // layer 1 transposed
        v4bf h[4];
        for (int cb = 0; cb < 4; ++cb) h[cb] = relu_bf16(mfma16(w.w1[cb], x, s_b1[cb * 4 + g]));
        const v8bf h0 = join(h[0], h[1]), h1 = join(h[2], h[3]);
        // layer 2 transposed, y of row r and its gradient
        float y = 0.0f;
        uint32_t m2 = 0;  // transposed: Z2 > 0
        for (int cb = 0; cb < 4; ++cb) {
            const v4f c = mfma32(w.w2[cb][1], h1, mfma32(w.w2[cb][0], h0, s_b2[cb * 4 + g]));
            const v4f w3 = s_w3[cb * 4 + g];
            for (int i = 0; i < 4; ++i) {
                m2 |= c[i] > 0.0f ? 1u << (cb * 4 + i) : 0u;
                y = __builtin_fmaf(fmaxf(c[i], 0.0f), w3[i], y);
            }
        }
        y += __shfl_xor(y, 16, 64);
        y += __shfl_xor(y, 32, 64);
        y += b3;
        float gy = 0.0f;  // rows past n contribute nothing
        if (row < n) {
            float l;
            if (loss_kind == 1) {
                const float e = expf(fminf(fmaxf(-2.0f * y, -80.0f), 80.0f)) * t * t;
                gy = (1.0f - e) * inv_total;
                l = y + 0.5f * e;
            } else {
                const float d = y - t;
                gy = 2.0f * d * inv_total;
                l = d * d;
            }
            if (g == 0) {
                lsum += l;
                db3 += gy;
            }
        }
        // dZ2 transposed, the A operand of dZ1 = dZ2 W2^T
        v4bf zt[4];
        for (int cb = 0; cb < 4; ++cb) {
            const v4f w3 = s_w3[cb * 4 + g];
            v4f d;
            for (int i = 0; i < 4; ++i) d[i] = (m2 >> (cb * 4 + i)) & 1u ? gy * w3[i] : 0.0f;
            zt[cb] = __builtin_convertvector(d, v4bf);
        }
        const v8bf z0 = join(zt[0], zt[1]), z1 = join(zt[2], zt[3]);
        // layer 2 plain: dw3, db2 and dZ2
        float gr[4];
        for (int i = 0; i < 4; ++i) gr[i] = __shfl(gy, 4 * g + i, 64);
        v4bf zn[4];
        for (int cb = 0; cb < 4; ++cb) {
            const v4f c =
                mfma32(h1, w.w2[cb][1], mfma32(h0, w.w2[cb][0], (v4f){b2n[cb], b2n[cb], b2n[cb], b2n[cb]}));
            v4f d;
            for (int i = 0; i < 4; ++i) {
                dw3[cb] = __builtin_fmaf(gr[i], fmaxf(c[i], 0.0f), dw3[cb]);
                d[i] = c[i] > 0.0f ? gr[i] * w3n[cb] : 0.0f;
                db2[cb] += d[i];
            }
            zn[cb] = __builtin_convertvector(d, v4bf);
        }
        // layer 1 and dZ1 plain, and the products over the rows
        for (int cb = 0; cb < 4; ++cb) {
            const v4f a1 = mfma16(x, w.w1[cb], (v4f){b1n[cb], b1n[cb], b1n[cb], b1n[cb]});
            const v4bf hn = relu_bf16(a1);
            for (int k = 0; k < 4; ++k) dw2[cb][k] = mfma16(hn, zn[k], dw2[cb][k]);
            v4f c = mfma32(z1, s_w2[cb][1][lane], mfma32(z0, s_w2[cb][0][lane], zero4));
            for (int i = 0; i < 4; ++i) {
                c[i] = a1[i] > 0.0f ? c[i] : 0.0f;
                db1[cb] += c[i];
            }
            dw1[cb] = mfma16(xn, __builtin_convertvector(c, v4bf), dw1[cb]);
        }
        x = xnext;
        t = tnext;
    }
    // Reduce over the workgroup without LDS float atomics (those took 57 us of
    // 82 at 65536 rows): the upper four waves hand their accumulators to the
    // lower four through LDS, those leave theirs there, and every thread sums
    // four and adds to grad.  Accumulator blocks hold D[4g+i][r].
    for (int cb = 0; cb < 4; ++cb)
        for (int o = 16; o < 64; o <<= 1) {
            db1[cb] += __shfl_xor(db1[cb], o, 64);
            db2[cb] += __shfl_xor(db2[cb], o, 64);
            dw3[cb] += __shfl_xor(dw3[cb], o, 64);
        }
    for (int o = 1; o < 64; o <<= 1) {
        db3 += __shfl_xor(db3, o, 64);
        lsum += __shfl_xor(lsum, o, 64);
    }
    if (g == 0)
        for (int cb = 0; cb < 4; ++cb) {
            s_vec[wid][cb * 16 + r] = db1[cb];
            s_vec[wid][64 + cb * 16 + r] = db2[cb];
            s_vec[wid][128 + cb * 16 + r] = dw3[cb];
        }
    if (lane == 0) {
        s_vec[wid][192] = db3;
        s_vec[wid][193] = lsum;
    }
    auto each = [&](auto f) {
        for (int kb = 0; kb < 4; ++kb) {
            for (int cb = 0; cb < 4; ++cb) f(kb * 4 + cb, dw2[kb][cb]);
            f(16 + kb, dw1[kb]);
        }
    };
    if (wid >= 4) each([&](int k, v4f &v) { s_part[wid - 4][k][lane] = v; });
    __syncthreads();
    if (wid < 4) each([&](int k, v4f &v) { s_part[wid][k][lane] = v + s_part[wid][k][lane]; });
    __syncthreads();
#pragma unroll 1
    for (int e = threadIdx.x; e < 20 * 256; e += kGradBlock) {
        // element i of block k's lane l, lanes of a row first
        const int k = e >> 8, l = ((e >> 6) & 3) * 16 + (e & 15), i = (e >> 4) & 3;
        const float v = (s_part[0][k][l][i] + s_part[1][k][l][i]) + (s_part[2][k][l][i] + s_part[3][k][l][i]);
        const int row = 4 * (l >> 4) + i;
        const int at = k < 16 ? kMlpW2 + ((k >> 2) * 16 + row) * 64 + (k & 3) * 16 + (l & 15)
                              : kMlpW1 + row * 64 + (k & 3) * 16 + (l & 15);
        if (v != 0.0f) atomicAdd(&grad[at], v);
    }
    if (threadIdx.x < 194) {
        float v = 0.0f;
        for (int q = 0; q < NW; ++q) v += s_vec[q][threadIdx.x];
        const int j = threadIdx.x & 63, which = threadIdx.x >> 6;
        float *dst = which == 0 ? grad + kMlpB1 + j
                     : which == 1 ? grad + kMlpB2 + j
                     : which == 2 ? grad + kMlpW3 + j
                                  : (j == 0 ? grad + kMlpB3 : loss);
        if (v != 0.0f) atomicAdd(dst, v);
    }
}

// Adam (Kingma & Ba 2015) with bias correction; rows 12..15 of W1 stay 0.
__global__ void mlp_adam_kernel(float *P, const float *grad, float *m, float *v, float lr, float b1, float b2,
                                float eps, float bc1, float bc2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kMlpParams) return;
    if (i >= kMlpW1 + 12 * 64 && i < kMlpW1 + 16 * 64) {
        P[i] = 0.0f;
        return;
    }
    const float gi = grad[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    P[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

// Features of output pixel (x, y) of a plane: the normalised intensity u of
// the input pixel it maps to (floor((x + 0.5) / zoom), clamped), the mean and
// variance of u over its 3x3 neighbourhood (edges clamped), the gradient
// magnitude (central differences), u (1 - u), the radius law, filter sigma and
// zoom (scaled to order one), and the channel one-hot.
// Bounded by its stores, 32 bytes a pixel: two 16-byte stores where the rows
// are so aligned (wide), and the pixel's row by a 32-bit division where the
// plane has fewer than 2^32 pixels (2.07M pixels: 18 us; 50 us with 16
// two-byte stores and a 64-bit division).
__global__ __launch_bounds__(256) void feature_kernel(const float *u, int in_w, int in_h, int out_w, int out_h,
                                                      float inv_zoom, float f_radius, float f_sd, float f_sigma,
                                                      float f_zoom, int channel, uint16_t *X, bool wide)
{
    const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)out_w * out_h;
    if (p >= n) return;
    const int y = n <= 0xFFFFFFFFLL ? (int)((uint32_t)p / (uint32_t)out_w) : (int)(p / out_w);
    const int x = (int)(p - (long long)y * out_w);
    const int ix = min(max((int)floorf(((float)x + 0.5f) * inv_zoom), 0), in_w - 1);
    const int iy = min(max((int)floorf(((float)y + 0.5f) * inv_zoom), 0), in_h - 1);
    auto at = [&](int dx, int dy) {
        const int xx = min(max(ix + dx, 0), in_w - 1), yy = min(max(iy + dy, 0), in_h - 1);
        return u[(size_t)yy * in_w + xx];
    };
    float s = 0.0f, s2 = 0.0f;
    for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
            const float v = at(dx, dy);
            s += v;
            s2 += v * v;
        }
    const float mean = s * (1.0f / 9.0f);
    const float var = fmaxf(s2 * (1.0f / 9.0f) - mean * mean, 0.0f);
    const float gx = 0.5f * (at(1, 0) - at(-1, 0)), gy = 0.5f * (at(0, 1) - at(0, -1));
    const float c = at(0, 0);
    float f[16] = {c,       mean,       sqrtf(var), sqrtf(gx * gx + gy * gy), c * (1.0f - c), f_radius, f_sd,
                   f_sigma, f_zoom,     channel == 0 ? 1.0f : 0.0f, channel == 1 ? 1.0f : 0.0f,
                   channel == 2 ? 1.0f : 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    uint16_t *dst = X + p * 16;
    if (wide) {
        v8bf lo, hi;
        for (int i = 0; i < 8; ++i) {
            lo[i] = (__bf16)f[i];
            hi[i] = (__bf16)f[8 + i];
        }
        reinterpret_cast<v8bf *>(dst)[0] = lo;
        reinterpret_cast<v8bf *>(dst)[1] = hi;
    } else {
        for (int i = 0; i < 16; ++i) dst[i] = __builtin_bit_cast(uint16_t, (__bf16)f[i]);
    }
}

// Sample budget n = clamp(ceil(c * s), nmin, nmax) per pixel, from s =
// exp(predicted log s) (pred != nullptr) or, for the allocator without the
// model, s = sqrt(u (1 - u)) from feature 4 of X.
// With dc != nullptr the scale is *dc (written by the scale search).
__global__ __launch_bounds__(256) void budget_kernel(const float *pred, const uint16_t *X, long long n, float c,
                                                     const float *dc, int nmin, int nmax, uint16_t *budget)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    if (dc) c = *dc;
    const float s = pred ? expf(pred[i]) : sqrtf(fmaxf(bf16_float(X[i * 16 + 4]), 0.0f));
    const float v = ceilf(c * s);
    const int b = v >= (float)nmax ? nmax : (v <= (float)nmin ? nmin : (int)v);
    budget[i] = (uint16_t)b;
}

hipError_t launch_budget(const float *pred, const uint16_t *X, long long n, float c, const float *dc, int nmin,
                         int nmax, uint16_t *budget, hipStream_t s)
{
    hipLaunchKernelGGL(budget_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, pred, X, n, c, dc, nmin,
                       nmax, budget);
    return hipGetLastError();
}

// ---- the budget scale search on the device ----
// Per-sample stds s_i = exp(pred[i * step]) * s_mult over the strided
// subsample i < m.  The smallest c whose budgets clamp(ceil(c s), nmin, nmax)
// have mean predicted squared error s^2 (1/n - 1/n_ref) <= target, by rounds
// of kScaleProbes geometric candidates between lo and hi (each round keeps the
// bracket of the first candidate that meets the target).
constexpr int kScaleProbes = 64;

__device__ __forceinline__ float scale_probe(float lo, float hi, int j)
{
    const float a = logf(lo), b = logf(hi);
    return expf(a + (b - a) * ((float)j / (float)(kScaleProbes - 1)));
}

// State: lo, hi, c, done (floats), the bits of the smallest positive s (a
// positive float orders as its bits do), then the probe sums.
__global__ void scale_clear_kernel(float *state, double *sums)
{
    if (threadIdx.x < kScaleProbes) sums[threadIdx.x] = 0.0;
    if (threadIdx.x == 0) reinterpret_cast<unsigned int *>(state)[4] = 0x7F800000u;  // +inf
}

__global__ __launch_bounds__(256) void scale_min_kernel(const float *pred, long long step, long long m, float s_mult,
                                                        float *state)
{
    float mn = INFINITY;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < m; i += (long long)gridDim.x * 256) {
        const float s = expf(pred[i * step]) * s_mult;
        if (s > 0.0f) mn = fminf(mn, s);
    }
    for (int o = 32; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o, 64));
    if ((threadIdx.x & 63) == 0 && mn < INFINITY)
        atomicMin(reinterpret_cast<unsigned int *>(state) + 4, __float_as_uint(mn));
}

__global__ void scale_setup_kernel(int nmax, float *state)
{
    if (threadIdx.x == 0) {
        const float mn = __uint_as_float(reinterpret_cast<const unsigned int *>(state)[4]);
        const float smin = mn < INFINITY ? fmaxf(mn, 1e-6f) : 1.0f;
        state[0] = 1e-2f;
        state[1] = 2.0f * (float)nmax / smin;
        state[2] = state[1];
        state[3] = 0.0f;
    }
}

__global__ __launch_bounds__(256) void scale_sums_kernel(const float *pred, long long step, long long m, float s_mult,
                                                         int nmin, int nmax, float inv_nref, const float *state,
                                                         double *sums)
{
    __shared__ float s_c[kScaleProbes];
    __shared__ float s_part[256 / 64][kScaleProbes];
    if (state[3] != 0.0f) return;
    if (threadIdx.x < kScaleProbes) s_c[threadIdx.x] = scale_probe(state[0], state[1], threadIdx.x);
    __syncthreads();
    float acc[kScaleProbes];
#pragma unroll
    for (int j = 0; j < kScaleProbes; ++j) acc[j] = 0.0f;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < m; i += (long long)gridDim.x * 256) {
        const float s = expf(pred[i * step]) * s_mult;
        const float s2 = s * s;
#pragma unroll
        for (int j = 0; j < kScaleProbes; ++j) {
            const float v = ceilf(s_c[j] * s);
            const float nj = fminf(fmaxf(v, (float)nmin), (float)nmax);
            acc[j] += s2 * (1.0f / nj - inv_nref);
        }
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < kScaleProbes; ++j) {
        float v = acc[j];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) s_part[wid][j] = v;
    }
    __syncthreads();
    if (threadIdx.x < kScaleProbes) {
        double t = 0.0;
        for (int w = 0; w < 256 / 64; ++w) t += (double)s_part[w][threadIdx.x];
        atomicAdd(&sums[threadIdx.x], t);
    }
}

__global__ void scale_pick_kernel(long long m, double target, int last, float *state, double *sums)
{
    __shared__ int s_first;
    if (threadIdx.x == 0) s_first = kScaleProbes;
    __syncthreads();
    if (state[3] == 0.0f && threadIdx.x < kScaleProbes && sums[threadIdx.x] / (double)m <= target)
        atomicMin(&s_first, (int)threadIdx.x);
    __syncthreads();
    if (threadIdx.x == 0 && state[3] == 0.0f) {
        const float lo = state[0], hi = state[1];
        const int k = s_first;
        if (k == kScaleProbes) {
            state[2] = scale_probe(lo, hi, kScaleProbes - 1);
            state[3] = 1.0f;
        } else if (k == 0) {
            state[2] = scale_probe(lo, hi, 0);
            state[3] = 1.0f;
        } else {
            state[0] = scale_probe(lo, hi, k - 1);
            state[1] = scale_probe(lo, hi, k);
            state[2] = state[1];
            if (last) state[3] = 1.0f;
        }
    }
    __syncthreads();
    if (threadIdx.x < kScaleProbes) sums[threadIdx.x] = 0.0;
}

__global__ void scale_out_kernel(const float *state, float s_mult, float *out)
{
    if (threadIdx.x == 0) {
        out[0] = state[2];
        out[1] = state[2] * s_mult;
    }
}

size_t budget_scale_state_bytes() { return 32 + sizeof(double) * kScaleProbes; }

hipError_t launch_budget_scale(const float *pred, long long n, float s_mult, double target, int nmin, int nmax,
                               int n_ref, int rounds, long long max_rows, void *state_buf, float *out, hipStream_t s)
{
    if (n < 1 || rounds < 1 || max_rows < 1) return hipErrorInvalidValue;
    const long long step = std::max<long long>(1, n / max_rows);
    const long long m = (n + step - 1) / step;
    float *state = static_cast<float *>(state_buf);
    double *sums = reinterpret_cast<double *>(static_cast<unsigned char *>(state_buf) + 32);
    const unsigned grid = (unsigned)std::min<long long>((m + 255) / 256, 1024);
    hipLaunchKernelGGL(scale_clear_kernel, dim3(1), dim3(kScaleProbes), 0, s, state, sums);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) {
        hipLaunchKernelGGL(scale_min_kernel, dim3(std::min(grid, 128u)), dim3(256), 0, s, pred, step, m, s_mult,
                           state);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(scale_setup_kernel, dim3(1), dim3(64), 0, s, nmax, state);
        e = hipGetLastError();
    }
    // each thread of the sums kernel folds several rows before the 64-probe
    // reduction across its wave, which costs about as much as 8 rows
    const unsigned sums_grid = (unsigned)std::min<long long>((m + 2047) / 2048, 128);
    for (int r = 0; r < rounds && e == hipSuccess; ++r) {
        hipLaunchKernelGGL(scale_sums_kernel, dim3(std::max(sums_grid, 1u)), dim3(256), 0, s, pred, step, m, s_mult,
                           nmin, nmax, 1.0f / (float)n_ref, state, sums);
        e = hipGetLastError();
        if (e != hipSuccess) break;
        hipLaunchKernelGGL(scale_pick_kernel, dim3(1), dim3(kScaleProbes), 0, s, m, target, r == rounds - 1 ? 1 : 0,
                           state, sums);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(scale_out_kernel, dim3(1), dim3(64), 0, s, state, s_mult, out);
        e = hipGetLastError();
    }
    return e;
}

hipError_t launch_mlp_forward(const float *P, const uint16_t *X, long long n, float *out, hipStream_t s)
{
    // waves loop over 16-row tiles.  Each wave first loads the whole network
    // into registers, so the grid is one resident round of waves (three
    // workgroups of 4 waves per CU on 256 CUs) and each wave amortises that
    // load over many tiles.
    const long long tiles = (n + 15) / 16;
    const unsigned grid = (unsigned)std::min<long long>((tiles + 4 * kTiles - 1) / (4 * kTiles), 768);
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(std::max(grid, 1u)), dim3(256), 0, s, P, X, n, out,
                       reinterpret_cast<uintptr_t>(X) % 8 == 0);
    return hipGetLastError();
}

hipError_t launch_mlp_grad(const float *P, const uint16_t *X, const float *target, long long n, float inv_total,
                           int loss_kind, float *grad, float *loss, hipStream_t s)
{
    const unsigned grid = (unsigned)std::min<long long>((n + 255) / 256, 256);
    hipLaunchKernelGGL(mlp_grad_kernel, dim3(std::max(grid, 1u)), dim3(kGradBlock), 0, s, P, X, target, n, inv_total,
                       loss_kind, grad, loss, reinterpret_cast<uintptr_t>(X) % 8 == 0);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(float *P, const float *grad, float *m, float *v, float lr, float b1, float b2, float eps,
                           float bc1, float bc2, hipStream_t s)
{
    hipLaunchKernelGGL(mlp_adam_kernel, dim3((kMlpParams + 255) / 256), dim3(256), 0, s, P, grad, m, v, lr, b1, b2,
                       eps, bc1, bc2);
    return hipGetLastError();
}

hipError_t launch_features(const float *u, int in_w, int in_h, int out_w, int out_h, float zoom, float radius,
                           float sd, float sigma, int channel, uint16_t *X, hipStream_t s)
{
    const long long n = (long long)out_w * out_h;
    hipLaunchKernelGGL(feature_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, u, in_w, in_h, out_w, out_h,
                       1.0f / zoom, radius / 0.3f, sd / 0.15f, sigma / 2.0f, zoom / 4.0f, channel, X,
                       reinterpret_cast<uintptr_t>(X) % 16 == 0);
    return hipGetLastError();
}

}  // namespace fg
