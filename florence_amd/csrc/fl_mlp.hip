// Warm-start predictor: a 3-layer MLP (in -> 128 -> 128 -> out, tanh) with FP32 master
// weights and BF16 MFMA GEMMs (v_mfma_f32_16x16x32_bf16, FP32 accumulation), forward,
// backward (MSE loss) and Adam, all on the device: one launch forward, two backward, one
// for Adam.  No reference counterpart.
//
// Parameter block (FP32, contiguous):  W1[IP][H] b1[H] W2[H][H] b2[H] W3[H][OP] b3[OP]
// with IP = 32 (inputs padded), H = 128, OP = 32 (outputs padded).  Activations are
// row-major [N][width] FP32.  Reductions are two-pass in a fixed order: bitwise
// reproducible.
#include <algorithm>
#include <cmath>

#include "fl_common.hpp"

namespace fl {

constexpr int MLP_IP = 32, MLP_H = 128, MLP_OP = 32;
constexpr int64_t OFF_W1 = 0, OFF_B1 = OFF_W1 + MLP_IP * MLP_H, OFF_W2 = OFF_B1 + MLP_H,
                  OFF_B2 = OFF_W2 + MLP_H * MLP_H, OFF_W3 = OFF_B2 + MLP_H, OFF_B3 = OFF_W3 + MLP_H * MLP_OP,
                  MLP_NPARAM = OFF_B3 + MLP_OP;

typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 b8_t __attribute__((ext_vector_type(8)));

typedef __bf16 b4_t __attribute__((ext_vector_type(4)));
// four floats at any float's alignment (rows of a caller's buffer)
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));

constexpr int MR = 32;                 // rows per workgroup step, and the MFMA's inner length in the weight gradients
constexpr int LDI = MLP_IP + 8;        // bf16 strides of the LDS tiles: 16-byte rows, two-way bank use at most
constexpr int LDH = MLP_H + 8, LDR = MR + 8;
constexpr int WS_NIN = 10;

__device__ __forceinline__ f4_t mfma_bf16(b8_t a, b8_t b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// B fragment of a [K][ld] matrix: column n, rows k0 .. k0 + 7
__device__ __forceinline__ b8_t frag_cols(const float *__restrict__ W, int ld, int k0, int n) {
    b8_t f;
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = (__bf16)W[(k0 + i) * ld + n];
    return f;
}

// B fragment of the transpose of a [N][ld] matrix: row n, columns k0 .. k0 + 7
__device__ __forceinline__ b8_t frag_rows(const float *__restrict__ W, int ld, int n, int k0) {
    const f4u_t lo = *reinterpret_cast<const f4u_t *>(W + n * ld + k0);
    const f4u_t hi = *reinterpret_cast<const f4u_t *>(W + n * ld + k0 + 4);
    b8_t f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[i] = (__bf16)lo[i];
        f[4 + i] = (__bf16)hi[i];
    }
    return f;
}

// The warm-start predictor's inputs and outputs around the network (PREDICT form).
struct WsArgs {
    const double *X, *u1, *u2;     // features: coordinates, the two last states
    double lam;
    const float *norm_in, *norm_out;
    const double *a, *b;           // the base 2 a - b the correction is added to
    const uint8_t *free_mask;
    const double *u_bc;
    double *u;
};

// One standardised input of node n: reference coordinates, the previous displacement, the
// last increment's step (u1 - u2) and the load factor; columns 10..31 are zero.  Feeding
// u1 - u2 rather than u2 keeps the step resolvable after BF16 rounding.
__device__ __forceinline__ float ws_feature(const double *__restrict__ X, const double *__restrict__ u1,
                                            const double *__restrict__ u2, double lam, const float *__restrict__ norm,
                                            int64_t n, int c) {
    double v = 0.0;
    if (c < 3) v = X[3 * n + c];
    else if (c < 6) v = u1[3 * n + c - 3];
    else if (c < 9) v = u1[3 * n + c - 6] - u2[3 * n + c - 6];
    else if (c == 9) v = lam;
    return c < WS_NIN ? (float)((v - (double)norm[c]) * (double)norm[WS_NIN + c]) : 0.f;
}

// u = free ? 2 a - b + (scale * Y + shift) : u_bc   (scale/shift = out_norm[0..2]/[3..5])
__device__ __forceinline__ double ws_corrected(double a, double b, float y, const float *__restrict__ out_norm, int c,
                                               bool free, double bc) {
    const double corr = (double)out_norm[c] * (double)y + (double)out_norm[3 + c];
    return free ? 2.0 * a - b + corr : bc;
}

// All three layers of MR rows per step, one workgroup of four waves.  Wave w owns the
// hidden columns [32 w, 32 w + 32) and keeps their weights in registers as BF16 fragments
// for every step it runs; only the activations pass through LDS.  A layer's sums run over
// k = 0, 32, ... in one accumulator, so the results do not depend on the split.  What
// bounds it is latency: at 11664 rows the three products are 0.6 GFLOP and 14 MB of
// activations.  As three 64 x 64-tile products through memory (one load per element,
// converted in the inner loop) they took 52 us; this kernel takes 9.5 us at 8192 rows and,
// with the inputs and outputs below fused in, 10.2 us at 11664 (56 us in five launches).
// PREDICT: the inputs are formed from the nodes' states and the outputs added to
// the extrapolation in the same launch (no activation reaches memory).
template <bool PREDICT>
__global__ __launch_bounds__(256) void mlp_forward_kernel(const float *__restrict__ P, const float *__restrict__ X,
                                                          int64_t N, float *__restrict__ H1, float *__restrict__ H2,
                                                          float *__restrict__ Y, WsArgs ws) {
    __shared__ __attribute__((aligned(16))) __bf16 sX[MR * LDI];
    __shared__ __attribute__((aligned(16))) __bf16 sH[2][MR * LDH];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int n0 = 32 * wave + li;                       // hidden columns n0, n0 + 16
    const int mt = wave >> 1, no = 16 * (wave & 1) + li;   // this wave's tile of the output layer
    b8_t w1[2], w2[4][2], w3[4];
    float b1[2], b2[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        w1[j] = frag_cols(P + OFF_W1, MLP_H, 8 * lk, n0 + 16 * j);
        b1[j] = P[OFF_B1 + n0 + 16 * j];
        b2[j] = P[OFF_B2 + n0 + 16 * j];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) w2[ks][j] = frag_cols(P + OFF_W2, MLP_H, 32 * ks + 8 * lk, n0 + 16 * j);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) w3[ks] = frag_cols(P + OFF_W3, MLP_OP, 32 * ks + 8 * lk, no);
    const float b3 = P[OFF_B3 + no];
    const int64_t nblk = (N + MR - 1) / MR;
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        const int64_t r0 = blk * MR;
        {
            const int r = tid >> 3, c = 4 * (tid & 7);
            const int64_t row = r0 + r;
            b4_t v = {(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
            if (row < N) {
                if constexpr (PREDICT) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float f = ws_feature(ws.X, ws.u1, ws.u2, ws.lam, ws.norm_in, row, c + i);
                        // rounded to FP32 first, as the feature array holds it: the compiler
                        // turns double -> float -> bf16 into one conversion, which rounds the
                        // doubles next to a bf16 tie the other way
                        asm volatile("" : "+v"(f));
                        v[i] = (__bf16)f;
                    }
                } else {
                    const f4u_t x = *reinterpret_cast<const f4u_t *>(X + row * MLP_IP + c);
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = (__bf16)x[i];
                }
            }
            *reinterpret_cast<b4_t *>(sX + r * LDI + c) = v;
        }
        __syncthreads();
#pragma unroll
        for (int layer = 0; layer < 2; ++layer) {
            f4_t acc[2][2] = {};
            if (layer == 0) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const b8_t a = *reinterpret_cast<const b8_t *>(sX + (16 * t + li) * LDI + 8 * lk);
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[t][j] = mfma_bf16(a, w1[j], acc[t][j]);
                }
            } else {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const b8_t a = *reinterpret_cast<const b8_t *>(sH[0] + (16 * t + li) * LDH + 32 * ks + 8 * lk);
#pragma unroll
                        for (int j = 0; j < 2; ++j) acc[t][j] = mfma_bf16(a, w2[ks][j], acc[t][j]);
                    }
            }
            float *H = layer ? H2 : H1;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int m = 16 * t + 4 * lk + r, n = n0 + 16 * j;
                        const float v = tanhf(acc[t][j][r] + (layer ? b2[j] : b1[j]));
                        sH[layer][m * LDH + n] = (__bf16)v;
                        if (!PREDICT && r0 + m < N) H[(r0 + m) * MLP_H + n] = v;
                    }
            __syncthreads();
        }
        f4_t acc = {};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            acc = mfma_bf16(*reinterpret_cast<const b8_t *>(sH[1] + (16 * mt + li) * LDH + 32 * ks + 8 * lk), w3[ks],
                            acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = r0 + 16 * mt + 4 * lk + r;
            const float v = acc[r] + b3;
            if (row >= N) continue;
            if constexpr (PREDICT) {
                if (no < 3) {
                    const int64_t d = 3 * row + no;
                    ws.u[d] = ws_corrected(ws.a[d], ws.b[d], v, ws.norm_out, no, ws.free_mask[d] != 0, ws.u_bc[d]);
                }
            } else {
                Y[row * MLP_OP + no] = v;
            }
        }
        // the next step's sX, sH[0] and sH[1] writes each follow a barrier after their last reads
    }
}

// The whole backward pass of the rows r = blockIdx.x MR + i, then the next gridDim.x MR
// rows: per step dY, dZ2 = (dY W3^T)(1 - H2^2) and dZ1 = (dZ2 W2^T)(1 - H1^2) stay in
// LDS, and the weight gradients A^T dZ of the step's rows (one MFMA step of inner length
// MR per 16 x 16 tile) are added up in registers, 24 tiles per wave.  Each workgroup
// writes its sums once, mlp_reduce_kernel adds the workgroups' in a fixed order.  Before,
// each weight gradient was one product with the whole batch as its inner length, four
// workgroups in all, and each bias sum eight: 2.6 of the 2.72 ms training step at 8192
// rows; here 16.6 us and 4.9 us for the sums (29 us the whole step).
// Wave w owns the hidden columns [32 w, 32 w + 32) of dZ2, dZ1, dW2, dW1 and the same
// rows of dW3.
constexpr int MLP_PARTS = 256;   // workgroups (and partial gradients) at most: one per CU
__global__ __launch_bounds__(256, 2) void mlp_backward_kernel(const float *__restrict__ P, const float *__restrict__ X,
                                                           const float *__restrict__ H1, const float *__restrict__ H2,
                                                           const float *__restrict__ Y, const float *__restrict__ T,
                                                           int64_t N, int nout, float *__restrict__ part,
                                                           double *__restrict__ lpart) {
    // [feature][row] tiles (operands whose inner index is the row) and [row][feature] ones
    __shared__ __attribute__((aligned(16))) __bf16 sXt[MLP_IP * LDR], sH1t[MLP_H * LDR], sH2t[MLP_H * LDR];
    __shared__ __attribute__((aligned(16))) __bf16 sdYt[MLP_OP * LDR], sZ2t[MLP_H * LDR], sZ1t[MLP_H * LDR];
    __shared__ __attribute__((aligned(16))) __bf16 sdY[MR * LDI], sZ2[MR * LDH];
    __shared__ double sl[256];
    __shared__ float s3[8][MLP_OP];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int n0 = 32 * wave + li;
    b8_t w3[2], w2[4][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        w3[j] = frag_rows(P + OFF_W3, MLP_OP, n0 + 16 * j, 8 * lk);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) w2[ks][j] = frag_rows(P + OFF_W2, MLP_H, n0 + 16 * j, 32 * ks + 8 * lk);
    }
    f4_t a2[8][2] = {}, a1[2][2] = {}, a3[2][2] = {};
    float c2[2] = {0.f, 0.f}, c1[2] = {0.f, 0.f}, c3 = 0.f;   // column sums of dZ2, dZ1, dY
    double loss = 0.0;
    const int64_t nblk = N / MR;
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        const int64_t r0 = blk * MR;
        {
            // 16 rows of one hidden feature per thread, coalesced over the features
            const int f = tid & 127, h = 16 * (tid >> 7);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const float *H = (s ? H2 : H1) + (r0 + h) * MLP_H + f;
                b8_t v[2];
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i >> 3][i & 7] = (__bf16)H[i * MLP_H];
                __bf16 *d = (s ? sH2t : sH1t) + f * LDR + h;
                *reinterpret_cast<b8_t *>(d) = v[0];
                *reinterpret_cast<b8_t *>(d + 8) = v[1];
            }
            const int c = tid & 31, q = 4 * (tid >> 5);
            b4_t xv, yv;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t k = (r0 + q + i) * MLP_IP + c;   // MLP_IP == MLP_OP
                xv[i] = (__bf16)X[k];
                float g = 0.f;
                if (c < nout) {
                    const float d = Y[k] - T[k];
                    g = 2.f * d / (float)(nout * N);
                    loss += (double)d * d;
                }
                c3 += g;
                yv[i] = (__bf16)g;
                sdY[(q + i) * LDI + c] = yv[i];
            }
            *reinterpret_cast<b4_t *>(sXt + c * LDR + q) = xv;
            *reinterpret_cast<b4_t *>(sdYt + c * LDR + q) = yv;
        }
        __syncthreads();
        // dZ2 and dW3
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const b8_t a = *reinterpret_cast<const b8_t *>(sdY + (16 * t + li) * LDI + 8 * lk);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f4_t d = mfma_bf16(a, w3[j], f4_t{0.f, 0.f, 0.f, 0.f});
                const int n = n0 + 16 * j, m = 16 * t + 4 * lk;
                b4_t zv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float h = H2[(r0 + m + r) * MLP_H + n];
                    const float z = d[r] * (1.f - h * h);
                    c2[j] += z;
                    zv[r] = (__bf16)z;
                    sZ2[(m + r) * LDH + n] = zv[r];
                }
                *reinterpret_cast<b4_t *>(sZ2t + n * LDR + m) = zv;
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const b8_t a = *reinterpret_cast<const b8_t *>(sH2t + (n0 + 16 * i) * LDR + 8 * lk);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                a3[i][j] = mfma_bf16(a, *reinterpret_cast<const b8_t *>(sdYt + (16 * j + li) * LDR + 8 * lk), a3[i][j]);
        }
        __syncthreads();
        // dZ1 and dW2
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f4_t d[2] = {};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const b8_t a = *reinterpret_cast<const b8_t *>(sZ2 + (16 * t + li) * LDH + 32 * ks + 8 * lk);
#pragma unroll
                for (int j = 0; j < 2; ++j) d[j] = mfma_bf16(a, w2[ks][j], d[j]);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int n = n0 + 16 * j, m = 16 * t + 4 * lk;
                b4_t zv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float h = H1[(r0 + m + r) * MLP_H + n];
                    const float z = d[j][r] * (1.f - h * h);
                    c1[j] += z;
                    zv[r] = (__bf16)z;
                }
                *reinterpret_cast<b4_t *>(sZ1t + n * LDR + m) = zv;
            }
        }
        {
            b8_t b[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const b8_t *>(sZ2t + (n0 + 16 * j) * LDR + 8 * lk);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const b8_t a = *reinterpret_cast<const b8_t *>(sH1t + (16 * i + li) * LDR + 8 * lk);
#pragma unroll
                for (int j = 0; j < 2; ++j) a2[i][j] = mfma_bf16(a, b[j], a2[i][j]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const b8_t a = *reinterpret_cast<const b8_t *>(sXt + (16 * i + li) * LDR + 8 * lk);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                a1[i][j] = mfma_bf16(a, *reinterpret_cast<const b8_t *>(sZ1t + (n0 + 16 * j) * LDR + 8 * lk), a1[i][j]);
        }
        __syncthreads();
    }
    float *o = part + (int64_t)blockIdx.x * MLP_NPARAM;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + 16 * j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int i = 0; i < 8; ++i) o[OFF_W2 + (16 * i + 4 * lk + r) * MLP_H + n] = a2[i][j][r];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                o[OFF_W1 + (16 * i + 4 * lk + r) * MLP_H + n] = a1[i][j][r];
                o[OFF_W3 + (32 * wave + 16 * i + 4 * lk + r) * MLP_OP + 16 * j + li] = a3[i][j][r];
            }
        }
        // the four lk groups hold the rows 4 lk + r of a column
        float t2 = c2[j], t1 = c1[j];
        t2 += __shfl_xor(t2, 16, 64);
        t1 += __shfl_xor(t1, 16, 64);
        t2 += __shfl_xor(t2, 32, 64);
        t1 += __shfl_xor(t1, 32, 64);
        if (lk == 0) {
            o[OFF_B2 + n] = t2;
            o[OFF_B1 + n] = t1;
        }
    }
    s3[tid >> 5][tid & 31] = c3;
    sl[tid] = loss;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (tid < off) sl[tid] += sl[tid + off];
        __syncthreads();
    }
    if (tid < MLP_OP) {
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) s += s3[q][tid];
        o[OFF_B3 + tid] = s;
    }
    if (tid == 0) lpart[blockIdx.x] = sl[0];
}

// Gr[i] = sum of the workgroups' partial gradients in a fixed order: 64 parameters per
// workgroup, wave g takes the partials g, g + 4, ...; the last workgroup sums the loss.
__global__ __launch_bounds__(256) void mlp_reduce_kernel(const float *__restrict__ part,
                                                         const double *__restrict__ lpart, int np, double scale,
                                                         float *__restrict__ Gr, float *__restrict__ loss) {
    __shared__ double sl[256];
    __shared__ float sg[4][64];
    const int tid = threadIdx.x;
    if (blockIdx.x == gridDim.x - 1) {
        sl[tid] = tid < np ? lpart[tid] : 0.0;
        __syncthreads();
        for (int off = 128; off > 0; off >>= 1) {
            if (tid < off) sl[tid] += sl[tid + off];
            __syncthreads();
        }
        if (tid == 0) *loss = (float)(sl[0] * scale);
        return;
    }
    const int64_t i = (int64_t)blockIdx.x * 64 + (tid & 63);
    float s = 0.f;
    if (i < MLP_NPARAM) {
#pragma unroll 16
        for (int p = tid >> 6; p < np; p += 4) s += part[(int64_t)p * MLP_NPARAM + i];
    }
    sg[tid >> 6][tid & 63] = s;
    __syncthreads();
    if (tid < 64 && i < MLP_NPARAM) Gr[i] = (sg[0][tid] + sg[1][tid]) + (sg[2][tid] + sg[3][tid]);
}

__global__ void adam_kernel(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, int64_t n, float lr, float b1, float b2, float eps, float c1,
                            float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ws_feature of every node and column
__global__ void ws_features_kernel(const double *__restrict__ X, const double *__restrict__ u1,
                                   const double *__restrict__ u2, double lam, int64_t nnode,
                                   const float *__restrict__ norm, float *__restrict__ F) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnode * MLP_IP) return;
    const int64_t n = i / MLP_IP;
    F[i] = ws_feature(X, u1, u2, lam, norm, n, (int)(i - n * MLP_IP));
}

__global__ void ws_apply_kernel(const double *__restrict__ u1, const double *__restrict__ u2,
                                const float *__restrict__ Y, int64_t nnode, const float *__restrict__ out_norm,
                                const uint8_t *__restrict__ free_mask, const double *__restrict__ u_bc,
                                double *__restrict__ u) {
    const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= 3 * nnode) return;
    const int64_t n = d / 3;
    const int c = (int)(d % 3);
    u[d] = ws_corrected(u1[d], u2[d], Y[n * MLP_OP + c], out_norm, c, free_mask[d] != 0, u_bc[d]);
}

// one workgroup per MR rows up to four per CU; above that each runs several steps on the
// weights it holds
static unsigned forward_grid(int64_t N) { return (unsigned)std::min<int64_t>((N + MR - 1) / MR, 1024); }

static int64_t backward_parts(int64_t N) { return std::min<int64_t>((N + MR - 1) / MR, MLP_PARTS); }

}  // namespace fl

using namespace fl;

extern "C" {

int64_t fl_mlp_param_count(void) { return MLP_NPARAM; }

int fl_mlp_forward(const float *P, const float *X, int64_t N, float *H1, float *H2, float *Y, void *stream) {
    if (!P || !X || !H1 || !H2 || !Y || N <= 0) {
        set_error("fl_mlp_forward: invalid argument");
        return FL_E_ARG;
    }
    mlp_forward_kernel<false><<<forward_grid(N), 256, 0, as_stream(stream)>>>(P, X, N, H1, H2, Y, WsArgs{});
    FL_LAUNCH_CHECK();
    return 0;
}

size_t fl_mlp_workspace_size(int64_t N) {
    const int64_t np = backward_parts(N);
    return align_up(sizeof(float) * np * MLP_NPARAM, 256) + align_up(sizeof(double) * np, 256) + 1024;
}

int fl_mlp_backward(const float *P, const float *X, const float *H1, const float *H2, const float *Y,
                    const float *Tgt, int64_t N, int32_t nout, float *Gr, float *loss, void *workspace,
                    size_t workspace_bytes, void *stream) {
    hipStream_t st = as_stream(stream);
    if (!P || !X || !H1 || !H2 || !Y || !Tgt || !Gr || !loss || N <= 0 || nout <= 0 || nout > MLP_OP) {
        set_error("fl_mlp_backward: invalid argument");
        return FL_E_ARG;
    }
    if (N % MR != 0) {
        set_error("fl_mlp_backward: batch size must be a multiple of %d", MR);
        return FL_E_ARG;
    }
    const int64_t np = backward_parts(N);
    Carve cv(workspace, workspace_bytes);
    float *part = cv.take<float>(np * MLP_NPARAM);
    double *lp = cv.take<double>(np);
    if (!cv.ok) {
        set_error("fl_mlp_backward: workspace too small");
        return FL_E_SPACE;
    }
    mlp_backward_kernel<<<(unsigned)np, 256, 0, st>>>(P, X, H1, H2, Y, Tgt, N, nout, part, lp);
    mlp_reduce_kernel<<<(unsigned)((MLP_NPARAM + 63) / 64 + 1), 256, 0, st>>>(part, lp, (int)np,
                                                                              1.0 / ((double)nout * N), Gr, loss);
    FL_LAUNCH_CHECK();
    return 0;
}

int fl_mlp_adam(float *P, const float *Gr, float *m, float *v, float lr, float beta1, float beta2, float eps,
                int32_t step, void *stream) {
    hipStream_t st = as_stream(stream);
    if (!P || !Gr || !m || !v || step <= 0) {
        set_error("fl_mlp_adam: invalid argument");
        return FL_E_ARG;
    }
    const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
    adam_kernel<<<(unsigned)((MLP_NPARAM + 255) / 256), 256, 0, st>>>(P, Gr, m, v, MLP_NPARAM, lr, beta1, beta2,
                                                                       eps, c1, c2);
    FL_LAUNCH_CHECK();
    return 0;
}

int fl_warmstart_features(const double *X, const double *u1, const double *u2, double load_factor, int64_t nnode,
                          const float *norm, float *F, void *stream) {
    if (!X || !u1 || !u2 || !norm || !F || nnode <= 0) {
        set_error("fl_warmstart_features: invalid argument");
        return FL_E_ARG;
    }
    const int64_t n = nnode * MLP_IP;
    ws_features_kernel<<<(unsigned)((n + 255) / 256), 256, 0, as_stream(stream)>>>(X, u1, u2, load_factor, nnode,
                                                                                   norm, F);
    FL_LAUNCH_CHECK();
    return 0;
}

int fl_warmstart_predict(const float *P, const double *X, const double *u1, const double *u2, double load_factor,
                         int64_t nnode, const float *norm_in, const float *norm_out, const double *a, const double *b,
                         const uint8_t *free_mask, const double *u_bc, double *u, void *stream) {
    if (!P || !X || !u1 || !u2 || !norm_in || !norm_out || !a || !b || !free_mask || !u_bc || !u || nnode <= 0) {
        set_error("fl_warmstart_predict: invalid argument");
        return FL_E_ARG;
    }
    const WsArgs ws = {X, u1, u2, load_factor, norm_in, norm_out, a, b, free_mask, u_bc, u};
    mlp_forward_kernel<true><<<forward_grid(nnode), 256, 0, as_stream(stream)>>>(P, nullptr, nnode, nullptr, nullptr,
                                                                                nullptr, ws);
    FL_LAUNCH_CHECK();
    return 0;
}

int fl_warmstart_apply(const double *u1, const double *u2, const float *Y, int64_t nnode, const float *out_norm,
                       const uint8_t *free_mask, const double *u_bc, double *u, void *stream) {
    if (!u1 || !u2 || !Y || !out_norm || !free_mask || !u_bc || !u || nnode <= 0) {
        set_error("fl_warmstart_apply: invalid argument");
        return FL_E_ARG;
    }
    ws_apply_kernel<<<(unsigned)((3 * nnode + 255) / 256), 256, 0, as_stream(stream)>>>(u1, u2, Y, nnode, out_norm,
                                                                                       free_mask, u_bc, u);
    FL_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
