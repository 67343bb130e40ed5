// mlp.hip -- ensemble MLP for the mouth-[Ca2+] surrogate: hand-written BF16
// MFMA GEMM (FP32 accumulation), fused bias/SiLU epilogues, backward pass and
// Adam, behind include/casim_surrogate.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../include/casim_surrogate.h"
#include "dyad_internal.hpp"

using namespace casim;

namespace casim {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

// float -> bf16 with round-to-nearest-even (finite inputs).
__host__ __device__ inline uint16_t f2bf(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(uint16_t h) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// ---------------------------------------------------------------------------
// C[M x N] = op(A) op(B) (+ beta C), BF16 operands, FP32 accumulation.
// 64 x 64 tile per workgroup of four waves; each wave owns a 32 x 32 quarter
// as 2 x 2 v_mfma_f32_16x16x32_bf16 tiles.  Both LDS tiles keep k contiguous
// ([m][k] and [n][k]), so a lane's eight k-values of one MFMA operand are one
// 16-byte LDS read; A lanes supply row (lane % 16), B lanes column (lane % 16),
// and the accumulator lane holds rows 4 (lane / 16) .. +3 of column lane % 16.
constexpr int GBM = 64, GBN = 64, GBK = 32, GPAD = 8;

__global__ __launch_bounds__(256) void k_gemm(const uint16_t *__restrict__ A, int lda, int ta,
                                              const uint16_t *__restrict__ B, int ldb, int tb, float *__restrict__ C,
                                              int ldc, int M, int N, int K, float beta) {
    __shared__ __attribute__((aligned(16))) uint16_t As[GBM][GBK + GPAD];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[GBN][GBK + GPAD];
    const int m0 = blockIdx.y * GBM, n0 = blockIdx.x * GBN;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    f32x4_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    for (int k0 = 0; k0 < K; k0 += GBK) {
        if (!ta) {
            const int m = t >> 2, kk = (t & 3) * 8;
            const int gm = m0 + m;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int gk = k0 + kk + e;
                As[m][kk + e] = (gm < M && gk < K) ? A[(size_t)gm * lda + gk] : (uint16_t)0;
            }
        } else {
            const int kk = t >> 3, m = (t & 7) * 8;
            const int gk = k0 + kk;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int gm = m0 + m + e;
                As[m + e][kk] = (gm < M && gk < K) ? A[(size_t)gk * lda + gm] : (uint16_t)0;
            }
        }
        if (!tb) {
            const int kk = t >> 3, n = (t & 7) * 8;
            const int gk = k0 + kk;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int gn = n0 + n + e;
                Bs[n + e][kk] = (gn < N && gk < K) ? B[(size_t)gk * ldb + gn] : (uint16_t)0;
            }
        } else {
            const int n = t >> 2, kk = (t & 3) * 8;
            const int gn = n0 + n;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int gk = k0 + kk + e;
                Bs[n][kk + e] = (gn < N && gk < K) ? B[(size_t)gn * ldb + gk] : (uint16_t)0;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bf16x8_t a = *reinterpret_cast<const bf16x8_t *>(&As[wm + i * 16 + (l & 15)][(l >> 4) * 8]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf16x8_t b = *reinterpret_cast<const bf16x8_t *>(&Bs[wn + j * 16 + (l & 15)][(l >> 4) * 8]);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wm + i * 16 + (l >> 4) * 4 + r;
                const int col = n0 + wn + j * 16 + (l & 15);
                if (row < M && col < N) {
                    float v = acc[i][j][r];
                    if (beta != 0.f) v += beta * C[(size_t)row * ldc + col];
                    C[(size_t)row * ldc + col] = v;
                }
            }
}

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + __expf(-z)); }

// sigmoidf_ of N values.  1 / d for 1 <= d <= 2^125 by the hardware's
// reciprocal and one Newton step, which gives the correctly rounded quotient,
// the compiler's result, for every float in that range (compared one by one);
// its general division takes 11 operations.  Below -86 the general one.
template <int N>
__device__ __forceinline__ void sigmoid_n(const float (&z)[N], float (&s)[N]) {
    float lo = z[0];
#pragma unroll
    for (int i = 1; i < N; ++i) lo = __builtin_fminf(lo, z[i]);
    if (lo < -86.f) {
#pragma unroll 1
        for (int i = 0; i < N; i += 4)
#pragma unroll
            for (int k = 0; k < N; k += 4)
                if (k == i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[k + r] = sigmoidf_(z[k + r]);
        return;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float d = 1.f + __expf(-z[i]), y = __builtin_amdgcn_rcpf(d);
        s[i] = __builtin_fmaf(__builtin_fmaf(-d, y, 1.f), y, y);
    }
}

// f2bf of four values by the conversion instruction (two values each, the same
// rounding)
__device__ __forceinline__ void f2bf4(const float (&f)[4], uint16_t (&h)[4]) {
    typedef float __attribute__((ext_vector_type(2))) f2_t;
    typedef __bf16 __attribute__((ext_vector_type(2))) b2_t;
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const b2_t b = __builtin_convertvector((f2_t{f[i], f[i + 1]}), b2_t);
        std::memcpy(h + i, &b, sizeof b);
    }
}

// Z += b (per column); H = bf16(SiLU(Z)) or bf16(Z) for the last layer.
__global__ void k_bias_act(float *__restrict__ Z, const float *__restrict__ b, uint16_t *__restrict__ H, int rows,
                           int cols, int act) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * cols) return;
    const float z = Z[i] + b[i % cols];
    Z[i] = z;
    if (H) H[i] = f2bf(act ? z * sigmoidf_(z) : z);
}

// Inference of one ensemble member for 16 RT rows per workgroup, every layer in
// one launch: the normalised BF16 input (k_gather's arithmetic), each hidden
// layer as BF16 MFMA products with FP32 accumulation (k_gemm's operand layout
// and k order), bias, SiLU and BF16 rounding (k_bias_act's), and the linear
// output, with the activations in LDS.  The weights come zero-padded in the
// order of MFMA operands (k_wt).  Per output element the operations and their
// order are those of k_gather + k_gemm + k_bias_act, so the outputs are the
// same bits.  Grid: (row tiles, members).
//
// Few rows: sixteen waves with 16 columns each, 32 rows.  A workgroup is a
// latency chain of layers, so a lane has all of the next layer's weights on
// their way while a layer runs.  Many rows: eight waves with 32 columns each, 64
// rows, two workgroups per CU.  The weights are then read half as often and the
// rows' operands from LDS feed two products; what bounds it is the SiLU, about
// 14 vector operations per activation (276 us with the compiler's division in
// it, 25 operations).  Times in us for five members of width
// 256, depth 4 (before: weights in plain rows, 32 rows per workgroup):
//   rows        512   2048   4096   8192   16384   55003
//   before       -      -      -      -      195     658
//   32 rows      15     26     42     66     126     424
//   64 rows      26     28     32     50      78     240
// so 64 rows from INFER_BIG workgroups on, one per CU.
constexpr int IMR = 32, IMAXW = 256, IPADK = 8, IMAXM = 8, IMAXL = 8, IWAVES = IMAXW / 16;
constexpr size_t INFER_BIG = 256;
struct InferArgs {
    const uint16_t *wt[IMAXM];  // member's transposed weights
    const float *p[IMAXM];      // member's FP32 parameters (biases at boff)
    int wtoff[IMAXL], boff[IMAXL], kp[IMAXL], fout[IMAXL];
    int nl, n_in;
    const float *mean, *istd;
    const int *rows_d;  // rows of this call, where only the device knows them (or null)
};

// Place of element (n, k) of a [n][k] operand with nk blocks of 32 in k, in the
// order in which an MFMA operand's lanes hold it: blocks of 16 n and 32 k, in
// them lane by lane eight consecutive k.  A wave's load of a block is 1 KiB in
// a row; with plain rows it is 16 half lines, and L2 moves each line twice.
__host__ __device__ inline int frag_at(int n, int k, int nk) {
    return (((n >> 4) * nk + (k >> 5)) << 9) + (((k >> 3 & 3) << 4 | (n & 15)) << 3) + (k & 7);
}

// Every layer's and member's W [fin][fout] -> zero-padded operands of the
// forward product (n over fout, k over fin) and of the product with W^T of the
// backward pass (n over fin, k over fout).  Grid: (elements, 2 layers, members).
struct WtArgs {
    const uint16_t *pb[IMAXM];
    uint16_t *wt[IMAXM];
    int woff[IMAXL], fin[IMAXL], fout[IMAXL], off[2 * IMAXL];  // off: operand of layer g / 2, backward if g % 2
};
__global__ void k_wt(const WtArgs a) {
    const int g = blockIdx.y, L = g >> 1, back = g & 1, e = blockIdx.z;
    const int nn = back ? a.fin[L] : a.fout[L], nk = back ? a.fout[L] : a.fin[L];
    const int kp = (nk + 31) & ~31, np = (nn + 15) & ~15;
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= np * kp) return;
    const int n = i / kp, k = i - n * kp;
    uint16_t v = 0;
    if (n < nn && k < nk) v = a.pb[e][a.woff[L] + (back ? n * a.fout[L] + k : k * a.fout[L] + n)];
    a.wt[e][a.off[g] + frag_at(n, k, kp >> 5)] = v;
}

template <int CT, int RT>
__global__ __launch_bounds__(64 * IWAVES / CT, 4) void k_mlp_infer(const float *__restrict__ X, int rows,
                                                                   float *__restrict__ out, int ostride, InferArgs a) {
    constexpr int R = 16 * RT, NT = 64 * IWAVES / CT;
    constexpr int GR = CT == 1 ? 2 : 1;  // row tiles whose activations are formed together, as registers allow
    __shared__ __attribute__((aligned(16))) uint16_t H[2][R][IMAXW + IPADK];
    const int m0 = blockIdx.x * R, e = blockIdx.y;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    if (a.rows_d) rows = min(rows, *a.rows_d);
    if (m0 >= rows) return;
    const uint16_t *wt = a.wt[e];
    const float *pe = a.p[e];
    // every k-block of the wave's columns for layer L, and their biases, issued
    // together (blocks past the layer's K repeat its last one, columns past its
    // width its last tile; neither is used)
    auto fetch = [&](int L, bf16x8_t (&b)[CT][IMAXW / 32], float (&bias)[CT]) {
        const int N = a.fout[L], nk = a.kp[L] >> 5, nt = (N + 15) >> 4;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int ct = min(w * CT + c, nt - 1);
            const uint16_t *wf = wt + a.wtoff[L] + ((ct * nk) << 9) + l * 8;
#pragma unroll
            for (int kb = 0; kb < IMAXW / 32; ++kb)
                b[c][kb] = *reinterpret_cast<const bf16x8_t *>(wf + ((kb < nk ? kb : nk - 1) << 9));
            bias[c] = pe[a.boff[L] + min(ct * 16 + (l & 15), N - 1)];
        }
    };
    bf16x8_t bw[CT][IMAXW / 32], bn[CT][IMAXW / 32];
    float bias[CT], bias_n[CT];
    fetch(0, bw, bias);  // in flight while the input is staged
    const int kp0 = a.kp[0];
    for (int i = t; i < R * kp0; i += NT) {
        const int r = i / kp0, f = i - r * kp0;
        uint16_t v = 0;
        if (m0 + r < rows && f < a.n_in) v = f2bf((X[(size_t)(m0 + r) * a.n_in + f] - a.mean[f]) * a.istd[f]);
        H[0][r][f] = v;
    }
    __syncthreads();
    for (int L = 0; L < a.nl; ++L) {
        const int src = L & 1, N = a.fout[L], nk = a.kp[L] >> 5;
        const bool last = L == a.nl - 1;
        // the next layer's weights are in flight during this layer (the last
        // layer fetches itself again, so that the count of loads in flight is
        // the same every layer); a wave with two column tiles has the registers
        // for them only once its products are done
        if (CT == 1) fetch(last ? L : L + 1, bn, bias_n);
        f32x4_t acc[CT][RT];
        const bool on = w * CT * 16 < N;
        if (on) {
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int i = 0; i < RT; ++i) acc[c][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < IMAXW / 32; ++kb) {
                if (kb >= nk) break;
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const bf16x8_t av =
                        *reinterpret_cast<const bf16x8_t *>(&H[src][i * 16 + (l & 15)][32 * kb + (l >> 4) * 8]);
#pragma unroll
                    for (int c = 0; c < CT; ++c)
                        acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bw[c][kb], acc[c][i], 0, 0, 0);
                }
            }
        }
        float b0[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) b0[c] = bias[c];
        if (CT > 1 && !last) fetch(L + 1, bw, bias);
        if (on) {
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const int col = (w * CT + c) * 16 + (l & 15);
                if (col >= N) break;
#pragma unroll
                for (int i0 = 0; i0 < RT; i0 += GR) {
                    const int row = i0 * 16 + (l >> 4) * 4;
                    float z[4 * GR], sg[4 * GR];
#pragma unroll
                    for (int i = 0; i < 4 * GR; ++i) z[i] = acc[c][i0 + i / 4][i % 4] + b0[c];
                    if (last) {
#pragma unroll
                        for (int i = 0; i < 4 * GR; ++i) {
                            const int m = m0 + row + i / 4 * 16 + i % 4;
                            if (m < rows) out[(size_t)e * ostride + m] = z[i];
                        }
                    } else {
                        sigmoid_n(z, sg);
#pragma unroll
                        for (int i = 0; i < GR; ++i) {
                            const float f[4] = {z[4 * i] * sg[4 * i], z[4 * i + 1] * sg[4 * i + 1],
                                                z[4 * i + 2] * sg[4 * i + 2], z[4 * i + 3] * sg[4 * i + 3]};
                            uint16_t h[4];
                            f2bf4(f, h);
#pragma unroll
                            for (int r = 0; r < 4; ++r) H[src ^ 1][row + 16 * i + r][col] = h[r];
                        }
                    }
                }
            }
        }
        __syncthreads();
        if (CT == 1) {
#pragma unroll
            for (int kb = 0; kb < IMAXW / 32; ++kb) bw[0][kb] = bn[0][kb];
            bias[0] = bias_n[0];
        }
    }
}

// dH * SiLU'(z), s the sigmoid of z
__device__ __forceinline__ float silu_back(float dH, float z, float s) { return dH * s * (1.f + z * (1.f - s)); }

// dZ = dH * SiLU'(Z), kept in FP32 (bias gradient) and BF16 (GEMM operand).
__global__ void k_silu_back(const float *__restrict__ dH, const float *__restrict__ Z, float *__restrict__ dZ,
                            uint16_t *__restrict__ dZb, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float d = silu_back(dH[i], Z[i], sigmoidf_(Z[i]));
    dZ[i] = d;
    dZb[i] = f2bf(d);
}

// out[c] = sum_r X[r][c]
__global__ void k_colsum(const float *__restrict__ X, float *__restrict__ out, int rows, int cols) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    float s = 0.f;
#pragma unroll 16
    for (int r = 0; r < rows; ++r) s += X[(size_t)r * cols + c];
    out[c] = s;
}

// Gather and normalise rows of the training set into a BF16 batch.
__global__ void k_gather(const float *__restrict__ X, const float *__restrict__ Y, const int *__restrict__ idx,
                         int rows, int F, const float *__restrict__ mean, const float *__restrict__ istd,
                         float ym, float yis, uint16_t *__restrict__ Xb, float *__restrict__ Yb) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * F) return;
    const int r = (int)(i / F), f = (int)(i % F);
    const int src = idx ? idx[r] : r;
    Xb[i] = f2bf((X[(size_t)src * F + f] - mean[f]) * istd[f]);
    if (f == 0 && Yb) Yb[r] = (Y[src] - ym) * yis;
}

// Mean squared error of pred vs target; dpred = 2 (pred - t) / rows.
__global__ void k_mse(const float *__restrict__ pred, const float *__restrict__ tgt, float *__restrict__ dpred,
                      uint16_t *__restrict__ dpredb, float *__restrict__ sq, int rows) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows) return;
    const float e = pred[i] - tgt[i];
    const float d = 2.f * e / (float)rows;
    dpred[i] = d;
    dpredb[i] = f2bf(d);
    sq[i] = e * e;
}

// Adam on one FP32 master weight w with moments m and v and gradient g; the
// fused operations are written out, so that every kernel rounds alike.
struct AdamArgs {
    float lr, b1, b2, eps;
};
__device__ __forceinline__ void adam_update(float &w, float &m, float &v, float g, const AdamArgs &a, float c1, float c2) {
#pragma clang fp contract(off)
    m = __builtin_fmaf(1.f - a.b1, g, a.b1 * m);
    v = __builtin_fmaf(g, (1.f - a.b2) * g, a.b2 * v);
    w = w - a.lr * (m / c1) / (sqrtf(v / c2) + a.eps);
}
// ... with a refresh of the BF16 copy.
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, uint16_t *__restrict__ pb, size_t n, AdamArgs a, float c1, float c2) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float w = p[i], mi = m[i], vi = v[i];
    adam_update(w, mi, vi, g[i], a, c1, c2);
    m[i] = mi;
    v[i] = vi;
    p[i] = w;
    pb[i] = f2bf(w);
}

// ---------------------------------------------------------------------------
// A training step of every member in two launches.
//
// k_train_rows: forward, loss and the chain of dZ down the layers for IMR rows
// per workgroup, which need nothing of any other row: the activations of a
// tile stay in LDS as in k_mlp_infer.  It leaves what the weight gradients
// contract over the batch, the layers' inputs X and dZ in BF16 as operands with
// the batch as k (frag_at's order: a wave's 32 x 16 results are one block of
// 1 KiB), and dZ in FP32, rows first, for the bias gradients.
// k_train_weights: a 64 x 64 tile of a layer's dW = X^T dZ, or the column sums
// of dZ for 64 biases, and Adam on what it formed: weights, moments, the BF16
// copy and its transposed copy for the next forward pass.
//
// Per element the operations and their order are those of k_gather, k_gemm,
// k_bias_act, k_mse, k_silu_back, k_colsum and k_adam (k ascending in blocks of
// 32, column sums from the first row on), which a layer at a time and a member
// at a time took 34 launches per member and step, most of the time in k_colsum
// (187 us for 256 columns: a chain of dependent loads).
struct TrainArgs {
    uint16_t *wt[IMAXM];
    float *p[IMAXM], *am[IMAXM], *av[IMAXM];
    float c1[IMAXM], c2[IMAXM];
    int wtoff[2 * IMAXL], woff[IMAXL], boff[IMAXL], kp[IMAXL], fin[IMAXL], fout[IMAXL];
    int xt0[IMAXL], zt0[IMAXL];    // first tile of 16 columns of a layer's X and dZ operands
    int xtiles, ztiles;            // tiles of a member's operands, `tiles` blocks of 32 batch rows each
    int zcol[IMAXL], zcols;        // first column of a layer's dZ in FP32; columns of a member
    int tile0[IMAXL + 1];          // first weight tile of a layer
    int mg, nsum;                  // members; workgroups that form a member's column sums, its first ones
    int nl, n_in, B, tiles;        // tiles: of IMR rows
    const float *mean, *istd, *X, *Y;
    const int *perm;  // [members][rows] + the batch's first row
    int64_t rows;
    float ym, yis;
    uint16_t *XT, *DZT;
    float *DZ, *Z, *sq;  // sq: [members][sqn] + the batch's first row
    int64_t sqn;
    AdamArgs adam;
};

// prediction less the normalised target, which k_gather rounds and stores
__device__ __forceinline__ float target_error(float pred, float y, float ym, float yis) {
#pragma clang fp contract(off)
    const float t = (y - ym) * yis;
    return pred - t;
}

// This workgroup's unit of `units`, dealt so that the workgroups of a chiplet
// (block index modulo 8) take units in a row, the same member's and layer's:
// what they share is then read into one L2.  -1: none.
__device__ __forceinline__ int chiplet_unit(int units) {
    const int per = (units + 7) / 8, u = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    return (int)(blockIdx.x >> 3) < per && u < units ? u : -1;
}
__host__ inline unsigned chiplet_grid(int units) { return (unsigned)(units + 7) / 8 * 8; }

__device__ __forceinline__ uint64_t pack4(const uint16_t (&h)[4]) {
    return (uint64_t)h[0] | (uint64_t)h[1] << 16 | (uint64_t)h[2] << 32 | (uint64_t)h[3] << 48;
}

// Latency-bound: 32 workgroups per member at 1024 rows, each a chain of 2 depth
// + 1 layers of eight MFMA pairs per wave between barriers, weights fetched a
// layer ahead.  Five members, 1024 rows, width 256, depth 4: 32 us; 49 with the
// weights in plain rows.
__global__ __launch_bounds__(64 * IWAVES) void k_train_rows(const TrainArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t H[2][IMR][IMAXW + IPADK];
    __shared__ int src[IMR];
    __shared__ float ty[IMR];
    const int unit = chiplet_unit(a.tiles * a.mg);
    if (unit < 0) return;
    const int e = unit / a.tiles, tile = unit - e * a.tiles, m0 = tile * IMR;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    const uint16_t *wt = a.wt[e];
    const float *pe = a.p[e];
    uint16_t *XT = a.XT + ((size_t)e * a.xtiles * a.tiles + tile) * 512;  // block `tile` of column tile 0
    uint16_t *DZT = a.DZT + ((size_t)e * a.ztiles * a.tiles + tile) * 512;
    float *DZ = a.DZ + ((size_t)e * a.tiles * IMR + m0) * a.zcols;
    const size_t ts = (size_t)a.tiles * 512;  // one column tile
    f32x4_t *Z = reinterpret_cast<f32x4_t *>(a.Z) + ((size_t)e * a.tiles + tile) * (a.nl - 1) * IWAVES * 128 + w * 128 + l;
    const int n0 = w * 16, c = n0 + (l & 15), kq = (l >> 4) * 8, rq = (l >> 4) * 4;
    // the wave's k-blocks of an operand (blocks past K repeat the last one,
    // columns past the width the last tile; neither is used)
    auto weights = [&](int g, int N, int K, bf16x8_t(&b)[IMAXW / 32]) {
        const int nk = (K + 31) >> 5;
        const uint16_t *wf = wt + a.wtoff[g] + ((min(w, (N - 1) >> 4) * nk) << 9) + l * 8;
#pragma unroll
        for (int kb = 0; kb < IMAXW / 32; ++kb) b[kb] = *reinterpret_cast<const bf16x8_t *>(wf + ((kb < nk ? kb : nk - 1) << 9));
    };
    auto forward_w = [&](int L, bf16x8_t(&b)[IMAXW / 32], float &bias) {
        weights(2 * L, a.fout[L], a.fin[L], b);
        bias = pe[a.boff[L] + min(c, a.fout[L] - 1)];
    };
    auto backward_w = [&](int L, bf16x8_t(&b)[IMAXW / 32]) { weights(2 * L + 1, a.fin[L], a.fout[L], b); };
    auto product = [&](int from, int nk, const bf16x8_t(&b)[IMAXW / 32], f32x4_t(&acc)[2]) {
        acc[0] = acc[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < IMAXW / 32; ++kb) {
            if (kb >= nk) break;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x8_t av = *reinterpret_cast<const bf16x8_t *>(&H[from][i * 16 + (l & 15)][32 * kb + kq]);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b[kb], acc[i], 0, 0, 0);
            }
        }
    };
    bf16x8_t bw[IMAXW / 32], bn[IMAXW / 32];
    float bias, bias_n = 0.f;
    forward_w(0, bw, bias);
    if (t < IMR) {
        const int r = src[t] = m0 + t < a.B ? a.perm[(size_t)e * a.rows + m0 + t] : -1;
        ty[t] = r >= 0 ? a.Y[r] : 0.f;
    }
    __syncthreads();
    const int kp0 = a.kp[0];
    for (int i = t; i < IMR * kp0; i += 64 * IWAVES) {
        const int r = i / kp0, f = i - r * kp0;
        uint16_t v = 0;
        if (src[r] >= 0 && f < a.n_in) v = f2bf((a.X[(size_t)src[r] * a.n_in + f] - a.mean[f]) * a.istd[f]);
        H[0][r][f] = v;
    }
    __syncthreads();
    for (int i = t; i < a.n_in * (IMR / 4); i += 64 * IWAVES) {
        const int f = i / (IMR / 4), r = i % (IMR / 4) * 4;
        const uint16_t h[4] = {H[0][r][f], H[0][r + 1][f], H[0][r + 2][f], H[0][r + 3][f]};
        *reinterpret_cast<uint64_t *>(XT + (a.xt0[0] + (f >> 4)) * ts + frag_at(f & 15, r, 1)) = pack4(h);
    }
    const int last = a.nl - 1;
    for (int L = 0; L < last; ++L) {
        forward_w(L + 1, bn, bias_n);
        if (n0 < a.fout[L]) {
            f32x4_t acc[2];
            product(L & 1, a.kp[L] >> 5, bw, acc);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f32x4_t zz;
                float z[4], f[4];
                uint16_t h[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) zz[r] = z[r] = acc[i][r] + bias;
                sigmoid_n(z, f);
#pragma unroll
                for (int r = 0; r < 4; ++r) f[r] *= z[r];
                f2bf4(f, h);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = i * 16 + rq + r;
                    H[(L & 1) ^ 1][row][c] = h[r];
                    if (m0 + row >= a.B) h[r] = 0;
                }
                Z[(L * IWAVES * 2 + i) * 64] = zz;
                *reinterpret_cast<uint64_t *>(XT + (a.xt0[L + 1] + w) * ts + frag_at(l & 15, i * 16 + rq, 1)) = pack4(h);
            }
        }
        __syncthreads();
#pragma unroll
        for (int kb = 0; kb < IMAXW / 32; ++kb) bw[kb] = bn[kb];
        bias = bias_n;
    }
    // output column, loss and its derivative; the other waves fetch what follows
    backward_w(last, bn);
    const int out = last & 1;
    if (w == 0) {
        f32x4_t acc[2];
        product(out, a.kp[last] >> 5, bw, acc);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = i * 16 + rq + r;
                const bool on = m0 + row < a.B;
                const float er = on ? target_error(acc[i][r] + bias, ty[row], a.ym, a.yis) : 0.f;
                const float d = on ? 2.f * er / (float)a.B : 0.f;
                if ((l & 15) == 0) DZ[(size_t)row * a.zcols + a.zcol[last]] = d;
                h[r] = f2bf(d);
                H[out ^ 1][row][l & 15] = (l & 15) == 0 ? h[r] : (uint16_t)0;
                H[out ^ 1][row][16 + (l & 15)] = 0;
                if (on && (l & 15) == 0) a.sq[e * a.sqn + m0 + row] = er * er;
            }
            if ((l & 15) == 0) *reinterpret_cast<uint64_t *>(DZT + a.zt0[last] * ts + frag_at(0, i * 16 + rq, 1)) = pack4(h);
        }
    }
    __syncthreads();
    for (int L = last; L > 0; --L) {
        const int from = (L & 1) ^ 1;
#pragma unroll
        for (int kb = 0; kb < IMAXW / 32; ++kb) bw[kb] = bn[kb];
        if (L > 1) backward_w(L - 1, bn);
        if (n0 < a.fin[L]) {
            f32x4_t zz[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) zz[i] = Z[((L - 1) * IWAVES * 2 + i) * 64];
            f32x4_t acc[2];
            product(from, (a.fout[L] + 31) >> 5, bw, acc);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float z[4] = {zz[i][0], zz[i][1], zz[i][2], zz[i][3]};
                float dz[4], sg[4];
                uint16_t h[4];
                sigmoid_n(z, sg);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = i * 16 + rq + r;
                    dz[r] = m0 + row < a.B ? silu_back(acc[i][r], z[r], sg[r]) : 0.f;
                    DZ[(size_t)row * a.zcols + a.zcol[L - 1] + c] = dz[r];
                }
                f2bf4(dz, h);
#pragma unroll
                for (int r = 0; r < 4; ++r) H[from ^ 1][i * 16 + rq + r][c] = h[r];
                *reinterpret_cast<uint64_t *>(DZT + (a.zt0[L - 1] + w) * ts + frag_at(l & 15, i * 16 + rq, 1)) = pack4(h);
            }
        }
        __syncthreads();
    }
}

// Latency-bound as well: a wave holds a 32 x 32 quarter of its tile and walks
// the batch in blocks of 32, TKU blocks' operands in flight; a column sum is a
// chain of B dependent additions, so a workgroup takes 64 columns and keeps the
// next TSR rows on their way.  The same shape: 20 us; 33 with a lane fetching
// its own column, 41 with X and dZ in rows of the batch besides, of which a load
// takes 16 half lines.
constexpr int TKU = 4, TSR = 128;
static_assert(IMR == 32 && TSR / 4 == IMR, "a row tile is one block of a weight gradient's k and one wave's rows of a column sum");
__global__ __launch_bounds__(256) void k_train_weights(const TrainArgs a) {
    const int ue = a.nsum + a.tile0[a.nl], unit = chiplet_unit(ue * a.mg);
    if (unit < 0) return;
    const int e = unit / ue, ub = unit - e * ue;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    const float c1 = a.c1[e], c2 = a.c2[e];
    float *const p = a.p[e], *const am = a.am[e], *const av = a.av[e];
    uint16_t *const wt = a.wt[e];
    if (ub < a.nsum) {
        // 64 columns: the four waves bring in TSR rows at a time, the first adds them
        __shared__ float rows[2][TSR][64];
        const int col = ub * 64 + l, nr = a.tiles * IMR;  // rows past the batch hold zeros
        const float *x = a.DZ + (size_t)e * nr * a.zcols + min(col, a.zcols - 1);
        float s = 0.f, v[TSR / 4];
        auto load = [&](int r0) {
            const int r = r0 + w * (TSR / 4);
#pragma unroll
            for (int q = 0; q < TSR / 4; ++q) v[q] = r < nr ? x[(size_t)(r + q) * a.zcols] : 0.f;
        };
        load(0);
        for (int r0 = 0, b = 0; r0 < nr; r0 += TSR, b ^= 1) {
#pragma unroll
            for (int q = 0; q < TSR / 4; ++q) rows[b][w * (TSR / 4) + q][l] = v[q];
            __syncthreads();
            load(r0 + TSR);
            if (w == 0)
#pragma unroll 16
                for (int q = 0; q < TSR; ++q) s += rows[b][q][l];
        }
        if (w != 0 || col >= a.zcols) return;
        int L = 0;
        while (L + 1 < a.nl && col >= a.zcol[L + 1]) ++L;
        const int q = a.boff[L] + (col - a.zcol[L]);
        float v1 = p[q], v2 = am[q], v3 = av[q];
        adam_update(v1, v2, v3, s, a.adam, c1, c2);
        p[q] = v1;
        am[q] = v2;
        av[q] = v3;
        return;
    }
    const int id = ub - a.nsum;
    int L = 0;
    while (L + 1 < a.nl && id >= a.tile0[L + 1]) ++L;
    const int M = a.fin[L], N = a.fout[L], nt = (N + 63) / 64, k = id - a.tile0[L];
    const int mt = k / nt * 64 + (w >> 1) * 32, nt0 = k % nt * 64 + (w & 1) * 32;
    if (mt >= M || nt0 >= N) return;
    const int nb = a.tiles;
    const uint16_t *xa[2], *zb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        xa[i] = a.XT + ((size_t)e * a.xtiles + a.xt0[L] + min(mt / 16 + i, (M - 1) / 16)) * nb * 512 + l * 8;
        zb[i] = a.DZT + ((size_t)e * a.ztiles + a.zt0[L] + min(nt0 / 16 + i, (N - 1) / 16)) * nb * 512 + l * 8;
    }
    f32x4_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int b0, bf16x8_t(&A)[TKU][2], bf16x8_t(&B)[TKU][2]) {
#pragma unroll
        for (int u = 0; u < TKU; ++u) {
            const int b = 512 * min(b0 + u, nb - 1);  // past the end: loaded again, not used
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                A[u][i] = *reinterpret_cast<const bf16x8_t *>(xa[i] + b);
                B[u][i] = *reinterpret_cast<const bf16x8_t *>(zb[i] + b);
            }
        }
    };
    bf16x8_t A[TKU][2], B[TKU][2], An[TKU][2], Bn[TKU][2];
    load(0, A, B);
    for (int b0 = 0; b0 < nb; b0 += TKU) {
        load(b0 + TKU, An, Bn);
#pragma unroll
        for (int u = 0; u < TKU; ++u) {
            if (b0 + u >= nb) break;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[u][i], B[u][j], acc[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < TKU; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                A[u][i] = An[u][i];
                B[u][i] = Bn[u][i];
            }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int m = mt + i * 16 + (l >> 4) * 4, n = nt0 + j * 16 + (l & 15);
            if (m >= M || n >= N) continue;
            const int q = a.woff[L] + m * N + n;
            float v1[4], v2[4], v3[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = q + (m + r < M ? r * N : 0);
                v1[r] = p[o];
                v2[r] = am[o];
                v3[r] = av[o];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) adam_update(v1[r], v2[r], v3[r], acc[i][j][r], a.adam, c1, c2);
            uint16_t h[4];
            f2bf4(v1, h);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (m + r < M) {
                    p[q + r * N] = v1[r];
                    am[q + r * N] = v2[r];
                    av[q + r * N] = v3[r];
                    if (L) wt[a.wtoff[2 * L + 1] + frag_at(m + r, n, (N + 31) >> 5)] = h[r];
                } else {
                    h[r] = 0;
                }
            *reinterpret_cast<uint64_t *>(wt + a.wtoff[2 * L] + frag_at(n, m, a.kp[L] >> 5)) = pack4(h);
        }
}

__global__ void k_to_bf16(const float *__restrict__ in, uint16_t *__restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f2bf(in[i]);
}

}  // namespace casim

struct CasimMLP {
    int dev = 0;
    hipStream_t stream = nullptr;
    int n_in = 0, width = 0, depth = 0, members = 0;
    std::vector<int> fin, fout;       // layer fan-in / fan-out
    std::vector<size_t> woff, boff;   // offsets of W_l and b_l in a member's parameters
    size_t P = 0;                     // parameters per member
    std::vector<float *> p, g, am, av;
    std::vector<uint16_t *> pb;
    std::vector<int> steps;
    float *mean = nullptr, *istd = nullptr;
    float ym = 0.f, ys = 1.f;
    float *X = nullptr, *Y = nullptr;
    int *perm_d = nullptr;  // [rows] shuffled row order of the current epoch
    int64_t rows = 0;
    // fused inference (k_mlp_infer): transposed weights, refreshed when the
    // parameters change (pver counts parameter updates, wt_ver the copy's)
    bool fused = true;
    uint16_t *wt = nullptr;  // [members][wt_per]
    size_t wt_per = 0;
    uint64_t pver = 1, wt_ver = 0;
    bool fused_ok() const;
    size_t wt_offsets(int *off) const;
    void refresh_wt();
    void infer(const float *x, int B, float *out, int ostride, const int *rows_d = nullptr);
    // batch workspace
    int cap = 0;
    std::vector<uint16_t *> Xl;  // [depth + 1] BF16 activations
    std::vector<float *> Zl;     // [depth + 1] FP32 pre-activations (last = output)
    float *dH = nullptr, *dZ = nullptr, *tgt = nullptr, *sq = nullptr;
    uint16_t *dZb = nullptr;
    int *idx = nullptr;
    // workspace of the two-launch training step (TrainArgs), for tr_members
    // members and tr_rows batch rows at a time
    int tr_members = 0, tr_rows = 0;
    int64_t tr_perm = 0;
    uint16_t *tr_x = nullptr, *tr_dzt = nullptr;
    float *tr_dz = nullptr, *tr_z = nullptr, *tr_sq = nullptr;
    int *tr_idx = nullptr;
    // features and outputs of casim_mlp_predict, two slots of pr_rows rows
    int pr_rows = 0;
    float *pr_x = nullptr, *pr_out = nullptr;
    float *pr_pin = nullptr;          // the same in pinned memory
    hipStream_t pr_stream = nullptr;  // its copies
    hipEvent_t pr_up = nullptr, pr_done[2] = {};
    void predict_reserve(int b);
    bool train_fused(int B) const;
    int train_members(int B) const;
    void train_reserve(int mg, int B);
    void train_free();
    void train_group(int e0, int mg, int epochs, int B, float lr, uint64_t seed, float *loss_out);

    void use() { HIPCK(hipSetDevice(dev)); }
    void reserve(int b);
    void gemm(const uint16_t *A, int lda, int ta, const uint16_t *B, int ldb, int tb, float *C, int ldc, int M, int N,
              int K, float beta = 0.f);
    void forward(int e, int B);
    void backward(int e, int B);
    void free_batch();
};

void CasimMLP::gemm(const uint16_t *A, int lda, int ta, const uint16_t *B, int ldb, int tb, float *C, int ldc, int M,
                    int N, int K, float beta) {
    dim3 grid((N + GBN - 1) / GBN, (M + GBM - 1) / GBM);
    hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, stream, A, lda, ta, B, ldb, tb, C, ldc, M, N, K, beta);
    HIPCK(hipGetLastError());
}

bool CasimMLP::fused_ok() const {
    return fused && members <= IMAXM && depth + 1 <= IMAXL && n_in <= IMAXW && width <= IMAXW && width % 64 == 0;
}

// Offsets of the operands of layer g / 2 (k_wt) in a member's copy; the bytes
// of a member's copy.
size_t CasimMLP::wt_offsets(int *off) const {
    size_t per = 0;
    for (int g = 0; g <= 2 * depth + 1; ++g) {
        const int n = g & 1 ? fin[g / 2] : fout[g / 2], k = g & 1 ? fout[g / 2] : fin[g / 2];
        off[g] = (int)per;
        per += (size_t)((n + 15) & ~15) * ((k + 31) & ~31);
    }
    return per;
}

void CasimMLP::refresh_wt() {
    if (wt && wt_ver == pver) return;
    WtArgs a{};
    const size_t per = wt_offsets(a.off);
    if (!wt) {
        HIPCK(hipMalloc(&wt, sizeof(uint16_t) * per * members));
        wt_per = per;
    }
    size_t most = 0;
    for (int l = 0; l <= depth; ++l) {
        a.woff[l] = (int)woff[l];
        a.fin[l] = fin[l];
        a.fout[l] = fout[l];
        most = std::max(most, (size_t)((fout[l] + 31) & ~31) * ((fin[l] + 31) & ~31));
    }
    for (int e = 0; e < members; ++e) {
        a.pb[e] = pb[e];
        a.wt[e] = wt + (size_t)e * wt_per;
    }
    hipLaunchKernelGGL(k_wt, dim3((unsigned)((most + 255) / 256), (unsigned)(2 * depth + 2), (unsigned)members), dim3(256), 0,
                       stream, a);
    HIPCK(hipGetLastError());
    wt_ver = pver;
}

// Every member's output (normalised units) for B raw rows x -> out[e * ostride + row].
void CasimMLP::infer(const float *x, int B, float *out, int ostride, const int *rows_d) {
    refresh_wt();
    InferArgs a{};
    int off[2 * IMAXL];
    (void)wt_offsets(off);
    for (int l = 0; l <= depth; ++l) {
        a.wtoff[l] = off[2 * l];
        a.kp[l] = (fin[l] + 31) & ~31;
        a.fout[l] = fout[l];
        a.boff[l] = (int)boff[l];
    }
    for (int e = 0; e < members; ++e) {
        a.wt[e] = wt + (size_t)e * wt_per;
        a.p[e] = p[e];
    }
    a.nl = depth + 1;
    a.n_in = n_in;
    a.mean = mean;
    a.istd = istd;
    a.rows_d = rows_d;
    const int big = (B + 63) / 64;
    if ((size_t)big * members >= INFER_BIG)
        hipLaunchKernelGGL((k_mlp_infer<2, 4>), dim3((unsigned)big, (unsigned)members), dim3(32 * IWAVES), 0, stream, x, B, out,
                           ostride, a);
    else
        hipLaunchKernelGGL((k_mlp_infer<1, 2>), dim3((unsigned)((B + IMR - 1) / IMR), (unsigned)members), dim3(64 * IWAVES), 0,
                           stream, x, B, out, ostride, a);
    HIPCK(hipGetLastError());
}

// Batch rows in whole tiles; columns of a member's X and dZ operands in tiles of 16.
struct TrainSize {
    size_t bp, x = 0, z = 0, zc = 0;
    TrainSize(const CasimMLP *m, int B) : bp((size_t)(B + IMR - 1) / IMR * IMR) {
        for (int l = 0; l <= m->depth; ++l) {
            x += (m->fin[l] + 15) / 16 * 16;
            z += (m->fout[l] + 15) / 16 * 16;
            zc += m->fout[l];
        }
    }
};
// Bytes of a member's workspace of the two-launch training step.
static size_t train_bytes(const CasimMLP *m, int B) {
    const TrainSize t(m, B);
    return t.bp * (2 * t.x + 2 * t.z + 4 * t.zc + 4 * (size_t)m->depth * IMAXW);
}

// The two launches take the shapes of k_mlp_infer; batches past 1 GiB of
// workspace per member go a layer at a time.
bool CasimMLP::train_fused(int B) const {
    return fused_ok() && train_bytes(this, B) <= ((size_t)1 << 30);
}

// Members that step together: all of them while their workspace is within 1 GiB.
int CasimMLP::train_members(int B) const {
    return (int)std::min<size_t>(members, std::max<size_t>(1, ((size_t)1 << 30) / train_bytes(this, B)));
}

// Rows of a chunk of casim_mlp_predict, which bounds what a handle keeps for it;
// enough to fill the chip (80 us of the ensemble kernel at five members).
constexpr int PREDICT_ROWS = 16384;

void CasimMLP::predict_reserve(int b) {
    if (!pr_stream) {
        HIPCK(hipStreamCreateWithFlags(&pr_stream, hipStreamNonBlocking));
        for (hipEvent_t *e : {&pr_up, &pr_done[0], &pr_done[1]}) HIPCK(hipEventCreateWithFlags(e, hipEventDisableTiming));
    }
    if (b <= pr_rows) return;
    // whole powers of two, so that a caller whose batches grow does not allocate each time
    int n = 256;
    while (n < b) n *= 2;
    if (pr_x) (void)hipFree(pr_x);
    if (pr_out) (void)hipFree(pr_out);
    if (pr_pin) (void)hipHostFree(pr_pin);
    pr_x = pr_out = pr_pin = nullptr;
    pr_rows = 0;
    HIPCK(hipMalloc(&pr_x, sizeof(float) * 2 * (size_t)n * n_in));
    HIPCK(hipMalloc(&pr_out, sizeof(float) * 2 * (size_t)n * members));
    HIPCK(hipHostMalloc((void **)&pr_pin, sizeof(float) * 2 * (size_t)n * (n_in + members + 2), hipHostMallocDefault));
    pr_rows = n;
}

void CasimMLP::train_free() {
    for (void *q : {(void *)tr_x, (void *)tr_dzt, (void *)tr_dz, (void *)tr_z, (void *)tr_sq, (void *)tr_idx})
        if (q) (void)hipFree(q);
    tr_x = tr_dzt = nullptr;
    tr_dz = tr_z = tr_sq = nullptr;
    tr_idx = nullptr;
    tr_members = tr_rows = tr_perm = 0;
}

void CasimMLP::train_reserve(int mg, int B) {
    if (mg <= tr_members && B <= tr_rows && rows <= tr_perm) return;
    HIPCK(hipStreamSynchronize(stream));
    train_free();
    const TrainSize t(this, B);
    HIPCK(hipMalloc(&tr_x, sizeof(uint16_t) * mg * t.x * t.bp));
    HIPCK(hipMalloc(&tr_dzt, sizeof(uint16_t) * mg * t.z * t.bp));
    HIPCK(hipMalloc(&tr_dz, sizeof(float) * mg * t.zc * t.bp));
    HIPCK(hipMalloc(&tr_z, sizeof(float) * mg * t.bp * depth * IMAXW));
    HIPCK(hipMalloc(&tr_sq, sizeof(float) * mg * rows));
    HIPCK(hipMalloc(&tr_idx, sizeof(int) * mg * rows));
    tr_members = mg;
    tr_rows = B;
    tr_perm = rows;
}

void CasimMLP::free_batch() {
    for (auto q : Xl) (void)hipFree(q);
    for (auto q : Zl) (void)hipFree(q);
    Xl.clear();
    Zl.clear();
    for (void *q : {(void *)dH, (void *)dZ, (void *)tgt, (void *)sq, (void *)dZb, (void *)idx})
        if (q) (void)hipFree(q);
    dH = dZ = tgt = sq = nullptr;
    dZb = nullptr;
    idx = nullptr;
    cap = 0;
}

void CasimMLP::reserve(int b) {
    if (b <= cap) return;
    free_batch();
    cap = b;
    Xl.resize(depth + 1);
    Zl.resize(depth + 1);
    for (int l = 0; l <= depth; ++l) {
        HIPCK(hipMalloc(&Xl[l], sizeof(uint16_t) * (size_t)b * std::max(fin[l], 1)));
        HIPCK(hipMalloc(&Zl[l], sizeof(float) * (size_t)b * fout[l]));
    }
    const int wmax = std::max(width, n_in);
    HIPCK(hipMalloc(&dH, sizeof(float) * (size_t)b * wmax));
    HIPCK(hipMalloc(&dZ, sizeof(float) * (size_t)b * wmax));
    HIPCK(hipMalloc(&dZb, sizeof(uint16_t) * (size_t)b * wmax));
    HIPCK(hipMalloc(&tgt, sizeof(float) * b));
    HIPCK(hipMalloc(&sq, sizeof(float) * b));
    HIPCK(hipMalloc(&idx, sizeof(int) * b));
}

// Activations of member e for the B rows already in Xl[0].
void CasimMLP::forward(int e, int B) {
    for (int l = 0; l <= depth; ++l) {
        const uint16_t *W = pb[e] + woff[l];
        gemm(Xl[l], fin[l], 0, W, fout[l], 0, Zl[l], fout[l], B, fout[l], fin[l]);
        const size_t n = (size_t)B * fout[l];
        const bool last = l == depth;
        hipLaunchKernelGGL(k_bias_act, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, Zl[l], p[e] + boff[l],
                           last ? (uint16_t *)nullptr : Xl[l + 1], B, fout[l], last ? 0 : 1);
        HIPCK(hipGetLastError());
    }
}

// Gradients of member e into g[e] given dZb/dZ of the output layer.
void CasimMLP::backward(int e, int B) {
    for (int l = depth; l >= 0; --l) {
        // dW_l = X_l^T dZ_l, db_l = column sums of dZ_l
        gemm(Xl[l], fin[l], 1, dZb, fout[l], 0, g[e] + woff[l], fout[l], fin[l], fout[l], B);
        hipLaunchKernelGGL(k_colsum, dim3((fout[l] + 255) / 256), dim3(256), 0, stream, dZ, g[e] + boff[l], B,
                           fout[l]);
        HIPCK(hipGetLastError());
        if (l == 0) break;
        // dH_{l} = dZ_l W_l^T  (the activation feeding layer l)
        gemm(dZb, fout[l], 0, pb[e] + woff[l], fout[l], 1, dH, fin[l], B, fin[l], fout[l]);
        const size_t n = (size_t)B * fin[l];
        hipLaunchKernelGGL(k_silu_back, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, dH, Zl[l - 1], dZ,
                           dZb, n);
        HIPCK(hipGetLastError());
    }
}

// Epochs of members e0 .. e0 + mg - 1, which step together.  Each keeps its
// own row order, as if it were trained alone.
void CasimMLP::train_group(int e0, int mg, int epochs, int B, float lr, uint64_t seed, float *loss_out) {
    refresh_wt();  // k_train_weights keeps the transposed weights up to date
    ++pver;
    TrainArgs a{};
    (void)wt_offsets(a.wtoff);
    for (int l = 0; l <= depth; ++l) {
        a.kp[l] = (fin[l] + 31) & ~31;
        a.fin[l] = fin[l];
        a.fout[l] = fout[l];
        a.woff[l] = (int)woff[l];
        a.boff[l] = (int)boff[l];
        a.xt0[l] = a.xtiles;
        a.zt0[l] = a.ztiles;
        a.zcol[l] = a.zcols;
        a.xtiles += (fin[l] + 15) / 16;
        a.ztiles += (fout[l] + 15) / 16;
        a.zcols += fout[l];
        a.tile0[l + 1] = a.tile0[l] + (fin[l] + 63) / 64 * ((fout[l] + 63) / 64);
    }
    for (int e = 0; e < mg; ++e) {
        a.wt[e] = wt + (size_t)(e0 + e) * wt_per;
        a.p[e] = p[e0 + e];
        a.am[e] = am[e0 + e];
        a.av[e] = av[e0 + e];
    }
    a.nl = depth + 1;
    a.mg = mg;
    a.nsum = (a.zcols + 63) / 64;
    a.n_in = n_in;
    a.B = B;
    a.tiles = (B + IMR - 1) / IMR;
    a.mean = mean, a.istd = istd, a.X = X, a.Y = Y;
    a.rows = a.sqn = rows;
    a.ym = ym;
    a.yis = 1.f / ys;
    a.XT = tr_x, a.DZT = tr_dzt, a.DZ = tr_dz, a.Z = tr_z;
    a.adam = {lr, 0.9f, 0.999f, 1e-8f};
    std::vector<std::mt19937_64> gen;
    for (int e = e0; e < e0 + mg; ++e) gen.emplace_back(seed * 1315423911ull + (uint64_t)e * 2654435761ull + 17);
    std::vector<int> perm((size_t)mg * rows);
    const int64_t nb = rows / B;
    struct Event {
        hipEvent_t e = nullptr;
        ~Event() {
            if (e) (void)hipEventDestroy(e);
        }
    } copied;
    HIPCK(hipEventCreateWithFlags(&copied.e, hipEventDisableTiming));
    for (int ep = 0; ep < epochs; ++ep) {
        // the last epoch's order has left the host buffer; its batches still run
        if (ep) HIPCK(hipEventSynchronize(copied.e));
        for (int e = 0; e < mg; ++e) {
            int *q = perm.data() + (size_t)e * rows;
            std::iota(q, q + rows, 0);
            std::shuffle(q, q + rows, gen[e]);
        }
        HIPCK(hipMemcpyAsync(tr_idx, perm.data(), sizeof(int) * perm.size(), hipMemcpyHostToDevice, stream));
        HIPCK(hipEventRecord(copied.e, stream));
        for (int64_t b = 0; b < nb; ++b) {
            a.perm = tr_idx + b * B;
            a.sq = tr_sq + b * B;
            for (int e = 0; e < mg; ++e) {
                const int t = ++steps[e0 + e];
                a.c1[e] = 1.f - std::pow(a.adam.b1, (float)t);
                a.c2[e] = 1.f - std::pow(a.adam.b2, (float)t);
            }
            hipLaunchKernelGGL(k_train_rows, dim3(chiplet_grid(a.tiles * mg)), dim3(64 * IWAVES), 0, stream, a);
            HIPCK(hipGetLastError());
            hipLaunchKernelGGL(k_train_weights, dim3(chiplet_grid((a.nsum + a.tile0[a.nl]) * mg)), dim3(256), 0, stream,
                               a);
            HIPCK(hipGetLastError());
        }
    }
    for (int e = e0; e < e0 + mg; ++e) {
        hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, stream, p[e], pb[e], P);
        HIPCK(hipGetLastError());
    }
    std::vector<float> sq((size_t)mg * rows);
    HIPCK(hipMemcpyAsync(sq.data(), tr_sq, sizeof(float) * sq.size(), hipMemcpyDeviceToHost, stream));
    HIPCK(hipStreamSynchronize(stream));
    wt_ver = pver;
    for (int e = 0; e < mg && loss_out; ++e) {
        double sum = 0.0;
        for (int64_t i = 0; i < nb * B; ++i) sum += sq[(size_t)e * rows + i];
        loss_out[e0 + e] = (float)(sum / (double)(nb * B));
    }
}

namespace casim {

// Every member's output (normalised units) for `rows` raw feature rows on the
// device: x [rows x n_in] -> out [members x ostride].  Runs on `stream` after
// the MLP's own stream has drained.  rows_d: the number of rows in device
// memory, at most `rows`; only with mlp_rows_on_device.
void mlp_forward_device(CasimMLP *m, const float *x, int64_t rows, float *out, int64_t ostride, const int *rows_d,
                        hipStream_t stream) {
    m->use();
    HIPCK(hipStreamSynchronize(m->stream));
    hipStream_t keep = m->stream;
    m->stream = stream;
    try {
        if (m->fused_ok()) {
            m->infer(x, (int)rows, out, (int)ostride, rows_d);
        } else {
            const int chunk = (int)std::min<int64_t>(rows, 65536);
            m->reserve(chunk);
            for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
                const int B = (int)std::min<int64_t>(chunk, rows - r0);
                const size_t n = (size_t)B * m->n_in;
                hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, x + r0 * m->n_in,
                                   (const float *)nullptr, (const int *)nullptr, B, m->n_in, m->mean, m->istd, 0.f, 1.f,
                                   m->Xl[0], (float *)nullptr);
                HIPCK(hipGetLastError());
                for (int e = 0; e < m->members; ++e) {
                    m->forward(e, B);
                    HIPCK(hipMemcpyAsync(out + (size_t)e * ostride + r0, m->Zl[m->depth], sizeof(float) * B,
                                         hipMemcpyDeviceToDevice, stream));
                }
            }
        }
    } catch (...) {
        m->stream = keep;
        throw;
    }
    m->stream = keep;
}

bool mlp_rows_on_device(const CasimMLP *m) { return m->fused_ok(); }
int mlp_members(const CasimMLP *m) { return m->members; }
int mlp_inputs(const CasimMLP *m) { return m->n_in; }
float mlp_out_mean(const CasimMLP *m) { return m->ym; }
float mlp_out_std(const CasimMLP *m) { return m->ys; }

}  // namespace casim

// ---------------------------------------------------------------------------
// Ensemble prediction that allocates nothing: the activations live in a fixed
// workspace, one per GPU, held from the library's first use of that GPU until
// the process ends.  Layout for up to CASIM_MLP_NOALLOC_MAX_ROWS rows: two BF16
// activation buffers [rows x CASIM_MLP_NOALLOC_MAX_WIDTH] (ping-pong), one FP32
// pre-activation buffer [rows x CASIM_MLP_NOALLOC_MAX_WIDTH], and the members'
// outputs [CASIM_MLP_NOALLOC_MAX_MEMBERS x rows].

namespace casim {
namespace {
constexpr size_t NA_ACT = (size_t)CASIM_MLP_NOALLOC_MAX_ROWS * CASIM_MLP_NOALLOC_MAX_WIDTH;  // elements per activation buffer
constexpr size_t NA_OFF_XB = NA_ACT * sizeof(uint16_t);
constexpr size_t NA_OFF_Z = 2 * NA_ACT * sizeof(uint16_t);
constexpr size_t NA_OFF_OUT = NA_OFF_Z + NA_ACT * sizeof(float);
constexpr size_t NA_BYTES = NA_OFF_OUT + (size_t)CASIM_MLP_NOALLOC_MAX_MEMBERS * CASIM_MLP_NOALLOC_MAX_ROWS * sizeof(float);
static_assert(NA_OFF_XB % 256 == 0 && NA_OFF_Z % 256 == 0 && NA_OFF_OUT % 256 == 0, "workspace alignment");
static_assert(NA_BYTES == CASIM_MLP_NOALLOC_BYTES, "workspace size as declared in casim_surrogate.h");

// The workspace.  In host code this name stands for the symbol only; its
// device address comes from hipGetSymbolAddress (noalloc_workspace below).
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

constexpr int NA_MAX_DEVICES = 64;
std::mutex na_mutex;
void *na_ptr[NA_MAX_DEVICES] = {};

// Device address of this GPU's workspace, looked up once per device with that
// device current.
void *noalloc_workspace(int dev) {
    REQUIRE(dev >= 0 && dev < NA_MAX_DEVICES, CASIM_E_DEVICE, "device index out of range for the MLP workspace");
    std::lock_guard<std::mutex> lock(na_mutex);
    if (!na_ptr[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            throw Err(CASIM_E_DEVICE, std::string("hipGetSymbolAddress of the MLP workspace: ") + hipGetErrorString(e));
        na_ptr[dev] = ptr;
    }
    return na_ptr[dev];
}

// out[e * cap + r] = z[r] (the output layer's column) for member e.
__global__ void k_na_collect(const float *__restrict__ z, float *__restrict__ out, int rows) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < rows) out[r] = z[r];
}

// Mean and relative spread of exp(y * ys + ym) over the members; raw (out, or
// null: not wanted) receives y * ys + ym.  4 us for 55003 rows of five members;
// on the host, member by member after a copy of its outputs, 1 ms.
__global__ void k_na_reduce(const float *out, int members, int cap, int rows, float ys, float ym,
                            float *__restrict__ mean, float *__restrict__ spread, float *raw, int rcap) {
#pragma clang fp contract(off)
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    double s = 0, s2 = 0;
    for (int e = 0; e < members; ++e) {
        const float o = out[(size_t)e * cap + r] * ys + ym;
        if (raw) raw[(size_t)e * rcap + r] = o;
        const double v = exp((double)o);
        s += v;
        s2 += v * v;
    }
    const double mu = s / members;
    const double var = fmax(0.0, s2 / members - mu * mu);
    if (mean) mean[r] = (float)mu;
    if (spread) spread[r] = (float)(mu > 0 ? sqrt(var) / mu : 0.0);
}
}  // namespace
}  // namespace casim

extern "C" {

int casim_mlp_create(int32_t n_in, int32_t width, int32_t depth, int32_t members, uint64_t seed, CasimMLP **out) {
    CasimMLP *m = nullptr;
    int rc = guard([&] {
        REQUIRE(out && n_in >= 1 && width >= 1 && depth >= 1 && members >= 1, CASIM_E_INVALID, "bad MLP shape");
        *out = nullptr;
        m = new CasimMLP();
        HIPCK(hipGetDevice(&m->dev));
        HIPCK(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
        (void)casim::noalloc_workspace(m->dev);  // this GPU's workspace of casim_mlp_predict_noalloc
        m->n_in = n_in;
        m->width = width;
        m->depth = depth;
        m->members = members;
        for (int l = 0; l <= depth; ++l) {
            m->fin.push_back(l == 0 ? n_in : width);
            m->fout.push_back(l == depth ? 1 : width);
        }
        size_t off = 0;
        for (int l = 0; l <= depth; ++l) {
            m->woff.push_back(off);
            off += (size_t)m->fin[l] * m->fout[l];
            m->boff.push_back(off);
            off += m->fout[l];
        }
        m->P = off;
        std::mt19937_64 gen(seed);
        std::vector<float> h(m->P);
        for (int e = 0; e < members; ++e) {
            for (int l = 0; l <= depth; ++l) {
                const float lim = std::sqrt(6.f / (float)m->fin[l]);
                std::uniform_real_distribution<float> U(-lim, lim);
                for (size_t i = 0; i < (size_t)m->fin[l] * m->fout[l]; ++i) h[m->woff[l] + i] = U(gen);
                for (int i = 0; i < m->fout[l]; ++i) h[m->boff[l] + i] = 0.f;
            }
            float *pp, *gg, *mm, *vv;
            uint16_t *bb;
            HIPCK(hipMalloc(&pp, sizeof(float) * m->P));
            HIPCK(hipMalloc(&gg, sizeof(float) * m->P));
            HIPCK(hipMalloc(&mm, sizeof(float) * m->P));
            HIPCK(hipMalloc(&vv, sizeof(float) * m->P));
            HIPCK(hipMalloc(&bb, sizeof(uint16_t) * m->P));
            m->p.push_back(pp);
            m->g.push_back(gg);
            m->am.push_back(mm);
            m->av.push_back(vv);
            m->pb.push_back(bb);
            m->steps.push_back(0);
            HIPCK(hipMemcpyAsync(pp, h.data(), sizeof(float) * m->P, hipMemcpyHostToDevice, m->stream));
            HIPCK(hipMemsetAsync(mm, 0, sizeof(float) * m->P, m->stream));
            HIPCK(hipMemsetAsync(vv, 0, sizeof(float) * m->P, m->stream));
            hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((m->P + 255) / 256)), dim3(256), 0, m->stream, pp, bb,
                               m->P);
            HIPCK(hipGetLastError());
        }
        std::vector<float> zero(n_in, 0.f), one(n_in, 1.f);
        HIPCK(hipMalloc(&m->mean, sizeof(float) * n_in));
        HIPCK(hipMalloc(&m->istd, sizeof(float) * n_in));
        HIPCK(hipMemcpyAsync(m->mean, zero.data(), sizeof(float) * n_in, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipMemcpyAsync(m->istd, one.data(), sizeof(float) * n_in, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipStreamSynchronize(m->stream));
        *out = m;
    });
    if (rc != CASIM_OK && m) {
        std::string keep = last_error();
        casim_mlp_destroy(m);
        last_error() = keep;
    }
    return rc;
}

int casim_mlp_destroy(CasimMLP *m) {
    if (!m) return CASIM_OK;
    (void)hipSetDevice(m->dev);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    m->free_batch();
    m->train_free();
    if (m->pr_stream) (void)hipStreamDestroy(m->pr_stream);
    if (m->pr_pin) (void)hipHostFree(m->pr_pin);
    for (hipEvent_t e : {m->pr_up, m->pr_done[0], m->pr_done[1]})
        if (e) (void)hipEventDestroy(e);
    for (auto v : {&m->p, &m->g, &m->am, &m->av})
        for (float *q : *v) (void)hipFree(q);
    for (uint16_t *q : m->pb) (void)hipFree(q);
    if (m->wt) (void)hipFree(m->wt);
    for (void *q : {(void *)m->mean, (void *)m->istd, (void *)m->X, (void *)m->Y, (void *)m->perm_d, (void *)m->pr_x, (void *)m->pr_out})
        if (q) (void)hipFree(q);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return CASIM_OK;
}

int64_t casim_mlp_param_count(const CasimMLP *m) { return m ? (int64_t)m->P : 0; }

int casim_mlp_get_params(CasimMLP *m, int32_t member, float *out) {
    return guard([&] {
        REQUIRE(m && out, CASIM_E_INVALID, "null argument");
        REQUIRE(member >= 0 && member < m->members, CASIM_E_RANGE, "member out of range");
        m->use();
        HIPCK(hipMemcpyAsync(out, m->p[member], sizeof(float) * m->P, hipMemcpyDeviceToHost, m->stream));
        HIPCK(hipStreamSynchronize(m->stream));
    });
}

int casim_mlp_set_params(CasimMLP *m, int32_t member, const float *in) {
    return guard([&] {
        REQUIRE(m && in, CASIM_E_INVALID, "null argument");
        REQUIRE(member >= 0 && member < m->members, CASIM_E_RANGE, "member out of range");
        m->use();
        HIPCK(hipMemcpyAsync(m->p[member], in, sizeof(float) * m->P, hipMemcpyHostToDevice, m->stream));
        hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((m->P + 255) / 256)), dim3(256), 0, m->stream, m->p[member],
                           m->pb[member], m->P);
        HIPCK(hipGetLastError());
        HIPCK(hipStreamSynchronize(m->stream));
        ++m->pver;
    });
}

int casim_mlp_set_normalization(CasimMLP *m, const float *in_mean, const float *in_std, float out_mean,
                                float out_std) {
    return guard([&] {
        REQUIRE(m && in_mean && in_std && out_std > 0.f, CASIM_E_INVALID, "bad normalisation");
        m->use();
        std::vector<float> is(m->n_in);
        for (int i = 0; i < m->n_in; ++i) is[i] = in_std[i] > 0.f ? 1.f / in_std[i] : 1.f;
        HIPCK(hipMemcpyAsync(m->mean, in_mean, sizeof(float) * m->n_in, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipMemcpyAsync(m->istd, is.data(), sizeof(float) * m->n_in, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipStreamSynchronize(m->stream));
        m->ym = out_mean;
        m->ys = out_std;
    });
}

int casim_mlp_set_data(CasimMLP *m, const float *x, const float *y, int64_t rows) {
    return guard([&] {
        REQUIRE(m && x && y && rows >= 1, CASIM_E_INVALID, "bad training data");
        m->use();
        if (m->X) (void)hipFree(m->X);
        if (m->Y) (void)hipFree(m->Y);
        if (m->perm_d) (void)hipFree(m->perm_d);
        m->X = m->Y = nullptr;
        m->perm_d = nullptr;
        HIPCK(hipMalloc(&m->X, sizeof(float) * rows * m->n_in));
        HIPCK(hipMalloc(&m->Y, sizeof(float) * rows));
        HIPCK(hipMalloc(&m->perm_d, sizeof(int) * rows));
        HIPCK(hipMemcpyAsync(m->X, x, sizeof(float) * rows * m->n_in, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipMemcpyAsync(m->Y, y, sizeof(float) * rows, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipStreamSynchronize(m->stream));
        m->rows = rows;
    });
}

int casim_mlp_train(CasimMLP *m, int32_t epochs, int32_t batch, float lr, uint64_t seed, float *loss_out) {
    return guard([&] {
        REQUIRE(m && m->X, CASIM_E_STATE, "no training data");
        REQUIRE(epochs >= 1 && batch >= 1, CASIM_E_INVALID, "bad epochs/batch");
        m->use();
        const int B = (int)std::min<int64_t>(batch, m->rows);
        if (m->train_fused(B)) {
            const int mg = m->train_members(B);
            m->train_reserve(mg, B);
            for (int e0 = 0; e0 < m->members; e0 += mg)
                m->train_group(e0, std::min(mg, m->members - e0), epochs, B, lr, seed, loss_out);
            return;
        }
        m->reserve(B);
        std::vector<int> perm(m->rows);
        const AdamArgs adam{lr, 0.9f, 0.999f, 1e-8f};
        const float yis = 1.f / m->ys;
        std::vector<float> sq(B);
        ++m->pver;  // the transposed inference weights follow the parameters
        for (int e = 0; e < m->members; ++e) {
            std::mt19937_64 gen(seed * 1315423911ull + (uint64_t)e * 2654435761ull + 17);
            double last = 0.0;
            for (int ep = 0; ep < epochs; ++ep) {
                std::iota(perm.begin(), perm.end(), 0);
                std::shuffle(perm.begin(), perm.end(), gen);
                HIPCK(hipMemcpyAsync(m->perm_d, perm.data(), sizeof(int) * m->rows, hipMemcpyHostToDevice,
                                     m->stream));
                double sum = 0.0;
                int64_t cnt = 0;
                const bool keep = ep == epochs - 1;
                for (int64_t r0 = 0; r0 + B <= m->rows; r0 += B) {
                    const size_t n = (size_t)B * m->n_in;
                    hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, m->X,
                                       m->Y, (const int *)(m->perm_d + r0), B, m->n_in, m->mean, m->istd, m->ym, yis,
                                       m->Xl[0], m->tgt);
                    HIPCK(hipGetLastError());
                    m->forward(e, B);
                    hipLaunchKernelGGL(k_mse, dim3((B + 255) / 256), dim3(256), 0, m->stream, m->Zl[m->depth], m->tgt,
                                       m->dZ, m->dZb, m->sq, B);
                    HIPCK(hipGetLastError());
                    m->backward(e, B);
                    const int t = ++m->steps[e];
                    const float c1 = 1.f - std::pow(adam.b1, (float)t), c2 = 1.f - std::pow(adam.b2, (float)t);
                    hipLaunchKernelGGL(k_adam, dim3((unsigned)((m->P + 255) / 256)), dim3(256), 0, m->stream, m->p[e],
                                       m->g[e], m->am[e], m->av[e], m->pb[e], m->P, adam, c1, c2);
                    HIPCK(hipGetLastError());
                    if (keep) {
                        HIPCK(hipMemcpyAsync(sq.data(), m->sq, sizeof(float) * B, hipMemcpyDeviceToHost, m->stream));
                        HIPCK(hipStreamSynchronize(m->stream));
                        for (int i = 0; i < B; ++i) sum += sq[i];
                        cnt += B;
                    }
                }
                if (keep) last = cnt ? sum / (double)cnt : 0.0;
            }
            HIPCK(hipStreamSynchronize(m->stream));
            if (loss_out) loss_out[e] = (float)last;
        }
    });
}

int casim_mlp_gradient(CasimMLP *m, int32_t member, const float *x, const float *y, int64_t rows, float *grad,
                       float *loss) {
    return guard([&] {
        REQUIRE(m && x && y && grad && rows >= 1, CASIM_E_INVALID, "bad arguments");
        REQUIRE(member >= 0 && member < m->members, CASIM_E_RANGE, "member out of range");
        m->use();
        const int B = (int)rows;
        m->reserve(B);
        float *dx = nullptr, *dy = nullptr;
        HIPCK(hipMalloc(&dx, sizeof(float) * rows * m->n_in));
        HIPCK(hipMalloc(&dy, sizeof(float) * rows));
        HIPCK(hipMemcpyAsync(dx, x, sizeof(float) * rows * m->n_in, hipMemcpyHostToDevice, m->stream));
        HIPCK(hipMemcpyAsync(dy, y, sizeof(float) * rows, hipMemcpyHostToDevice, m->stream));
        const size_t n = (size_t)B * m->n_in;
        hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, dx, dy,
                           (const int *)nullptr, B, m->n_in, m->mean, m->istd, m->ym, 1.f / m->ys, m->Xl[0], m->tgt);
        m->forward(member, B);
        hipLaunchKernelGGL(k_mse, dim3((B + 255) / 256), dim3(256), 0, m->stream, m->Zl[m->depth], m->tgt, m->dZ,
                           m->dZb, m->sq, B);
        m->backward(member, B);
        std::vector<float> sq(B);
        HIPCK(hipMemcpyAsync(grad, m->g[member], sizeof(float) * m->P, hipMemcpyDeviceToHost, m->stream));
        HIPCK(hipMemcpyAsync(sq.data(), m->sq, sizeof(float) * B, hipMemcpyDeviceToHost, m->stream));
        HIPCK(hipStreamSynchronize(m->stream));
        (void)hipFree(dx);
        (void)hipFree(dy);
        if (loss) {
            double s = 0;
            for (float v : sq) s += v;
            *loss = (float)(s / B);
        }
    });
}

int casim_mlp_predict(CasimMLP *m, const float *x, int64_t rows, float *mean, float *spread, float *member_out) {
    return guard([&] {
        REQUIRE(m && x && rows >= 1, CASIM_E_INVALID, "bad arguments");
        m->use();
        const int E = m->members;
        // halved where a row is wide, so that a slot stays within 32 MiB of pinned
        // memory (from about 500 features on; 256 rows at the least)
        int most = PREDICT_ROWS;
        while (most > 256 && (int64_t)most * ((int64_t)m->n_in + E + 2) > (8 << 20)) most /= 2;
        const int chunk = (int)std::min<int64_t>(rows, most);
        const bool fused = m->fused_ok();
        if (!fused) m->reserve(chunk);
        m->predict_reserve(chunk);
        // two slots: while a chunk is evaluated, the next one is copied to pinned
        // memory and on to the device, and the outputs, which the kernel writes to
        // pinned memory, go to the caller (five members, us: 55003 rows 530, 690 where
        // every call brings an array that was not used before, 740 and more with one
        // copy each from and to pageable memory; 100 rows 39, 150)
        const int cap = m->pr_rows, nc = (int)((rows + chunk - 1) / chunk);
        const size_t slot = (size_t)cap * (m->n_in + E + 2);
        auto take = [&](int c) {
            const int64_t r0 = (int64_t)c * chunk;
            const int B = (int)std::min<int64_t>(chunk, rows - r0);
            const float *h = m->pr_pin + (c & 1) * slot + (size_t)cap * m->n_in;
            HIPCK(hipEventSynchronize(m->pr_done[c & 1]));
            for (int e = 0; member_out && e < E; ++e)
                std::memcpy(member_out + (size_t)e * rows + r0, h + (size_t)e * B, sizeof(float) * B);
            if (mean) std::memcpy(mean + r0, h + (size_t)E * B, sizeof(float) * B);
            if (spread) std::memcpy(spread + r0, h + (size_t)(E + 1) * B, sizeof(float) * B);
        };
        for (int c = 0; c < nc; ++c) {
            if (c >= 2) take(c - 2);
            const int64_t r0 = (int64_t)c * chunk;
            const int B = (int)std::min<int64_t>(chunk, rows - r0);
            float *const hx = m->pr_pin + (c & 1) * slot, *const ho = hx + (size_t)cap * m->n_in;
            float *const px = m->pr_x + (size_t)(c & 1) * cap * m->n_in, *const raw = m->pr_out + (size_t)(c & 1) * cap * E;
            std::memcpy(hx, x + r0 * m->n_in, sizeof(float) * (size_t)B * m->n_in);
            // alone, a chunk is copied on the stream that evaluates it
            hipStream_t up = nc > 1 ? m->pr_stream : m->stream;
            HIPCK(hipMemcpyAsync(px, hx, sizeof(float) * (size_t)B * m->n_in, hipMemcpyHostToDevice, up));
            if (nc > 1) {
                HIPCK(hipEventRecord(m->pr_up, up));
                HIPCK(hipStreamWaitEvent(m->stream, m->pr_up, 0));
            }
            if (fused) {
                m->infer(px, B, raw, B);
            } else {
                const size_t n = (size_t)B * m->n_in;
                hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, px,
                                   (const float *)nullptr, (const int *)nullptr, B, m->n_in, m->mean, m->istd, 0.f, 1.f,
                                   m->Xl[0], (float *)nullptr);
                HIPCK(hipGetLastError());
                for (int e = 0; e < E; ++e) {
                    m->forward(e, B);
                    HIPCK(hipMemcpyAsync(raw + (size_t)e * B, m->Zl[m->depth], sizeof(float) * B, hipMemcpyDeviceToDevice,
                                         m->stream));
                }
            }
            hipLaunchKernelGGL(casim::k_na_reduce, dim3((B + 255) / 256), dim3(256), 0, m->stream, (const float *)raw, E, B, B,
                               m->ys, m->ym, ho + (size_t)E * B, ho + (size_t)(E + 1) * B, ho, B);
            HIPCK(hipGetLastError());
            HIPCK(hipEventRecord(m->pr_done[c & 1], m->stream));
        }
        for (int c = std::max(0, nc - 2); c < nc; ++c) take(c);
    });
}

int casim_mlp_set_fused_inference(CasimMLP *m, int32_t on) {
    return guard([&] {
        REQUIRE(m, CASIM_E_INVALID, "null handle");
        REQUIRE(on == 0 || on == 1, CASIM_E_INVALID, "on must be 0 or 1");
        m->fused = on != 0;
    });
}

int casim_mlp_predict_noalloc(CasimMLP *m, const float *x, int64_t rows, float *mean, float *spread, void *stream) {
    return guard([&] {
        REQUIRE(m && x && rows >= 1, CASIM_E_INVALID, "bad arguments");
        REQUIRE(rows <= CASIM_MLP_NOALLOC_MAX_ROWS, CASIM_E_RANGE,
                "rows exceed the workspace of casim_mlp_predict_noalloc (" + std::to_string(CASIM_MLP_NOALLOC_MAX_ROWS) +
                    "); split the call");
        REQUIRE(m->width <= CASIM_MLP_NOALLOC_MAX_WIDTH && m->n_in <= CASIM_MLP_NOALLOC_MAX_WIDTH, CASIM_E_RANGE,
                "layer wider than the workspace of casim_mlp_predict_noalloc (" +
                    std::to_string(CASIM_MLP_NOALLOC_MAX_WIDTH) + ")");
        REQUIRE(m->members <= CASIM_MLP_NOALLOC_MAX_MEMBERS, CASIM_E_RANGE,
                "more members than the workspace of casim_mlp_predict_noalloc holds (" +
                    std::to_string(CASIM_MLP_NOALLOC_MAX_MEMBERS) + ")");
        REQUIRE(m->mean && m->istd, CASIM_E_STATE, "normalisation not set");
        m->use();
        hipStream_t st = stream ? (hipStream_t)stream : m->stream;
        unsigned char *ws = (unsigned char *)casim::noalloc_workspace(m->dev);
        uint16_t *xa = (uint16_t *)ws;
        uint16_t *xb = (uint16_t *)(ws + casim::NA_OFF_XB);
        float *z = (float *)(ws + casim::NA_OFF_Z);
        float *outm = (float *)(ws + casim::NA_OFF_OUT);
        const int B = (int)rows;
        const int cap = CASIM_MLP_NOALLOC_MAX_ROWS;
        const size_t n = (size_t)B * m->n_in;
        for (int e = 0; e < m->members; ++e) {
            hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, (const float *)nullptr,
                               (const int *)nullptr, B, m->n_in, m->mean, m->istd, 0.f, 1.f, xa, (float *)nullptr);
            HIPCK(hipGetLastError());
            uint16_t *in = xa, *nxt = xb;
            for (int l = 0; l <= m->depth; ++l) {
                const int fi = m->fin[l], fo = m->fout[l];
                dim3 grid((fo + GBN - 1) / GBN, (B + GBM - 1) / GBM);
                hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, st, in, fi, 0, m->pb[e] + m->woff[l], fo, 0, z, fo, B,
                                   fo, fi, 0.f);
                HIPCK(hipGetLastError());
                const bool last = l == m->depth;
                const size_t nz = (size_t)B * fo;
                hipLaunchKernelGGL(k_bias_act, dim3((unsigned)((nz + 255) / 256)), dim3(256), 0, st, z,
                                   m->p[e] + m->boff[l], last ? (uint16_t *)nullptr : nxt, B, fo, last ? 0 : 1);
                HIPCK(hipGetLastError());
                std::swap(in, nxt);
            }
            hipLaunchKernelGGL(casim::k_na_collect, dim3((B + 255) / 256), dim3(256), 0, st, (const float *)z,
                               outm + (size_t)e * cap, B);
            HIPCK(hipGetLastError());
        }
        hipLaunchKernelGGL(casim::k_na_reduce, dim3((B + 255) / 256), dim3(256), 0, st, outm, m->members, cap, B, m->ys, m->ym,
                           mean, spread, (float *)nullptr, 0);
        HIPCK(hipGetLastError());
    });
}

int casim_gemm_bf16(const void *a, int32_t lda, int32_t trans_a, const void *b, int32_t ldb, int32_t trans_b,
                    float *c, int32_t ldc, int32_t M, int32_t N, int32_t K, float beta, void *stream) {
    return guard([&] {
        REQUIRE(a && b && c && M >= 0 && N >= 0 && K >= 0, CASIM_E_INVALID, "bad GEMM arguments");
        dim3 grid((N + GBN - 1) / GBN, (M + GBM - 1) / GBM);
        if (M == 0 || N == 0) return;
        hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t *)a, lda, trans_a,
                           (const uint16_t *)b, ldb, trans_b, c, ldc, M, N, K, beta);
        HIPCK(hipGetLastError());
        HIPCK(hipStreamSynchronize((hipStream_t)stream));
    });
}

}  // extern "C"
