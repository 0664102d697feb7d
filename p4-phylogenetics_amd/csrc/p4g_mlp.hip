// p4g_mlp.hip -- the learned proposal's network: a 3-layer MLP
// (F -> H -> H -> O, ReLU) with BF16 weights and BF16 MFMA operands,
// FP32 accumulation, FP32 master weights and an FP32 Adam update, all on
// the GPU.  It maps per-branch (and per-composition) features to the mean
// and log standard deviation of a Gaussian proposal; it is trained by
// minimising the Gaussian negative log likelihood of samples from
// plain-proposal chains.  The proposal that uses it is Metropolis-Hastings
// corrected (p4gpu/learned.py), so the network only affects mixing.
//
// Networks up to MLP_MAX_H hidden units, MLP_MAX_F inputs and MLP_MAX_O
// outputs run in three launches (k_mlpRows, k_mlpWgrad, k_mlpUpdate; one for
// a forward pass); larger ones on one GEMM kernel per product (k_gemm), on
// v_mfma_f32_16x16x16bf16_1k, one wavefront per 16x16 output tile.  There
// lane l holds A[l%16][4*(l/16)+i], B[4*(l/16)+i][l%16] (i < 4) and D rows
// 4*(l/16)+r of column l%16.
#include "../../include/p4gpu.h"
#include "p4g_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

namespace p4g {

typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4m __attribute__((ext_vector_type(4)));

__host__ __device__ inline unsigned short f2bf(float f)
{
    unsigned u;
    std::memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float bf2f(unsigned short h)
{
    return __uint_as_float(((unsigned)h) << 16);
}

// Element (m, k) of A and (k, n) of B; each operand is FP32 (rounded to
// BF16 for the MFMA) or BF16, row-major with a leading dimension, and may
// be transposed.
struct GemmOp {
    const void *p;
    int ld;
    int trans;   // 0: [rows][ld], 1: stored transposed
    int isBf16;
};

__device__ __forceinline__ unsigned short opLoad(const GemmOp &o, int r, int c, int R, int C)
{
    if (r >= R || c >= C) return 0;
    const size_t idx = o.trans ? (size_t)c * o.ld + r : (size_t)r * o.ld + c;
    if (o.isBf16) return ((const unsigned short *)o.p)[idx];
    return f2bf(((const float *)o.p)[idx]);
}

// C[M][N] = A[M][K] . B[K][N] (+ bias[n]) (ReLU) -- FP32 result.
__global__ __launch_bounds__(64) void k_gemm(GemmOp A, GemmOp B, float *C, int ldc, int M, int N, int K,
                                             const float *bias, float *reluOut)
{
    const int lane = threadIdx.x;
    const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
    const int row = lane & 15, kq = (lane >> 4) * 4;
    f4m acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 16) {
        s4v a, b;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            a[i] = (short)opLoad(A, m0 + row, k0 + kq + i, M, K);
            b[i] = (short)opLoad(B, k0 + kq + i, n0 + row, K, N);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    const int n = n0 + row;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int m = m0 + kq + r;
        if (m < M && n < N) {
            const float v = acc[r] + (bias ? bias[n] : 0.f);
            C[(size_t)m * ldc + n] = v;
            if (reluOut) reluOut[(size_t)m * ldc + n] = fmaxf(v, 0.f);
        }
    }
}

// Gaussian negative log likelihood of targets y under (mu = out[:, :D],
// s = log sigma = out[:, D:2D]), masked per coordinate; writes dL/dout and
// the per-row loss.  Loss per row: sum_d mask (s + 0.5 (y - mu)^2 e^{-2s}).
__global__ void k_nll(const float *out, const float *y, const float *mask, int n, int D, float invCount,
                      float *dOut, float *rowLoss)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float L = 0.f;
    for (int d = 0; d < D; d++) {
        const float mk = mask[(size_t)i * D + d];
        const float mu = out[(size_t)i * 2 * D + d];
        const float s = out[(size_t)i * 2 * D + D + d];
        const float r = y[(size_t)i * D + d] - mu;
        const float w = expf(-2.f * s);
        L += mk * (s + 0.5f * r * r * w);
        dOut[(size_t)i * 2 * D + d] = -mk * r * w * invCount;
        dOut[(size_t)i * 2 * D + D + d] = mk * (1.f - r * r * w) * invCount;
    }
    rowLoss[i] = L;
}

// dZ = dH * (Z > 0)
__global__ void k_reluBack(float *dH, const float *Z, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !(Z[i] > 0.f)) dH[i] = 0.f;
}

// column sums of X[n][N] (bias gradients)
__global__ void k_colsum(const float *X, int n, int N, float *out)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= N) return;
    float s = 0.f;
    for (int i = 0; i < n; i++) s += X[(size_t)i * N + c];
    out[c] = s;
}

__global__ void k_sum(const float *x, int n, float *out)
{
    __shared__ float sh[256];
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += 256) s += x[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0];
}

// Adam on the FP32 masters, then refresh the BF16 copies.
__global__ void k_adam(float *w, unsigned short *wb, const float *g, float *m, float *v, size_t n, float lr,
                       float b1, float b2, float eps, float c1, float c2)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (wb) wb[i] = f2bf(wi);
}

__global__ void k_tobf16(const float *w, unsigned short *wb, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wb[i] = f2bf(w[i]);
}

// ------------------------------------------------------- the fused path
// All widths are padded in the packed BF16 weight copies (zeros), so any
// size up to these limits takes it: the limits are what one workgroup's LDS
// rows and a wave's accumulators hold.
constexpr int MLP_MAX_H = 512, MLP_MAX_F = 512, MLP_MAX_O = 64;
constexpr int MLP_ROWS = 16;      // batch rows per workgroup (one MFMA tile)
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

// Widths: H to 64 (four waves of 16-column tiles), F and the contraction
// over outputs to 32 (one MFMA step), outputs as rows to 32.
struct MlpDims {
    int F, H, O, Fp, Hp, Op, n, nPad;
};
// Packed BF16 copies: W1p [Hp][Fp], W2p [Hp][Hp], W2t its transpose, W3p
// [Op][Hp], W3t [Hp][Op].
struct MlpPack {
    unsigned short *W1p, *W2p, *W2t, *W3p, *W3t;
};

// Copy parameter i of the master vector into its packed places.
__device__ __forceinline__ void packParam(const MlpDims &d, const MlpPack &p, size_t i, float w)
{
    const unsigned short b = f2bf(w);
    const size_t nW1 = (size_t)d.H * d.F, nW2 = (size_t)d.H * d.H, nW3 = (size_t)d.O * d.H;
    if (i < nW1) {
        const int h = (int)(i / d.F), f = (int)(i - (size_t)h * d.F);
        p.W1p[(size_t)h * d.Fp + f] = b;
        return;
    }
    if (i < nW1 + d.H) return;
    i -= nW1 + d.H;
    if (i < nW2) {
        const int h = (int)(i / d.H), j = (int)(i - (size_t)h * d.H);
        p.W2p[(size_t)h * d.Hp + j] = b;
        p.W2t[(size_t)j * d.Hp + h] = b;
        return;
    }
    if (i < nW2 + d.H) return;
    i -= nW2 + d.H;
    if (i < nW3) {
        const int o = (int)(i / d.H), h = (int)(i - (size_t)o * d.H);
        p.W3p[(size_t)o * d.Hp + h] = b;
        p.W3t[(size_t)h * d.Op + o] = b;
    }
}

__global__ void k_mlpPack(MlpDims d, MlpPack p, const float *w, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) packParam(d, p, i, w[i]);
}

struct MlpRowArgs {
    MlpDims d;
    MlpPack p;
    const float *X, *Y, *MASK;        // [n][F], [n][D], [n][D]
    const float *b1, *b2, *b3;
    float *OUT;                       // [n][O] (forward only)
    float invCount;
    // backward: the weight-gradient operands, row-transposed, BF16, nPad rows
    unsigned short *XT, *H1T, *H2T, *Z1T, *Z2T, *OT;   // [Fp], [Hp] x 4, [Op] rows of [nPad]
    float *db1, *db2, *db3, *blockLoss;                // per workgroup: [Hp], [Hp], [Op], one
};

// NT tiles of 16 columns per wave: acc[c] += A (16 rows in LDS, BF16) . B^T
// with B's rows (output columns) contiguous over the contraction.
template <int NT>
__device__ __forceinline__ void rowGemm(const unsigned short *A, int lda, const unsigned short *B, int ldb, int K,
                                        int n0, f4m (&acc)[NT])
{
    const int lane = threadIdx.x & 63;
    const int pl = lane & 15, q8 = (lane >> 4) * 8;
    for (int k0 = 0; k0 < K; k0 += 32) {
        const bf8v a = *reinterpret_cast<const bf8v *>(A + pl * lda + k0 + q8);
#pragma unroll
        for (int c = 0; c < NT; c++) {
            const bf8v b = *reinterpret_cast<const bf8v *>(B + (size_t)(n0 + 16 * c + pl) * ldb + k0 + q8);
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[c], 0, 0, 0);
        }
    }
}

// Forward, loss and the backward pass to the activations for 16 rows per
// workgroup.  Latency-bound: a batch of 4,096 rows is 256 workgroups, one
// per CU, and each is a chain of five small products whose activations stay
// in LDS; the weights (BF16, 0.3 MB in all) come from L2.  The four waves
// split the hidden columns, so a wave's A operand (16 rows) is read once for
// its NT column tiles, and a result's column owner keeps the ReLU mask in
// registers for the backward pass.  Every operand is rounded to BF16 exactly
// where the one-kernel-per-product path rounds it; sums stay FP32.  Before:
// eight k_gemm launches with element gathers and FP32 activations through
// HBM, 1,845 us of a 4,096 x (24-256-256-6) gradient, and the bias sums
// 2,110 us more; now 23 us here and 11 us in k_mlpWgrad (HIP trace).
template <int NT>
__global__ __launch_bounds__(256) void k_mlpRows(MlpRowArgs a, int backward)
{
    extern __shared__ __align__(16) unsigned char mlpSm[];
    const MlpDims d = a.d;
    const int ldx = d.Fp + 8, ldh = d.Hp + 8, ldo = d.Op + 8;   // +8: rows start on different banks
    unsigned short *sX = reinterpret_cast<unsigned short *>(mlpSm);
    unsigned short *sH1 = sX + MLP_ROWS * ldx;
    unsigned short *sH2 = sH1 + MLP_ROWS * ldh;     // H2, then dZ2
    unsigned short *sDo = sH2 + MLP_ROWS * ldh;     // dL/dout, BF16
    float *sOut = reinterpret_cast<float *>(sDo + MLP_ROWS * ldo);   // [16][Op]
    float *sDoF = sOut + MLP_ROWS * d.Op;           // dL/dout, FP32
    float *sLoss = sDoF + MLP_ROWS * d.Op;          // [16]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int pl = lane & 15, q = lane >> 4;
    const int row0 = blockIdx.x * MLP_ROWS;
    for (int i = tid; i < MLP_ROWS * d.Fp; i += 256) {
        const int r = i / d.Fp, f = i - r * d.Fp;
        const bool in = row0 + r < d.n && f < d.F;
        sX[r * ldx + f] = in ? f2bf(a.X[(size_t)(row0 + r) * d.F + f]) : (unsigned short)0;
    }
    __syncthreads();
    if (backward)
        for (int i = tid; i < d.Fp * 2; i += 256) {
            const int f = i >> 1, r0 = (i & 1) * 8;
            union { unsigned short h[8]; uint4 v; } u;
            for (int r = 0; r < 8; r++) u.h[r] = sX[(r0 + r) * ldx + f];
            *reinterpret_cast<uint4 *>(a.XT + (size_t)f * d.nPad + row0 + r0) = u.v;
        }
    const int n0 = wave * NT * 16;
    // four rows (4q..) of one column, rounded: LDS row-major and the
    // transposed copy
    auto put = [&](unsigned short *S, unsigned short *GT, int col, const float (&v)[4]) {
        union { unsigned short h[4]; uint2 v; } u;
        for (int r = 0; r < 4; r++) {
            u.h[r] = f2bf(v[r]);
            S[(4 * q + r) * ldh + col] = u.h[r];
        }
        if (backward) *reinterpret_cast<uint2 *>(GT + (size_t)col * d.nPad + row0 + 4 * q) = u.v;
    };
    unsigned m1 = 0, m2 = 0;   // ReLU masks, 4 bits per tile
    auto hidden = [&](const f4m (&acc)[NT], const float *bias, unsigned short *S, unsigned short *GT) -> unsigned {
        unsigned m = 0;
#pragma unroll
        for (int c = 0; c < NT; c++) {
            const int col = n0 + 16 * c + pl;
            const float b = col < d.H ? bias[col] : 0.f;
            float v[4];
            for (int r = 0; r < 4; r++) {
                const float z = acc[c][r] + b;
                if (z > 0.f) m |= 1u << (4 * c + r);
                v[r] = row0 + 4 * q + r < d.n ? fmaxf(z, 0.f) : 0.f;
            }
            put(S, GT, col, v);
        }
        return m;
    };
    {
        f4m acc[NT] = {};
        rowGemm<NT>(sX, ldx, a.p.W1p, d.Fp, d.Fp, n0, acc);
        m1 = hidden(acc, a.b1, sH1, a.H1T);
    }
    __syncthreads();
    {
        f4m acc[NT] = {};
        rowGemm<NT>(sH1, ldh, a.p.W2p, d.Hp, d.Hp, n0, acc);
        m2 = hidden(acc, a.b2, sH2, a.H2T);
    }
    __syncthreads();
    for (int t = wave; t < d.Op / 16; t += 4) {
        f4m acc[1] = {};
        rowGemm<1>(sH2, ldh, a.p.W3p, d.Hp, d.Hp, 16 * t, acc);
        const int o = 16 * t + pl;
        for (int r = 0; r < 4; r++) {
            const float v = acc[0][r] + (o < d.O ? a.b3[o] : 0.f);
            sOut[(4 * q + r) * d.Op + o] = v;
            if (!backward && o < d.O && row0 + 4 * q + r < d.n) a.OUT[(size_t)(row0 + 4 * q + r) * d.O + o] = v;
        }
    }
    if (!backward) return;
    __syncthreads();
    // dL/dout and the rows' losses (k_nll's formulas)
    const int D = d.O / 2;
    for (int i = tid; i < MLP_ROWS * d.Op; i += 256) {
        sDoF[i] = 0.f;
        sDo[(i / d.Op) * ldo + i % d.Op] = 0;
    }
    __syncthreads();
    if (tid < MLP_ROWS) {
        const int i = row0 + tid;
        float L = 0.f;
        if (i < d.n)
            for (int c = 0; c < D; c++) {
                const float mk = a.MASK[(size_t)i * D + c];
                const float mu = sOut[tid * d.Op + c], s = sOut[tid * d.Op + D + c];
                const float r = a.Y[(size_t)i * D + c] - mu;
                const float w = expf(-2.f * s);
                L += mk * (s + 0.5f * r * r * w);
                const float g0 = -mk * r * w * a.invCount, g1 = mk * (1.f - r * r * w) * a.invCount;
                sDoF[tid * d.Op + c] = g0;
                sDoF[tid * d.Op + D + c] = g1;
                sDo[tid * ldo + c] = f2bf(g0);
                sDo[tid * ldo + D + c] = f2bf(g1);
            }
        sLoss[tid] = L;
    }
    __syncthreads();
    for (int i = tid; i < d.Op; i += 256) {
        float s = 0.f;
        for (int r = 0; r < MLP_ROWS; r++) s += sDoF[r * d.Op + i];
        a.db3[(size_t)blockIdx.x * d.Op + i] = s;
        for (int h = 0; h < 2; h++) {
            union { unsigned short h[8]; uint4 v; } u;
            for (int r = 0; r < 8; r++) u.h[r] = sDo[(8 * h + r) * ldo + i];
            *reinterpret_cast<uint4 *>(a.OT + (size_t)i * d.nPad + row0 + 8 * h) = u.v;
        }
    }
    if (tid == 0) {
        float s = 0.f;
        for (int r = 0; r < MLP_ROWS; r++) s += sLoss[r];
        a.blockLoss[blockIdx.x] = s;
    }
    // dZ = (dY . W) masked; its column sums are the bias gradients
    auto back = [&](const f4m (&acc)[NT], unsigned m, float *db, unsigned short *S, unsigned short *GT) {
#pragma unroll
        for (int c = 0; c < NT; c++) {
            const int col = n0 + 16 * c + pl;
            float v[4], s = 0.f;
            for (int r = 0; r < 4; r++) {
                v[r] = (m >> (4 * c + r)) & 1u ? acc[c][r] : 0.f;
                s += v[r];
            }
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (q == 0) db[(size_t)blockIdx.x * d.Hp + col] = s;
            put(S, GT, col, v);
        }
    };
    {
        f4m acc[NT] = {};
        rowGemm<NT>(sDo, ldo, a.p.W3t, d.Op, d.Op, n0, acc);
        back(acc, m2, a.db2, sH2, a.Z2T);   // every wave is past its reads of H2
    }
    __syncthreads();
    {
        f4m acc[NT] = {};
        rowGemm<NT>(sH2, ldh, a.p.W2t, d.Hp, d.Hp, n0, acc);
        back(acc, m1, a.db1, sH1, a.Z1T);   // and of H1 (dZ1's LDS copy is not read)
    }
}

// Weight gradients: dW2 = dZ2^T H1, dW1 = dZ1^T X, dW3 = dOut^T H2, each a
// contraction over the batch of two row-transposed operands.  One wave owns
// a 32 x 32 block of a gradient and a slice of the batch; the workgroup's
// four waves add their slices in LDS, and nSplit workgroups per block write
// partial sums (a 4,096-row batch with 256 hidden units: 80 blocks x 4
// workgroups, where one wave per block would leave two thirds of the CUs
// idle on a chain of 128 steps).  The last blocks sum the bias gradients
// and the loss over k_mlpRows' workgroups (one thread per column over every
// row took 703 us per layer).  All sums in a fixed order.
struct MlpWgradArgs {
    MlpDims d;
    const unsigned short *XT, *H1T, *H2T, *Z1T, *Z2T, *OT;
    const float *db1, *db2, *db3, *blockLoss;
    float *part;          // [nSplit][nParams], weights only
    float *g;             // biases
    float *loss;
    int nSplit, nUnits;
    size_t nParams;
};

constexpr int MLP_BIAS_COLS = 32;   // columns per workgroup of the bias sums

__global__ __launch_bounds__(256) void k_mlpWgrad(MlpWgradArgs a)
{
    const MlpDims d = a.d;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nBlk = d.nPad / MLP_ROWS;
    const size_t oB1 = (size_t)d.H * d.F, oW2 = oB1 + d.H, oB2 = oW2 + (size_t)d.H * d.H, oW3 = oB2 + d.H,
                 oB3 = oW3 + (size_t)d.O * d.H;
    if ((int)blockIdx.x >= a.nUnits * a.nSplit) {
        // bias columns: 32 per workgroup, eight slices of the row blocks
        __shared__ float sb[8][MLP_BIAS_COLS];
        const int c = ((int)blockIdx.x - a.nUnits * a.nSplit) * MLP_BIAS_COLS + (tid & 31), sl = tid >> 5;
        const int total = 2 * d.Hp + d.Op + 1;
        float s = 0.f;
        const float *src = nullptr;
        int ld = 1;
        if (c < d.Hp) src = a.db1 + c, ld = d.Hp;
        else if (c < 2 * d.Hp) src = a.db2 + (c - d.Hp), ld = d.Hp;
        else if (c < 2 * d.Hp + d.Op) src = a.db3 + (c - 2 * d.Hp), ld = d.Op;
        else if (c < total) src = a.blockLoss;
        if (src)
            for (int b = sl; b < nBlk; b += 8) s += src[(size_t)b * ld];
        sb[sl][tid & 31] = s;
        __syncthreads();
        if (sl) return;
        for (int i = 1; i < 8; i++) s += sb[i][tid & 31];
        if (c < d.Hp) {
            if (c < d.H) a.g[oB1 + c] = s;
        } else if (c < 2 * d.Hp) {
            if (c - d.Hp < d.H) a.g[oB2 + c - d.Hp] = s;
        } else if (c < 2 * d.Hp + d.Op) {
            if (c - 2 * d.Hp < d.O) a.g[oB3 + c - 2 * d.Hp] = s;
        } else if (c < total) {
            *a.loss = s;
        }
        return;
    }
    const int unit = (int)blockIdx.x / a.nSplit, split = (int)blockIdx.x - unit * a.nSplit;
    const int hU = d.Hp / 32, fU = d.Fp / 32;
    const unsigned short *A, *B;
    float *P = a.part + (size_t)split * a.nParams;
    int M, N, m0, n0;
    if (unit < hU * hU) {
        A = a.Z2T, B = a.H1T, M = N = d.H, m0 = unit / hU * 32, n0 = unit % hU * 32;
        P += oW2;
    } else if (unit < hU * hU + hU * fU) {
        const int u = unit - hU * hU;
        A = a.Z1T, B = a.XT, M = d.H, N = d.F, m0 = u / fU * 32, n0 = u % fU * 32;
    } else {
        const int u = unit - hU * hU - hU * fU;
        A = a.OT, B = a.H2T, M = d.O, N = d.H, m0 = u / hU * 32, n0 = u % hU * 32;
        P += oW3;
    }
    const int pl = lane & 15, q = lane >> 4;
    const int nk = d.nPad / 32, w = split * 4 + wave, nw = a.nSplit * 4;
    const int k0 = (int)((long)nk * w / nw), k1 = (int)((long)nk * (w + 1) / nw);
    f4m acc[2][2] = {};
    const unsigned short *Ap = A + (size_t)(m0 + pl) * d.nPad + q * 8, *Bp = B + (size_t)(n0 + pl) * d.nPad + q * 8;
    for (int k = k0; k < k1; k++) {
        bf8v av[2], bv[2];
        for (int i = 0; i < 2; i++) {
            av[i] = *reinterpret_cast<const bf8v *>(Ap + (size_t)(16 * i) * d.nPad + 32 * k);
            bv[i] = *reinterpret_cast<const bf8v *>(Bp + (size_t)(16 * i) * d.nPad + 32 * k);
        }
        for (int i = 0; i < 2; i++)
            for (int j = 0; j < 2; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
    __shared__ f4m sp[4][4][64];
    for (int i = 0; i < 4; i++) sp[wave][i][lane] = acc[i >> 1][i & 1];
    __syncthreads();
    // wave i adds block i (of the four 16 x 16) over the slices
    f4m s = sp[0][wave][lane];
    for (int i = 1; i < 4; i++) s += sp[i][wave][lane];
    const int n = n0 + 16 * (wave & 1) + pl;
    for (int r = 0; r < 4; r++) {
        const int m = m0 + 16 * (wave >> 1) + 4 * q + r;
        if (m < M && n < N) P[(size_t)m * N + n] = s[r];
    }
}

// The gradients from the partial sums, and with `adam` the update of the
// FP32 masters (k_adam's formulas) and of the packed BF16 copies.
__global__ __launch_bounds__(256) void k_mlpUpdate(MlpDims d, MlpPack p, const float *part, int nSplit, float *g,
                                                   size_t n, int adam, float *w, float *m, float *v, float lr,
                                                   float b1, float b2, float eps, float c1, float c2)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t oB1 = (size_t)d.H * d.F, oW2 = oB1 + d.H, oB2 = oW2 + (size_t)d.H * d.H, oW3 = oB2 + d.H,
                 oB3 = oW3 + (size_t)d.O * d.H;
    const bool bias = (i >= oB1 && i < oW2) || (i >= oB2 && i < oW3) || i >= oB3;
    float gi;
    if (bias) {
        gi = g[i];
    } else {
        gi = part[i];
        for (int s = 1; s < nSplit; s++) gi += part[(size_t)s * n + i];
        g[i] = gi;
    }
    if (!adam) return;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    packParam(d, p, i, wi);
}

}  // namespace p4g

using namespace p4g;

// Parameter block layout (FP32 masters, one contiguous array):
//   W1 [H][F], b1 [H], W2 [H][H], b2 [H], W3 [O][H], b3 [O]
struct p4g_mlp {
    int F = 0, H = 0, O = 0;
    size_t nW1, nW2, nW3, nParams;
    float *w = nullptr;           // masters
    unsigned short *wb = nullptr; // BF16 copy (biases unused)
    float *g = nullptr, *m = nullptr, *v = nullptr;
    long step = 0;
    // activations for a batch of up to cap rows
    int cap = 0;
    float *X = nullptr, *Z1 = nullptr, *Z2 = nullptr, *OUT = nullptr, *Y = nullptr, *MASK = nullptr;
    float *dOUT = nullptr, *dH2 = nullptr, *dH1 = nullptr, *rowLoss = nullptr, *loss = nullptr;
    // the fused path: packed weights; row-transposed operands and
    // per-workgroup sums for up to capPad rows
    bool fused = false;
    int Fp = 0, Hp = 0, Op = 0, capPad = 0;
    unsigned short *pack = nullptr, *rowsT = nullptr;
    float *sums = nullptr, *part = nullptr;
    MlpDims dims(int n) const { return MlpDims{F, H, O, Fp, Hp, Op, n, (n + 31) & ~31}; }
    size_t packElems() const { return (size_t)Hp * Fp + 2 * (size_t)Hp * Hp + 2 * (size_t)Op * Hp; }
    MlpPack packs() const
    {
        MlpPack p;
        p.W1p = pack;
        p.W2p = p.W1p + (size_t)Hp * Fp;
        p.W2t = p.W2p + (size_t)Hp * Hp;
        p.W3p = p.W2t + (size_t)Hp * Hp;
        p.W3t = p.W3p + (size_t)Op * Hp;
        return p;
    }
    size_t off(int which) const
    {
        switch (which) {
        case 0: return 0;                                  // W1
        case 1: return nW1;                                // b1
        case 2: return nW1 + H;                            // W2
        case 3: return nW1 + H + nW2;                      // b2
        case 4: return nW1 + H + nW2 + H;                  // W3
        default: return nW1 + H + nW2 + H + nW3;           // b3
        }
    }
};

namespace {

constexpr int MLP_MAX_SPLIT = 4;   // workgroups per weight-gradient block

// a batch slice of four MFMA steps per wave before the batch is split
// further: shorter slices do not pay for their partial sums
int mlpSplits(int nPad) { return std::max(1, std::min(MLP_MAX_SPLIT, nPad / (32 * 4 * 4))); }

// Buffers of the fused path for n rows; the gradients' only when asked.
bool ensureFused(p4g_mlp *m, int n, bool backward)
{
    if (n > m->cap) {
        float **bufs[] = {&m->X, &m->OUT, &m->Y, &m->MASK};
        const int D = m->O / 2;
        const size_t sizes[] = {(size_t)n * m->F, (size_t)n * m->O, (size_t)n * D, (size_t)n * D};
        m->cap = 0;
        for (auto b : bufs)
            if (*b) {
                (void)hipFree(*b);
                *b = nullptr;
            }
        for (int i = 0; i < 4; i++)
            if (!hipOk(hipMalloc((void **)bufs[i], sizes[i] * sizeof(float)), "hipMalloc mlp buffers")) return false;
        m->cap = n;
    }
    const int nPad = (n + 31) & ~31;
    if (!backward || nPad <= m->capPad) return true;
    m->capPad = 0;
    if (m->rowsT) (void)hipFree(m->rowsT);
    if (m->sums) (void)hipFree(m->sums);
    m->rowsT = nullptr;
    m->sums = nullptr;
    if (!m->part && !hipOk(hipMalloc((void **)&m->part, sizeof(float) * MLP_MAX_SPLIT * m->nParams), "hipMalloc mlp sums"))
        return false;
    if (!hipOk(hipMalloc((void **)&m->rowsT, sizeof(short) * (size_t)nPad * (m->Fp + 4 * m->Hp + m->Op)),
               "hipMalloc mlp rows") ||
        !hipOk(hipMalloc((void **)&m->sums, sizeof(float) * (size_t)(nPad / MLP_ROWS) * (2 * m->Hp + m->Op + 1)),
               "hipMalloc mlp sums"))
        return false;
    m->capPad = nPad;
    return true;
}

MlpRowArgs rowArgs(p4g_mlp *m, int n)
{
    MlpRowArgs a{};
    a.d = m->dims(n);
    a.p = m->packs();
    a.X = m->X;
    a.Y = m->Y;
    a.MASK = m->MASK;
    a.b1 = m->w + m->off(1);
    a.b2 = m->w + m->off(3);
    a.b3 = m->w + m->off(5);
    a.OUT = m->OUT;
    a.invCount = 1.0f / (float)n;
    const size_t nP = a.d.nPad, nB = nP / MLP_ROWS;
    if (m->rowsT) {
        a.H1T = m->rowsT;
        a.H2T = a.H1T + nP * m->Hp;
        a.Z1T = a.H2T + nP * m->Hp;
        a.Z2T = a.Z1T + nP * m->Hp;
        a.XT = a.Z2T + nP * m->Hp;
        a.OT = a.XT + nP * m->Fp;
        a.db1 = m->sums;
        a.db2 = a.db1 + nB * m->Hp;
        a.db3 = a.db2 + nB * m->Hp;
        a.blockLoss = a.db3 + nB * m->Op;
    }
    return a;
}

bool launchRows(p4g_mlp *m, const MlpRowArgs &a, int backward)
{
    const MlpDims &d = a.d;
    const size_t lds = sizeof(short) * MLP_ROWS * ((size_t)d.Fp + 8 + 2 * ((size_t)d.Hp + 8) + d.Op + 8) +
                       sizeof(float) * MLP_ROWS * (2 * (size_t)d.Op + 1);
    const dim3 grid(backward ? d.nPad / MLP_ROWS : (d.n + MLP_ROWS - 1) / MLP_ROWS);
    hipStream_t s = stream();
    switch (d.Hp / 64) {
    case 1: hipLaunchKernelGGL(k_mlpRows<1>, grid, dim3(256), lds, s, a, backward); break;
    case 2: hipLaunchKernelGGL(k_mlpRows<2>, grid, dim3(256), lds, s, a, backward); break;
    case 3: hipLaunchKernelGGL(k_mlpRows<3>, grid, dim3(256), lds, s, a, backward); break;
    case 4: hipLaunchKernelGGL(k_mlpRows<4>, grid, dim3(256), lds, s, a, backward); break;
    case 5: hipLaunchKernelGGL(k_mlpRows<5>, grid, dim3(256), lds, s, a, backward); break;
    case 6: hipLaunchKernelGGL(k_mlpRows<6>, grid, dim3(256), lds, s, a, backward); break;
    case 7: hipLaunchKernelGGL(k_mlpRows<7>, grid, dim3(256), lds, s, a, backward); break;
    default: hipLaunchKernelGGL(k_mlpRows<8>, grid, dim3(256), lds, s, a, backward); break;
    }
    return hipOk(hipGetLastError(), "mlp rows");
}

// loss, gradients and with `adam` the update, n rows in X, Y, MASK
bool fusedBackward(p4g_mlp *m, int n, bool adam, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const MlpRowArgs r = rowArgs(m, n);
    if (!launchRows(m, r, 1)) return false;
    MlpWgradArgs a{};
    a.d = r.d;
    a.XT = r.XT;
    a.H1T = r.H1T;
    a.H2T = r.H2T;
    a.Z1T = r.Z1T;
    a.Z2T = r.Z2T;
    a.OT = r.OT;
    a.db1 = r.db1;
    a.db2 = r.db2;
    a.db3 = r.db3;
    a.blockLoss = r.blockLoss;
    a.part = m->part;
    a.g = m->g;
    a.loss = m->loss;
    a.nSplit = mlpSplits(r.d.nPad);
    a.nUnits = (m->Hp / 32) * (m->Hp / 32 + m->Fp / 32 + m->Op / 32);
    a.nParams = m->nParams;
    const int biasBlocks = (2 * m->Hp + m->Op + 1 + MLP_BIAS_COLS - 1) / MLP_BIAS_COLS;
    hipStream_t s = stream();
    hipLaunchKernelGGL(k_mlpWgrad, dim3(a.nUnits * a.nSplit + biasBlocks), dim3(256), 0, s, a);
    if (!hipOk(hipGetLastError(), "mlp weight gradients")) return false;
    hipLaunchKernelGGL(k_mlpUpdate, dim3((m->nParams + 255) / 256), dim3(256), 0, s, r.d, r.p, m->part, a.nSplit, m->g,
                       m->nParams, adam ? 1 : 0, m->w, m->m, m->v, lr, b1, b2, eps, c1, c2);
    return hipOk(hipGetLastError(), "mlp update");
}

// the masters' BF16 copies, for whichever path the network takes
void repack(p4g_mlp *m)
{
    const size_t n = m->nParams;
    if (m->fused)
        hipLaunchKernelGGL(k_mlpPack, dim3((n + 255) / 256), dim3(256), 0, stream(), m->dims(1), m->packs(), m->w, n);
    else
        hipLaunchKernelGGL(k_tobf16, dim3((n + 255) / 256), dim3(256), 0, stream(), m->w, m->wb, n);
}

bool ensureCap(p4g_mlp *m, int n, bool backward)
{
    if (m->fused) return ensureFused(m, n, backward);
    if (n <= m->cap) return true;
    float **bufs[] = {&m->X, &m->Z1, &m->Z2, &m->OUT, &m->Y, &m->MASK, &m->dOUT, &m->dH2, &m->dH1, &m->rowLoss};
    for (auto b : bufs)
        if (*b) {
            (void)hipFree(*b);
            *b = nullptr;
        }
    const int D = m->O / 2;
    const size_t sizes[] = {(size_t)n * m->F, (size_t)n * m->H, (size_t)n * m->H, (size_t)n * m->O,
                            (size_t)n * D, (size_t)n * D, (size_t)n * m->O, (size_t)n * m->H,
                            (size_t)n * m->H, (size_t)n};
    for (int i = 0; i < 10; i++)
        if (!hipOk(hipMalloc((void **)bufs[i], sizes[i] * sizeof(float)), "hipMalloc mlp buffers")) return false;
    m->cap = n;
    return true;
}

hipError_t gemm(GemmOp A, GemmOp B, float *C, int ldc, int M, int N, int K, const float *bias,
                float *reluOut = nullptr)
{
    dim3 grid((M + 15) / 16, (N + 15) / 16);
    hipLaunchKernelGGL(k_gemm, grid, dim3(64), 0, stream(), A, B, C, ldc, M, N, K, bias, reluOut);
    return hipGetLastError();
}

// forward of n rows already in m->X
bool forward(p4g_mlp *m, int n)
{
    if (m->fused) return launchRows(m, rowArgs(m, n), 0);
    const unsigned short *wb = m->wb;
    const float *w = m->w;
    GemmOp X{m->X, m->F, 0, 0};
    GemmOp W1t{wb + m->off(0), m->F, 1, 1};  // B(k=f, n=h) = W1[h][f]
    // Z1 is kept for the backward pass, H1 = relu(Z1) goes to dH1's storage
    if (!hipOk(gemm(X, W1t, m->Z1, m->H, n, m->H, m->F, w + m->off(1), m->dH1), "mlp layer 1")) return false;
    GemmOp H1{m->dH1, m->H, 0, 0};
    GemmOp W2t{wb + m->off(2), m->H, 1, 1};
    if (!hipOk(gemm(H1, W2t, m->Z2, m->H, n, m->H, m->H, w + m->off(3), m->dH2), "mlp layer 2")) return false;
    GemmOp H2{m->dH2, m->H, 0, 0};
    GemmOp W3t{wb + m->off(4), m->H, 1, 1};
    return hipOk(gemm(H2, W3t, m->OUT, m->O, n, m->O, m->H, w + m->off(5)), "mlp layer 3");
}

// forward + loss + gradients into m->g for n rows in X, Y, MASK
bool backward(p4g_mlp *m, int n)
{
    if (m->fused) return fusedBackward(m, n, false, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f);
    if (!forward(m, n)) return false;
    const int D = m->O / 2;
    hipStream_t s = stream();
    hipLaunchKernelGGL(k_nll, dim3((n + 255) / 256), dim3(256), 0, s, m->OUT, m->Y, m->MASK, n, D,
                       1.0f / (float)n, m->dOUT, m->rowLoss);
    hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, s, m->rowLoss, n, m->loss);
    float *g = m->g;
    // H1 (relu(Z1)) is in dH1, H2 (relu(Z2)) in dH2 after forward(); layer-3
    // gradients first, then overwrite dH2/dH1 with the backpropagated values
    GemmOp dOutT{m->dOUT, m->O, 1, 0};  // A(m=o, k=row) = dOUT[row][o]
    GemmOp H2{m->dH2, m->H, 0, 0};      // B(k=row, n=h)
    if (!hipOk(gemm(dOutT, H2, g + m->off(4), m->H, m->O, m->H, n, nullptr), "mlp dW3")) return false;
    hipLaunchKernelGGL(k_colsum, dim3((m->O + 63) / 64), dim3(64), 0, s, m->dOUT, n, m->O, g + m->off(5));
    GemmOp H1{m->dH1, m->H, 0, 0};
    // dH2 = dOUT . W3   (W3 [O][H]: B(k=o, n=h))
    GemmOp dOut{m->dOUT, m->O, 0, 0};
    GemmOp W3{m->wb + m->off(4), m->H, 0, 1};
    // dH2 must not overwrite H2 before dW3 is done: same stream, ordered
    if (!hipOk(gemm(dOut, W3, m->dH2, m->H, n, m->H, m->O, nullptr), "mlp dH2")) return false;
    const size_t cnt = (size_t)n * m->H;
    hipLaunchKernelGGL(k_reluBack, dim3((cnt + 255) / 256), dim3(256), 0, s, m->dH2, m->Z2, cnt);
    GemmOp dZ2T{m->dH2, m->H, 1, 0};
    if (!hipOk(gemm(dZ2T, H1, g + m->off(2), m->H, m->H, m->H, n, nullptr), "mlp dW2")) return false;
    hipLaunchKernelGGL(k_colsum, dim3((m->H + 63) / 64), dim3(64), 0, s, m->dH2, n, m->H, g + m->off(3));
    GemmOp dZ2{m->dH2, m->H, 0, 0};
    GemmOp W2{m->wb + m->off(2), m->H, 0, 1};
    if (!hipOk(gemm(dZ2, W2, m->dH1, m->H, n, m->H, m->H, nullptr), "mlp dH1")) return false;
    hipLaunchKernelGGL(k_reluBack, dim3((cnt + 255) / 256), dim3(256), 0, s, m->dH1, m->Z1, cnt);
    GemmOp dZ1T{m->dH1, m->H, 1, 0};
    GemmOp X{m->X, m->F, 0, 0};
    if (!hipOk(gemm(dZ1T, X, g + m->off(0), m->F, m->H, m->F, n, nullptr), "mlp dW1")) return false;
    hipLaunchKernelGGL(k_colsum, dim3((m->H + 63) / 64), dim3(64), 0, s, m->dH1, n, m->H, g + m->off(1));
    return hipOk(hipGetLastError(), "mlp backward");
}

}  // namespace

extern "C" {

p4g_mlp *p4g_mlpNew(int nIn, int nHidden, int nOut, unsigned long long seed)
{
    clearError();
    if (!deviceReady()) return nullptr;
    if (nIn < 1 || nHidden < 16 || nOut < 2 || (nOut & 1)) {
        setError("mlpNew: bad sizes (nOut holds means and log sds: even)");
        return nullptr;
    }
    auto *m = new p4g_mlp();
    m->F = nIn;
    m->H = nHidden;
    m->O = nOut;
    m->nW1 = (size_t)nHidden * nIn;
    m->nW2 = (size_t)nHidden * nHidden;
    m->nW3 = (size_t)nOut * nHidden;
    m->nParams = m->nW1 + nHidden + m->nW2 + nHidden + m->nW3 + nOut;
    std::vector<float> h(m->nParams, 0.f);
    std::mt19937_64 rng(seed);
    auto fill = [&](size_t off, size_t n, int fanIn, float gain) {
        std::normal_distribution<float> nd(0.f, gain * std::sqrt(2.0f / (float)fanIn));
        for (size_t i = 0; i < n; i++) h[off + i] = nd(rng);
    };
    fill(m->off(0), m->nW1, nIn, 1.f);
    fill(m->off(2), m->nW2, nHidden, 1.f);
    fill(m->off(4), m->nW3, nHidden, 0.1f);
    const size_t n = m->nParams;
    m->fused = nHidden <= MLP_MAX_H && nIn <= MLP_MAX_F && nOut <= MLP_MAX_O;
    m->Fp = (nIn + 31) & ~31;
    m->Hp = (nHidden + 63) & ~63;
    m->Op = (nOut + 31) & ~31;
    if (m->fused && (!hipOk(hipMalloc((void **)&m->pack, m->packElems() * 2), "hipMalloc mlp") ||
                     !hipOk(hipMemsetAsync(m->pack, 0, m->packElems() * 2, stream()), "mlp pack"))) {
        p4g_mlpFree(m);
        return nullptr;
    }
    if (!hipOk(hipMalloc((void **)&m->w, n * 4), "hipMalloc mlp") ||
        !hipOk(hipMalloc((void **)&m->wb, n * 2), "hipMalloc mlp") ||
        !hipOk(hipMalloc((void **)&m->g, n * 4), "hipMalloc mlp") ||
        !hipOk(hipMalloc((void **)&m->m, n * 4), "hipMalloc mlp") ||
        !hipOk(hipMalloc((void **)&m->v, n * 4), "hipMalloc mlp") ||
        !hipOk(hipMalloc((void **)&m->loss, 8), "hipMalloc mlp")) {
        p4g_mlpFree(m);
        return nullptr;
    }
    hipStream_t s = stream();
    (void)hipMemcpyAsync(m->w, h.data(), n * 4, hipMemcpyHostToDevice, s);
    (void)hipMemsetAsync(m->m, 0, n * 4, s);
    (void)hipMemsetAsync(m->v, 0, n * 4, s);
    repack(m);
    if (!hipOk(hipStreamSynchronize(s), "mlp init")) {
        p4g_mlpFree(m);
        return nullptr;
    }
    return m;
}

void p4g_mlpFree(p4g_mlp *m)
{
    if (!m) return;
    (void)hipStreamSynchronize(stream());
    float *fs[] = {m->w, m->g, m->m, m->v, m->loss, m->X, m->Z1, m->Z2, m->OUT, m->Y, m->MASK, m->dOUT, m->dH2,
                   m->dH1, m->rowLoss, m->sums, m->part};
    for (auto p : fs)
        if (p) (void)hipFree(p);
    unsigned short *us[] = {m->wb, m->pack, m->rowsT};
    for (auto p : us)
        if (p) (void)hipFree(p);
    delete m;
}

int p4g_mlpNumParams(const p4g_mlp *m) { return m ? (int)m->nParams : -1; }

int p4g_mlpGetParams(p4g_mlp *m, float *out)
{
    clearError();
    if (!m || !out) return 1;
    return hipOk(hipMemcpy(out, m->w, m->nParams * 4, hipMemcpyDeviceToHost), "mlp get params") ? 0 : 1;
}

int p4g_mlpSetParams(p4g_mlp *m, const float *in)
{
    clearError();
    if (!m || !in) return 1;
    hipStream_t s = stream();
    if (!hipOk(hipMemcpyAsync(m->w, in, m->nParams * 4, hipMemcpyHostToDevice, s), "mlp set params")) return 1;
    repack(m);
    return hipOk(hipStreamSynchronize(s), "mlp set params") ? 0 : 1;
}

int p4g_mlpForward(p4g_mlp *m, const float *x, int n, float *out)
{
    clearError();
    if (!m || !x || !out || n < 1) return 1;
    if (!ensureCap(m, n, false)) return 1;
    hipStream_t s = stream();
    if (!hipOk(hipMemcpyAsync(m->X, x, sizeof(float) * (size_t)n * m->F, hipMemcpyHostToDevice, s), "mlp input") ||
        !forward(m, n) ||
        !hipOk(hipMemcpyAsync(out, m->OUT, sizeof(float) * (size_t)n * m->O, hipMemcpyDeviceToHost, s), "mlp out"))
        return 1;
    return hipOk(hipStreamSynchronize(s), "mlp forward") ? 0 : 1;
}

static int uploadBatch(p4g_mlp *m, const float *x, const float *y, const float *mask, int n)
{
    const int D = m->O / 2;
    if (!ensureCap(m, n, true)) return 1;
    hipStream_t s = stream();
    if (!hipOk(hipMemcpyAsync(m->X, x, sizeof(float) * (size_t)n * m->F, hipMemcpyHostToDevice, s), "mlp x") ||
        !hipOk(hipMemcpyAsync(m->Y, y, sizeof(float) * (size_t)n * D, hipMemcpyHostToDevice, s), "mlp y") ||
        !hipOk(hipMemcpyAsync(m->MASK, mask, sizeof(float) * (size_t)n * D, hipMemcpyHostToDevice, s), "mlp mask"))
        return 1;
    return 0;
}

int p4g_mlpGradients(p4g_mlp *m, const float *x, const float *y, const float *mask, int n, float *grads,
                     float *loss)
{
    clearError();
    if (!m || !x || !y || !mask || n < 1) return 1;
    if (uploadBatch(m, x, y, mask, n) || !backward(m, n)) return 1;
    hipStream_t s = stream();
    if (grads && !hipOk(hipMemcpyAsync(grads, m->g, m->nParams * 4, hipMemcpyDeviceToHost, s), "mlp grads"))
        return 1;
    if (loss && !hipOk(hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, s), "mlp loss")) return 1;
    return hipOk(hipStreamSynchronize(s), "mlp gradients") ? 0 : 1;
}

int p4g_mlpTrainStep(p4g_mlp *m, const float *x, const float *y, const float *mask, int n, float lr,
                     float *loss)
{
    clearError();
    if (!m || !x || !y || !mask || n < 1) return 1;
    if (uploadBatch(m, x, y, mask, n)) return 1;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float step = (float)(m->step + 1);
    const float c1 = 1.f - std::pow(b1, step), c2 = 1.f - std::pow(b2, step);
    hipStream_t s = stream();
    if (m->fused ? !fusedBackward(m, n, true, lr, b1, b2, eps, c1, c2) : !backward(m, n)) return 1;
    m->step++;
    if (!m->fused)
        hipLaunchKernelGGL(k_adam, dim3((m->nParams + 255) / 256), dim3(256), 0, s, m->w, m->wb, m->g, m->m, m->v,
                       m->nParams, lr, b1, b2, eps, c1, c2);
    if (loss && !hipOk(hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, s), "mlp loss")) return 1;
    return hipOk(hipStreamSynchronize(s), "mlp train step") ? 0 : 1;
}

}  // extern "C"
