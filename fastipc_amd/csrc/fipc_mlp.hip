// fipc_mlp.hip -- per-vertex MLP of the learned Newton warm start on gfx950:
// products on the BF16 matrix cores (v_mfma_f32_32x32x16_bf16) with FP32
// accumulation, FP32 master weights trained with Adam, and a device-resident
// dataset of (feature, target) rows captured from solver trajectories.
//
// Network: n_in -> depth hidden layers of `width` (SiLU) -> n_out (linear).
// Parameters are packed per layer as W_l [fan_in][fan_out] (row-major, so a
// layer is H_out = act(H_in W_l + b_l)) followed by b_l [fan_out].
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>
#include "fipc_ctx.h"
#include "fipc_mlp.h"

#define TPB 256
static inline int nblk(long n, int t = TPB) { return (int)((n + t - 1) / t); }

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

enum { EPI_NONE = 0, EPI_BIAS_SILU = 1, EPI_BIAS = 2, EPI_DSILU = 3 };

// ---------------------------------------------------------------------------
// GEMM: C[M][N] = epilogue(A[M][K] B[K][N]).  A and B are FP32 in memory with
// arbitrary strides (A(m,k) = A[m sam + k sak], B(k,n) = B[k sbk + n sbn]), so
// transposed operands cost nothing; tiles are rounded to BF16 when staged in
// LDS.  A block of 4 waves computes a 64 x 64 tile, each wave one 32 x 32
// MFMA tile.  Operand layout of v_mfma_f32_32x32x16_bf16 (wave64): lane l
// supplies A[l % 32][8 (l / 32) + i] and B[8 (l / 32) + i][l % 32], i < 8;
// accumulator element j of lane l is D[8 (j / 4) + 4 (l / 32) + j % 4][l % 32].
// gridDim.z > 1 splits K: slice z covers [z kslice, (z + 1) kslice) and
// writes its partial product to C + z c_slice (EPI_NONE only).
// ---------------------------------------------------------------------------
#define GBM 64
#define GBN 64
#define GBK 32
#define LDSK (GBK + 8)

struct GemmArgs {
    int M, N, K;
    const float* A;
    long sam, sak;
    const float* B;
    long sbk, sbn;
    float* C;
    long ldc;
    long c_slice;
    int kslice;
    int epi;
    const float* bias;   // EPI_BIAS, EPI_BIAS_SILU
    const float* Z;      // EPI_DSILU: pre-activation, leading dimension ldc
    float* Zout;         // EPI_BIAS_SILU: pre-activation output (may be null)
};

// logistic sigmoid with the hardware reciprocal (about 1 ulp): the products
// that consume it round to BF16
__device__ __forceinline__ float sigm(float z) { return __builtin_amdgcn_rcpf(1.f + __expf(-z)); }

__global__ void __launch_bounds__(256) k_gemm_bf16(GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) __bf16 As[GBM][LDSK];
    __shared__ __attribute__((aligned(16))) __bf16 Bs[GBN][LDSK];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w >> 1, wn = w & 1;
    const int m0 = blockIdx.x * GBM, n0 = blockIdx.y * GBN;
    const int kbeg = blockIdx.z * g.kslice;
    const int kend = min(g.K, kbeg + g.kslice);
    floatx16 acc;
#pragma unroll
    for (int j = 0; j < 16; j++) acc[j] = 0.f;
    // staging: thread -> tile row sr (0..63), k offsets sk..sk+7
    const int sr = tid >> 2, sk = (tid & 3) * 8;
    const int am = m0 + sr, bn = n0 + sr;
    for (int k0 = kbeg; k0 < kend; k0 += GBK) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            int k = k0 + sk + j;
            bool kin = k < kend;
            float a = (am < g.M && kin) ? g.A[(long)am * g.sam + (long)k * g.sak] : 0.f;
            float b = (bn < g.N && kin) ? g.B[(long)k * g.sbk + (long)bn * g.sbn] : 0.f;
            As[sr][sk + j] = (__bf16)a;
            Bs[sr][sk + j] = (__bf16)b;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GBK; kk += 16) {
            bf16x8 a = *(const bf16x8*)&As[wm * 32 + (lane & 31)][kk + (lane >> 5) * 8];
            bf16x8 b = *(const bf16x8*)&Bs[wn * 32 + (lane & 31)][kk + (lane >> 5) * 8];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    float* C = g.C + (long)blockIdx.z * g.c_slice;
    const int col = n0 + wn * 32 + (lane & 31);
    if (col >= g.N) return;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        int row = m0 + wm * 32 + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
        if (row >= g.M) continue;
        long o = (long)row * g.ldc + col;
        float v = acc[j];
        if (g.epi == EPI_BIAS_SILU) {
            v += g.bias[col];
            if (g.Zout) g.Zout[o] = v;
            v = v * sigm(v);
        } else if (g.epi == EPI_BIAS) {
            v += g.bias[col];
        } else if (g.epi == EPI_DSILU) {
            float z = g.Z[o], s = sigm(z);
            v *= s * (1.f + z * (1.f - s));
        }
        C[o] = v;
    }
}

static int gemm(hipStream_t s, int M, int N, int K, const float* A, long sam, long sak, const float* B, long sbk,
                long sbn, float* C, long ldc, int epi, const float* bias, const float* Z, float* Zout, int splits = 1,
                long c_slice = 0)
{
    if (M <= 0 || N <= 0) return FIPC_OK;
    GemmArgs g;
    g.M = M; g.N = N; g.K = K;
    g.A = A; g.sam = sam; g.sak = sak;
    g.B = B; g.sbk = sbk; g.sbn = sbn;
    g.C = C; g.ldc = ldc; g.c_slice = c_slice;
    int per = (K + splits - 1) / splits;
    g.kslice = ((per + GBK - 1) / GBK) * GBK;
    g.epi = epi; g.bias = bias; g.Z = Z; g.Zout = Zout;
    dim3 grid((M + GBM - 1) / GBM, (N + GBN - 1) / GBN, splits);
    k_gemm_bf16<<<grid, 256, 0, s>>>(g);
    HIPCHK(hipGetLastError());
    return FIPC_OK;
}

// ---------------------------------------------------------------------------
// elementwise and reduction kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long mix64(unsigned long long z)
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ float unif(unsigned long long seed, unsigned long long i)
{
    return (float)((mix64(seed * 0x2545f4914f6cdd1dull + i) >> 40) * (1.0 / 16777216.0));  // [0, 1)
}
// W uniform in (-a, a), b = 0
__global__ void k_init_layer(long nw, int nb, float* W, float* b, float a, unsigned long long seed)
{
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < nw) W[i] = (2.f * unif(seed, i) - 1.f) * a;
    if (i < nb) b[i] = 0.f;
}
// out[i] = sum over slices of P[s n + i], in slice order
__global__ void k_sum_slices(long n, int S, const float* P, float* out)
{
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = 0.f;
    for (int s = 0; s < S; s++) v += P[s * n + i];
    out[i] = v;
}
// column sums of slices of A[M][N]: out[z N + c] = sum of A[m][c] over the rows of
// slice z = blockIdx.y
__global__ void k_colsum(int M, int N, int slice, const float* A, float* out)
{
    __shared__ float sh[4][64];
    int c = blockIdx.x * 64 + (threadIdx.x & 63), r0 = threadIdx.x >> 6;
    int m0 = blockIdx.y * slice, m1 = min(M, m0 + slice);
    float v = 0.f;
    if (c < N)
        for (int m = m0 + r0; m < m1; m += 4) v += A[(long)m * N + c];
    sh[r0][threadIdx.x & 63] = v;
    __syncthreads();
    if (r0 == 0 && c < N)
        out[(long)blockIdx.y * N + c] = sh[0][threadIdx.x] + sh[1][threadIdx.x] + sh[2][threadIdx.x] + sh[3][threadIdx.x];
}
// dY = 2 (Y - T) / (M N); per-block partial sums of (Y - T)^2 / (M N)
__global__ void k_mse(long n, float inv, const float* Y, const float* T, float* dY, float* part)
{
    __shared__ float sh[TPB];
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    float e = 0.f;
    if (i < n) {
        float d = Y[i] - T[i];
        dY[i] = 2.f * d * inv;
        e = d * d * inv;
    }
    sh[threadIdx.x] = e;
    __syncthreads();
    for (int o = TPB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}
__global__ void k_adam(long n, float* p, const float* g, float* m, float* v, float lr, float b1, float b2, float eps,
                       float c1, float c2)
{
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gi = g[i];
    float mi = b1 * m[i] + (1.f - b1) * gi;
    float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
// batch of B rows drawn uniformly (with replacement) from the dataset
__global__ void k_gather_batch(int B, long nds, unsigned long long seed, int nin, int nout, const float* dsX,
                               const float* dsT, float* X, float* T)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    long r = (long)(mix64(seed * 0x9e3779b97f4a7c15ull + (unsigned long long)i) % (unsigned long long)nds);
    for (int k = 0; k < nin; k++) X[(long)i * nin + k] = dsX[r * nin + k];
    for (int k = 0; k < nout; k++) T[(long)i * nout + k] = dsT[r * nout + k];
}

#ifndef FI_RT
#define FI_RT 4
#endif
#ifndef FI_ROWS
#define FI_ROWS (32 * FI_RT)
#endif
// a wave takes 64 output features (two 32-feature tiles) of FI_RT 32-row
// tiles: wave w takes features 64 (w % 4) .. +64 of rows 32 FI_RT (w / 4) ..
constexpr int FI_WROWS = 32 * FI_RT;
static_assert(FI_ROWS % FI_WROWS == 0, "rows per block");
constexpr int FI_THREADS = 4 * (FI_ROWS / FI_WROWS) * 64;
#define FI_W 256
#define FI_LDS (FI_W + 8)
// D[feature][row] += W[feature][k..k+15] . H[row][k..k+15] over the layer's
// fan-in KIN for NF 32-feature tiles from f0 and RT 32-row tiles from rbase.
// The A operand is a weight fragment (8 consecutive k of one output feature,
// one 16-byte load from the packed BF16 weights), the B operand an
// activation fragment (8 consecutive k of one row, one 16-byte LDS read);
// the next k step's weight fragments are loaded before this step's products.
template <int NF, int RT>
__device__ __forceinline__ void fi_step(const bf16x8 (&a)[NF], const __bf16 (*H)[FI_LDS], int rbase, int lane, int k0,
                                        floatx16 (&acc)[NF][RT])
{
    bf16x8 b[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) b[rt] = *(const bf16x8*)&H[rbase + rt * 32 + (lane & 31)][k0 + (lane >> 5) * 8];
#pragma unroll
    for (int f = 0; f < NF; f++)
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
            acc[f][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[f], b[rt], acc[f][rt], 0, 0, 0);
}
template <int KIN, int NF, int RT>
__device__ __forceinline__ void fi_layer(const __bf16* __restrict__ W, const __bf16 (*H)[FI_LDS], int f0, int rbase,
                                         int lane, floatx16 (&acc)[NF][RT])
{
    static_assert(KIN == 16 || KIN % 32 == 0, "fan-in");
    const __bf16* wp[NF];
    bf16x8 a[NF], an[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        wp[f] = W + (long)(f0 / 32 + f) * 32 * KIN + lane * 8;
        a[f] = *(const bf16x8*)wp[f];
    }
    if (KIN == 16) {
        fi_step<NF, RT>(a, H, rbase, lane, 0, acc);
        return;
    }
    // two k steps per pass in alternating registers: the fragments of the
    // next step are in flight during this step's products (the last pass
    // reloads its own last step rather than read past the row)
    for (int k0 = 0; k0 < KIN; k0 += 32) {
#pragma unroll
        for (int f = 0; f < NF; f++) an[f] = *(const bf16x8*)(wp[f] + 32 * (k0 + 16));
        fi_step<NF, RT>(a, H, rbase, lane, k0, acc);
        const int kn = k0 + 32 < KIN ? k0 + 32 : KIN - 16;
#pragma unroll
        for (int f = 0; f < NF; f++) a[f] = *(const bf16x8*)(wp[f] + 32 * kn);
        fi_step<NF, RT>(an, H, rbase, lane, k0 + 16, acc);
    }
}
__device__ __forceinline__ unsigned int bf16_bits(float v)
{
    return (unsigned int)__builtin_bit_cast(unsigned short, (__bf16)v);
}
// hidden-layer epilogue: bias, SiLU, BF16 into the activation tile.  Lane l
// holds features f + 8 (j / 4) + 4 (l / 32) + j % 4 of row (l % 32) of each
// tile, so each group of four j is four consecutive features of one row:
// one 8-byte LDS store
template <int RT>
__device__ __forceinline__ void fi_silu_store(const floatx16 (&acc)[2][RT], const float* __restrict__ bias,
                                              __bf16 (*H)[FI_LDS], int f0, int rbase, int lane)
{
#pragma unroll
    for (int ft = 0; ft < 2; ft++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int m = f0 + ft * 32 + 8 * g + 4 * (lane >> 5);
            const float b0 = bias[m], b1 = bias[m + 1], b2 = bias[m + 2], b3 = bias[m + 3];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                float z0 = acc[ft][rt][4 * g] + b0, z1 = acc[ft][rt][4 * g + 1] + b1;
                float z2 = acc[ft][rt][4 * g + 2] + b2, z3 = acc[ft][rt][4 * g + 3] + b3;
                uint2 pk;
                pk.x = bf16_bits(z0 * sigm(z0)) | (bf16_bits(z1 * sigm(z1)) << 16);
                pk.y = bf16_bits(z2 * sigm(z2)) | (bf16_bits(z3 * sigm(z3)) << 16);
                *(uint2*)&H[rbase + rt * 32 + (lane & 31)][m] = pk;
            }
        }
}
// ---------------------------------------------------------------------------
// Fused inference for the warm-start shape (16 -> 4 x 256 SiLU -> 3): a block
// takes FI_ROWS rows through all five layers; the activations stay in LDS as
// BF16 (the products' input precision) and never touch HBM.  Weights are read
// from L2 as BF16 fragments per layer (k_pack_weights; the last layer padded to
// 32 rows of zeros).  In the hidden layers wave w owns output features
// 64 (w % 4) .. +64 (two 32-feature MFMA tiles) of its FI_RT 32-row tiles:
// each weight fragment feeds FI_RT MFMAs, each activation fragment two.  The
// output layer's 32-row tiles are shared out over all the block's waves.
// The weight fragments come from L1/L2, so rows per wave set the loads per
// product: 200k rows take 199 us with 2 row tiles (108 VGPRs, 4 waves per
// SIMD), 159 us with 3, 151 us with 4 (192 VGPRs, 2 waves per SIMD, two
// 128-row blocks per CU), all with the same bits and with weights row by row (132
// us as fragments); 5 or more row tiles fit only one wave per SIMD.  The accumulation order over k is the generic GEMM's.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(FI_THREADS) __attribute__((amdgpu_waves_per_eu(FI_RT <= 2 ? 4 : 2)))
k_mlp_infer(int n, const float* __restrict__ X, const __bf16* __restrict__ Wt, const float* __restrict__ params,
            const long* __restrict__ boff, float* __restrict__ Y)
{
    __shared__ __attribute__((aligned(16))) __bf16 H[FI_ROWS][FI_LDS];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int f0 = (w & 3) * 64, rbase = (w >> 2) * FI_WROWS;
    const long r0 = (long)blockIdx.x * FI_ROWS;
    // input tile: FI_ROWS rows x 16 features
    for (int e = tid; e < FI_ROWS * 16; e += blockDim.x) {
        int r = e >> 4, k = e & 15;
        long gr = r0 + r;
        H[r][k] = (__bf16)(gr < n ? X[gr * 16 + k] : 0.f);
    }
    __syncthreads();
    const __bf16* W = Wt;
    for (int l = 0; l < 4; l++) {
        floatx16 acc[2][FI_RT];
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int rt = 0; rt < FI_RT; rt++)
#pragma unroll
                for (int j = 0; j < 16; j++) acc[f][rt][j] = 0.f;
        if (l == 0) fi_layer<16, 2, FI_RT>(W, H, f0, rbase, lane, acc);
        else fi_layer<FI_W, 2, FI_RT>(W, H, f0, rbase, lane, acc);
        __syncthreads();  // every wave has read this layer's input
        fi_silu_store<FI_RT>(acc, params + boff[l], H, f0, rbase, lane);
        __syncthreads();
        W += (long)FI_W * (l == 0 ? 16 : FI_W);
    }
    // output layer: features 0..2 of the first 32-feature tile, one 32-row
    // tile per wave at a time
    const float* bias = params + boff[4];
    for (int t = w; t < FI_ROWS / 32; t += FI_THREADS / 64) {
        floatx16 acc[1][1];
#pragma unroll
        for (int j = 0; j < 16; j++) acc[0][0][j] = 0.f;
        fi_layer<FI_W, 1, 1>(W, H, 0, t * 32, lane, acc);
        const long gr = r0 + t * 32 + lane;
        if (lane < 32 && gr < n)
#pragma unroll
            for (int i = 0; i < 3; i++) Y[gr * 3 + i] = acc[0][0][i] + bias[i];
    }
}
// BF16 weights of the warm-start shape from the FP32 parameters, one launch: per
// layer Wt[n][k] (transposed, the last padded to 32 rows), then, for the
// backward products, W[k][n] of layers 1 to 4 (the last padded to 16 columns).
// Each matrix is stored as its A fragments: 32 rows by 16 columns, 8 consecutive
// columns per lane, lane after lane, so a wave's load is 1 KB in a row.  Row by
// row, a load touched 32 bytes of each of 32 lines, and the lines of two blocks
// did not stay in L1 until their next quarter was read: inference of 200k rows
// 151 us row by row, 132 in fragments.
constexpr int FI_L = 5, FI_IN = 16, FI_OUT = 3;
constexpr long FI_WT = (long)FI_W * FI_IN + 3L * FI_W * FI_W + 32L * FI_W;  // elements of the first part
constexpr long FI_WN = 3L * FI_W * FI_W + 16L * FI_W;                       // and of the second
// row and column of the j-th element of a matrix of ld columns in fragment order
__device__ __forceinline__ void fi_frag(int j, int ld, int& row, int& col)
{
    const int lane = (j >> 3) & 63, t = j >> 9, steps = ld / 16;
    row = t / steps * 32 + (lane & 31);
    col = t % steps * 16 + (lane >> 5) * 8 + (j & 7);
}
__global__ void k_pack_weights(const float* __restrict__ params, const long* __restrict__ boff, __bf16* __restrict__ w,
                               long total)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= total) return;
    long j = i;
    float v = 0.f;
    if (i < FI_WT) {
        int l = 0;
        long size = (long)FI_W * FI_IN;
        while (j >= size) { j -= size; l++; size = l == FI_L - 1 ? 32L * FI_W : (long)FI_W * FI_W; }
        const int fi = l == 0 ? FI_IN : FI_W, fo = l == FI_L - 1 ? FI_OUT : FI_W;
        int n, k;
        fi_frag((int)j, fi, n, k);
        if (n < fo) v = params[boff[l] - (long)fi * fo + (long)k * fo + n];
    } else {
        j -= FI_WT;
        const int l = j < 3L * FI_W * FI_W ? 1 + (int)(j / (FI_W * FI_W)) : FI_L - 1;
        j -= (l - 1L) * FI_W * FI_W;
        const int fo = l == FI_L - 1 ? FI_OUT : FI_W, ld = l == FI_L - 1 ? 16 : FI_W;
        int k, n;
        fi_frag((int)j, ld, k, n);
        if (n < fo) v = params[boff[l] - (long)FI_W * fo + (long)k * fo + n];
    }
    w[i] = (__bf16)v;
}

// ---------------------------------------------------------------------------
// Fused training for the warm-start shape, in three launches after the packing:
//  - k_mlp_fwdbwd: a block takes 32 rows through the five layers and back.  A
//    wave owns 64 features: their pre-activations stay in its registers (4 x 32
//    floats), activations and gradients pass between waves through one LDS tile
//    in BF16 (the precision of the products' inputs).  What the weight gradients
//    need, the inputs A_l of the layers and the gradients G_l at their outputs, is
//    written in BF16, transposed ([feature][row]), so that the next launch's
//    fragments (8 consecutive rows of a feature) are 16-byte loads; the bias
//    gradients' FP32 column sums and the loss are written per block;
//  - k_mlp_dw: dW_l = A_l^T G_l in 64 x 64 tiles over row slices;
//  - k_mlp_sum: the slices' and the blocks' sums.
// Layer by layer, with FP32 activations in HBM and a column sum of 8,192 rows
// in four workgroups (385 us a layer), loss and gradient of 8,192 rows took
// 3.0 ms of kernels; like this 69 us (35 + 28 + 6; the packing, once the
// parameters changed, 8 more).
// ---------------------------------------------------------------------------
struct TrainBufs {
    __bf16* A;      // A_0 [16][ld], then A_1 .. A_4 [256][ld]
    __bf16* G;      // G_0 .. G_3 [256][ld], then G_4 [32][ld]
    float* bias;    // per block 4 x 256 + 3 column sums
    float* loss;    // per block
    long ld;        // rows, a multiple of 32
};
constexpr int FI_NB = 4 * FI_W + FI_OUT;  // bias parameters
__device__ __forceinline__ long fi_a(int l, long ld) { return l == 0 ? 0 : (FI_IN + (l - 1L) * FI_W) * ld; }
// D[feature][row] for this wave's 64 features of the block's 32 rows; four k
// steps of weight fragments are in flight ahead of the products.  The chunks stay
// a loop: unrolled, with the fragments' addresses spelled out, the kernel of 8,192
// rows takes 61 us, as a loop 36 (51 unrolled with row-by-row weights).
template <int KIN>
__device__ __forceinline__ void ft_layer(const __bf16* __restrict__ W, const __bf16 (*H)[FI_LDS], int f0, int lane,
                                         floatx16 (&acc)[2])
{
    constexpr int CH = KIN == 16 ? 1 : 4;  // k steps per chunk
    const __bf16* wp[2];
#pragma unroll
    for (int f = 0; f < 2; f++) {
        wp[f] = W + (long)(f0 / 32 + f) * 32 * KIN + lane * 8;
#pragma unroll
        for (int j = 0; j < 16; j++) acc[f][j] = 0.f;
    }
    bf16x8 a[2][CH], an[2][CH];
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int c = 0; c < CH; c++) a[f][c] = *(const bf16x8*)(wp[f] + 32 * (16 * c));
#pragma unroll 1
    for (int k0 = 0; k0 < KIN; k0 += 16 * CH) {
        if (k0 + 16 * CH < KIN)
#pragma unroll
            for (int f = 0; f < 2; f++)
#pragma unroll
                for (int c = 0; c < CH; c++) an[f][c] = *(const bf16x8*)(wp[f] + 32 * (k0 + 16 * (CH + c)));
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const bf16x8 b = *(const bf16x8*)&H[lane & 31][k0 + 16 * c + (lane >> 5) * 8];
#pragma unroll
            for (int f = 0; f < 2; f++) acc[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[f][c], b, acc[f], 0, 0, 0);
        }
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int c = 0; c < CH; c++) a[f][c] = an[f][c];
    }
}
// value j of tile f of a lane belongs to feature f0 + 32 f + 8 (j / 4) + 4 (lane / 32)
// + j % 4 of row lane % 32: to the LDS tile ([row][feature]) and, transposed, to
// dst ([feature][ld])
__device__ __forceinline__ void ft_store(const float (&v)[2][16], __bf16 (*H)[FI_LDS], __bf16* __restrict__ dst, long ld,
                                         long r0, int f0, int lane)
{
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int m = f0 + 32 * f + 8 * g + 4 * (lane >> 5);
            uint2 pk;
            unsigned int b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                b[i] = bf16_bits(v[f][4 * g + i]);
                ((unsigned short*)dst)[(m + i) * ld + r0 + (lane & 31)] = (unsigned short)b[i];
            }
            pk.x = b[0] | (b[1] << 16);
            pk.y = b[2] | (b[3] << 16);
            *(uint2*)&H[lane & 31][m] = pk;
        }
}
// The last block's rows past n are zeros in every layer and gradient: what the
// biases alone give there may overflow though no row does, and its product with a
// zero gradient would be NaN.  In a branch of that block: 64 selects a layer in
// every block cost 2 us of 8,192 rows' 177.
__device__ __forceinline__ void ft_mask(float (&v)[2][16], bool row, bool partial)
{
    if (partial)
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int j = 0; j < 16; j++) v[f][j] = row ? v[f][j] : 0.f;
}
// column sums over the block's 32 rows: each step hands half of the values to the
// lane across, so 31 exchanges reduce 32 values; lane l % 32 ends with value l % 32
template <int N>
__device__ __forceinline__ float ft_fold(const float (&w)[2 * N], int lane)
{
    float h[N];
    const bool up = lane & N;
#pragma unroll
    for (int k = 0; k < N; k++) {
        const float lo = w[k], hi = w[k + N];
        h[k] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, N, 64);
    }
    if constexpr (N == 1) return h[0];
    else return ft_fold<N / 2>(h, lane);
}
__device__ __forceinline__ void ft_colsum(const float (&v)[2][16], float* __restrict__ out, int f0, int lane)
{
    float w[32];
#pragma unroll
    for (int k = 0; k < 32; k++) w[k] = v[k >> 4][k & 15];
    const float sum = ft_fold<16>(w, lane);
    const int k = lane & 31, j = k & 15;
    out[f0 + 32 * (k >> 4) + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3)] = sum;
}
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1)))
k_mlp_fwdbwd(int n, const float* __restrict__ X, const float* __restrict__ T, const __bf16* __restrict__ Wt,
             const float* __restrict__ params, const long* __restrict__ boff, float inv, TrainBufs tb)
{
    __shared__ __attribute__((aligned(16))) __bf16 H[32][FI_LDS];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int f0 = w * 64;
    const long r0 = (long)blockIdx.x * 32, ld = tb.ld;
    const __bf16* Wn = Wt + FI_WT;
    float* bias = tb.bias + (long)blockIdx.x * FI_NB;
    for (int e = tid; e < 32 * FI_IN; e += 256) {
        const int r = e >> 4, k = e & 15;
        H[r][k] = (__bf16)(r0 + r < n ? X[(r0 + r) * FI_IN + k] : 0.f);
    }
    __syncthreads();
    for (int e = tid; e < 32 * FI_IN; e += 256) tb.A[(long)(e >> 5) * ld + r0 + (e & 31)] = H[e & 31][e >> 5];
    // forward
    float z[4][2][16], v[2][16];
    floatx16 acc[2];
    const __bf16* W = Wt;
#pragma unroll
    for (int l = 0; l < 4; l++) {
        if (l == 0) ft_layer<FI_IN>(W, H, f0, lane, acc);
        else ft_layer<FI_W>(W, H, f0, lane, acc);
        const float* b = params + boff[l];
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const float zz = acc[f][j] + b[f0 + 32 * f + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3)];
                z[l][f][j] = zz;
                v[f][j] = zz * sigm(zz);
            }
        ft_mask(v, r0 + (lane & 31) < n, r0 + 32 > n);
        __syncthreads();  // every wave has read this layer's input
        ft_store(v, H, tb.A + fi_a(l + 1, ld), ld, r0, f0, lane);
        __syncthreads();
        W += (long)FI_W * (l == 0 ? FI_IN : FI_W);
    }
    // output layer (its first 32-feature tile, on the first wave): loss and G_4
    float dy[3] = {0.f, 0.f, 0.f};
    if (w == 0) {
        floatx16 y[1][1];
#pragma unroll
        for (int j = 0; j < 16; j++) y[0][0][j] = 0.f;
        fi_layer<FI_W, 1, 1>(W, H, 0, 0, lane, y);
        const long gr = r0 + (lane & 31);
        const float* b = params + boff[4];
        float e = 0.f;
        if (lane < 32 && gr < n)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const float d = y[0][0][i] + b[i] - T[gr * 3 + i];
                dy[i] = 2.f * d * inv;
                e += d * d * inv;
            }
        float s[4] = {e, dy[0], dy[1], dy[2]};
#pragma unroll
        for (int o = 16; o > 0; o >>= 1)
#pragma unroll
            for (int i = 0; i < 4; i++) s[i] += __shfl_xor(s[i], o, 64);
        if (lane == 0) {
            tb.loss[blockIdx.x] = s[0];
#pragma unroll
            for (int i = 0; i < 3; i++) bias[4 * FI_W + i] = s[1 + i];
        }
    }
    __syncthreads();
    if (w == 0) {
        // the gradient as the next product's input (16 columns, 3 used), and G_4
        __bf16* g4 = tb.G + 4L * FI_W * ld;
        if (lane < 32) {
#pragma unroll
            for (int k = 0; k < 16; k++) H[lane][k] = (__bf16)(k < 3 ? dy[k] : 0.f);
#pragma unroll
            for (int k = 0; k < 32; k++) g4[k * ld + r0 + lane] = (__bf16)(k < 3 ? dy[k] : 0.f);
        }
    }
    __syncthreads();
    // backward: G_{l-1} = (G_l W_l^T) silu'(z_{l-1})
#pragma unroll
    for (int l = 4; l >= 1; l--) {
        const __bf16* B = Wn + (l - 1L) * FI_W * FI_W;
        if (l == 4) ft_layer<16>(B, H, f0, lane, acc);
        else ft_layer<FI_W>(B, H, f0, lane, acc);
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const float zz = z[l - 1][f][j], s = sigm(zz);
                v[f][j] = acc[f][j] * (s * (1.f + zz * (1.f - s)));
            }
        ft_mask(v, r0 + (lane & 31) < n, r0 + 32 > n);
        __syncthreads();  // every wave has read G_l
        ft_store(v, H, tb.G + (l - 1L) * FI_W * ld, ld, r0, f0, lane);
        ft_colsum(v, bias + (l - 1) * FI_W, f0, lane);
        __syncthreads();
    }
}
// dW_l tiles: 64 inputs x 64 outputs of one layer over one slice of rows; the
// four waves take every fourth k step and add their tiles in LDS in order.
// Blocks of a slice: 4 tiles of layer 0 (16 inputs), 16 each of layers 1 to 3,
// 4 of layer 4 (3 outputs)
constexpr int FI_TILES = 4 + 3 * 16 + 4;
__global__ void __launch_bounds__(256) k_mlp_dw(TrainBufs tb, int slice, const long* __restrict__ boff, long nparams,
                                                float* __restrict__ part)
{
    __shared__ float S[64][65];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int t = blockIdx.x;
    const int l = t < 4 ? 0 : (t < 52 ? 1 + (t - 4) / 16 : 4);
    const int fi = l == 0 ? FI_IN : FI_W, fo = l == 4 ? FI_OUT : FI_W, fog = l == 4 ? 32 : FI_W;
    const int tt = t < 4 ? t : (t < 52 ? (t - 4) % 16 : t - 52);
    const int m0 = l == 0 ? 0 : (l == 4 ? tt * 64 : (tt >> 2) * 64), n0 = l == 4 ? 0 : (l == 0 ? tt : tt & 3) * 64;
    const long ld = tb.ld, k0 = (long)blockIdx.y * slice, k1 = min(ld, k0 + slice);
    const __bf16* A = tb.A + fi_a(l, ld);
    const __bf16* G = tb.G + (long)l * FI_W * ld;
    floatx16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int j = 0; j < 16; j++) acc[a][b][j] = 0.f;
    const __bf16 *pa[2], *pb[2];
    bool ina[2], inb[2];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int m = m0 + 32 * a + (lane & 31), c = n0 + 32 * a + (lane & 31);
        ina[a] = m < fi;
        inb[a] = c < fog;
        pa[a] = A + (ina[a] ? m : 0) * ld + (lane >> 5) * 8;
        pb[a] = G + (inb[a] ? c : 0) * ld + (lane >> 5) * 8;
    }
    bf16x8 zero;
#pragma unroll
    for (int i = 0; i < 8; i++) zero[i] = (__bf16)0.f;
#pragma unroll 4
    for (long k = k0 + 16 * w; k < k1; k += 64) {
        bf16x8 fa[2], fb[2];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            fa[a] = ina[a] ? *(const bf16x8*)(pa[a] + k) : zero;
            fb[a] = inb[a] ? *(const bf16x8*)(pb[a] + k) : zero;
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
    }
    for (int v = 0; v < 4; v++) {
        if (w == v)
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        float& s = S[32 * a + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3)][32 * b + (lane & 31)];
                        s = v == 0 ? acc[a][b][j] : s + acc[a][b][j];
                    }
        __syncthreads();
    }
    float* out = part + (long)blockIdx.y * nparams + boff[l] - (long)fi * fo;
    for (int e = tid; e < 64 * 64; e += 256) {
        const int m = m0 + (e >> 6), c = n0 + (e & 63);
        if (m < fi && c < fo) out[(long)m * fo + c] = S[e >> 6][e & 63];
    }
}
// grads: weights from S slices, biases from nb blocks' column sums (the first
// nwb blocks take 64 biases each, 16 rows of threads over the blocks)
__global__ void __launch_bounds__(1024) k_mlp_sum(long nparams, int S, const float* __restrict__ part, int nb,
                                                  const float* __restrict__ bias, const long* __restrict__ boff,
                                                  int nwb, float* __restrict__ grads)
{
    __shared__ float sh[16][64];
    if ((int)blockIdx.x < nwb) {
        const int c = (int)blockIdx.x * 64 + (threadIdx.x & 63), r = threadIdx.x >> 6;
        float v = 0.f;
        if (c < FI_NB)
#pragma unroll 8
            for (int b = r; b < nb; b += 16) v += bias[(long)b * FI_NB + c];
        sh[r][threadIdx.x & 63] = v;
        __syncthreads();
        if (r == 0 && c < FI_NB) {
            float t = 0.f;
            for (int k = 0; k < 16; k++) t += sh[k][threadIdx.x];
            grads[boff[min(c / FI_W, 4)] + (c < 4 * FI_W ? c % FI_W : c - 4 * FI_W)] = t;
        }
        return;
    }
    const long i = ((long)blockIdx.x - nwb) * 1024 + threadIdx.x;
    if (i >= nparams) return;
    for (int l = 0; l < FI_L; l++)
        if (i >= boff[l] && i < boff[l] + (l == 4 ? FI_OUT : FI_W)) return;  // a bias
    float v = 0.f;
#pragma unroll 8
    for (int s = 0; s < S; s++) v += part[s * nparams + i];
    grads[i] = v;
}

// ---------------------------------------------------------------------------
// the network object
// ---------------------------------------------------------------------------
struct fipc_mlp {
    int n_in = 0, width = 0, depth = 0, n_out = 0, L = 0;
    std::vector<int> dim;          // dim[0] = n_in, ..., dim[L] = n_out
    std::vector<long> woff, boff;  // offsets of W_l and b_l in the packed parameters
    long nparams = 0;
    DVec<float> params, grads, am, av;
    long adam_t = 0;
    int cap = 0;                   // rows the layer outputs H hold
    int tcap = 0;                  // rows the training buffers (Z, gradients, X, T) hold
    std::vector<DVec<float>> H, Z; // H[l] (l >= 1) layer outputs, Z[l] hidden pre-activations
    DVec<float> X, T, dA, dB, part, loss;
    // fused inference (warm-start shape only): packed BF16 weights, stale
    // after any parameter change
    bool fused = false;
    bool wt_ok = false;
    DVec<__bf16> wt;
    // fused training: layer inputs and output gradients in BF16, transposed, and
    // the blocks' bias sums
    DVec<__bf16> tA, tG;
    DVec<float> tbias;
    DVec<long> dboff;
    // dataset
    DVec<float> dsX, dsT;
    long ds_n = 0;
    hipStream_t s = nullptr;
};

static int mlp_reserve(fipc_mlp* m, int rows, bool train)
{
    if (rows > m->cap) {
        // the fused kernels keep the hidden layers on the chip
        for (int l = m->fused ? m->L : 1; l <= m->L; l++) STCHK(ensure(m->H[l], (size_t)rows * m->dim[l]));
        m->cap = rows;
    }
    if (train && rows > m->tcap) {
        if (!m->fused) {
            for (int l = 1; l < m->L; l++) STCHK(ensure(m->Z[l], (size_t)rows * m->dim[l]));
            int wmax = *std::max_element(m->dim.begin(), m->dim.end());
            STCHK(ensure(m->dA, (size_t)rows * wmax));
            STCHK(ensure(m->dB, (size_t)rows * wmax));
        }
        STCHK(ensure(m->X, (size_t)rows * m->n_in));
        STCHK(ensure(m->T, (size_t)rows * m->n_out));
        STCHK(ensure(m->loss, (size_t)std::max(nblk((long)rows * m->n_out), (rows + 31) / 32) + 8));
        m->tcap = rows;
    }
    return FIPC_OK;
}

// forward of n rows from device X; Y (device, n x n_out) in the network's buffer.
// With train != 0 the hidden pre-activations are kept for the backward pass.
static int mlp_forward(fipc_mlp* m, hipStream_t s, int n, const float* X, bool train)
{
    STCHK(mlp_reserve(m, n, train));
    const float* in = X;
    for (int l = 0; l < m->L; l++) {
        int fi = m->dim[l], fo = m->dim[l + 1];
        const float* W = m->params.p + m->woff[l];
        const float* b = m->params.p + m->boff[l];
        bool last = l == m->L - 1;
        STCHK(gemm(s, n, fo, fi, in, fi, 1, W, fo, 1, m->H[l + 1].p, fo, last ? EPI_BIAS : EPI_BIAS_SILU, b, nullptr,
                   (!last && train) ? m->Z[l + 1].p : nullptr));
        in = m->H[l + 1].p;
    }
    return FIPC_OK;
}

static int mlp_pack(fipc_mlp* m, hipStream_t s);
// loss partials of n rows: per block of the fused kernel, or of k_mse
static int mlp_loss_parts(const fipc_mlp* m, int n) { return m->fused ? (n + 31) / 32 : nblk((long)n * m->n_out); }
static int mlp_backward_fused(fipc_mlp* m, hipStream_t s, int n, const float* X, const float* T)
{
    const int nb = (n + 31) / 32;
    // the weight gradients' row slices, at most 32: one below 1,024 rows, then of
    // at least 512, rounded up to the four waves' 64 rows.  So the last ones may be
    // short or empty (16,416 rows: 28 of 576, one of 288, three that store zeros)
    const long ld = 32L * nb;
    const int S = (int)std::max(1L, std::min(32L, ld / 512));
    const int slice = (int)((ld + 64L * S - 1) / (64L * S)) * 64;
    STCHK(mlp_pack(m, s));
    STCHK(ensure(m->tA, (size_t)ld * (FI_IN + 4 * FI_W)));
    STCHK(ensure(m->tG, (size_t)ld * (4 * FI_W + 32)));
    STCHK(ensure(m->tbias, (size_t)nb * FI_NB));
    STCHK(ensure(m->part, (size_t)S * m->nparams));
    const TrainBufs tb{m->tA.p, m->tG.p, m->tbias.p, m->loss.p, ld};
    k_mlp_fwdbwd<<<nb, 256, 0, s>>>(n, X, T, m->wt.p, m->params.p, m->dboff.p, 1.f / (float)((long)n * m->n_out), tb);
    k_mlp_dw<<<dim3(FI_TILES, S), 256, 0, s>>>(tb, slice, m->dboff.p, m->nparams, m->part.p);
    const int nwb = (FI_NB + 63) / 64;
    k_mlp_sum<<<nwb + (int)((m->nparams + 1023) / 1024), 1024, 0, s>>>(m->nparams, S, m->part.p, nb, m->tbias.p,
                                                                      m->dboff.p, nwb, m->grads.p);
    HIPCHK(hipGetLastError());
    return FIPC_OK;
}

// gradient of the mean squared error over n rows (X, T on the device) into
// m->grads; the loss partials are left in m->loss (mlp_loss_parts floats)
static int mlp_backward(fipc_mlp* m, hipStream_t s, int n, const float* X, const float* T)
{
    if (m->fused) return mlp_backward_fused(m, s, n, X, T);
    STCHK(mlp_forward(m, s, n, X, true));
    long ny = (long)n * m->n_out;
    float* dZ = m->dA.p;   // gradient at the current layer's pre-activation
    float* dH = m->dB.p;
    k_mse<<<nblk(ny), TPB, 0, s>>>(ny, 1.f / (float)ny, m->H[m->L].p, T, dZ, m->loss.p);
    HIPCHK(hipGetLastError());
    // split-K partials of dW and of the bias gradients: slices of at most 1024 rows
    int S = std::max(1, std::min(32, (n + 1023) / 1024));
    for (int l = m->L - 1; l >= 0; l--) {
        int fi = m->dim[l], fo = m->dim[l + 1];
        const float* Hin = l == 0 ? X : m->H[l].p;
        // dW_l = H_in^T dZ  (fi x fo), K = n rows
        STCHK(ensure(m->part, (size_t)S * fi * fo));
        STCHK(gemm(s, fi, fo, n, Hin, 1, fi, dZ, fo, 1, m->part.p, fo, EPI_NONE, nullptr, nullptr, nullptr, S,
                   (long)fi * fo));
        k_sum_slices<<<nblk((long)fi * fo), TPB, 0, s>>>((long)fi * fo, S, m->part.p, m->grads.p + m->woff[l]);
        // up to 1,024 rows are one slice, whose sums are the gradient (a launch to
        // sum one slice: 8 us of 97 with one hidden layer, 18 of 262 with eight)
        float* gb = m->grads.p + m->boff[l];
        k_colsum<<<dim3((fo + 63) / 64, S), 256, 0, s>>>(n, fo, (n + S - 1) / S, dZ, S == 1 ? gb : m->part.p);
        if (S > 1) k_sum_slices<<<nblk(fo), TPB, 0, s>>>(fo, S, m->part.p, gb);
        HIPCHK(hipGetLastError());
        if (l > 0) {
            // dZ_{l} = (dZ W_l^T) * silu'(Z_l)
            const float* W = m->params.p + m->woff[l];
            STCHK(gemm(s, n, fi, fo, dZ, fo, 1, W, 1, fo, dH, fi, EPI_DSILU, nullptr, m->Z[l].p, nullptr));
            std::swap(dZ, dH);
        }
    }
    return FIPC_OK;
}

int mlp_dims(const fipc_mlp* m, int* n_in, int* n_out)
{
    *n_in = m->n_in;
    *n_out = m->n_out;
    return FIPC_OK;
}
static int mlp_pack(fipc_mlp* m, hipStream_t s)
{
    if (m->wt_ok) return FIPC_OK;
    const long total = FI_WT + FI_WN;
    STCHK(ensure(m->wt, total));
    k_pack_weights<<<nblk(total), TPB, 0, s>>>(m->params.p, m->dboff.p, m->wt.p, total);
    HIPCHK(hipGetLastError());
    m->wt_ok = true;
    return FIPC_OK;
}
// forward of n rows of device X on stream s: the fused kernel for the
// warm-start shape, the layer-by-layer GEMMs otherwise
static int mlp_infer(fipc_mlp* m, hipStream_t s, int n, const float* X, const float** Y)
{
    if (!m->fused) {
        STCHK(mlp_forward(m, s, n, X, false));
        *Y = m->H[m->L].p;
        return FIPC_OK;
    }
    STCHK(mlp_pack(m, s));
    STCHK(ensure(m->H[m->L], (size_t)n * m->n_out));
    k_mlp_infer<<<(n + FI_ROWS - 1) / FI_ROWS, FI_THREADS, 0, s>>>(n, X, m->wt.p, m->params.p, m->dboff.p,
                                                                  m->H[m->L].p);
    HIPCHK(hipGetLastError());
    *Y = m->H[m->L].p;
    return FIPC_OK;
}
int mlp_forward_dev(fipc_mlp* m, hipStream_t s, int n, const float* X, const float** Y)
{
    return mlp_infer(m, s, n, X, Y);
}
int mlp_dataset_append_dev(fipc_mlp* m, hipStream_t s, int n, const float* X, const float* T)
{
    if (n <= 0) return FIPC_OK;
    long need = m->ds_n + n;
    if ((size_t)need * m->n_in > m->dsX.cap) {
        // grow, keeping the rows already captured
        DVec<float> nx, nt;
        STCHK(ensure(nx, (size_t)need * 2 * m->n_in));
        STCHK(ensure(nt, (size_t)need * 2 * m->n_out));
        if (m->ds_n) {
            HIPCHK(hipMemcpyAsync(nx.p, m->dsX.p, (size_t)m->ds_n * m->n_in * 4, hipMemcpyDeviceToDevice, s));
            HIPCHK(hipMemcpyAsync(nt.p, m->dsT.p, (size_t)m->ds_n * m->n_out * 4, hipMemcpyDeviceToDevice, s));
        }
        HIPCHK(hipStreamSynchronize(s));
        release(m->dsX);
        release(m->dsT);
        m->dsX = nx;
        m->dsT = nt;
    }
    HIPCHK(hipMemcpyAsync(m->dsX.p + m->ds_n * m->n_in, X, (size_t)n * m->n_in * 4, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(m->dsT.p + m->ds_n * m->n_out, T, (size_t)n * m->n_out * 4, hipMemcpyDeviceToDevice, s));
    m->ds_n = need;
    return FIPC_OK;
}
hipStream_t mlp_stream(fipc_mlp* m) { return m->s; }

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
extern "C" int fipc_mlp_create(fipc_mlp** out, int n_in, int width, int depth, int n_out, unsigned long long seed)
{
    if (!out || n_in <= 0 || width <= 0 || depth < 0 || n_out <= 0) return FIPC_ERR_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return FIPC_ERR_HIP;
    fipc_mlp* m = new fipc_mlp();
    m->n_in = n_in; m->width = width; m->depth = depth; m->n_out = n_out;
    m->L = depth + 1;
    m->dim.push_back(n_in);
    for (int i = 0; i < depth; i++) m->dim.push_back(width);
    m->dim.push_back(n_out);
    long off = 0;
    for (int l = 0; l < m->L; l++) {
        m->woff.push_back(off);
        off += (long)m->dim[l] * m->dim[l + 1];
        m->boff.push_back(off);
        off += m->dim[l + 1];
    }
    m->nparams = off;
    m->H.resize(m->L + 1);
    m->Z.resize(m->L + 1);
    if (hipStreamCreate(&m->s) != hipSuccess) { delete m; return FIPC_ERR_HIP; }
    int st = FIPC_OK;
    if (!st) st = ensure(m->params, off);
    if (!st) st = ensure(m->grads, off);
    if (!st) st = ensure(m->am, off);
    if (!st) st = ensure(m->av, off);
    if (st) { fipc_mlp_destroy(m); return st; }
    for (int l = 0; l < m->L; l++) {
        long nw = (long)m->dim[l] * m->dim[l + 1];
        // variance 1 / fan_in; the output layer starts 10x smaller so an
        // untrained network predicts almost no correction
        float a = sqrtf(3.f / (float)m->dim[l]) * (l == m->L - 1 ? 0.1f : 1.f);
        k_init_layer<<<nblk(std::max<long>(nw, m->dim[l + 1])), TPB, 0, m->s>>>(
            nw, m->dim[l + 1], m->params.p + m->woff[l], m->params.p + m->boff[l], a, seed + 7919ull * l);
    }
    if (hipGetLastError() != hipSuccess) { fipc_mlp_destroy(m); return FIPC_ERR_HIP; }
    m->fused = n_in == 16 && width == FI_W && depth == 4 && n_out == 3;
    if (m->fused) {
        if (ensure(m->dboff, m->L) != FIPC_OK) { fipc_mlp_destroy(m); return FIPC_ERR_HIP; }
        (void)hipMemcpyAsync(m->dboff.p, m->boff.data(), m->L * sizeof(long), hipMemcpyHostToDevice, m->s);
    }
    (void)hipMemsetAsync(m->am.p, 0, off * 4, m->s);
    (void)hipMemsetAsync(m->av.p, 0, off * 4, m->s);
    if (hipStreamSynchronize(m->s) != hipSuccess) { fipc_mlp_destroy(m); return FIPC_ERR_HIP; }
    *out = m;
    return FIPC_OK;
}

extern "C" int fipc_mlp_destroy(fipc_mlp* m)
{
    if (!m) return FIPC_OK;
    if (m->s) (void)hipStreamSynchronize(m->s);
    release(m->params); release(m->grads); release(m->am); release(m->av);
    for (auto& v : m->H) release(v);
    for (auto& v : m->Z) release(v);
    release(m->X); release(m->T); release(m->dA); release(m->dB); release(m->part); release(m->loss);
    release(m->dsX); release(m->dsT); release(m->wt); release(m->dboff);
    release(m->tA); release(m->tG); release(m->tbias);
    if (m->s) (void)hipStreamDestroy(m->s);
    delete m;
    return FIPC_OK;
}

extern "C" int fipc_mlp_nparams(fipc_mlp* m, long* n)
{
    if (!m || !n) return FIPC_ERR_ARG;
    *n = m->nparams;
    return FIPC_OK;
}
extern "C" int fipc_mlp_get_params(fipc_mlp* m, float* w)
{
    if (!m || !w) return FIPC_ERR_ARG;
    HIPCHK(hipMemcpyAsync(w, m->params.p, m->nparams * 4, hipMemcpyDeviceToHost, m->s));
    HIPCHK(hipStreamSynchronize(m->s));
    return FIPC_OK;
}
extern "C" int fipc_mlp_set_params(fipc_mlp* m, const float* w)
{
    if (!m || !w) return FIPC_ERR_ARG;
    HIPCHK(hipMemcpyAsync(m->params.p, w, m->nparams * 4, hipMemcpyHostToDevice, m->s));
    m->wt_ok = false;
    HIPCHK(hipMemsetAsync(m->am.p, 0, m->nparams * 4, m->s));
    HIPCHK(hipMemsetAsync(m->av.p, 0, m->nparams * 4, m->s));
    m->adam_t = 0;
    HIPCHK(hipStreamSynchronize(m->s));
    return FIPC_OK;
}

extern "C" int fipc_mlp_forward(fipc_mlp* m, int n, const float* X, float* Y)
{
    if (!m || n < 0 || (n && (!X || !Y))) return FIPC_ERR_ARG;
    if (!n) return FIPC_OK;
    STCHK(mlp_reserve(m, n, true));
    HIPCHK(hipMemcpyAsync(m->X.p, X, (size_t)n * m->n_in * 4, hipMemcpyHostToDevice, m->s));
    const float* Yd = nullptr;
    STCHK(mlp_infer(m, m->s, n, m->X.p, &Yd));
    HIPCHK(hipMemcpyAsync(Y, Yd, (size_t)n * m->n_out * 4, hipMemcpyDeviceToHost, m->s));
    HIPCHK(hipStreamSynchronize(m->s));
    return FIPC_OK;
}

extern "C" int fipc_mlp_grad(fipc_mlp* m, int n, const float* X, const float* T, float* loss, float* grad)
{
    if (!m || n <= 0 || !X || !T) return FIPC_ERR_ARG;
    STCHK(mlp_reserve(m, n, true));
    HIPCHK(hipMemcpyAsync(m->X.p, X, (size_t)n * m->n_in * 4, hipMemcpyHostToDevice, m->s));
    HIPCHK(hipMemcpyAsync(m->T.p, T, (size_t)n * m->n_out * 4, hipMemcpyHostToDevice, m->s));
    STCHK(mlp_backward(m, m->s, n, m->X.p, m->T.p));
    int nb = mlp_loss_parts(m, n);
    std::vector<float> lp(nb);
    HIPCHK(hipMemcpyAsync(lp.data(), m->loss.p, nb * 4, hipMemcpyDeviceToHost, m->s));
    if (grad) HIPCHK(hipMemcpyAsync(grad, m->grads.p, m->nparams * 4, hipMemcpyDeviceToHost, m->s));
    HIPCHK(hipStreamSynchronize(m->s));
    double l = 0.0;
    for (float v : lp) l += v;
    if (loss) *loss = (float)l;
    return FIPC_OK;
}

extern "C" int fipc_mlp_dataset_clear(fipc_mlp* m)
{
    if (!m) return FIPC_ERR_ARG;
    m->ds_n = 0;
    return FIPC_OK;
}
extern "C" int fipc_mlp_dataset_size(fipc_mlp* m, long* n)
{
    if (!m || !n) return FIPC_ERR_ARG;
    *n = m->ds_n;
    return FIPC_OK;
}
extern "C" int fipc_mlp_dataset_add(fipc_mlp* m, int n, const float* X, const float* T)
{
    if (!m || n < 0 || (n && (!X || !T))) return FIPC_ERR_ARG;
    if (!n) return FIPC_OK;
    DVec<float> dx, dt;
    STCHK(ensure(dx, (size_t)n * m->n_in));
    STCHK(ensure(dt, (size_t)n * m->n_out));
    HIPCHK(hipMemcpyAsync(dx.p, X, (size_t)n * m->n_in * 4, hipMemcpyHostToDevice, m->s));
    HIPCHK(hipMemcpyAsync(dt.p, T, (size_t)n * m->n_out * 4, hipMemcpyHostToDevice, m->s));
    int st = mlp_dataset_append_dev(m, m->s, n, dx.p, dt.p);
    (void)hipStreamSynchronize(m->s);
    release(dx);
    release(dt);
    return st;
}
extern "C" int fipc_mlp_dataset_get(fipc_mlp* m, long first, long n, float* X, float* T)
{
    if (!m || first < 0 || n < 0 || first + n > m->ds_n) return FIPC_ERR_ARG;
    if (!n) return FIPC_OK;
    if (X) HIPCHK(hipMemcpyAsync(X, m->dsX.p + first * m->n_in, (size_t)n * m->n_in * 4, hipMemcpyDeviceToHost, m->s));
    if (T) HIPCHK(hipMemcpyAsync(T, m->dsT.p + first * m->n_out, (size_t)n * m->n_out * 4, hipMemcpyDeviceToHost, m->s));
    HIPCHK(hipStreamSynchronize(m->s));
    return FIPC_OK;
}

// iters Adam steps (beta1 0.9, beta2 0.999, eps 1e-8) on batches drawn from
// the dataset; losses[i] = mean squared error of batch i before its update
extern "C" int fipc_mlp_train(fipc_mlp* m, int iters, int batch, float lr, unsigned long long seed, float* losses)
{
    if (!m || iters < 0 || batch <= 0 || m->ds_n == 0) return FIPC_ERR_ARG;
    STCHK(mlp_reserve(m, batch, true));
    int nb = mlp_loss_parts(m, batch);
    DVec<float> lossall;
    STCHK(ensure(lossall, (size_t)iters * nb + 1));
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int it = 0; it < iters; it++) {
        k_gather_batch<<<nblk(batch), TPB, 0, m->s>>>(batch, m->ds_n, seed + 1000003ull * (unsigned long long)it,
                                                      m->n_in, m->n_out, m->dsX.p, m->dsT.p, m->X.p, m->T.p);
        HIPCHK(hipGetLastError());
        STCHK(mlp_backward(m, m->s, batch, m->X.p, m->T.p));
        HIPCHK(hipMemcpyAsync(lossall.p + (size_t)it * nb, m->loss.p, nb * 4, hipMemcpyDeviceToDevice, m->s));
        m->adam_t++;
        float c1 = 1.f - powf(b1, (float)m->adam_t), c2 = 1.f - powf(b2, (float)m->adam_t);
        k_adam<<<nblk(m->nparams), TPB, 0, m->s>>>(m->nparams, m->params.p, m->grads.p, m->am.p, m->av.p, lr, b1, b2,
                                                    eps, c1, c2);
        m->wt_ok = false;
        HIPCHK(hipGetLastError());
    }
    std::vector<float> lp((size_t)iters * nb);
    if (iters) HIPCHK(hipMemcpyAsync(lp.data(), lossall.p, lp.size() * 4, hipMemcpyDeviceToHost, m->s));
    HIPCHK(hipStreamSynchronize(m->s));
    release(lossall);
    if (losses)
        for (int it = 0; it < iters; it++) {
            double l = 0.0;
            for (int b = 0; b < nb; b++) l += lp[(size_t)it * nb + b];
            losses[it] = (float)l;
        }
    return FIPC_OK;
}
