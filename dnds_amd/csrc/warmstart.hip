// Learned warm start of the VR reconstruction (gfx950).  No counterpart in
// the reference: a small MLP maps a cell's stencil of cell means and its
// geometry moments to an initial guess of its 9 x 4 rec coefficients; plain
// Jacobi sweeps then iterate to the same tolerance, so the method decides the
// result and remains the fallback.
//
// Network (58 -> 128 -> 128 -> 36, GELU): inputs are the mean differences
// u_j - u_i of 12 stencil cells (per variable divided by s_v, the largest of
// them but at least 1e-3 max_v |u_i,v|), the 9 base moments of the cell and
// 0.5 log(volume); outputs are the
// rec coefficients divided by s_v (the reconstruction is linear in the means,
// so this scaling makes the map scale-free).  The stencil is the first 12
// cells met by a breadth-first walk over faces (cell2face order); missing
// cells repeat the cell itself.
//
// Training and inference use hand-written kernels on gfx950's matrix cores
// (v_mfma_f32_16x16x32_bf16: BF16 operands, FP32 accumulation), FP32
// otherwise.  A training step is three launches: the rows' forward and
// backward pass, the weight and bias gradients' partial sums over the rows,
// and their sums with Adam.  Inference is one fused kernel that keeps the
// three layers' BF16 weights in LDS and the hidden activations on chip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>
#include <vector>

#include "ctx.hpp"

using namespace dndsmi_dev;
using namespace dndsmi_host;

namespace {

constexpr int kIn = 58, kHid = 128, kOut = 36, kSten = 12;
// parameter block: W1 [58][128], b1 [128], W2 [128][128], b2 [128], W3 [128][36], b3 [36]
constexpr int64_t oW1 = 0, ob1 = oW1 + kIn * kHid, oW2 = ob1 + kHid, ob2 = oW2 + kHid * kHid, oW3 = ob2 + kHid,
                  ob3 = oW3 + kHid * kOut, kNParam = ob3 + kOut;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (finite inputs)
__device__ inline unsigned short to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

__device__ __forceinline__ floatx4 mfma(bf16x8 a, bf16x8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Operand layout of v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][k] and
// B[k][l % 16] for the eight k = 8 (l / 16) + 0..7 (a product is the same
// under any assignment of k that A and B share); it receives
// D[4 (l / 16) + 0..3][l % 16].
//
// The weight matrices as training's B operands in BF16: fragment f of wave w
// (columns 16 w .. 16 w + 15) is 64 lanes x 8 values; zeros where the matrix
// ends.  Fragments 0-1 are W1's K steps, 2-5 W2's, 6-9 W3's, 10-11 those of
// W3's transpose, 12-15 those of W2's.  The parameters' update writes them with
// the parameters: rounded by every workgroup of the rows' pass from strided
// loads, they were 9 of its 23 us at 4096 rows.
constexpr int kRowWaves = 8, kFragments = 16, kPacked = kFragments * kRowWaves * 64 * 8;
__device__ __forceinline__ int packed_at(int f, int k, int n) {
    return (((f + k / 32) * kRowWaves + n / 16) * 64 + 16 * (k % 32 / 8) + n % 16) * 8 + k % 8;
}
__device__ __forceinline__ void pack_parameter(int i, float p, unsigned short *__restrict__ packed) {
    const unsigned short h = to_bf16(p);
    if (i < ob1) {
        packed[packed_at(0, i / kHid, i % kHid)] = h;
    } else if (i >= oW2 && i < ob2) {
        const int a = (i - oW2) / kHid, b = (i - oW2) % kHid;
        packed[packed_at(2, a, b)] = packed[packed_at(12, b, a)] = h;
    } else if (i >= oW3 && i < ob3) {
        const int a = (i - oW3) / kOut, b = (i - oW3) % kOut;
        packed[packed_at(6, a, b)] = packed[packed_at(10, b, a)] = h;
    }
}
__global__ __launch_bounds__(256) void k_pack(const float *__restrict__ P, unsigned short *__restrict__ packed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kNParam)
        pack_parameter(i, P[i], packed);
}

// The operands of the weight gradients, BF16, transposed: column c's rows
// contiguous, [column][ld] with ld a multiple of 32 and zeros from the batch's
// last row on, so that a lane's eight k (rows) are one 16-byte load.
struct TrainCols {
    int64_t ld;
    unsigned short *X, *H1, *H2, *dY, *dZ2, *dZ1; // 64, 128, 128, 64, 128, 128 columns
};
constexpr int kColsX = 0, kColsH1 = 64, kColsH2 = 192, kColsdY = 320, kColsdZ2 = 384, kColsdZ1 = 512, kColsAll = 640;

constexpr int kInPad = 64, kOutPad = 48, kLdX = kInPad + 8, kLdH = kHid + 8;

// Forward and backward pass of the batch, 16 rows per workgroup and turn: row
// r is row idx[r] (r without idx) of X and T.  Wave w owns columns 16 w .. 16
// w + 15 of the hidden layers (waves 0 .. 2 the outputs) and holds its columns
// of the three weight matrices and of the two transposed ones as BF16 operands
// in registers for all its turns; a layer's output goes through LDS to the
// next, z1 and z2 stay in registers for the GELU's derivative.  Out come the
// weight gradients' operands (TrainCols) and the FP32 columns the bias
// gradients sum; Y where the loss is asked for (else null).
//
// The chain of six small products is bound by latency (LDS, barriers, the
// GELUs); five separate products through memory took 18 + 20 + 18 + 16 + 16
// us at 4096 rows besides two gathers and the loss gradient.
__global__ __launch_bounds__(64 * kRowWaves) void k_train_rows(int32_t rows, const int32_t *__restrict__ idx,
                                                               const float *__restrict__ X,
                                                               const float *__restrict__ T,
                                                               const float *__restrict__ P,
                                                               const unsigned short *__restrict__ packed, float scale,
                                                               TrainCols tc,
                                                               float *__restrict__ Y, float *__restrict__ dY,
                                                               float *__restrict__ dZ2, float *__restrict__ dZ1) {
    __shared__ __attribute__((aligned(16))) unsigned short Xs[16][kLdX], Ds[16][kLdX];
    __shared__ __attribute__((aligned(16))) unsigned short H1s[16][kLdH], H2s[16][kLdH], Gs[16][kLdH];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, lr = lane % 16, lg = lane / 16;
    const int n = 16 * wave + lr;
    bf16x8 w1[2], w2[4], w3[4], w3t[2], w2t[4];
    auto weights = [&](int f) {
        return __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const shortx8 *>(packed + ((f * kRowWaves + wave) * 64 + lane) * 8));
    };
#pragma unroll
    for (int s = 0; s < 2; s++)
        w1[s] = weights(s), w3t[s] = weights(10 + s);
#pragma unroll
    for (int s = 0; s < 4; s++)
        w2[s] = weights(2 + s), w3[s] = weights(6 + s), w2t[s] = weights(12 + s);
    const float bias1 = P[ob1 + n], bias2 = P[ob2 + n], bias3 = n < kOut ? P[ob3 + n] : 0.f;
    const floatx4 zero = floatx4{0.f, 0.f, 0.f, 0.f};
    const int64_t ntile = tc.ld / 16;
    for (int64_t tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        const int64_t r0 = 16 * tile, rl = r0 + 4 * lg; // the lane's four rows of every result
        // a fragment of the tile's K step s, and a column's four rows to memory
        auto frag = [&](const auto &S, int s) {
            return __builtin_bit_cast(bf16x8, *reinterpret_cast<const shortx8 *>(&S[lr][32 * s + 8 * lg]));
        };
        auto to_cols = [&](unsigned short *cols, int c, const unsigned short v[4]) {
            *reinterpret_cast<ushort4 *>(cols + c * tc.ld + rl) = make_ushort4(v[0], v[1], v[2], v[3]);
        };
        float t[4] = {0.f, 0.f, 0.f, 0.f};
        if (n < kOut)
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (rl + j < rows)
                    t[j] = T[(idx ? idx[rl + j] : rl + j) * int64_t(kOut) + n];
#pragma unroll
        for (int q = 0; q < 16 * kInPad / (64 * kRowWaves); q++) {
            const int e = tid + 64 * kRowWaves * q, r = e / kInPad, k = e % kInPad;
            float v = 0.f;
            if (r0 + r < rows && k < kIn)
                v = X[(idx ? idx[r0 + r] : r0 + r) * int64_t(kIn) + k];
            Xs[r][k] = to_bf16(v);
        }
        __syncthreads();
        if (wave < kInPad / 16) {
            unsigned short o[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
                o[j] = Xs[4 * lg + j][n];
            to_cols(tc.X, n, o);
        }
        floatx4 z1 = zero, z2 = zero, acc = zero;
#pragma unroll
        for (int s = 0; s < 2; s++)
            z1 = mfma(frag(Xs, s), w1[s], z1);
        unsigned short o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            z1[j] = z1[j] + bias1;
            H1s[4 * lg + j][n] = to_bf16(gelu(z1[j]));
            o[j] = rl + j < rows ? H1s[4 * lg + j][n] : (unsigned short)(0);
        }
        to_cols(tc.H1, n, o);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; s++)
            z2 = mfma(frag(H1s, s), w2[s], z2);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            z2[j] = z2[j] + bias2;
            H2s[4 * lg + j][n] = to_bf16(gelu(z2[j]));
            o[j] = rl + j < rows ? H2s[4 * lg + j][n] : (unsigned short)(0);
        }
        to_cols(tc.H2, n, o);
        __syncthreads();
        // outputs, and the loss's gradient 2 (Y - T) / (rows 36)
        if (wave < kInPad / 16) {
            if (wave < kOutPad / 16)
#pragma unroll
                for (int s = 0; s < 4; s++)
                    acc = mfma(frag(H2s, s), w3[s], acc);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float y = acc[j] + bias3;
                float d = 0.f;
                if (n < kOut && rl + j < rows) {
                    d = scale * (y - t[j]);
                    dY[(rl + j) * kOut + n] = d;
                    if (Y)
                        Y[(rl + j) * kOut + n] = y;
                }
                Ds[4 * lg + j][n] = o[j] = to_bf16(d);
            }
            to_cols(tc.dY, n, o);
        }
        __syncthreads();
        acc = zero;
#pragma unroll
        for (int s = 0; s < 2; s++)
            acc = mfma(frag(Ds, s), w3t[s], acc);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float d = rl + j < rows ? acc[j] * gelu_grad(z2[j]) : 0.f;
            if (rl + j < rows)
                dZ2[(rl + j) * kHid + n] = d;
            Gs[4 * lg + j][n] = o[j] = to_bf16(d);
        }
        to_cols(tc.dZ2, n, o);
        __syncthreads();
        acc = zero;
#pragma unroll
        for (int s = 0; s < 4; s++)
            acc = mfma(frag(Gs, s), w2t[s], acc);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float d = rl + j < rows ? acc[j] * gelu_grad(z1[j]) : 0.f;
            if (rl + j < rows)
                dZ1[(rl + j) * kHid + n] = d;
            o[j] = to_bf16(d);
        }
        to_cols(tc.dZ1, n, o);
    }
}

// Partial weight and bias gradients over chunks of the rows.
//
// Workgroups of one wave: the first nz * kWTiles take a 32 x 32 tile of one
// weight matrix's A^T B (A the layer's input, B its output's gradient) over
// rows [z kchunk, (z + 1) kchunk), 2 x 2 MFMA blocks, K in steps of 32, into
// part[z] laid out like the parameters; eight steps' operands (16 bytes a
// lane) are in flight at a time, for the wave waits for nothing else.  The
// others sum 64 columns over one chunk of rows in order, into bpart[chunk].
// (Products of 64 x 64 tiles with operands rounded on the way into LDS, one
// step's at a time, took 40 us each at 4096 rows, the column sums 13.)
constexpr int kWTiles = 8 + 16 + 8, kBias = 2 * kHid + kOut, kBiasBlocks = 5;

__global__ __launch_bounds__(64) void k_train_grads(int32_t rows, int32_t nz, int32_t kchunk, int32_t bchunk,
                                                    TrainCols tc, const float *__restrict__ dY,
                                                    const float *__restrict__ dZ2, const float *__restrict__ dZ1,
                                                    float *__restrict__ part, float *__restrict__ bpart) {
    const int lane = threadIdx.x, lr = lane % 16, lg = lane / 16;
    const int32_t blk = blockIdx.x;
    if (blk >= nz * kWTiles) {
        const int32_t z = (blk - nz * kWTiles) / kBiasBlocks, q = (blk - nz * kWTiles) % kBiasBlocks;
        const int w = q < 4 ? kHid : kOut, c = q < 4 ? 64 * (q % 2) + lane : lane;
        if (c >= w)
            return;
        const float *src = (q < 2 ? dZ1 : q < 4 ? dZ2 : dY) + c;
        const int32_t r0 = z * bchunk, r1 = min(rows, r0 + bchunk);
        float sum = 0.f;
        int32_t r = r0;
        for (; r + 32 <= r1; r += 32) {
            float v[32];
#pragma unroll
            for (int e = 0; e < 32; e++)
                v[e] = src[int64_t(r + e) * w];
#pragma unroll
            for (int e = 0; e < 32; e++)
                sum += v[e];
        }
        for (; r < r1; r++)
            sum += src[int64_t(r) * w];
        bpart[int64_t(z) * kBias + (q < 2 ? 0 : q < 4 ? kHid : 2 * kHid) + c] = sum;
        return;
    }
    const int32_t z = blk / kWTiles, t = blk % kWTiles;
    // W2: 4 x 4 tiles, W1: 2 x 4 (58 of 64 rows), W3: 4 x 2 (36 of 64 columns)
    const unsigned short *A, *B;
    int M, N, m0, n0;
    int64_t o;
    if (t < 16)
        A = tc.H1, B = tc.dZ2, M = kHid, N = kHid, m0 = 32 * (t / 4), n0 = 32 * (t % 4), o = oW2;
    else if (t < 24)
        A = tc.X, B = tc.dZ1, M = kIn, N = kHid, m0 = 32 * ((t - 16) / 4), n0 = 32 * (t % 4), o = oW1;
    else
        A = tc.H2, B = tc.dY, M = kHid, N = kOut, m0 = 32 * ((t - 24) / 2), n0 = 32 * (t % 2), o = oW3;
    const int32_t kbeg = z * kchunk, kend = min(rows, kbeg + kchunk);
    floatx4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
            acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    constexpr int kSteps = 8;
    for (int32_t k0 = kbeg; k0 < kend; k0 += 32 * kSteps) {
        shortx8 fa[kSteps][2], fb[kSteps][2];
#pragma unroll
        for (int s = 0; s < kSteps; s++)
#pragma unroll
            for (int a = 0; a < 2; a++) {
                const int64_t k = k0 + 32 * s + 8 * lg;
                fa[s][a] = fb[s][a] = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
                if (k < kend) {
                    fa[s][a] = *reinterpret_cast<const shortx8 *>(A + (m0 + 16 * a + lr) * tc.ld + k);
                    fb[s][a] = *reinterpret_cast<const shortx8 *>(B + (n0 + 16 * a + lr) * tc.ld + k);
                }
            }
#pragma unroll
        for (int s = 0; s < kSteps; s++)
            if (k0 + 32 * s < kend)
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 2; b++)
                        acc[a][b] = mfma(__builtin_bit_cast(bf16x8, fa[s][a]), __builtin_bit_cast(bf16x8, fb[s][b]),
                                         acc[a][b]);
    }
    float *C = part + int64_t(z) * kNParam + o;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int m = m0 + 16 * a + 4 * lg + j, n = n0 + 16 * b + lr;
                if (m < M && n < N)
                    C[m * N + n] = acc[a][b][j];
            }
}

// Adam (Kingma & Ba 2015) with bias correction folded into the step size
struct AdamStep {
    float lr_t, b1, b2, eps_t;
};
__device__ __forceinline__ void adam_update(int64_t i, float g, const AdamStep &a, float *__restrict__ P,
                                            float *__restrict__ Mm, float *__restrict__ Vv) {
    const float m = a.b1 * Mm[i] + (1.f - a.b1) * g;
    const float v = a.b2 * Vv[i] + (1.f - a.b2) * g * g;
    Mm[i] = m, Vv[i] = v;
    P[i] -= a.lr_t * m / (sqrtf(v) + a.eps_t);
}

// Gradient of every parameter, its partial sums added in order; into G, or
// (without G) straight into Adam's step
__global__ __launch_bounds__(256) void k_train_update(int32_t nz, int32_t nb, const float *__restrict__ part,
                                                      const float *__restrict__ bpart, float *__restrict__ G,
                                                      AdamStep a, float *__restrict__ P, float *__restrict__ Mm,
                                                      float *__restrict__ Vv, unsigned short *__restrict__ packed) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= kNParam)
        return;
    const float *src = part + i;
    int64_t ld = kNParam;
    int32_t cnt = nz;
    const bool b1 = i >= ob1 && i < oW2, b2 = i >= ob2 && i < oW3, b3 = i >= ob3;
    if (b1 || b2 || b3)
        src = bpart + (b1 ? i - ob1 : b2 ? kHid + i - ob2 : 2 * kHid + i - ob3), ld = kBias, cnt = nb;
    float acc = 0.f;
    int32_t z = 0;
    for (; z + 16 <= cnt; z += 16) {
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; e++)
            v[e] = src[(z + e) * ld];
#pragma unroll
        for (int e = 0; e < 16; e++)
            acc += v[e];
    }
    for (; z < cnt; z++)
        acc += src[z * ld];
    if (G) {
        G[i] = acc;
    } else {
        adam_update(i, acc, a, P, Mm, Vv);
        pack_parameter(int(i), P[i], packed);
    }
}

__global__ __launch_bounds__(256) void k_adam(int64_t n, float *__restrict__ P, const float *__restrict__ G,
                                              float *__restrict__ Mm, float *__restrict__ Vv, AdamStep a) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        adam_update(i, G[i], a, P, Mm, Vv);
}

// Inference of the whole network, Y = W3^T g(W2^T g(W1^T x + b1) + b2) + b3
// per row (g = GELU), in one kernel.  Each workgroup (8 waves) stages the
// three weight matrices once, transposed to [n][k] and rounded to BF16, in
// LDS (about 66 KB), then walks its rows 16 at a time per wave: layer 1 reads
// the row's features from memory, every hidden layer's output (bias and GELU
// applied in FP32, then rounded to BF16, as the operand of the next GEMM
// would be) goes through the wave's own 16 x 128 LDS tile, and only the 36
// outputs reach memory.  The arithmetic is that of training's forward pass
// (BF16 operands, FP32 accumulation, FP32 epilogues).
constexpr int kLdW1 = kInPad + 8, kInferWaves = 16;

__global__ __launch_bounds__(64 * kInferWaves) void k_mlp_infer(int32_t rows, const float *__restrict__ X,
                                                                  const float *__restrict__ P,
                                                                  float *__restrict__ Y) {
    __shared__ __attribute__((aligned(16))) unsigned short W1t[kHid][kLdW1];
    __shared__ __attribute__((aligned(16))) unsigned short W2t[kHid][kLdH];
    __shared__ __attribute__((aligned(16))) unsigned short W3t[kOutPad][kLdH];
    __shared__ float bs[2 * kHid + kOutPad];
    __shared__ __attribute__((aligned(16))) unsigned short H[kInferWaves][16][kLdH];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    for (int e = tid; e < kHid * kInPad; e += 64 * kInferWaves) {
        const int n = e % kHid, k = e / kHid; // consecutive threads: consecutive n of one row of W1
        W1t[n][k] = to_bf16(k < kIn ? P[oW1 + k * kHid + n] : 0.f);
    }
    for (int e = tid; e < kHid * kHid; e += 64 * kInferWaves) {
        const int n = e % kHid, k = e / kHid;
        W2t[n][k] = to_bf16(P[oW2 + k * kHid + n]);
    }
    for (int e = tid; e < kOutPad * kHid; e += 64 * kInferWaves) {
        const int n = e % kOutPad, k = e / kOutPad;
        W3t[n][k] = to_bf16(n < kOut ? P[oW3 + k * kOut + n] : 0.f);
    }
    for (int e = tid; e < 2 * kHid + kOutPad; e += 64 * kInferWaves)
        bs[e] = e < kHid ? P[ob1 + e] : (e < 2 * kHid ? P[ob2 + e - kHid] : (e - 2 * kHid < kOut ? P[ob3 + e - 2 * kHid] : 0.f));
    __syncthreads();
    const int kb = 8 * (lane / 16), lr = lane % 16;
    const int64_t ntile = (int64_t(rows) + 15) / 16;
    // the loop bound depends on the workgroup only, so every wave reaches
    // every __syncthreads (a wave past the last tile computes on zeros and
    // stores nothing)
    float xc[kInPad / 32][8];
    {
        const int64_t row = (int64_t(blockIdx.x) * kInferWaves + wave) * 16 + lr;
#pragma unroll
        for (int s2 = 0; s2 < kInPad / 32; s2++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int k = 32 * s2 + kb + e;
                xc[s2][e] = row < rows && k < kIn ? X[row * kIn + k] : 0.f;
            }
    }
    for (int64_t t0 = int64_t(blockIdx.x) * kInferWaves; t0 < ntile; t0 += int64_t(gridDim.x) * kInferWaves) {
        const int64_t r0 = (t0 + wave) * 16;
        // layer 1: A operand straight from the features (58 per row, zero
        // padded); the next tile's features are loaded while this one runs
        floatx4 acc[8];
#pragma unroll
        for (int b = 0; b < 8; b++)
            acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
        float xn[kInPad / 32][8];
        {
            const int64_t nrow = r0 + int64_t(gridDim.x) * kInferWaves * 16 + lr;
#pragma unroll
            for (int s2 = 0; s2 < kInPad / 32; s2++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int k = 32 * s2 + kb + e;
                    xn[s2][e] = nrow < rows && k < kIn ? X[nrow * kIn + k] : 0.f;
                }
        }
#pragma unroll
        for (int s2 = 0; s2 < kInPad / 32; s2++) {
            shortx8 av;
#pragma unroll
            for (int e = 0; e < 8; e++)
                av[e] = short(to_bf16(xc[s2][e]));
            const bf16x8 a = __builtin_bit_cast(bf16x8, av);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, *reinterpret_cast<const shortx8 *>(&W1t[16 * b + lr][32 * s2 + kb]));
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w, acc[b], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < 8; b++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                H[wave][4 * (lane / 16) + j][16 * b + lr] = to_bf16(gelu(acc[b][j] + bs[16 * b + lr]));
        __syncthreads();
        // layer 2
#pragma unroll
        for (int b = 0; b < 8; b++)
            acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s2 = 0; s2 < kHid / 32; s2++) {
            const bf16x8 a = __builtin_bit_cast(bf16x8, *reinterpret_cast<const shortx8 *>(&H[wave][lr][32 * s2 + kb]));
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, *reinterpret_cast<const shortx8 *>(&W2t[16 * b + lr][32 * s2 + kb]));
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w, acc[b], 0, 0, 0);
            }
        }
        __syncthreads(); // every wave has read its layer-1 tile
#pragma unroll
        for (int b = 0; b < 8; b++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                H[wave][4 * (lane / 16) + j][16 * b + lr] = to_bf16(gelu(acc[b][j] + bs[kHid + 16 * b + lr]));
        __syncthreads();
        // layer 3
        floatx4 out[3];
#pragma unroll
        for (int b = 0; b < 3; b++)
            out[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s2 = 0; s2 < kHid / 32; s2++) {
            const bf16x8 a = __builtin_bit_cast(bf16x8, *reinterpret_cast<const shortx8 *>(&H[wave][lr][32 * s2 + kb]));
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const bf16x8 w = __builtin_bit_cast(bf16x8, *reinterpret_cast<const shortx8 *>(&W3t[16 * b + lr][32 * s2 + kb]));
                out[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w, out[b], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int64_t m = r0 + 4 * (lane / 16) + j;
                const int n = 16 * b + lr;
                if (m < rows && n < kOut)
                    Y[m * kOut + n] = out[b][j] + bs[2 * kHid + n];
            }
        __syncthreads(); // the tile is free for the next rows
#pragma unroll
        for (int s2 = 0; s2 < kInPad / 32; s2++)
#pragma unroll
            for (int e = 0; e < 8; e++)
                xc[s2][e] = xn[s2][e];
    }
}

// MSE loss: per-block sums of (Y - T)^2 over the n = rows * 36 outputs
__global__ __launch_bounds__(256) void k_mse(int64_t n, const int32_t *__restrict__ idx, const float *__restrict__ Y,
                                             const float *__restrict__ T, float *__restrict__ part) {
    __shared__ float red[256];
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    float e = 0.f;
    if (i < n) {
        const float d = Y[i] - T[idx ? idx[i / kOut] * int64_t(kOut) + i % kOut : i];
        e = d * d;
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        part[blockIdx.x] = red[0];
}

// features and scales of cell i: the row goes to `row` (58 floats), the
// scales to S
__device__ inline void features_row(int32_t i, int64_t ldc, const int32_t *__restrict__ sten,
                                    const double *__restrict__ u, const float *__restrict__ mom,
                                    const float *__restrict__ logsz, float *row, float *__restrict__ S) {
    double ui[4], d[kSten][4];
#pragma unroll
    for (int v = 0; v < 4; v++)
        ui[v] = u[4 * int64_t(i) + v];
    double s[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < kSten; k++) {
        const int32_t j = sten[k * ldc + i];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            d[k][v] = u[4 * int64_t(j) + v] - ui[v];
            s[v] = fmax(s[v], fabs(d[k][v]));
        }
    }
    // floor: a thousandth of the cell's largest |u_v|, so that nearly uniform
    // stencils (whose coefficients are set by distant cells) stay bounded
    double umax = 0;
#pragma unroll
    for (int v = 0; v < 4; v++)
        umax = fmax(umax, fabs(ui[v]));
#pragma unroll
    for (int v = 0; v < 4; v++) {
        s[v] = fmax(s[v], 1e-3 * umax);
        s[v] = s[v] > 0 ? s[v] : 1.0;
    }
#pragma unroll
    for (int k = 0; k < kSten; k++)
#pragma unroll
        for (int v = 0; v < 4; v++)
            row[4 * k + v] = float(d[k][v] / s[v]);
#pragma unroll
    for (int k = 0; k < 9; k++)
        row[48 + k] = mom[k * ldc + i];
    row[57] = logsz[i];
#pragma unroll
    for (int v = 0; v < 4; v++)
        S[4 * int64_t(i) + v] = float(s[v]);
}

// features and scales of every cell (see the file comment).  The block's
// rows are formed in LDS and written out as one contiguous run: a row is 58
// floats, so stores of whole rows by single threads would not coalesce.
__global__ __launch_bounds__(256) void k_features(int32_t nc, int64_t ldc, const int32_t *__restrict__ sten,
                                                  const double *__restrict__ u, const float *__restrict__ mom,
                                                  const float *__restrict__ logsz, float *__restrict__ X,
                                                  float *__restrict__ S) {
    __shared__ float tile[256][kIn + 1];
    const int64_t i0 = int64_t(blockIdx.x) * 256;
    const int32_t i = int32_t(i0) + int32_t(threadIdx.x);
    if (i < nc)
        features_row(i, ldc, sten, u, mom, logsz, tile[threadIdx.x], S);
    __syncthreads();
    const int64_t nrow = min(int64_t(256), int64_t(nc) - i0);
    for (int64_t e = threadIdx.x; e < nrow * kIn; e += 256)
        X[i0 * kIn + e] = tile[e / kIn][e % kIn];
}

// targets: converged rec coefficients x (k = r + 9 v) divided by
// s_v, rows of 36 formed in LDS and written contiguously; x is read, and in
// k_unscale written, in whole 32-byte elements (predict on 1 M cells, value by
// value -> now: 589 -> 574 us)
__global__ __launch_bounds__(256) void k_targets(int32_t nc, int64_t ldc, const double *__restrict__ x,
                                                 const float *__restrict__ S, float *__restrict__ T) {
    __shared__ float tile[256][kOut + 1];
    const int64_t i0 = int64_t(blockIdx.x) * 256;
    const int32_t i = int32_t(i0) + int32_t(threadIdx.x);
    if (i < nc) {
        const floatx4 sv = reinterpret_cast<const floatx4 *>(S)[i];
#pragma unroll
        for (int r = 0; r < 9; r++) {
            const dbl2 *xq = reinterpret_cast<const dbl2 *>(x + rec(i, r, 0));
            const dbl2 a = xq[0], b = xq[1];
            const double e[4] = {a.x, a.y, b.x, b.y};
#pragma unroll
            for (int v = 0; v < 4; v++)
                tile[threadIdx.x][r + 9 * v] = float(e[v] / double(sv[v]));
        }
    }
    __syncthreads();
    const int64_t nrow = min(int64_t(256), int64_t(nc) - i0);
    for (int64_t e = threadIdx.x; e < nrow * kOut; e += 256)
        T[i0 * kOut + e] = tile[e / kOut][e % kOut];
}

// prediction back to rec coefficients, x = Y s_v (ADD: x += Y s_v, the stage
// correction of the learned warm start inside the mixed-precision step).
// The block's rows of Y are read contiguously into LDS first.
template <bool ADD>
__global__ __launch_bounds__(256) void k_unscale(int32_t nc, int64_t ldc, const float *__restrict__ Y,
                                                 const float *__restrict__ S, double *__restrict__ x) {
    __shared__ float tile[256][kOut + 1];
    const int64_t i0 = int64_t(blockIdx.x) * 256;
    const int64_t nrow = min(int64_t(256), int64_t(nc) - i0);
    for (int64_t e = threadIdx.x; e < nrow * kOut; e += 256)
        tile[e / kOut][e % kOut] = Y[i0 * kOut + e];
    __syncthreads();
    const int32_t i = int32_t(i0) + int32_t(threadIdx.x);
    if (i >= nc)
        return;
    const floatx4 sv = reinterpret_cast<const floatx4 *>(S)[i];
#pragma unroll
    for (int r = 0; r < 9; r++) {
        dbl2 *xq = reinterpret_cast<dbl2 *>(x + rec(i, r, 0));
        double e[4];
#pragma unroll
        for (int v = 0; v < 4; v++)
            e[v] = double(tile[threadIdx.x][r + 9 * v]) * double(sv[v]);
        if (ADD) {
            const dbl2 a = xq[0], b = xq[1];
            e[0] = a.x + e[0], e[1] = a.y + e[1], e[2] = b.x + e[2], e[3] = b.y + e[3];
        }
        xq[0] = dbl2{e[0], e[1]}, xq[1] = dbl2{e[2], e[3]};
    }
}

// du = u - u_prev, then u_prev = u (cell means, [cell][4])
__global__ __launch_bounds__(256) void k_mean_change(int32_t nc, const double *__restrict__ u,
                                                     double *__restrict__ uprev, double *__restrict__ du) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4 * nc)
        return;
    const double v = u[i];
    du[i] = v - uprev[i];
    uprev[i] = v;
}

// per block: sum of (a - b)^2 and of b^2 over n doubles (the corrected state
// against the plain one at the end of a check window)
__global__ __launch_bounds__(256) void k_diff2(int64_t n, const double *__restrict__ a, const double *__restrict__ b,
                                               double *__restrict__ part) {
    __shared__ double red[2][256];
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    double d2 = 0.0, b2 = 0.0;
    if (i < n) {
        const double d = a[i] - b[i];
        d2 = d * d, b2 = b[i] * b[i];
    }
    red[0][threadIdx.x] = d2, red[1][threadIdx.x] = b2;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st)
            red[0][threadIdx.x] += red[0][threadIdx.x + st], red[1][threadIdx.x] += red[1][threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        part[2 * blockIdx.x] = red[0][0], part[2 * blockIdx.x + 1] = red[1][0];
}

} // namespace

struct dndsmi_warmstart {
    dndsmi_ctx *ctx = nullptr;
    int64_t nc = 0, ldc = 0;
    std::vector<void *> allocs;
    int32_t *sten = nullptr; // [12][ldc]
    float *mom = nullptr;    // [9][ldc]
    float *logsz = nullptr;  // [ldc]
    float *P = nullptr, *G = nullptr, *Mm = nullptr, *Vv = nullptr; // [kNParam]
    int64_t adam_t = 0;
    // training set
    float *X = nullptr, *T = nullptr;
    int64_t n_samples = 0, capacity = 0;
    // per-call work: Y up to max_rows, the batch's up to max_batch rows
    int64_t max_rows = 0, max_batch = 0;
    float *bX = nullptr, *bT = nullptr, *Y = nullptr, *dY = nullptr, *dZ2 = nullptr, *dZ1 = nullptr, *part = nullptr;
    int32_t *perm = nullptr; // [max_perm] the epoch's order of the samples
    int64_t max_perm = 0;
    unsigned short *packed = nullptr; // [kPacked] the weights as training's operands
    unsigned short *cols = nullptr;   // [kColsAll][max_batch up to a multiple of 32]
    float *fX = nullptr, *fS = nullptr; // features / scales of all cells
    float *kpart = nullptr, *bpart = nullptr; // [kMaxSplit][kNParam], [kMaxBiasChunks][kBias] partial sums
    std::mt19937_64 rng;

    template <class T>
    int alloc(T *&p, int64_t n) {
        void *q = nullptr;
        if (hipMalloc(&q, sizeof(T) * size_t(std::max<int64_t>(n, 1))) != hipSuccess) {
            (void)hipGetLastError();
            ctx->err = "hipMalloc failed (warm start)";
            return DNDSMI_ERR_OUT_OF_MEMORY;
        }
        allocs.push_back(q);
        p = static_cast<T *>(q);
        return DNDSMI_OK;
    }
    ~dndsmi_warmstart() {
        for (void *q : allocs)
            (void)hipFree(q);
    }
};

namespace {

int ensure_rows(dndsmi_warmstart *w, int64_t rows) {
    if (rows <= w->max_rows)
        return DNDSMI_OK;
    // growth frees nothing: old buffers stay in the allocation list until destroy
    const int64_t r = std::max<int64_t>(rows, 256);
    DNDSMI_TRY(w->alloc(w->Y, r * kOut));
    w->max_rows = r;
    return DNDSMI_OK;
}

constexpr int kSplitChunk = 256, kMaxSplit = 64, kMaxBiasChunks = 1024;

int ensure_batch(dndsmi_warmstart *w, int64_t rows) {
    DNDSMI_TRY(ensure_rows(w, rows));
    if (!w->packed) {
        unsigned short *packed = nullptr;
        DNDSMI_TRY(w->alloc(w->bpart, int64_t(kMaxBiasChunks) * kBias));
        DNDSMI_TRY(w->alloc(w->kpart, int64_t(kMaxSplit) * kNParam));
        DNDSMI_TRY(w->alloc(packed, kPacked));
        DNDSMI_TRY(w->ctx->upload(packed, std::vector<unsigned short>(kPacked, 0)));
        w->packed = packed;
    }
    if (rows <= w->max_batch)
        return DNDSMI_OK;
    const int64_t r = (std::max<int64_t>(rows, 256) + 31) / 32 * 32;
    DNDSMI_TRY(w->alloc(w->bX, r * kIn));
    DNDSMI_TRY(w->alloc(w->bT, r * kOut));
    DNDSMI_TRY(w->alloc(w->dY, r * kOut));
    DNDSMI_TRY(w->alloc(w->dZ2, r * kHid));
    DNDSMI_TRY(w->alloc(w->dZ1, r * kHid));
    DNDSMI_TRY(w->alloc(w->cols, r * kColsAll));
    DNDSMI_TRY(w->alloc(w->part, (r * kOut + 255) / 256 + 1));
    w->max_batch = r;
    return DNDSMI_OK;
}

// the network's output for `rows` rows of X into Y (fused kernel, inference
// only: the hidden activations are not kept)
int infer(dndsmi_warmstart *w, const float *X, int32_t rows) {
    const int64_t ntile = (int64_t(rows) + 15) / 16;
    const unsigned grid = unsigned(std::max<int64_t>(1, std::min<int64_t>((ntile + kInferWaves - 1) / kInferWaves, 512)));
    hipLaunchKernelGGL(k_mlp_infer, dim3(grid), dim3(64 * kInferWaves), 0, w->ctx->stream, rows, X, w->P, w->Y);
    return w->ctx->launch_check("k_mlp_infer");
}

// the weights as BF16 operands, before the first loss_grad on parameters as
// they are now
int pack_weights(dndsmi_warmstart *w) {
    hipLaunchKernelGGL(k_pack, dim3(unsigned((kNParam + 255) / 256)), dim3(256), 0, w->ctx->stream, w->P, w->packed);
    return w->ctx->launch_check("k_pack");
}

// loss and gradients of `rows` rows of (X, T), those of idx or the first
// ones, with the weights last packed; the gradients go into G, or with `step` into that step of Adam
int loss_grad(dndsmi_warmstart *w, const float *X, const float *T, const int32_t *idx, int32_t rows, double *loss,
              const AdamStep *step) {
    hipStream_t s = w->ctx->stream;
    const int64_t ny = int64_t(rows) * kOut, ld = (int64_t(rows) + 31) / 32 * 32;
    const TrainCols tc{ld,
                       w->cols + kColsX * ld,
                       w->cols + kColsH1 * ld,
                       w->cols + kColsH2 * ld,
                       w->cols + kColsdY * ld,
                       w->cols + kColsdZ2 * ld,
                       w->cols + kColsdZ1 * ld};
    const unsigned gr = unsigned(std::min<int64_t>(ld / 16, 512));
    hipLaunchKernelGGL(k_train_rows, dim3(gr), dim3(64 * kRowWaves), 0, s, rows, idx, X, T, w->P,
                       w->packed, float(2.0 / double(ny)), tc, loss ? w->Y : nullptr, w->dY, w->dZ2, w->dZ1);
    // the rows split into at most kMaxSplit chunks for the weights and
    // kMaxBiasChunks for the biases
    const int32_t kchunk = std::max<int32_t>(kSplitChunk, (rows + kMaxSplit - 1) / kMaxSplit / 16 * 16 + 16);
    const int32_t bchunk = std::max<int32_t>(64, (rows + kMaxBiasChunks - 1) / kMaxBiasChunks);
    const int32_t nz = (rows + kchunk - 1) / kchunk, nb = (rows + bchunk - 1) / bchunk;
    hipLaunchKernelGGL(k_train_grads, dim3(unsigned(nz * kWTiles + nb * kBiasBlocks)), dim3(64), 0, s, rows, nz,
                       kchunk, bchunk, tc, w->dY, w->dZ2, w->dZ1, w->kpart, w->bpart);
    hipLaunchKernelGGL(k_train_update, dim3(unsigned((kNParam + 255) / 256)), dim3(256), 0, s, nz, nb, w->kpart,
                       w->bpart, step ? nullptr : w->G, step ? *step : AdamStep{}, w->P, w->Mm, w->Vv,
                       w->packed);
    DNDSMI_TRY(w->ctx->launch_check("warm-start training step"));
    if (loss) {
        const unsigned nblk = unsigned((ny + 255) / 256);
        hipLaunchKernelGGL(k_mse, dim3(nblk), dim3(256), 0, s, ny, idx, w->Y, T, w->part);
        DNDSMI_TRY(w->ctx->launch_check("k_mse"));
        std::vector<float> h(nblk);
        DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(h.data(), w->part, sizeof(float) * nblk, hipMemcpyDeviceToHost, s),
                               "hipMemcpyAsync"));
        DNDSMI_TRY(w->ctx->hip(hipStreamSynchronize(s), "hipStreamSynchronize"));
        double acc = 0;
        for (float v : h)
            acc += v;
        *loss = acc / double(ny);
    }
    return DNDSMI_OK;
}

AdamStep adam_step(dndsmi_warmstart *w, double lr) {
    const double b1 = 0.9, b2 = 0.999, eps = 1e-8;
    w->adam_t++;
    const double c1 = 1 - std::pow(b1, double(w->adam_t)), c2 = 1 - std::pow(b2, double(w->adam_t));
    // step lr sqrt(c2) / c1 on m / (sqrt(v) + eps sqrt(c2)), the bias-corrected update
    return {float(lr * std::sqrt(c2) / c1), float(b1), float(b2), float(eps * std::sqrt(c2))};
}

int features(dndsmi_warmstart *w, const double *u) {
    if (!w->fS)
        DNDSMI_TRY(w->alloc(w->fS, w->nc * 4));
    if (!w->fX)
        DNDSMI_TRY(w->alloc(w->fX, w->nc * kIn));
    hipLaunchKernelGGL(k_features, dim3(grid_for(w->nc)), dim3(256), 0, w->ctx->stream, int32_t(w->nc), w->ldc,
                       w->sten, u, w->mom, w->logsz, w->fX, w->fS);
    return w->ctx->launch_check("k_features");
}

} // namespace

extern "C" int dndsmi_warmstart_create(dndsmi_ctx *c, const dndsmi_mesh_view *mesh, const dndsmi_vr_view *vr,
                                       uint64_t seed, int64_t capacity, dndsmi_warmstart **out) {
    if (!c || !mesh || !vr || !out || mesh->n_cell != c->nc || vr->n_cell != c->nc || capacity < 0)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    {
        std::string why;
        if (check_mesh_view(mesh, why) != DNDSMI_OK)
            return DNDSMI_ERR_INVALID_ARGUMENT;
    }
    *out = nullptr;
    auto *w = new (std::nothrow) dndsmi_warmstart();
    if (!w)
        return DNDSMI_ERR_OUT_OF_MEMORY;
    w->ctx = c, w->nc = c->nc, w->ldc = c->ldc;
    w->rng.seed(seed);
    auto fail = [&](int rc) {
        delete w;
        return rc;
    };
    const int64_t nc = c->nc, ldc = c->ldc;
    // stencil: breadth-first over faces, cell2face order, first 12 cells
    std::vector<int32_t> sten(size_t(kSten) * ldc, 0);
    std::vector<float> mom(size_t(9) * ldc, 0.f), lsz(size_t(ldc), 0.f);
    std::vector<int64_t> ring, next;
    std::vector<int64_t> seen;
    for (int64_t i = 0; i < nc; i++) {
        seen.assign(1, i);
        ring.assign(1, i);
        std::vector<int64_t> got;
        while (int(got.size()) < kSten && !ring.empty()) {
            next.clear();
            for (int64_t a : ring)
                for (int64_t q = mesh->cell_ptr[a]; q < mesh->cell_ptr[a + 1]; q++) {
                    const int64_t f = mesh->cell2face[q];
                    const int64_t L = mesh->face2cell[2 * f], R = mesh->face2cell[2 * f + 1];
                    const int64_t b = L == a ? R : L;
                    if (b == DNDSMI_NO_CELL || std::find(seen.begin(), seen.end(), b) != seen.end())
                        continue;
                    seen.push_back(b);
                    next.push_back(b);
                    if (int(got.size()) < kSten)
                        got.push_back(b);
                }
            ring = next;
        }
        const int64_t ci = c->c2d[i]; // device numbering
        for (int k = 0; k < kSten; k++)
            sten[k * ldc + ci] = c->c2d[k < int(got.size()) ? got[k] : i];
        for (int k = 0; k < 9; k++)
            mom[k * ldc + ci] = float(vr->base_moment[10 * i + 1 + k]);
        lsz[ci] = float(0.5 * std::log(vr->volume[i]));
    }
    try {
        if (w->alloc(w->sten, kSten * ldc) || w->alloc(w->mom, 9 * ldc) || w->alloc(w->logsz, ldc) ||
            w->alloc(w->P, kNParam) || w->alloc(w->G, kNParam) || w->alloc(w->Mm, kNParam) ||
            w->alloc(w->Vv, kNParam) || w->alloc(w->X, capacity * kIn) || w->alloc(w->T, capacity * kOut))
            return fail(DNDSMI_ERR_OUT_OF_MEMORY);
    } catch (...) {
        return fail(DNDSMI_ERR_OUT_OF_MEMORY);
    }
    w->capacity = capacity;
    // He-style initialisation, seeded: weights U(-sqrt(6/fan_in), ...), zero biases
    std::vector<float> P(kNParam, 0.f);
    auto init = [&](int64_t o, int fin, int fout) {
        std::uniform_real_distribution<float> d(-std::sqrt(6.f / fin), std::sqrt(6.f / fin));
        for (int64_t k = 0; k < int64_t(fin) * fout; k++)
            P[o + k] = d(w->rng);
    };
    init(oW1, kIn, kHid), init(oW2, kHid, kHid), init(oW3, kHid, kOut);
    for (int64_t k = oW3; k < oW3 + kHid * kOut; k++)
        P[k] *= 0.1f; // small initial output
    std::vector<float> zero(kNParam, 0.f);
    int rc = DNDSMI_OK;
    rc = rc ? rc : c->upload(w->sten, sten);
    rc = rc ? rc : c->upload(w->mom, mom);
    rc = rc ? rc : c->upload(w->logsz, lsz);
    rc = rc ? rc : c->upload(w->P, P);
    rc = rc ? rc : c->upload(w->Mm, zero);
    rc = rc ? rc : c->upload(w->Vv, zero);
    if (rc)
        return fail(rc);
    c->warmstarts.insert(w);
    *out = w;
    return DNDSMI_OK;
}

void dndsmi_warmstart_detach(dndsmi_warmstart *w) { w->ctx = nullptr; } // keeps its own allocations

extern "C" void dndsmi_warmstart_destroy(dndsmi_warmstart *w) {
    if (w && w->ctx) {
        (void)hipStreamSynchronize(w->ctx->stream);
        w->ctx->warmstarts.erase(w);
        if (w->ctx->step_ws == w)
            w->ctx->step_ws = nullptr;
    }
    delete w;
}

// ---- the learned warm start inside the mixed-precision step ------------
//
// Every stage of dndsmi_ssprk3_step_mixed starts its sweeps from the uRec the
// previous stage left (the reference's own warm start).  With a network
// attached, the stage first adds the network's prediction on the change of
// the cell means since the previous stage.  The plain method judges it: in a
// check window every step runs twice, plain on shadow copies of u and uRec
// and then with the correction, with the plain run's time step; at the
// window's end the corrected state must lie within the tolerance of the
// plain one (relative L2 over all cells), else u and uRec become the plain
// run's and the correction stays off until the next attach.  A corrected
// run that meets a non-positive state inside a window is replaced the same
// way.

namespace dndsmi_host {

int ws_stage_begin(dndsmi_ctx *c, const double *u, double *x, bool use) {
    dndsmi_warmstart *w = c->step_ws;
    DNDSMI_TRY(c->ensure(c->ws_uprev, 4 * c->ldc));
    DNDSMI_TRY(c->ensure(c->ws_du, 4 * c->ldc));
    if (!c->ws_have_prev) {
        DNDSMI_TRY(c->hip(hipMemcpyAsync(c->ws_uprev, u, sizeof(double) * 4 * c->nc, hipMemcpyDeviceToDevice,
                                         c->stream),
                          "copy u"));
        c->ws_have_prev = true;
        return DNDSMI_OK;
    }
    hipLaunchKernelGGL(k_mean_change, dim3(grid_for(4 * c->nc)), dim3(256), 0, c->stream, int32_t(c->nc), u,
                       c->ws_uprev, c->ws_du);
    DNDSMI_TRY(c->launch_check("k_mean_change"));
    if (!use)
        return DNDSMI_OK;
    DNDSMI_TRY(features(w, c->ws_du));
    DNDSMI_TRY(ensure_rows(w, w->nc));
    DNDSMI_TRY(infer(w, w->fX, int32_t(w->nc)));
    hipLaunchKernelGGL(k_unscale<true>, dim3(grid_for(w->nc)), dim3(256), 0, c->stream, int32_t(w->nc), w->ldc, w->Y,
                       w->fS, x);
    DNDSMI_TRY(c->launch_check("warm-start stage correction"));
    c->ws_stats[0]++;
    return DNDSMI_OK;
}

int ws_window_begin(dndsmi_ctx *c, const double *u, const double *x) {
    DNDSMI_TRY(c->ensure(c->ws_sh_u, 4 * c->ldc));
    DNDSMI_TRY(c->ensure(c->ws_sh_x, 36 * c->ldc));
    DNDSMI_TRY(c->ensure(c->ws_part, 2 * int64_t(grid_for(36 * c->ldc)) + 2));
    DNDSMI_TRY(c->hip(hipMemcpyAsync(c->ws_sh_u, u, sizeof(double) * 4 * c->ldc, hipMemcpyDeviceToDevice, c->stream),
                      "copy u to the shadow"));
    return c->hip(hipMemcpyAsync(c->ws_sh_x, x, sizeof(double) * 36 * c->ldc, hipMemcpyDeviceToDevice, c->stream),
                  "copy uRec to the shadow");
}

int ws_window_end(dndsmi_ctx *c, double *u, double *x, bool failed) {
    bool reject = failed;
    if (!reject) {
        const int64_t n = 4 * c->nc;
        const unsigned g = grid_for(n, 256);
        hipLaunchKernelGGL(k_diff2, dim3(g), dim3(256), 0, c->stream, n, u, c->ws_sh_u, c->ws_part);
        DNDSMI_TRY(c->launch_check("k_diff2"));
        std::vector<double> part(2 * size_t(g));
        DNDSMI_TRY(c->hip(hipMemcpyAsync(part.data(), c->ws_part, sizeof(double) * part.size(), hipMemcpyDeviceToHost,
                                         c->stream),
                          "hipMemcpyAsync"));
        DNDSMI_TRY(c->hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
        double d2 = 0, b2 = 0;
        for (unsigned k = 0; k < g; k++)
            d2 += part[2 * k], b2 += part[2 * k + 1];
        c->ws_last_dev = std::sqrt(d2 / (b2 > 0 ? b2 : 1.0));
        reject = !(c->ws_last_dev <= c->ws_tol);
    }
    if (reject) {
        DNDSMI_TRY(c->hip(hipMemcpyAsync(u, c->ws_sh_u, sizeof(double) * 4 * c->ldc, hipMemcpyDeviceToDevice,
                                         c->stream),
                          "restore u"));
        DNDSMI_TRY(c->hip(hipMemcpyAsync(x, c->ws_sh_x, sizeof(double) * 36 * c->ldc, hipMemcpyDeviceToDevice,
                                         c->stream),
                          "restore uRec"));
        c->ws_rejected = true;
        c->ws_stats[2]++;
    } else {
        c->ws_stats[1]++;
    }
    return DNDSMI_OK;
}

} // namespace dndsmi_host

extern "C" int dndsmi_ssprk3_set_warm_start(dndsmi_ctx *c, dndsmi_warmstart *ws, int32_t check_steps,
                                            int32_t recheck_interval, double tolerance) {
    if (!c || (ws && ws->ctx != c) || check_steps < 1 || recheck_interval < 0 || !(tolerance >= 0))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    c->step_ws = ws;
    c->ws_check_steps = check_steps;
    c->ws_recheck = recheck_interval;
    c->ws_tol = tolerance;
    c->ws_have_prev = false;
    c->ws_rejected = false;
    c->ws_win_left = 0;
    c->ws_since_check = 0;
    c->ws_first = true;
    c->ws_last_dev = -1.0;
    for (int k = 0; k < 3; k++)
        c->ws_stats[k] = 0;
    return DNDSMI_OK;
}

extern "C" int dndsmi_ssprk3_warm_start_stats(const dndsmi_ctx *c, int64_t stats[3], double *last_deviation) {
    if (!c || !stats)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    for (int k = 0; k < 3; k++)
        stats[k] = c->ws_stats[k];
    if (last_deviation)
        *last_deviation = c->ws_last_dev;
    return DNDSMI_OK;
}

extern "C" int64_t dndsmi_warmstart_num_params(void) { return kNParam; }

extern "C" int dndsmi_warmstart_get_params(dndsmi_warmstart *w, float *host) {
    if (!w || !host)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(host, w->P, sizeof(float) * kNParam, hipMemcpyDeviceToHost, w->ctx->stream),
                           "hipMemcpyAsync"));
    return w->ctx->hip(hipStreamSynchronize(w->ctx->stream), "hipStreamSynchronize");
}

extern "C" int dndsmi_warmstart_set_params(dndsmi_warmstart *w, const float *host) {
    if (!w || !host)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->P, host, sizeof(float) * kNParam, hipMemcpyHostToDevice, w->ctx->stream),
                           "hipMemcpyAsync"));
    w->adam_t = 0;
    std::vector<float> zero(kNParam, 0.f);
    DNDSMI_TRY(w->ctx->upload(w->Mm, zero));
    return w->ctx->upload(w->Vv, zero);
}

extern "C" int dndsmi_warmstart_loss_grad(dndsmi_warmstart *w, const float *X, const float *T, int32_t rows,
                                          float *grad, double *loss) {
    if (!w || !X || !T || rows < 1)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(ensure_batch(w, rows));
    hipStream_t s = w->ctx->stream;
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->bX, X, sizeof(float) * rows * kIn, hipMemcpyHostToDevice, s), "copy"));
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->bT, T, sizeof(float) * rows * kOut, hipMemcpyHostToDevice, s), "copy"));
    DNDSMI_TRY(pack_weights(w));
    DNDSMI_TRY(loss_grad(w, w->bX, w->bT, nullptr, rows, loss, nullptr));
    if (grad) {
        DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(grad, w->G, sizeof(float) * kNParam, hipMemcpyDeviceToHost, s), "copy"));
        DNDSMI_TRY(w->ctx->hip(hipStreamSynchronize(s), "hipStreamSynchronize"));
    }
    return DNDSMI_OK;
}

extern "C" int dndsmi_warmstart_adam_step(dndsmi_warmstart *w, const float *grad, double lr) {
    if (!w || !grad)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->G, grad, sizeof(float) * kNParam, hipMemcpyHostToDevice, w->ctx->stream),
                           "copy"));
    hipLaunchKernelGGL(k_adam, dim3(unsigned((kNParam + 255) / 256)), dim3(256), 0, w->ctx->stream, kNParam, w->P,
                       w->G, w->Mm, w->Vv, adam_step(w, lr));
    return w->ctx->launch_check("k_adam");
}

extern "C" int dndsmi_warmstart_features(dndsmi_warmstart *w, const dndsmi_array *u, float *X, float *S) {
    if (!w || !same_ctx(w->ctx, u, DNDSMI_ARRAY_DOF))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(features(w, u->d));
    hipStream_t s = w->ctx->stream;
    std::vector<float> hx(size_t(w->nc) * kIn), hs(size_t(w->nc) * 4);
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(hx.data(), w->fX, sizeof(float) * hx.size(), hipMemcpyDeviceToHost, s),
                           "copy"));
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(hs.data(), w->fS, sizeof(float) * hs.size(), hipMemcpyDeviceToHost, s),
                           "copy"));
    DNDSMI_TRY(w->ctx->hip(hipStreamSynchronize(s), "hipStreamSynchronize"));
    for (int64_t i = 0; i < w->nc; i++) { // rows back in mesh numbering
        const int64_t d = w->ctx->c2d[i];
        if (X)
            std::memcpy(X + i * kIn, hx.data() + d * kIn, sizeof(float) * kIn);
        if (S)
            std::memcpy(S + i * 4, hs.data() + d * 4, sizeof(float) * 4);
    }
    return DNDSMI_OK;
}

extern "C" int dndsmi_warmstart_add_samples(dndsmi_warmstart *w, const dndsmi_array *u, const dndsmi_array *uRec) {
    if (!w || !same_ctx(w->ctx, u, DNDSMI_ARRAY_DOF) || !same_ctx(w->ctx, uRec, DNDSMI_ARRAY_REC))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (w->n_samples + w->nc > w->capacity) {
        w->ctx->err = "warm-start training set is full";
        return DNDSMI_ERR_INVALID_ARGUMENT;
    }
    DNDSMI_TRY(features(w, u->d));
    hipStream_t s = w->ctx->stream;
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->X + w->n_samples * kIn, w->fX, sizeof(float) * w->nc * kIn,
                                          hipMemcpyDeviceToDevice, s),
                           "copy"));
    hipLaunchKernelGGL(k_targets, dim3(grid_for(w->nc)), dim3(256), 0, s, int32_t(w->nc), w->ldc, uRec->d, w->fS,
                       w->T + w->n_samples * kOut);
    DNDSMI_TRY(w->ctx->launch_check("k_targets"));
    w->n_samples += w->nc;
    return DNDSMI_OK;
}

extern "C" int dndsmi_warmstart_add_rows(dndsmi_warmstart *w, const float *X, const float *T, int64_t rows) {
    if (!w || !X || !T || rows < 0)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    if (w->n_samples + rows > w->capacity) {
        w->ctx->err = "warm-start training set is full";
        return DNDSMI_ERR_INVALID_ARGUMENT;
    }
    hipStream_t s = w->ctx->stream;
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->X + w->n_samples * kIn, X, sizeof(float) * rows * kIn,
                                          hipMemcpyHostToDevice, s),
                           "copy"));
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(w->T + w->n_samples * kOut, T, sizeof(float) * rows * kOut,
                                          hipMemcpyHostToDevice, s),
                           "copy"));
    DNDSMI_TRY(w->ctx->hip(hipStreamSynchronize(s), "hipStreamSynchronize"));
    w->n_samples += rows;
    return DNDSMI_OK;
}

extern "C" int dndsmi_warmstart_targets(dndsmi_warmstart *w, const dndsmi_array *u, const dndsmi_array *uRec,
                                        float *T) {
    if (!w || !T || !same_ctx(w->ctx, u, DNDSMI_ARRAY_DOF) || !same_ctx(w->ctx, uRec, DNDSMI_ARRAY_REC))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(features(w, u->d));
    DNDSMI_TRY(ensure_rows(w, w->nc));
    hipStream_t s = w->ctx->stream;
    hipLaunchKernelGGL(k_targets, dim3(grid_for(w->nc)), dim3(256), 0, s, int32_t(w->nc), w->ldc, uRec->d, w->fS,
                       w->Y);
    DNDSMI_TRY(w->ctx->launch_check("k_targets"));
    std::vector<float> ht(size_t(w->nc) * kOut);
    DNDSMI_TRY(w->ctx->hip(hipMemcpyAsync(ht.data(), w->Y, sizeof(float) * ht.size(), hipMemcpyDeviceToHost, s),
                           "copy"));
    DNDSMI_TRY(w->ctx->hip(hipStreamSynchronize(s), "hipStreamSynchronize"));
    for (int64_t i = 0; i < w->nc; i++)
        std::memcpy(T + i * kOut, ht.data() + int64_t(w->ctx->c2d[i]) * kOut, sizeof(float) * kOut);
    return DNDSMI_OK;
}

extern "C" int64_t dndsmi_warmstart_num_samples(const dndsmi_warmstart *w) { return w ? w->n_samples : -1; }

extern "C" int dndsmi_warmstart_train(dndsmi_warmstart *w, int32_t epochs, int32_t batch, double lr, double lr_final,
                                      double *loss_hist) {
    if (!w || epochs < 1 || batch < 1 || w->n_samples < 1)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    const int64_t n = w->n_samples;
    const int32_t b = int32_t(std::min<int64_t>(batch, n));
    DNDSMI_TRY(ensure_batch(w, b));
    if (n > w->max_perm) {
        DNDSMI_TRY(w->alloc(w->perm, w->capacity));
        w->max_perm = w->capacity;
    }
    int32_t *perm = w->perm;
    DNDSMI_TRY(pack_weights(w));
    std::vector<int32_t> hp(static_cast<size_t>(n));
    std::iota(hp.begin(), hp.end(), 0);
    hipStream_t s = w->ctx->stream;
    const int64_t steps_per_epoch = n / b, total = steps_per_epoch * epochs;
    int64_t step = 0;
    for (int32_t e = 0; e < epochs; e++) {
        std::shuffle(hp.begin(), hp.end(), w->rng);
        DNDSMI_TRY(w->ctx->upload(perm, hp));
        double acc = 0;
        for (int64_t q = 0; q < steps_per_epoch; q++, step++) {
            const int32_t *ix = perm + q * b;
            double l = 0;
            const bool last = q == steps_per_epoch - 1;
            // cosine decay from lr to lr_final
            const double f = 0.5 * (1 + std::cos(M_PI * double(step) / double(std::max<int64_t>(total, 1))));
            const AdamStep as = adam_step(w, lr_final + (lr - lr_final) * f);
            DNDSMI_TRY(loss_grad(w, w->X, w->T, ix, b, last ? &l : nullptr, &as));
            if (last)
                acc = l;
        }
        DNDSMI_TRY(w->ctx->launch_check("warm-start training"));
        if (loss_hist)
            loss_hist[e] = acc;
    }
    return w->ctx->hip(hipStreamSynchronize(s), "hipStreamSynchronize");
}

extern "C" int dndsmi_warmstart_predict(dndsmi_warmstart *w, const dndsmi_array *u, dndsmi_array *uRec) {
    if (!w || !same_ctx(w->ctx, u, DNDSMI_ARRAY_DOF) || !same_ctx(w->ctx, uRec, DNDSMI_ARRAY_REC))
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(features(w, u->d));
    DNDSMI_TRY(ensure_rows(w, w->nc));
    DNDSMI_TRY(infer(w, w->fX, int32_t(w->nc)));
    hipLaunchKernelGGL(k_unscale<false>, dim3(grid_for(w->nc)), dim3(256), 0, w->ctx->stream, int32_t(w->nc), w->ldc, w->Y,
                       w->fS, uRec->d);
    return w->ctx->launch_check("warm-start predict");
}

extern "C" int dndsmi_reconstruct_to_tolerance(dndsmi_ctx *c, const dndsmi_array *u, dndsmi_array *uRec,
                                               dndsmi_array *uRecNewBuf, double tol, int32_t max_sweeps, double t,
                                               int32_t *sweeps, double *res_out) {
    if (!c || !same_ctx(c, u, DNDSMI_ARRAY_DOF) || !same_ctx(c, uRec, DNDSMI_ARRAY_REC) ||
        !same_ctx(c, uRecNewBuf, DNDSMI_ARRAY_REC) || uRec == uRecNewBuf || max_sweeps < 1)
        return DNDSMI_ERR_INVALID_ARGUMENT;
    DNDSMI_TRY(ensure_increment(c));
    double res = 0;
    int32_t k = 0;
    while (k < max_sweeps) {
        DNDSMI_TRY(launch_increment(c, u->d, uRec->d, uRecNewBuf->d, t));
        std::swap(uRec->d, uRecNewBuf->d);
        k++;
        DNDSMI_TRY(check_errw(c));
        res = 0;
        for (unsigned b = 0; b < grid_for(c->nc, 256); b++)
            res += c->host_sums[b];
        res /= double(c->nc);
        if (res < tol)
            break;
    }
    if (sweeps)
        *sweeps = k;
    if (res_out)
        *res_out = res;
    return DNDSMI_OK;
}
