// nsfv1_mlp.hip -- learned Newton initial guess: a per-node MLP
// 24 -> 128 -> 128 -> 4 (ReLU), BF16 weights and activations with FP32
// accumulation on the MFMA units (v_mfma_f32_16x16x32_bf16), plus the
// backward pass on the MFMA units with FP32 operands
// (v_mfma_f32_16x16x4_f32), deterministic gradient reduction and Adam used to train it
// on trajectories of the plain solver, and the feature / guess kernels that
// connect it to the discretisation.  No counterpart in the reference.
//
// Parameter blob (FP32 master copy, MLP_NPARAM floats):
//   W1 [128][32] (inputs padded 24 -> 32 with zero columns), b1 [128],
//   W2 [128][128], b2 [128], W3 [16][128] (outputs padded 4 -> 16 with zero
//   rows), b3 [16].
// The BF16 copy (MLP_NPARAM uint16) uses the same offsets; only its weight
// matrices are read.
//
// MFMA mapping (one wavefront = 16 nodes).  The layers are evaluated in
// transposed form, H^T = W X^T, so that the accumulators of two tiles of one
// layer (lane l holds rows 4*(l/16)+j, column l%16 of each) are the B operand
// of the next (8 products per lane, column l%16), the weights being loaded in
// the same order: activations never leave registers.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nsfv1_mlp.hpp"

namespace nsfv1 {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __host__ inline uint16_t f2bf(float f)
{
    // round to nearest even (finite inputs)
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ inline float bf2f(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

__device__ inline float relu_bf(float z) { return bf2f(f2bf(z > 0.f ? z : 0.f)); }

// ---------------------------------------------------------------------
// forward: y[n][0..3] = W3 relu(W2 relu(W1 x + b1) + b2) + b3
//
// A wave holds the weights of layers 2 and 3 as MFMA A operands in registers
// (144 VGPRs, two waves per SIMD), loaded once from the BF16 copy, and walks
// 16-node blocks; layer 1 (a tile is 1 KB in lane order, read without bank
// conflicts) and the biases, which start the accumulators, sit in LDS.
// Bound by the conversions between layers and the matrix products, 44 MFMA of
// 16x16x32 a block: 65536 nodes with the cached pre-activations (68 MB
// written) 43.5 -> 31 us, 233000 nodes without them 66 -> 34 us against 64 nodes
// a workgroup with weights and activations in LDS.
// ---------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// four weights at p and four at q (8-byte aligned) as one A operand
__device__ __forceinline__ bf16x8 load_a(const uint16_t* __restrict__ p, const uint16_t* __restrict__ q)
{
    const uint2 lo = *reinterpret_cast<const uint2*>(p), hi = *reinterpret_cast<const uint2*>(q);
    return __builtin_bit_cast(bf16x8, make_uint4(lo.x, lo.y, hi.x, hi.y));
}

__global__ void __launch_bounds__(256, 2)
mlp_forward(const float* __restrict__ P, const uint16_t* __restrict__ WB, const float* __restrict__ X, int64_t n,
            float* __restrict__ Y, float* __restrict__ Z1, float* __restrict__ Z2)
{
    __shared__ __align__(16) float bias[2 * MLP_H + MLP_KOUT];
    __shared__ __align__(16) uint16_t w1[MLP_H * MLP_KIN];
    for (int i = threadIdx.x; i < MLP_H * MLP_KIN / 2; i += blockDim.x)
        reinterpret_cast<uint32_t*>(w1)[i] = reinterpret_cast<const uint32_t*>(WB + MLP_OFF_W1)[i];
    for (int i = threadIdx.x; i < MLP_H; i += blockDim.x) {
        bias[i] = P[MLP_OFF_B1 + i];
        bias[MLP_H + i] = P[MLP_OFF_B2 + i];
    }
    if (threadIdx.x < MLP_KOUT) bias[2 * MLP_H + threadIdx.x] = P[MLP_OFF_B3 + threadIdx.x];
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    // A operands: row col of the tile; the 8 products of lane group g sum over
    // inputs 8 g .. (layer 1) and, so that an accumulator pair is the next
    // layer's B operand as it stands, over hidden units 32 m + 4 g .. and
    // 32 m + 16 + 4 g .. (layers 2 and 3)
    bf16x8 a2[MLP_H / 16][MLP_H / 32], a3[MLP_H / 32];
#pragma unroll
    for (int t = 0; t < MLP_H / 16; ++t) {
#pragma unroll
        for (int m = 0; m < MLP_H / 32; ++m) {
            const uint16_t* w2 = WB + MLP_OFF_W2 + (t * 16 + col) * MLP_H + 32 * m + 4 * g;
            a2[t][m] = load_a(w2, w2 + 16);
        }
    }
#pragma unroll
    for (int m = 0; m < MLP_H / 32; ++m) {
        const uint16_t* w3 = WB + MLP_OFF_W3 + col * MLP_H + 32 * m + 4 * g;
        a3[m] = load_a(w3, w3 + 16);
    }
    __syncthreads();

    const int64_t nblk = (n + 15) / 16, nw = (int64_t)gridDim.x * 4;
    for (int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); blk < nblk; blk += nw) {
        asm volatile("" ::: "memory");  // layer 1 and the biases stay in LDS: hoisted, they spill
        const int64_t node = blk * 16 + col;
        const bool valid = node < n;
        // columns past the end repeat the last node (their results are dropped)
        const float* xp = X + (valid ? node : n - 1) * MLP_KIN + 8 * g;
        const float4 x0 = *reinterpret_cast<const float4*>(xp), x1 = *reinterpret_cast<const float4*>(xp + 4);
        bf16x8 xb;
        xb[0] = (__bf16)x0.x; xb[1] = (__bf16)x0.y; xb[2] = (__bf16)x0.z; xb[3] = (__bf16)x0.w;
        xb[4] = (__bf16)x1.x; xb[5] = (__bf16)x1.y; xb[6] = (__bf16)x1.z; xb[7] = (__bf16)x1.w;
        bf16x8 h1[MLP_H / 32], h2[MLP_H / 32];
#pragma unroll
        for (int t = 0; t < MLP_H / 16; ++t) {
            f32x4 acc = *reinterpret_cast<const f32x4*>(&bias[t * 16 + 4 * g]);
            const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&w1[(t * 16 + col) * MLP_KIN + 8 * g]);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, xb, acc, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; ++j) h1[t >> 1][(t & 1) * 4 + j] = (__bf16)(acc[j] > 0.f ? acc[j] : 0.f);
            if (Z1 && valid) *reinterpret_cast<f32x4*>(Z1 + node * MLP_H + t * 16 + 4 * g) = acc;
        }
#pragma unroll
        for (int t = 0; t < MLP_H / 16; ++t) {
            f32x4 acc = *reinterpret_cast<const f32x4*>(&bias[MLP_H + t * 16 + 4 * g]);
#pragma unroll
            for (int m = 0; m < MLP_H / 32; ++m) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[t][m], h1[m], acc, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; ++j) h2[t >> 1][(t & 1) * 4 + j] = (__bf16)(acc[j] > 0.f ? acc[j] : 0.f);
            if (Z2 && valid) *reinterpret_cast<f32x4*>(Z2 + node * MLP_H + t * 16 + 4 * g) = acc;
        }
        // layer 3 (rows 0..3 of the padded 16-row output)
        f32x4 acc = *reinterpret_cast<const f32x4*>(&bias[2 * MLP_H + 4 * g]);
#pragma unroll
        for (int m = 0; m < MLP_H / 32; ++m) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a3[m], h2[m], acc, 0, 0, 0);
        if (valid && g == 0) *reinterpret_cast<f32x4*>(Y + node * MLP_OUT) = acc;
    }
}

// ---------------------------------------------------------------------
// backward through the activations on the MFMA units (FP32 operands,
// v_mfma_f32_16x16x4_f32), one wavefront per 16 nodes, transposed form:
//   dZ2^T = (W3^T dY^T) * [z2 > 0],  dZ1^T = (W2^T dZ2^T) * [z1 > 0]
// with the BF16-rounded weights the forward used (straight-through for the
// activation rounding).  16x16x4 layouts: A[i][k] in lane (i + 16 k),
// B[k][j] in lane (j + 16 k), D[4 g + r][j] in lane (j + 16 g), element r.
// The dZ2 accumulators feed the W2^T product as B operands without leaving
// registers: MFMA (ot, r) sums over the hidden rows k = 16 ot + 4 g + r
// held by lane group g, and its A operand is gathered for the same k.
// ---------------------------------------------------------------------
__global__ void __launch_bounds__(256)
mlp_backward_act(const uint16_t* __restrict__ WB, const float* __restrict__ Z1, const float* __restrict__ Z2,
                 const float* __restrict__ DY, int64_t n, float* __restrict__ DZ1, float* __restrict__ DZ2)
{
    __shared__ __align__(16) uint16_t w2[MLP_H * MLP_H];
    __shared__ __align__(16) uint16_t w3[MLP_OUT * MLP_H];
    for (int i = threadIdx.x; i < MLP_H * MLP_H; i += blockDim.x) w2[i] = WB[MLP_OFF_W2 + i];
    for (int i = threadIdx.x; i < MLP_OUT * MLP_H; i += blockDim.x) w3[i] = WB[MLP_OFF_W3 + i];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, g = lane >> 4;
    const int64_t node = ((int64_t)blockIdx.x * 4 + wave) * 16 + col;
    const bool valid = node < n;
    // B of the first product: dY^T (k = output 0..3 = g, column = node)
    const float dyv = valid ? DY[node * MLP_OUT + g] : 0.f;
    f32x4 dz2[MLP_H / 16];
#pragma unroll
    for (int ot = 0; ot < MLP_H / 16; ++ot) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(bf2f(w3[g * MLP_H + ot * 16 + col]), dyv, acc, 0, 0, 0);
        float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        if (valid) z = *reinterpret_cast<const float4*>(Z2 + node * MLP_H + ot * 16 + 4 * g);
        dz2[ot][0] = z.x > 0.f ? acc[0] : 0.f;
        dz2[ot][1] = z.y > 0.f ? acc[1] : 0.f;
        dz2[ot][2] = z.z > 0.f ? acc[2] : 0.f;
        dz2[ot][3] = z.w > 0.f ? acc[3] : 0.f;
        if (valid)
            *reinterpret_cast<float4*>(DZ2 + node * MLP_H + ot * 16 + 4 * g) =
                make_float4(dz2[ot][0], dz2[ot][1], dz2[ot][2], dz2[ot][3]);
    }
#pragma unroll
    for (int o1 = 0; o1 < MLP_H / 16; ++o1) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ot = 0; ot < MLP_H / 16; ++ot) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float a = bf2f(w2[(ot * 16 + 4 * g + r) * MLP_H + o1 * 16 + col]);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, dz2[ot][r], acc, 0, 0, 0);
            }
        }
        float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        if (valid) z = *reinterpret_cast<const float4*>(Z1 + node * MLP_H + o1 * 16 + 4 * g);
        if (valid)
            *reinterpret_cast<float4*>(DZ1 + node * MLP_H + o1 * 16 + 4 * g) =
                make_float4(z.x > 0.f ? acc[0] : 0.f, z.y > 0.f ? acc[1] : 0.f, z.z > 0.f ? acc[2] : 0.f,
                            z.w > 0.f ? acc[3] : 0.f);
    }
}

// ---------------------------------------------------------------------
// weight gradients on the MFMA units (FP32 operands, 16x16x4):
//   dW1 = dZ1^T X,  dW2 = dZ2^T H1,  dW3 = dY^T H2
// as 88 16x16 tiles (W1 8x2, W2 8x8, W3 1x8 with rows 4..15 zero) summed over
// the nodes (k = node, 4 per MFMA).  A wave holds all 88 accumulators (352
// registers, one wave per SIMD) and takes its operands straight from memory:
// lane (col, g) reads entry col of a tile of node g, 64 contiguous bytes per
// node, which is the operand layout of both sides, so every value is read
// once and nothing is staged in LDS.  The next four nodes are loaded beside
// the products of the current ones.  The bias sums ride on the operands.
// The waves' tiles are added through LDS, partials go to
// part[block][MLP_NPARAM] and are reduced in block order (deterministic).
// Bound by the FP32 products (88 tiles, 2.95 GFLOP for 65536 nodes): 203 -> 59 us
// at 65536 nodes against tiles staged in LDS.
// ---------------------------------------------------------------------
constexpr int WG_T1 = 16, WG_T2 = 64, WG_TILES = WG_T1 + WG_T2 + 8;  // tiles of W1, W2, all
constexpr int WG_GROUP = 8;                                          // tiles combined at a time

struct WgradNode {
    float dz1[8], dz2[8], z1[8], z2[8], x[2], dy;
};

__device__ __forceinline__ void wgrad_load(WgradNode& N, const float* __restrict__ X, const float* __restrict__ Z1,
                                           const float* __restrict__ Z2, const float* __restrict__ DY,
                                           const float* __restrict__ DZ1, const float* __restrict__ DZ2, int64_t node,
                                           int64_t end, int64_t n, int col)
{
    // nodes past the end read the last one and contribute zero gradients
    const bool ok = node < end;
    const int64_t r = ok ? node : n - 1;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const float a = DZ1[r * MLP_H + 16 * t + col], b = DZ2[r * MLP_H + 16 * t + col];
        N.dz1[t] = ok ? a : 0.f;
        N.dz2[t] = ok ? b : 0.f;
        N.z1[t] = Z1[r * MLP_H + 16 * t + col];
        N.z2[t] = Z2[r * MLP_H + 16 * t + col];
    }
    N.x[0] = X[r * MLP_KIN + col];
    N.x[1] = X[r * MLP_KIN + 16 + col];
    const float d = DY[r * MLP_OUT + (col & 3)];
    N.dy = ok && col < MLP_OUT ? d : 0.f;
}

// parameter of element (tile, r, lane)
__device__ __forceinline__ int wgrad_param(int tile, int r, int lane)
{
    const int row = 4 * (lane >> 4) + r, col = lane & 15;
    if (tile < WG_T1) return MLP_OFF_W1 + ((tile >> 1) * 16 + row) * MLP_KIN + (tile & 1) * 16 + col;
    if (tile < WG_T1 + WG_T2)
        return MLP_OFF_W2 + (((tile - WG_T1) >> 3) * 16 + row) * MLP_H + ((tile - WG_T1) & 7) * 16 + col;
    return MLP_OFF_W3 + row * MLP_H + (tile - WG_T1 - WG_T2) * 16 + col;
}

__global__ void __launch_bounds__(256, 1)
mlp_wgrad_partial(const float* __restrict__ X, const float* __restrict__ Z1, const float* __restrict__ Z2,
                  const float* __restrict__ DY, const float* __restrict__ DZ1, const float* __restrict__ DZ2,
                  int64_t n, int64_t chunk, float* __restrict__ part)
{
    __shared__ float sh[4][WG_GROUP][4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int col = lane & 15, g = lane >> 4;
    f32x4 acc[WG_TILES];
#pragma unroll
    for (int q = 0; q < WG_TILES; ++q) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    float b1[8], b2[8], b3 = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) b1[t] = b2[t] = 0.f;
    const int64_t a = (int64_t)blockIdx.x * chunk;
    const int64_t b = a + chunk < n ? a + chunk : n;
    WgradNode N;
    if (a < b) wgrad_load(N, X, Z1, Z2, DY, DZ1, DZ2, a + 4 * wave + g, b, n, col);
#pragma unroll 1
    for (int64_t s0 = a; s0 < b; s0 += 16) {
        WgradNode C = N;
        if (s0 + 16 < b) wgrad_load(N, X, Z1, Z2, DY, DZ1, DZ2, s0 + 16 + 4 * wave + g, b, n, col);
        const float x0 = bf2f(f2bf(C.x[0])), x1 = bf2f(f2bf(C.x[1]));
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            b1[t] += C.dz1[t];
            b2[t] += C.dz2[t];
            C.z1[t] = relu_bf(C.z1[t]);
            C.z2[t] = relu_bf(C.z2[t]);
        }
        b3 += C.dy;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            acc[2 * t] = __builtin_amdgcn_mfma_f32_16x16x4f32(C.dz1[t], x0, acc[2 * t], 0, 0, 0);
            acc[2 * t + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(C.dz1[t], x1, acc[2 * t + 1], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                acc[WG_T1 + 8 * t + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(C.dz2[t], C.z1[i], acc[WG_T1 + 8 * t + i], 0, 0, 0);
            acc[WG_T1 + WG_T2 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(C.dy, C.z2[t], acc[WG_T1 + WG_T2 + t], 0, 0, 0);
        }
    }
    float* out = part + (int64_t)blockIdx.x * MLP_NPARAM;
    // tiles of the four waves, WG_GROUP at a time
#pragma unroll
    for (int q0 = 0; q0 < WG_TILES; q0 += WG_GROUP) {
#pragma unroll
        for (int q = 0; q < WG_GROUP; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) sh[wave][q][r][lane] = acc[q0 + q][r];
        __syncthreads();
        for (int i = threadIdx.x; i < WG_GROUP * 256; i += 256) {
            const int q = i >> 8, r = (i >> 6) & 3, l = i & 63;
            out[wgrad_param(q0 + q, r, l)] = ((sh[0][q][r][l] + sh[1][q][r][l]) + sh[2][q][r][l]) + sh[3][q][r][l];
        }
        __syncthreads();
    }
    // biases: over the four nodes of a wave, then over the waves
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        b1[t] += __shfl_xor(b1[t], 16, 64);
        b1[t] += __shfl_xor(b1[t], 32, 64);
        b2[t] += __shfl_xor(b2[t], 16, 64);
        b2[t] += __shfl_xor(b2[t], 32, 64);
    }
    b3 += __shfl_xor(b3, 16, 64);
    b3 += __shfl_xor(b3, 32, 64);
    float* sb = &sh[0][0][0][0] + wave * (2 * MLP_H + MLP_KOUT);
    if (g == 0) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            sb[16 * t + col] = b1[t];
            sb[MLP_H + 16 * t + col] = b2[t];
        }
        sb[2 * MLP_H + col] = b3;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * MLP_H + MLP_KOUT; i += 256) {
        const float* q = &sh[0][0][0][0] + i;
        constexpr int S = 2 * MLP_H + MLP_KOUT;
        const float v = ((q[0] + q[S]) + q[2 * S]) + q[3 * S];
        out[i < MLP_H ? MLP_OFF_B1 + i : (i < 2 * MLP_H ? MLP_OFF_B2 + i - MLP_H : MLP_OFF_B3 + i - 2 * MLP_H)] = v;
    }
}

// grad = sum of the block partials: 64 parameters a workgroup, a quarter of
// the blocks per wave, the quarters added in order (61 -> 5.6 us for 256
// blocks: one thread walked all blocks of its parameter)
__global__ void __launch_bounds__(256)
mlp_reduce(const float* __restrict__ part, int nblk, float* __restrict__ grad)
{
    __shared__ float sh[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    const int per = (nblk + 3) / 4, b0 = wave * per, b1 = b0 + per < nblk ? b0 + per : nblk;
    float s = 0.f;
    if (p < MLP_NPARAM) {
#pragma unroll 16
        for (int b = b0; b < b1; ++b) s += part[(int64_t)b * MLP_NPARAM + p];
    }
    sh[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && p < MLP_NPARAM) grad[p] = ((sh[0][lane] + sh[1][lane]) + sh[2][lane]) + sh[3][lane];
}

// MSE loss gradient on the 4 outputs: dy = 2 (y - t) / (4 n); loss partials
__global__ void mlp_mse(const float* __restrict__ Y, const float* __restrict__ T, int64_t n, float* __restrict__ DY,
                        float* __restrict__ lpart)
{
    __shared__ float sh[256];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (i < n * MLP_OUT) {
        const float e = Y[i] - T[i];
        DY[i] = 2.f * e / (float)(n * MLP_OUT);
        l = e * e;
    }
    sh[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = sh[0];
}

// Adam on the FP32 master copy; refreshes the BF16 copy.  Padding entries
// (zero columns of W1, zero rows of W3 and b3) stay zero.
__global__ void mlp_adam(float* __restrict__ P, float* __restrict__ M, float* __restrict__ V,
                         const float* __restrict__ G, float lr, float b1, float b2, float eps, float c1, float c2,
                         uint16_t* __restrict__ WB)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= MLP_NPARAM) return;
    bool pad = false;
    if (p < MLP_OFF_B1) pad = (p % MLP_KIN) >= MLP_IN;
    else if (p >= MLP_OFF_W3 && p < MLP_OFF_B3) pad = (p - MLP_OFF_W3) / MLP_H >= MLP_OUT;
    else if (p >= MLP_OFF_B3) pad = (p - MLP_OFF_B3) >= MLP_OUT;
    float w = P[p];
    if (!pad) {
        const float g = G[p];
        const float m = b1 * M[p] + (1.f - b1) * g;
        const float v = b2 * V[p] + (1.f - b2) * g * g;
        M[p] = m;
        V[p] = v;
        w -= lr * (m * c1) / (sqrtf(v * c2) + eps);
    } else {
        w = 0.f;
    }
    P[p] = w;
    WB[p] = f2bf(w);
}

__global__ void mlp_pack(const float* __restrict__ P, uint16_t* __restrict__ WB)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < MLP_NPARAM) WB[p] = f2bf(P[p]);
}

// ---------------------------------------------------------------------
// features, guess and target (node-major states [nv][4], FP64)
//
// With the three previous states u1 = u^{n-1}, u2 = u^{n-2}, u3 = u^{n-3},
// the backward differences are evaluated as nested differences,
//   d1 = u - u1,  e1 = u1 - u2,  f1 = u2 - u3,
//   d2 = d1 - e1 (= u - 2 u1 + u2),  d3 = d2 - (e1 - f1) (= u - 3 u1 + 3 u2 - u3),
// (exactly 0 for equal states, no products to contract), the quadratic
// extrapolation is q = u + d1 + d2 (= 3 u - 3 u1 + u2),
// and the step's scale sigma = max(rms of d3 over the velocity components
// of all nodes, 1e-30).  Differences enter the features divided by sigma,
// so one network sees slow and fast phases of a trajectory on one scale.
// ---------------------------------------------------------------------
__device__ inline float clampf(float x) { return fminf(fmaxf(x, -PRED_CLAMP), PRED_CLAMP); }

// partial sums of d3^2 over the velocity components, one per workgroup
// (grid-stride over the nodes, fixed grid: the sum order is fixed)
__global__ void __launch_bounds__(256)
predict_scale_partial(const double* __restrict__ u, const double* __restrict__ u1, const double* __restrict__ u2,
                      const double* __restrict__ u3, int64_t nv, double* __restrict__ part)
{
    __shared__ double sh[256];
    double acc = 0.0;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int64_t i = v * 4 + c;
            const double a = u1[i], b = u2[i], e1 = a - b;
            const double d3 = ((u[i] - a) - e1) - (e1 - (b - u3[i]));
            acc += d3 * d3;
        }
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void __launch_bounds__(256)
predict_scale_final(const double* __restrict__ part, int nparts, int64_t nv, double* __restrict__ sigma)
{
    __shared__ double sh[256];
    double acc = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) acc += part[i];
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double r = nv > 0 ? sqrt(sh[0] / (3.0 * (double)nv)) : 0.0;
        *sigma = r > 1e-30 ? r : 1e-30;
    }
}

// x[v] = clamp(( u, d1 / sigma, d2 / sigma, d3 / sigma,
//                1-ring mean of u - u, (1-ring mean of d1 - d1) / sigma ) * scale),
// 24 values padded to 32.  The 1-ring is the node's neighbours in the pattern,
// the node itself excluded.
// Four lanes per node, one per component: a neighbour's state is 32
// contiguous bytes, and neighbours come from the node-block list (one index
// each) in ascending order, four in flight.  Latency and L2 bound:
// 233000 nodes of the tetrahedral channel 78 -> 38 us against one lane per node that walked
// the columns of its first CSR row.
__global__ void __launch_bounds__(256)
predict_features(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ adj, const double* __restrict__ u,
                 const double* __restrict__ u1, const double* __restrict__ u2, const double* __restrict__ u3,
                 int64_t nv, const float* __restrict__ scale, const double* __restrict__ sigma, float* __restrict__ X)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t v = t >> 2;
    const int c = (int)(t & 3);
    if (v >= nv) return;
    const double is = 1.0 / *sigma;
    const int64_t i = v * 4 + c;
    const double un = u[i], a = u1[i], b = u2[i], e1 = a - b;
    const double d1 = un - a, d2 = d1 - e1, d3 = d2 - (e1 - (b - u3[i]));
    const int64_t r0 = rowptr[v * 4];
    const int nb = (int)((rowptr[v * 4 + 1] - r0) >> 2);
    const int32_t* ad = adj + (r0 >> 4);
    double m0 = 0.0, m1 = 0.0;
    int cnt = 0;
#pragma unroll 4
    for (int k = 0; k < nb; ++k) {
        const int64_t w = ad[k];
        const double x = u[w * 4 + c], y = u1[w * 4 + c];
        if (w != v) {
            m0 += x;
            m1 += x - y;
            ++cnt;
        }
    }
    const double ic = cnt > 0 ? 1.0 / cnt : 0.0;
    float out[MLP_KIN / 4];
    out[0] = clampf((float)un * scale[c]);
    out[1] = clampf((float)(d1 * is) * scale[4 + c]);
    out[2] = clampf((float)(d2 * is) * scale[8 + c]);
    out[3] = clampf((float)(d3 * is) * scale[12 + c]);
    out[4] = clampf((float)(cnt > 0 ? m0 * ic - un : 0.0) * scale[16 + c]);
    out[5] = clampf((float)(cnt > 0 ? (m1 * ic - d1) * is : 0.0) * scale[20 + c]);
    out[6] = out[7] = 0.f;
#pragma unroll
    for (int q = 0; q < MLP_KIN / 4; ++q) X[v * MLP_KIN + 4 * q + c] = out[q];
}

// guess = u + d1 + d2 + y * out_scale * sigma (per component)
__global__ void predict_guess(const double* __restrict__ u, const double* __restrict__ u1,
                              const double* __restrict__ u2, const float* __restrict__ Y,
                              const float* __restrict__ oscale, const double* __restrict__ sigma, int64_t nv,
                              double* __restrict__ g)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nv * 4) return;
    const int c = (int)(t & 3);
    const double d1 = u[t] - u1[t];
    const double d2 = d1 - (u1[t] - u2[t]);
    g[t] = u[t] + d1 + d2 + (double)Y[t] * (double)oscale[c] * *sigma;
}

// training target: t = clamp(((u^{n+1} - u) - d1 - d2) / (sigma * out_scale)),
// 0 for a component whose out_scale is 0 (not corrected)
__global__ void predict_target(const double* __restrict__ un1, const double* __restrict__ u,
                               const double* __restrict__ u1, const double* __restrict__ u2,
                               const float* __restrict__ oscale, const double* __restrict__ sigma, int64_t nv,
                               float* __restrict__ T)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nv * 4) return;
    const int c = (int)(t & 3);
    const double os = (double)oscale[c];
    const double d1 = u[t] - u1[t];
    const double d2 = d1 - (u1[t] - u2[t]);
    const double r = ((un1[t] - u[t]) - d1) - d2;
    T[t] = os > 0.0 ? clampf((float)(r / (*sigma * os))) : 0.f;
}

// ---------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------
static inline unsigned nblocks(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_mlp_forward(const float* P, const uint16_t* WB, const float* X, int64_t n, float* Y, float* Z1,
                              float* Z2, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    // two workgroups per CU (256 CUs): each wave holds the weights in
    // registers (two waves per SIMD) and walks its share of the 16-node blocks
    const unsigned g = nblocks(n, 64) < 512u ? nblocks(n, 64) : 512u;
    mlp_forward<<<g, 256, 0, s>>>(P, WB, X, n, Y, Z1, Z2);
    return hipGetLastError();
}

int64_t mlp_work_floats(int64_t n) { return 2 * n * MLP_H + (int64_t)MLP_WG_BLOCKS * MLP_NPARAM + n * MLP_OUT + 1024; }

hipError_t launch_mlp_backward(const uint16_t* WB, const float* X, const float* Z1, const float* Z2, const float* DY,
                               int64_t n, float* grad, float* work, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    float* dz1 = work;
    float* dz2 = dz1 + n * MLP_H;
    float* part = dz2 + n * MLP_H;
    mlp_backward_act<<<nblocks(n, 64), 256, 0, s>>>(WB, Z1, Z2, DY, n, dz1, dz2);
    const int64_t chunk = (n + MLP_WG_BLOCKS - 1) / MLP_WG_BLOCKS;
    mlp_wgrad_partial<<<MLP_WG_BLOCKS, 256, 0, s>>>(X, Z1, Z2, DY, dz1, dz2, n, chunk, part);
    mlp_reduce<<<nblocks(MLP_NPARAM, 64), 256, 0, s>>>(part, MLP_WG_BLOCKS, grad);
    return hipGetLastError();
}

hipError_t launch_mlp_mse(const float* Y, const float* T, int64_t n, float* DY, float* lpart, int* nparts,
                          hipStream_t s)
{
    const unsigned nb = nblocks(n * MLP_OUT, 256);
    *nparts = (int)nb;
    mlp_mse<<<nb, 256, 0, s>>>(Y, T, n, DY, lpart);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(float* P, float* M, float* V, const float* G, int step, float lr, float b1, float b2,
                           float eps, uint16_t* WB, hipStream_t s)
{
    const float c1 = 1.f / (1.f - powf(b1, (float)step)), c2 = 1.f / (1.f - powf(b2, (float)step));
    mlp_adam<<<nblocks(MLP_NPARAM, 256), 256, 0, s>>>(P, M, V, G, lr, b1, b2, eps, c1, c2, WB);
    return hipGetLastError();
}

hipError_t launch_mlp_pack(const float* P, uint16_t* WB, hipStream_t s)
{
    mlp_pack<<<nblocks(MLP_NPARAM, 256), 256, 0, s>>>(P, WB);
    return hipGetLastError();
}

hipError_t launch_predict_scale(const double* u, const double* u1, const double* u2, const double* u3, int64_t nv,
                                double* part, double* sigma, hipStream_t s)
{
    predict_scale_partial<<<PRED_SCALE_BLOCKS, 256, 0, s>>>(u, u1, u2, u3, nv, part);
    predict_scale_final<<<1, 256, 0, s>>>(part, PRED_SCALE_BLOCKS, nv, sigma);
    return hipGetLastError();
}

hipError_t launch_predict_features(const int64_t* rowptr, const int32_t* adj, const double* u, const double* u1,
                                   const double* u2, const double* u3, int64_t nv, const float* scale,
                                   const double* sigma, float* X, hipStream_t s)
{
    if (nv <= 0) return hipSuccess;
    predict_features<<<nblocks(nv * 4, 256), 256, 0, s>>>(rowptr, adj, u, u1, u2, u3, nv, scale, sigma, X);
    return hipGetLastError();
}

hipError_t launch_predict_guess(const double* u, const double* u1, const double* u2, const float* Y,
                                const float* oscale, const double* sigma, int64_t nv, double* g, hipStream_t s)
{
    if (nv <= 0) return hipSuccess;
    predict_guess<<<nblocks(nv * 4, 256), 256, 0, s>>>(u, u1, u2, Y, oscale, sigma, nv, g);
    return hipGetLastError();
}

hipError_t launch_predict_target(const double* un1, const double* u, const double* u1, const double* u2,
                                 const float* oscale, const double* sigma, int64_t nv, float* T, hipStream_t s)
{
    if (nv <= 0) return hipSuccess;
    predict_target<<<nblocks(nv * 4, 256), 256, 0, s>>>(un1, u, u1, u2, oscale, sigma, nv, T);
    return hipGetLastError();
}

}  // namespace nsfv1
