// lee_mlp.hip -- the learned ground model: a small MLP (4 -> 64 -> 64 -> 64 -> 8, GELU) that
// maps ground parameters to the residues of the ground impedance's poles, trained and run on
// the GPU with BF16 MFMA products and FP32 accumulation, FP32 master weights and Adam.
//
// Every product of the network is one kernel, C[M x N] = A[M x K] B[K x N] with strided
// operands (forward: activations x weights^T; backward: dZ^T x activations and dZ x weights),
// one 64-lane wave per 16 x 16 tile of C, gfx950's v_mfma_f32_16x16x32_bf16 over K in steps
// of 32 (and v_mfma_f32_16x16x16_bf16 for a last step of 16 when K is an odd multiple of 16);
// the FP32 operands are rounded to BF16 (nearest even, NaN kept) as they are loaded.  Elementwise
// kernels do the bias, GELU and its derivative, the loss gradient, the bias sums and Adam.
// Training with batches of up to 64 rows runs whole steps in one kernel (k_train).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/lee_abi.h"

namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// FP32 -> BF16 bits, round to nearest even; a NaN stays a (quiet) NaN instead of rounding
// into the exponent field.
__device__ __forceinline__ short to_bf16(float x)
{
    unsigned u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (short)((u >> 16) | 0x0040u);
    u = u + 0x7fffu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}

// C(m, n) = sum_k A(m, k) B(k, n) [+ bias(n)]; A(m, k) = pa[m*am + k*ak], B(k, n) = pb[k*bk + n*bn].
// M, N, K multiples of 16.  Block: 4 waves, one 16x16 tile each.  With r = l % 16 and
// q = l / 16, lane l of a wave holds A(r, k0+8q .. k0+8q+7) and B(k0+8q .. +7, r) in a step of
// 32 (A(r, k0+4q .. +3), B(k0+4q .. +3, r) in a step of 16) and receives C(4q .. 4q+3, r).
__global__ __launch_bounds__(256) void k_gemm_bf16(const float *__restrict__ pa, long am, long ak,
                                                   const float *__restrict__ pb, long bk, long bn,
                                                   float *__restrict__ pc, long cm, const float *__restrict__ bias,
                                                   int M, int N, int K)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tiles_n = N >> 4;
    const int tile = blockIdx.x * 4 + wave;
    if (tile >= (M >> 4) * tiles_n) return;
    const int m0 = (tile / tiles_n) << 4, n0 = (tile % tiles_n) << 4;
    const int r = lane & 15, q = lane >> 4;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    int k0 = 0;
    for (; k0 + 32 <= K; k0 += 32) {
        v8s a, b;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int k = k0 + 8 * q + t;
            a[t] = to_bf16(pa[(long)(m0 + r) * am + (long)k * ak]);
            b[t] = to_bf16(pb[(long)k * bk + (long)(n0 + r) * bn]);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0, 0, 0);
    }
    if (k0 < K) {
        v4s a, b;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = k0 + 4 * q + t;
            a[t] = to_bf16(pa[(long)(m0 + r) * am + (long)k * ak]);
            b[t] = to_bf16(pb[(long)k * bk + (long)(n0 + r) * bn]);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int m = m0 + 4 * q + t, n = n0 + r;
        pc[(long)m * cm + n] = acc[t] + (bias ? bias[n] : 0.f);
    }
}

__device__ __forceinline__ float gelu(float x)
{
    const float c = 0.7978845608028654f;  // sqrt(2/pi)
    return 0.5f * x * (1.f + tanhf(c * (x + 0.044715f * x * x * x)));
}
__device__ __forceinline__ float gelu_d(float x)
{
    const float c = 0.7978845608028654f;
    const float u = c * (x + 0.044715f * x * x * x);
    const float th = tanhf(u);
    return 0.5f * (1.f + th) + 0.5f * x * (1.f - th * th) * c * (1.f + 3.f * 0.044715f * x * x);
}

__global__ void k_gelu(const float *z, float *a, long n)
{
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) a[t] = gelu(z[t]);
}
// dz = da * gelu'(z)
__global__ void k_gelu_back(const float *z, const float *da, float *dz, long n)
{
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x)
        dz[t] = da[t] * gelu_d(z[t]);
}
// loss gradient of the mean squared error over the valid rows (< n) and columns (< nout) of a
// [rows x ld] output: dy = 2 (y - t) / (n nout), zero elsewhere; loss partial sums per block
__global__ void k_mse_back(const float *y, const float *t, float *dy, int rows, int ld, int n, int nout, float *loss)
{
    __shared__ float part[256];
    float s = 0.f;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < (long)rows * ld; e += (long)gridDim.x * blockDim.x) {
        const int i = (int)(e / ld), j = (int)(e % ld);
        float g = 0.f;
        if (i < n && j < nout) {
            const float d = y[e] - t[(long)i * nout + j];
            s += d * d;
            g = 2.f * d / ((float)n * nout);
        }
        dy[e] = g;
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss[blockIdx.x] = part[0];
}
// db(n) = sum over rows of dz(row, n): one 64-lane wave per column, lanes stride the rows,
// then a butterfly over the wave
__global__ __launch_bounds__(256) void k_colsum(const float *dz, float *db, int rows, int cols)
{
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (n >= cols) return;
    float s = 0.f;
    for (int i = lane; i < rows; i += 64) s += dz[(long)i * cols + n];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) db[n] = s;
}
// Adam on FP32 parameters (m, v moments), step t (1-based)
__global__ void k_adam(float *w, const float *g, float *m, float *v, long n, float lr, float b1, float b2, float eps,
                       float c1, float c2)
{
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        const float gg = g[e];
        const float mm = b1 * m[e] + (1.f - b1) * gg;
        const float vv = b2 * v[e] + (1.f - b2) * gg * gg;
        m[e] = mm;
        v[e] = vv;
        w[e] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    }
}

// ------------------------------------------------------------------------------------
// Training steps in one kernel: one workgroup of 16 waves runs `nsteps` whole steps (forward,
// loss, backward, Adam) of batches of up to 64 rows.
//
// A step by single products is 22 launches, two copies and two waits for the GPU: 150 us for
// 2 MFLOP in batches of 32; here 10 us (256 rows, 10 epochs: 12.2 -> 0.86 ms), bound by the
// vector instructions of one CU, half of them Adam's divisions and square roots.  Every step is eight phases between workgroup barriers: FP32 weights and
// Adam moments live in registers (a wave owns a 16 x 16 tile of each 64 x 64 matrix, and a
// quarter of the first or the last), their BF16 copies and the batch's activations in LDS,
// in the two orders the products read along K (16-byte reads, rows padded to 144 bytes).
// A batch of 64 takes 148 of the 160 KB, so larger batches keep the single products.  The same
// MFMA steps along K, the same order of every sum and the same elementwise expressions as the
// single kernels: the same bits.  The steps' batches come from host memory that the kernel
// reads one step ahead.
// ------------------------------------------------------------------------------------
constexpr int TR = 64, TW = 72, TN = 24;      // rows at most; shorts per 64-wide and per 16-wide row
constexpr int W0 = 0, B0 = 1024, W1 = 1088, B1 = 5184, W2 = 5248, B2 = 9344, W3 = 9408, B3 = 10432, NP = 10448;

struct TrainLds {
    short w0[64 * TN], w1[64 * TW], w2[64 * TW], w3[16 * TW];  // [out][in]
    short w1t[64 * TW], w2t[64 * TW], w3t[64 * TN];            // [in][out]
    short x[TR * TN], xt[16 * TW];                             // batch, [row][in] and [in][row]
    short h[2][TR * TW];                                       // activations, then dZ, [row][col]
    short at[3][64 * TW];                                      // activations [col][row]
    short dzt[2][64 * TW];                                     // dZ [col][row]
    short dy[TR * TN], dyt[16 * TW];
    v4f s[2][12][64], sy[4][64];                               // FP32 dZ and dY by tile and lane, for the bias sums
    float b[208], bm[208], bv[208];                            // biases and their moments
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "LDS of a workgroup");

// C tile from A(r, k) and B(k, r): a and b point at the lane's rows along K.
__device__ __forceinline__ v4f tile_mul(const short *a, const short *b, int q, int K)
{
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    int k0 = 0;
    for (; k0 + 32 <= K; k0 += 32)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, *(const v8s *)(a + k0 + 8 * q)),
                                                      __builtin_bit_cast(v8bf, *(const v8s *)(b + k0 + 8 * q)), acc, 0, 0, 0);
    if (k0 < K)
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*(const v4s *)(a + k0 + 4 * q), *(const v4s *)(b + k0 + 4 * q), acc, 0, 0, 0);
    return acc;
}
// Tile C(4q + t, r) as BF16 into [row][col] (p, stride ld; null: not kept) and [col][row] (pt).
__device__ __forceinline__ void tile_put(short *p, int ld, short *pt, int ldt, int r, int q, const float (&v)[4])
{
    v4s h;
#pragma unroll
    for (int t = 0; t < 4; ++t) h[t] = to_bf16(v[t]);
    if (p)
#pragma unroll
        for (int t = 0; t < 4; ++t) p[(4 * q + t) * ld + r] = h[t];
    if (pt) *(v4s *)(pt + r * ldt + 4 * q) = h;
}
// k_adam's update of one parameter
__device__ __forceinline__ void adam_one(float &w, float &m, float &v, float g, float lr, float c1, float c2)
{
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mm = b1 * m + (1.f - b1) * g;
    const float vv = b2 * v + (1.f - b2) * g * g;
    m = mm;
    v = vv;
    w -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
}
struct TrainTile {
    float w[4], m[4], v[4];
    __device__ __forceinline__ void load(const float *pw, const float *pm, const float *pv, int e, int ld)
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) { w[t] = pw[e + t * ld]; m[t] = pm[e + t * ld]; v[t] = pv[e + t * ld]; }
    }
    __device__ __forceinline__ void store(float *pw, float *pm, float *pv, int e, int ld) const
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) { pw[e + t * ld] = w[t]; pm[e + t * ld] = m[t]; pv[e + t * ld] = v[t]; }
    }
    __device__ __forceinline__ void adam(v4f g, float lr, float c1, float c2)
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) adam_one(w[t], m[t], v[t], g[t], lr, c1, c2);
    }
};
// Column sum of a tile column from its row tiles, in k_colsum's order: rows 32, 16, 8, 4, 2, 1 apart.
__device__ __forceinline__ float tile_colsum(v4f d0, v4f d1, v4f d2, v4f d3)
{
    float s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        s[t] = (d0[t] + d2[t]) + (d1[t] + d3[t]);
        s[t] += __shfl_xor(s[t], 32, 64);
        s[t] += __shfl_xor(s[t], 16, 64);
    }
    return (s[0] + s[2]) + (s[1] + s[3]);
}
// LDS visible to the workgroup; loads from memory stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// data: per step c1, c2 (Adam's bias corrections), x [batch][4], t [batch][8].  loss: partial
// sums of the last step's squared error per row tile, or null.
__global__ __launch_bounds__(1024) void k_train(float *__restrict__ pw, float *__restrict__ pm, float *__restrict__ pv,
                                                const float *__restrict__ data, int nsteps, int batch, float lr,
                                                float *__restrict__ loss)
{
    __shared__ TrainLds S;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int mt = wave >> 2, nt = wave & 3;
    const int R = (batch + 15) & ~15, rt = R >> 4;
    int r = lane & 15, q = lane >> 4;
    const bool act = mt < rt;                       // owns row tile mt, column tile nt of the activations
    const bool out = mt == nt && act;               // owns row tile mt of the output
    int col = 16 * nt + r, row = 16 * mt + 4 * q;
    // Before each phase: the compiler forms the phase's LDS addresses anew (a few instructions)
    // instead of keeping all of them across the loop, which takes the kernel past 128 registers
    // (71 spilled).
    auto phase = [&]() {
        int l = lane;
        asm("" : "+v"(l));
        r = l & 15; q = l >> 4;
        col = 16 * nt + r; row = 16 * mt + 4 * q;
    };
    const size_t stride = 2 + (size_t)batch * 12;

    for (int e = tid; e < TR * TN; e += 1024) S.x[e] = 0;
    for (int e = tid; e < 16 * TW; e += 1024) S.xt[e] = 0;
    // parameters: rows 16 mt + 4 q + t, column 16 nt + r of the 64 x 64 matrices; waves 8-11 a
    // column tile of the last, waves 12-15 a row tile of the first; waves 0-3 update the biases
    TrainTile p1, p2, p3;
    const int e1 = W1 + row * 64 + col, e2 = W2 + row * 64 + col;
    const int e3 = mt == 3 ? W0 + (16 * nt + 4 * q) * 16 + r : W3 + 4 * q * 64 + col, l3 = mt == 3 ? 16 : 64;
    p1.load(pw, pm, pv, e1, 64);
    p2.load(pw, pm, pv, e2, 64);
    tile_put(S.w1 + 16 * mt * TW + 16 * nt, TW, S.w1t + 16 * nt * TW + 16 * mt, TW, r, q, p1.w);
    tile_put(S.w2 + 16 * mt * TW + 16 * nt, TW, S.w2t + 16 * nt * TW + 16 * mt, TW, r, q, p2.w);
    if (mt >= 2) p3.load(pw, pm, pv, e3, l3);
    if (mt == 2) tile_put(S.w3 + 16 * nt, TW, S.w3t + 16 * nt * TN, TN, r, q, p3.w);
    if (mt == 3) tile_put(S.w0 + 16 * nt * TN, TN, nullptr, 0, r, q, p3.w);
    constexpr int eb[4] = {B0, B1, B2, B3};
    if (mt == 0 && q == 0)
#pragma unroll
        for (int l = 0; l < 4; ++l)
            if (l < 3 || nt == 0) {
                S.b[64 * l + col] = pw[eb[l] + col];
                S.bm[64 * l + col] = pm[eb[l] + col];
                S.bv[64 * l + col] = pv[eb[l] + col];
            }
    // the first batch
    const bool hasx = tid < batch * 4;
    float xc = hasx ? data[2 + tid] : 0.f, xn = 0.f, c1 = data[0], c2 = data[1], c1n = 1.f, c2n = 1.f;
    float tc[4] = {}, tn[4] = {};
    const bool hast = out && r < 8;
    auto targets = [&](const float *d, float (&t)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (hast && row + e < batch) t[e] = d[2 + 4 * batch + (row + e) * 8 + r];
    };
    targets(data, tc);
    __syncthreads();
    if (hasx) S.x[(tid >> 2) * TN + (tid & 3)] = to_bf16(xc);
    lds_barrier();

    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < nsteps; ++s) {
        if (s + 1 < nsteps) {
            const float *d = data + (size_t)(s + 1) * stride;
            if (hasx) xn = d[2 + tid];
            targets(d, tn);
            c1n = d[0]; c2n = d[1];
        }
        // hidden layers: a wave's tile of the activations and of GELU's derivative
        float gd[3][4];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            phase();
            if (act) {
                const v4f acc = l == 0 ? tile_mul(S.x + (16 * mt + r) * TN, S.w0 + col * TN, q, 16)
                                       : tile_mul(S.h[(l + 1) & 1] + (16 * mt + r) * TW, (l == 1 ? S.w1 : S.w2) + col * TW, q, 64);
                const float bias = S.b[64 * l + col];
                float a[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float z = acc[t] + bias, c = 0.7978845608028654f;
                    const float th = tanhf(c * (z + 0.044715f * z * z * z));
                    a[t] = 0.5f * z * (1.f + th);
                    gd[l][t] = 0.5f * (1.f + th) + 0.5f * z * (1.f - th * th) * c * (1.f + 3.f * 0.044715f * z * z);
                }
                tile_put(S.h[l & 1] + 16 * mt * TW + 16 * nt, TW, S.at[l] + 16 * nt * TW + 16 * mt, TW, r, q, a);
            }
            if (l == 1 && hasx) S.xt[(tid & 3) * TW + (tid >> 2)] = to_bf16(xc);
            lds_barrier();
        }
        // output and the loss gradient
        phase();
        if (out) {
            const v4f acc = tile_mul(S.h[0] + (16 * mt + r) * TW, S.w3 + r * TW, q, 64);
            const float bias = S.b[192 + r];
            float g[4], sq[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float z = acc[t] + bias;
                g[t] = sq[t] = 0.f;
                if (r < 8 && row + t < batch) {
                    const float d = z - tc[t];
                    sq[t] = d * d;
                    g[t] = 2.f * d / ((float)batch * 8);
                }
            }
            tile_put(S.dy + 16 * mt * TN, TN, S.dyt + 16 * mt, TW, r, q, g);
            S.sy[mt][lane] = v4f{g[0], g[1], g[2], g[3]};
            if (loss && s == nsteps - 1) {  // k_mse_back's order: a row tile is one of its blocks
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    sq[t] += __shfl_xor(sq[t], 32, 64);
                    sq[t] += __shfl_xor(sq[t], 16, 64);
                }
                float v = (sq[0] + sq[2]) + (sq[1] + sq[3]);
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
                if (lane == 0) loss[mt] = v;
            }
        }
        lds_barrier();
        // backward; phase l leaves dZ of layer l - 1, updates layer l's parameters and publishes
        // the weights that the phases before it have read for the last time
        v4f dz = zero;
#pragma unroll
        for (int l = 3; l >= 0; --l) {
            phase();
            const int cur = l == 1 ? 1 : 0;  // buffer of layer l's dZ (layers 2, 1, 0)
            v4f dn = zero;
            if (l > 0 && act) {
                const v4f da = l == 3 ? tile_mul(S.dy + (16 * mt + r) * TN, S.w3t + col * TN, q, 16)
                                      : tile_mul(S.h[l & 1 ? 0 : 1] + (16 * mt + r) * TW, (l == 2 ? S.w2t : S.w1t) + col * TW, q, 64);
                float v[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) v[t] = dn[t] = da[t] * gd[l - 1][t];
                const int nb = l == 2 ? 1 : 0;
                tile_put(l > 1 ? S.h[l & 1] + 16 * mt * TW + 16 * nt : nullptr, TW, S.dzt[nb] + 16 * nt * TW + 16 * mt, TW, r, q, v);
                if (mt > 0) S.s[nb][4 * (mt - 1) + nt][lane] = dn;
            }
            if (l == 3 && mt == 2) p3.adam(tile_mul(S.dyt + r * TW, S.at[2] + col * TW, q, R), lr, c1, c2);
            if (l == 2) p2.adam(tile_mul(S.dzt[cur] + (16 * mt + r) * TW, S.at[1] + col * TW, q, R), lr, c1, c2);
            if (l == 1) p1.adam(tile_mul(S.dzt[cur] + (16 * mt + r) * TW, S.at[0] + col * TW, q, R), lr, c1, c2);
            if (l == 0 && mt == 3) p3.adam(tile_mul(S.dzt[cur] + col * TW, S.xt + r * TW, q, R), lr, c1, c2);
            if (mt == 0 && (l < 3 || nt == 0)) {
                float db;
                if (l == 3)
                    db = tile_colsum(S.sy[0][lane], rt > 1 ? S.sy[1][lane] : zero, rt > 2 ? S.sy[2][lane] : zero, rt > 3 ? S.sy[3][lane] : zero);
                else
                    db = tile_colsum(dz, rt > 1 ? S.s[cur][nt][lane] : zero, rt > 2 ? S.s[cur][4 + nt][lane] : zero,
                                     rt > 3 ? S.s[cur][8 + nt][lane] : zero);
                if (q == 0) adam_one(S.b[64 * l + col], S.bm[64 * l + col], S.bv[64 * l + col], db, lr, c1, c2);
            }
            if (l == 2 && mt == 2) tile_put(S.w3 + 16 * nt, TW, S.w3t + 16 * nt * TN, TN, r, q, p3.w);
            if (l == 1) tile_put(S.w2 + 16 * mt * TW + 16 * nt, TW, S.w2t + 16 * nt * TW + 16 * mt, TW, r, q, p2.w);
            if (l == 0) {
                tile_put(S.w1 + 16 * mt * TW + 16 * nt, TW, S.w1t + 16 * nt * TW + 16 * mt, TW, r, q, p1.w);
                if (mt == 3) tile_put(S.w0 + 16 * nt * TN, TN, nullptr, 0, r, q, p3.w);
                if (hasx) S.x[(tid >> 2) * TN + (tid & 3)] = to_bf16(xn);
            }
            dz = dn;
            lds_barrier();
        }
        xc = xn;
        c1 = c1n; c2 = c2n;
#pragma unroll
        for (int t = 0; t < 4; ++t) tc[t] = tn[t];
    }
    p1.store(pw, pm, pv, e1, 64);
    p2.store(pw, pm, pv, e2, 64);
    if (mt >= 2) p3.store(pw, pm, pv, e3, l3);
    if (mt == 0 && q == 0)
#pragma unroll
        for (int l = 0; l < 4; ++l)
            if (l < 3 || nt == 0) {
                pw[eb[l] + col] = S.b[64 * l + col];
                pm[eb[l] + col] = S.bm[64 * l + col];
                pv[eb[l] + col] = S.bv[64 * l + col];
            }
}

unsigned blocks_for(long n) { long b = (n + 255) / 256; return (unsigned)(b > 4096 ? 4096 : (b ? b : 1)); }

}  // namespace

// ------------------------------------------------------------------------------------
// Network object
// ------------------------------------------------------------------------------------
struct lee_mlp {
    static constexpr int L = 4;
    int din[L] = {16, 64, 64, 64};    // padded inputs of each layer (4 real inputs)
    int dout[L] = {64, 64, 64, 16};   // padded outputs (8 real outputs)
    int n_in = 4, n_out = 8;
    hipStream_t stream = nullptr;
    std::string err;
    // parameters (FP32 master), gradients, Adam moments: one flat buffer each, layer offsets
    std::vector<long> woff, boff;
    long nparam = 0;
    float *w = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
    long step = 0;
    // activations for a batch capacity
    int cap = 0;
    float *x = nullptr, *t = nullptr, *dy = nullptr, *loss = nullptr;
    float *z[L] = {}, *a[L] = {}, *dz[L] = {}, *da[L] = {};
    std::vector<void *> allocs;
    // batches of the training kernel, in two host buffers of stage_cap floats
    float *stage[2] = {};
    hipEvent_t staged[2] = {};
    size_t stage_cap = 0;
    ~lee_mlp()
    {
        if (stream) (void)hipStreamSynchronize(stream);
        for (void *p : allocs) (void)hipFree(p);
        for (float *p : stage)
            if (p) (void)hipHostFree(p);
        for (hipEvent_t e : staged)
            if (e) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

int mlp_err(lee_mlp *n, int code, const std::string &m)
{
    if (n) n->err = m;
    return code;
}
#define MHIP(n, expr)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) return mlp_err((n), LEE_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

int mlp_alloc(lee_mlp *n, float **p, long count)
{
    void *q = nullptr;
    MHIP(n, hipMalloc(&q, (size_t)std::max(count, 1L) * sizeof(float)));
    MHIP(n, hipMemsetAsync(q, 0, (size_t)std::max(count, 1L) * sizeof(float), n->stream));
    n->allocs.push_back(q);
    *p = (float *)q;
    return LEE_OK;
}

// Give back a buffer of the batch (the stream must be idle).
void mlp_release(lee_mlp *n, float *&p)
{
    if (!p) return;
    for (auto it = n->allocs.begin(); it != n->allocs.end(); ++it)
        if (*it == (void *)p) {
            n->allocs.erase(it);
            break;
        }
    (void)hipFree(p);
    p = nullptr;
}

// Batch buffers for `rows` rows: kept while they are large enough; on growth the old set is
// freed and the new one sized with headroom (1.5x), so a run of growing batches reallocates
// a few times, not once per call.
int mlp_batch(lee_mlp *n, int rows)
{
    if (rows <= n->cap) return LEE_OK;
    int rc;
    const long want = n->cap > 0 ? std::max((long)rows, (long)n->cap * 3 / 2) : (long)rows;
    const int R = (int)((want + 15) / 16 * 16);
    MHIP(n, hipStreamSynchronize(n->stream));
    mlp_release(n, n->x); mlp_release(n, n->t); mlp_release(n, n->dy); mlp_release(n, n->loss);
    for (int l = 0; l < lee_mlp::L; ++l) {
        mlp_release(n, n->z[l]); mlp_release(n, n->a[l]); mlp_release(n, n->dz[l]); mlp_release(n, n->da[l]);
    }
    n->cap = 0;
    if ((rc = mlp_alloc(n, &n->x, (long)R * n->din[0])) || (rc = mlp_alloc(n, &n->t, (long)R * n->n_out)) ||
        (rc = mlp_alloc(n, &n->dy, (long)R * n->dout[lee_mlp::L - 1])) || (rc = mlp_alloc(n, &n->loss, 4096)))
        return rc;
    for (int l = 0; l < lee_mlp::L; ++l)
        if ((rc = mlp_alloc(n, &n->z[l], (long)R * n->dout[l])) || (rc = mlp_alloc(n, &n->a[l], (long)R * n->dout[l])) ||
            (rc = mlp_alloc(n, &n->dz[l], (long)R * n->dout[l])) || (rc = mlp_alloc(n, &n->da[l], (long)R * n->din[l])))
            return rc;
    n->cap = R;
    return LEE_OK;
}

// The two host buffers of the training kernel's batches: 64 steps each, the host packs one
// while the kernel runs the other.
constexpr int STAGE_STEPS = 64;
int mlp_stage(lee_mlp *n, int batch)
{
    const size_t want = STAGE_STEPS * (2 + (size_t)batch * 12) + TR / 16;  // and the loss partials
    for (hipEvent_t &e : n->staged)
        if (!e) MHIP(n, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (want <= n->stage_cap) return LEE_OK;
    MHIP(n, hipStreamSynchronize(n->stream));
    n->stage_cap = 0;
    for (float *&p : n->stage) {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        void *q = nullptr;
        MHIP(n, hipHostMalloc(&q, want * sizeof(float), hipHostMallocPortable));
        p = (float *)q;
    }
    n->stage_cap = want;
    return LEE_OK;
}

void gemm(lee_mlp *n, const float *A, long am, long ak, const float *B, long bk, long bn, float *C, long cm,
          const float *bias, int M, int N, int K)
{
    const int tiles = (M / 16) * (N / 16);
    hipLaunchKernelGGL(k_gemm_bf16, dim3((tiles + 3) / 4), dim3(256), 0, n->stream, A, am, ak, B, bk, bn, C, cm, bias, M, N, K);
}

// inputs [rows x n_in] (host) -> padded device batch
int mlp_load_x(lee_mlp *n, const float *x, int rows)
{
    const int R = (rows + 15) / 16 * 16;
    std::vector<float> h((size_t)R * n->din[0], 0.f);
    for (int i = 0; i < rows; ++i)
        for (int j = 0; j < n->n_in; ++j) h[(size_t)i * n->din[0] + j] = x[(size_t)i * n->n_in + j];
    MHIP(n, hipMemcpyAsync(n->x, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice, n->stream));
    MHIP(n, hipStreamSynchronize(n->stream));
    return LEE_OK;
}

void mlp_forward(lee_mlp *n, int R)
{
    const float *in = n->x;
    for (int l = 0; l < lee_mlp::L; ++l) {
        const float *W = n->w + n->woff[l], *b = n->w + n->boff[l];
        gemm(n, in, n->din[l], 1, W, 1, n->din[l], n->z[l], n->dout[l], b, R, n->dout[l], n->din[l]);
        const long cnt = (long)R * n->dout[l];
        if (l < lee_mlp::L - 1) {
            hipLaunchKernelGGL(k_gelu, dim3(blocks_for(cnt)), dim3(256), 0, n->stream, n->z[l], n->a[l], cnt);
            in = n->a[l];
        }
    }
}

// backward from dy (already in n->dy) into n->g
void mlp_backward(lee_mlp *n, int R)
{
    const float *dcur = n->dy;
    for (int l = lee_mlp::L - 1; l >= 0; --l) {
        const int o = n->dout[l], i = n->din[l];
        const float *dzl = n->dy;  // linear output layer: dZ = dY
        if (l < lee_mlp::L - 1) {
            const long cnt = (long)R * o;
            hipLaunchKernelGGL(k_gelu_back, dim3(blocks_for(cnt)), dim3(256), 0, n->stream, n->z[l], dcur, n->dz[l], cnt);
            dzl = n->dz[l];
        }
        const float *prev = l ? n->a[l - 1] : n->x;
        // dW [o x i] = dZ^T [o x R] * prev [R x i]
        gemm(n, dzl, 1, o, prev, i, 1, n->g + n->woff[l], i, nullptr, o, i, R);
        hipLaunchKernelGGL(k_colsum, dim3((o + 3) / 4), dim3(256), 0, n->stream, dzl, n->g + n->boff[l], R, o);
        if (l > 0) {
            // dA_prev [R x i] = dZ [R x o] * W [o x i]
            gemm(n, dzl, o, 1, n->w + n->woff[l], i, 1, n->da[l], i, nullptr, R, i, o);
            dcur = n->da[l];
        }
    }
}

// loss gradient for targets t [rows x n_out] (host); returns the mean squared error
int mlp_loss(lee_mlp *n, const float *t, int rows, double *mse)
{
    const int R = (rows + 15) / 16 * 16;
    MHIP(n, hipMemcpyAsync(n->t, t, (size_t)rows * n->n_out * sizeof(float), hipMemcpyHostToDevice, n->stream));
    const int last = lee_mlp::L - 1;
    const unsigned nb = 64;
    hipLaunchKernelGGL(k_mse_back, dim3(nb), dim3(256), 0, n->stream, n->z[last], n->t, n->dy, R, n->dout[last], rows,
                       n->n_out, n->loss);
    std::vector<float> part(nb);
    MHIP(n, hipMemcpyAsync(part.data(), n->loss, nb * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    MHIP(n, hipStreamSynchronize(n->stream));
    double s = 0;
    for (float v : part) s += v;
    if (mse) *mse = s / ((double)rows * n->n_out);
    return LEE_OK;
}

}  // namespace

extern "C" {

int lee_mlp_create(int device, unsigned long long seed, lee_mlp **out)
{
    if (!out) return LEE_ERR_ARG;
    *out = nullptr;
    std::unique_ptr<lee_mlp> n(new lee_mlp());
    lee_mlp *N = n.get();
    MHIP(N, hipSetDevice(device));
    MHIP(N, hipStreamCreateWithFlags(&N->stream, hipStreamNonBlocking));
    long off = 0;
    for (int l = 0; l < lee_mlp::L; ++l) {
        N->woff.push_back(off); off += (long)N->dout[l] * N->din[l];
        N->boff.push_back(off); off += N->dout[l];
    }
    N->nparam = off;
    int rc;
    if ((rc = mlp_alloc(N, &N->w, off)) || (rc = mlp_alloc(N, &N->g, off)) || (rc = mlp_alloc(N, &N->m1, off)) ||
        (rc = mlp_alloc(N, &N->m2, off)))
        return rc;
    // He-uniform initial weights over the real fan-in; padded rows and columns stay zero
    std::vector<float> h(off, 0.f);
    unsigned long long st = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto uni = [&]() {
        st = st * 6364136223846793005ULL + 1442695040888963407ULL;
        return (double)(st >> 11) * (1.0 / 9007199254740992.0);
    };
    const int real_in[lee_mlp::L] = {N->n_in, 64, 64, 64}, real_out[lee_mlp::L] = {64, 64, 64, N->n_out};
    for (int l = 0; l < lee_mlp::L; ++l) {
        const double lim = std::sqrt(6.0 / real_in[l]) * (l == lee_mlp::L - 1 ? 0.1 : 1.0);
        for (int o = 0; o < real_out[l]; ++o)
            for (int i = 0; i < real_in[l]; ++i) h[N->woff[l] + (long)o * N->din[l] + i] = (float)((2 * uni() - 1) * lim);
    }
    MHIP(N, hipMemcpyAsync(N->w, h.data(), off * sizeof(float), hipMemcpyHostToDevice, N->stream));
    MHIP(N, hipStreamSynchronize(N->stream));
    *out = n.release();
    return LEE_OK;
}

int lee_mlp_destroy(lee_mlp *n)
{
    delete n;
    return LEE_OK;
}

const char *lee_mlp_error(const lee_mlp *n) { return n ? n->err.c_str() : ""; }

long long lee_mlp_param_count(const lee_mlp *n) { return n ? n->nparam : 0; }

int lee_mlp_get_params(lee_mlp *n, float *w, long long cap)
{
    if (!n || !w || cap < n->nparam) return mlp_err(n, LEE_ERR_ARG, "buffer too small");
    MHIP(n, hipMemcpyAsync(w, n->w, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    MHIP(n, hipStreamSynchronize(n->stream));
    return LEE_OK;
}

int lee_mlp_set_params(lee_mlp *n, const float *w, long long count)
{
    if (!n || !w || count != n->nparam) return mlp_err(n, LEE_ERR_ARG, "parameter count mismatch");
    MHIP(n, hipMemcpyAsync(n->w, w, n->nparam * sizeof(float), hipMemcpyHostToDevice, n->stream));
    MHIP(n, hipStreamSynchronize(n->stream));
    return LEE_OK;
}

int lee_mlp_predict(lee_mlp *n, const float *x, int rows, float *y)
{
    if (!n || !x || !y || rows <= 0) return mlp_err(n, LEE_ERR_ARG, "bad arguments");
    int rc;
    if ((rc = mlp_batch(n, rows)) || (rc = mlp_load_x(n, x, rows))) return rc;
    const int R = (rows + 15) / 16 * 16, last = lee_mlp::L - 1;
    mlp_forward(n, R);
    std::vector<float> h((size_t)R * n->dout[last]);
    MHIP(n, hipMemcpyAsync(h.data(), n->z[last], h.size() * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    MHIP(n, hipStreamSynchronize(n->stream));
    for (int i = 0; i < rows; ++i)
        for (int j = 0; j < n->n_out; ++j) y[(size_t)i * n->n_out + j] = h[(size_t)i * n->dout[last] + j];
    return LEE_OK;
}

int lee_mlp_gradient(lee_mlp *n, const float *x, const float *t, int rows, float *grad, double *mse)
{
    if (!n || !x || !t || rows <= 0) return mlp_err(n, LEE_ERR_ARG, "bad arguments");
    int rc;
    if ((rc = mlp_batch(n, rows)) || (rc = mlp_load_x(n, x, rows))) return rc;
    const int R = (rows + 15) / 16 * 16;
    mlp_forward(n, R);
    if ((rc = mlp_loss(n, t, rows, mse))) return rc;
    mlp_backward(n, R);
    MHIP(n, hipGetLastError());
    if (grad) {
        MHIP(n, hipMemcpyAsync(grad, n->g, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
        MHIP(n, hipStreamSynchronize(n->stream));
    }
    return LEE_OK;
}

int lee_mlp_train(lee_mlp *n, const float *x, const float *t, int rows, int batch, int epochs, float lr,
                  unsigned long long seed, double *final_mse)
{
    if (!n || !x || !t || rows <= 0 || batch <= 0 || epochs < 0) return mlp_err(n, LEE_ERR_ARG, "bad arguments");
    batch = std::min(batch, rows);
    int rc;
    const bool fused = batch <= TR;  // what k_train's LDS holds
    if ((rc = fused ? mlp_stage(n, batch) : mlp_batch(n, batch))) return rc;
    std::vector<int> order(rows);
    for (int i = 0; i < rows; ++i) order[i] = i;
    unsigned long long st = seed + 0x9E3779B97F4A7C15ULL;
    const size_t stride = 2 + (size_t)batch * 12;
    std::vector<float> single(fused ? 0 : stride);
    const long steps = (long)epochs * (rows / batch);
    long done = 0;
    int buf = 0, held = 0;  // staging buffer in use, steps it holds
    double mse = 0;
    for (int ep = 0; ep < epochs; ++ep) {
        for (int i = rows - 1; i > 0; --i) {  // Fisher-Yates with a 64-bit LCG
            st = st * 6364136223846793005ULL + 1442695040888963407ULL;
            std::swap(order[i], order[(int)((st >> 33) % (unsigned long long)(i + 1))]);
        }
        for (int b0 = 0; b0 + batch <= rows; b0 += batch) {
            if (fused && held == 0) MHIP(n, hipEventSynchronize(n->staged[buf]));  // its last launch has read it
            float *d = fused ? n->stage[buf] + (size_t)held * stride : single.data();
            float *bx = d + 2, *bt = bx + (size_t)batch * n->n_in;
            for (int r = 0; r < batch; ++r) {
                std::memcpy(&bx[(size_t)r * n->n_in], &x[(size_t)order[b0 + r] * n->n_in], n->n_in * sizeof(float));
                std::memcpy(&bt[(size_t)r * n->n_out], &t[(size_t)order[b0 + r] * n->n_out], n->n_out * sizeof(float));
            }
            if (!fused && (rc = lee_mlp_gradient(n, bx, bt, batch, nullptr, &mse))) return rc;
            n->step += 1;
            ++done;
            const float b1 = 0.9f, b2 = 0.999f;
            const float c1 = 1.f - std::pow(b1, (float)n->step), c2 = 1.f - std::pow(b2, (float)n->step);
            if (!fused) {
                hipLaunchKernelGGL(k_adam, dim3(blocks_for(n->nparam)), dim3(256), 0, n->stream, n->w, n->g, n->m1, n->m2,
                                   (long)n->nparam, lr, b1, b2, 1e-8f, c1, c2);
                continue;
            }
            d[0] = c1;
            d[1] = c2;
            if (++held == STAGE_STEPS || done == steps) {
                float *loss = done == steps ? n->stage[buf] + STAGE_STEPS * stride : nullptr;
                hipLaunchKernelGGL(k_train, dim3(1), dim3(1024), 0, n->stream, n->w, n->m1, n->m2, n->stage[buf], held, batch,
                                   lr, loss);
                MHIP(n, hipGetLastError());
                MHIP(n, hipEventRecord(n->staged[buf], n->stream));
                if (loss) {
                    MHIP(n, hipStreamSynchronize(n->stream));
                    double sum = 0;
                    for (int b = 0; b < (batch + 15) / 16; ++b) sum += loss[b];
                    mse = sum / ((double)batch * n->n_out);
                }
                buf ^= 1;
                held = 0;
            }
        }
    }
    MHIP(n, hipStreamSynchronize(n->stream));
    if (final_mse) *final_mse = mse;
    return LEE_OK;
}

}  // extern "C"
