// Autoregressive proposal network for the Metropolis independence sampler:
// forward, backward and optimiser kernels (bf16 weights, fp32 arithmetic).
//
// No counterpart in the reference.  The model proposes an output state of n
// photons over m modes as a non-decreasing sequence of modes s_0 <= ... <=
// s_{n-1}; step p sees the counts of the modes drawn so far and a one-hot of
// p (D = m + n inputs), and emits logits over the m modes, masked below
// s_{p-1}.  The sequence is unique per Fock state, so q(state) is exact.
//   h = relu(x W1^T + b1)  (hidden H),  logits = h W2^T + b2.
// Matrices are row-major; W1 is H x D and W2 is m x H, stored as bf16 for the
// products with fp32 master copies for the optimiser.
#include "common.h"
#include "../../include/pcvl_hip.h"

#include <algorithm>

namespace pcvl {

__device__ __forceinline__ float bf16_to_f32(uint16_t b)
{
    return __uint_as_float(((uint32_t)b) << 16);
}

__device__ __forceinline__ uint16_t f32_to_bf16(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);   // round to nearest even
    return (uint16_t)(u >> 16);
}

template <typename T> __device__ __forceinline__ float ld(const T *p, size_t i);
template <> __device__ __forceinline__ float ld<float>(const float *p, size_t i) { return p[i]; }
template <> __device__ __forceinline__ float ld<uint16_t>(const uint16_t *p, size_t i) { return bf16_to_f32(p[i]); }

// Y[i][j] = act(alpha * sum_k A(i,k) B(k,j) + bias[j]) (+ Y[i][j] if accumulate)
// with A(i,k) = A[i*sai + k*sak], B(k,j) = B[k*sbk + j*sbj].  64 x 64 output
// tile per 256-thread block, 16-deep K slices staged through LDS, 4 x 4
// outputs per thread.
constexpr int GT = 64, GK = 16;

template <typename TB>
__global__ void __launch_bounds__(256) gemm_kernel(const float *__restrict__ A, int64_t sai, int64_t sak,
                                                   const TB *__restrict__ B, int64_t sbk, int64_t sbj,
                                                   float *__restrict__ Y, int64_t ldy, int M, int N, int K,
                                                   const float *__restrict__ bias, int relu, int accumulate)
{
    __shared__ float As[GK][GT + 1];
    __shared__ float Bs[GK][GT + 1];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int i0 = blockIdx.y * GT, j0 = blockIdx.x * GT;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += GK) {
        for (int e = threadIdx.x; e < GK * GT; e += 256) {
            const int kk = e / GT, ii = e % GT;
            const int i = i0 + ii, k = k0 + kk;
            As[kk][ii] = (i < M && k < K) ? A[i * sai + k * sak] : 0.0f;
            const int j = j0 + ii;
            Bs[kk][ii] = (j < N && k < K) ? ld<TB>(B, (size_t)(k * sbk + j * sbj)) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GK; kk++) {
            float a[4], b[4];
#pragma unroll
            for (int r = 0; r < 4; r++) a[r] = As[kk][ty + 16 * r];
#pragma unroll
            for (int c = 0; c < 4; c++) b[c] = Bs[kk][tx + 16 * c];
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int c = 0; c < 4; c++) acc[r][c] = fmaf(a[r], b[c], acc[r][c]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int i = i0 + ty + 16 * r;
        if (i >= M) continue;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int j = j0 + tx + 16 * c;
            if (j >= N) continue;
            float v = acc[r][c];
            if (bias) v += bias[j];
            if (accumulate) v += Y[(size_t)i * ldy + j];
            if (relu) v = v > 0.0f ? v : 0.0f;
            Y[(size_t)i * ldy + j] = v;
        }
    }
}

// Weight gradient over a long row dimension, split deterministically:
//   part[s][i][j] = sum_{r in split s} dY[r][i] * Xe[r][j],  j < No + 1,
// with Xe = [X | 1], so column No of the result is db = colsum(dY).  Split s
// covers rows [s*rows_per, min(R, (s+1)*rows_per)); the second kernel sums
// the splits in order, so the result does not depend on the launch.
constexpr int WG_ROWS = 16;

__global__ void __launch_bounds__(256) wgrad_partial_kernel(const float *__restrict__ dY, int64_t ldd,
                                                            const float *__restrict__ X, int64_t ldx, int R,
                                                            int Mo, int No, int rows_per, float *__restrict__ part)
{
    __shared__ float As[WG_ROWS][GT + 1];
    __shared__ float Bs[WG_ROWS][GT + 1];
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int i0 = blockIdx.y * GT, j0 = blockIdx.x * GT;
    const int split = blockIdx.z;
    const int r0 = split * rows_per;
    const int r1 = min(R, r0 + rows_per);
    const int Ne = No + 1;
    float acc[4][4] = {};
    for (int rb = r0; rb < r1; rb += WG_ROWS) {
        for (int e = threadIdx.x; e < WG_ROWS * GT; e += 256) {
            const int kk = e / GT, ii = e % GT;
            const int r = rb + kk;
            const bool rv = r < r1;
            const int i = i0 + ii, j = j0 + ii;
            As[kk][ii] = (rv && i < Mo) ? dY[(size_t)r * ldd + i] : 0.0f;
            Bs[kk][ii] = (rv && j < No) ? X[(size_t)r * ldx + j] : ((rv && j == No) ? 1.0f : 0.0f);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < WG_ROWS; kk++) {
            float a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) a[q] = As[kk][ty + 16 * q];
#pragma unroll
            for (int c = 0; c < 4; c++) b[c] = Bs[kk][tx + 16 * c];
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int c = 0; c < 4; c++) acc[q][c] = fmaf(a[q], b[c], acc[q][c]);
        }
        __syncthreads();
    }
    float *P = part + (size_t)split * Mo * Ne;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int i = i0 + ty + 16 * q;
        if (i >= Mo) continue;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int j = j0 + tx + 16 * c;
            if (j < Ne) P[(size_t)i * Ne + j] = acc[q][c];
        }
    }
}

__global__ void wgrad_reduce_kernel(const float *__restrict__ part, int splits, int Mo, int No,
                                    float *__restrict__ dW, float *__restrict__ db)
{
    const int Ne = No + 1;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)Mo * Ne) return;
    float s = 0.0f;
    for (int k = 0; k < splits; k++) s += part[(size_t)k * Mo * Ne + e];
    const int i = (int)(e / Ne), j = (int)(e % Ne);
    if (j < No) {
        if (dW) dW[(size_t)i * No + j] = s;
    } else if (db) {
        db[i] = s;
    }
}

// dH *= (H > 0)
__global__ void relu_bwd_kernel(float *__restrict__ dH, const float *__restrict__ H, int64_t count)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < count && !(H[e] > 0.0f)) dH[e] = 0.0f;
}

// db[j] = sum_i dY[i][j]: 64 columns per block, four row groups combined in
// a fixed order (coalesced rows; for long row counts use the weight-gradient
// kernels, which split the rows over many blocks).
__global__ void __launch_bounds__(256) colsum_kernel(const float *__restrict__ dY, int M, int N, float *__restrict__ db)
{
    __shared__ float part[4][64];
    const int c = threadIdx.x % 64, g = threadIdx.x / 64;
    const int j = blockIdx.x * 64 + c;
    float s = 0.0f;
    if (j < N)
        for (int i = g; i < M; i += 4) s += dY[(size_t)i * N + j];
    part[g][c] = s;
    __syncthreads();
    if (g == 0 && j < N) db[j] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

// Masked softmax cross-entropy of row i with target t[i], modes < lo[i]
// masked: loss[i] = -log q(t | row); dlogits = (softmax - onehot) * scale.
__global__ void ce_kernel(const float *__restrict__ logits, int M, int m, const int32_t *__restrict__ target,
                          const int32_t *__restrict__ lo, float scale, float *__restrict__ loss,
                          float *__restrict__ dlogits)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    const float *z = logits + (size_t)i * m;
    const int l0 = lo[i];
    const int t = target[i];
    if (t < l0 || t >= m || l0 < 0) {   // target outside the allowed modes: q = 0
        loss[i] = __int_as_float(0x7f800000);
        if (dlogits)
            for (int j = 0; j < m; j++) dlogits[(size_t)i * m + j] = 0.0f;
        return;
    }
    float mx = -3.0e38f;
    for (int j = l0; j < m; j++) mx = fmaxf(mx, z[j]);
    float se = 0.0f;
    for (int j = l0; j < m; j++) se += __expf(z[j] - mx);
    const float lse = mx + __logf(se);
    loss[i] = lse - z[t];
    if (dlogits) {
        float *d = dlogits + (size_t)i * m;
        for (int j = 0; j < m; j++) {
            const float p = (j >= l0) ? __expf(z[j] - lse) : 0.0f;
            d[j] = (p - (j == t ? 1.0f : 0.0f)) * scale;
        }
    }
}

// ---- loss and gradients in one launch ------------------------------------------
//
// The five products of a training step (h, logits, dh and the two weight
// gradients) on v_mfma_f32_16x16x4_f32, one workgroup of 8 waves per CU.  A
// workgroup walks over tiles of 32 rows; h, the logits and dh never leave the
// CU, and the weight gradients stay in accumulator registers over all of its
// tiles, so a pass reads x once and writes one partial gradient per workgroup.
//
// Wave w owns hidden columns 32w .. 32w + 31.  An MFMA lane (c16 = lane % 16,
// g = lane / 16) takes its four k values of a 16-deep slice as k = 4g + c, c =
// 0..3, one per instruction; with that order the result tile of one product
// (rows 4g + c, column c16) is already the operand of the products that sum
// over its rows, so h and dh go into the weight gradients from the registers
// that they were made in.  Only the logits sum over hidden columns: h crosses
// LDS once for them.  The weights stay in registers as bf16 pairs.
//   1. h[r][h]  = relu(x W1^T + b1)    K = D    -> registers and LDS
//   2. z[r][j]  = h W2^T + b2          K = H    one 16 x 16 tile per wave -> LDS
//   3. softmax, loss, dz               16 lanes per row, dz over z in LDS
//   4. dh[r][h] = (dz W2) (h > 0)      K = m
//   5. dW2 += dz^T h, dW1 += dh^T x    K = 32 rows
// Three barriers a tile; x of the next tile is loaded during this one.
// Sizes up to D = 96, H = 256, m = 64 (what the registers hold); shorter ones
// are padded with zeros, larger networks take the kernels above.
// Measured at 40,960 rows, D = 80, H = 256, m = 60: 84 us and 7 for the sum of
// the partials, against 468 us in eight launches (products 62 each, weight
// gradients 80 and their sums 32 each, softmax 38, ReLU 20) that passed h and
// dh, 42 MB each, through memory; a whole training step 490 -> 92 us.  What
// bounds it: the FP32 matrix unit, busy 53% of the kernel and 70% of a tile
// (13.3 us; 352 MFMAs of 32 cycles a wave are 9.4), then the 38 MB of partials.
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int TG_ROWS = 32;
constexpr int TG_H = 256, TG_M = 64, TG_DT = 6;   // D in 16s
constexpr int TG_THREADS = 512;
constexpr int TG_BLOCKS = 256;                    // one workgroup per CU
constexpr int TG_HS = TG_H + 4, TG_ZS = TG_M + 4; // row strides in LDS, conflict-free in 16-byte and 4-byte reads
constexpr int tg_xs(int dt) { return 16 * dt + 4; }
constexpr size_t tg_lds(int dt)
{
    const size_t tiles = sizeof(float) * TG_ROWS * (2 * tg_xs(dt) + TG_HS + TG_ZS);
    const size_t weights = sizeof(uint16_t) * (TG_H * tg_xs(dt) + TG_M * TG_HS);   // staged there first
    return tiles > weights ? tiles : weights;
}

// f4 entries of one workgroup's partial gradients
constexpr __host__ __device__ int tg_part(int dt) { return TG_THREADS * (2 * dt + 8) + (TG_H + TG_M) / 4; }

template <int CTRL>
__device__ __forceinline__ float row_dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

__device__ __forceinline__ float row_max(float v)   // over 16 lanes
{
    v = fmaxf(v, row_dpp<0xB1>(v));
    v = fmaxf(v, row_dpp<0x4E>(v));
    v = fmaxf(v, row_dpp<0x141>(v));
    return fmaxf(v, row_dpp<0x140>(v));
}

__device__ __forceinline__ float row_sum(float v)
{
    v += row_dpp<0xB1>(v);
    v += row_dpp<0x4E>(v);
    v += row_dpp<0x141>(v);
    return v + row_dpp<0x140>(v);
}

__device__ __forceinline__ f4 unpack4(uint2 v)
{
    // in the loop's registers the weights stay packed: the compiler must not unpack them ahead of it
    asm volatile("" : "+v"(v.x), "+v"(v.y));
    return f4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
              __uint_as_float(v.y & 0xffff0000u)};
}

#define TG_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0)

template <int DT>
__global__ void __launch_bounds__(TG_THREADS, 2) train_grads_kernel(
    const float *__restrict__ x, int R, int D, const uint16_t *__restrict__ W1, const float *__restrict__ b1, int H,
    const uint16_t *__restrict__ W2, const float *__restrict__ b2, int m, const int32_t *__restrict__ target,
    const int32_t *__restrict__ lo, float scale, float *__restrict__ loss, float *__restrict__ part)
{
    constexpr int XS = tg_xs(DT);
    extern __shared__ float s_tg[];
    float *xs = s_tg, *xn = xs + TG_ROWS * XS;       // this tile's rows of x and the next one's
    float *hs = xn + TG_ROWS * XS, *zs = hs + TG_ROWS * TG_HS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c16 = lane & 15, g = lane >> 4;
    const int h0 = 32 * wave;
    const int rt = wave & 1, jt0 = wave >> 1;        // this wave's tile of the logits

    uint2 w1[2][DT], w2k[TG_H / 16], w2j[2][TG_M / 16];
    {
        uint16_t *s1 = reinterpret_cast<uint16_t *>(s_tg), *s2 = s1 + TG_H * XS;
        constexpr int N1 = TG_H * 16 * DT / TG_THREADS, N2 = TG_M * TG_H / TG_THREADS;
        uint32_t v1[N1], v2[N2];
#pragma unroll
        for (int u = 0; u < N1; u++) {
            const int e = tid + TG_THREADS * u, h = e / (16 * DT), d = e % (16 * DT);
            v1[u] = W1[h < H && d < D ? h * D + d : 0];
        }
#pragma unroll
        for (int u = 0; u < N2; u++) {
            const int e = tid + TG_THREADS * u, j = e / TG_H, h = e % TG_H;
            v2[u] = W2[j < m && h < H ? j * H + h : 0];
        }
        __builtin_amdgcn_sched_barrier(0);   // every load is issued before the first store waits for one
#pragma unroll
        for (int u = 0; u < N1; u++) {
            const int e = tid + TG_THREADS * u, h = e / (16 * DT), d = e % (16 * DT);
            s1[h * XS + d] = (uint16_t)(h < H && d < D ? v1[u] : 0u);
        }
#pragma unroll
        for (int u = 0; u < N2; u++) {
            const int e = tid + TG_THREADS * u, j = e / TG_H, h = e % TG_H;
            s2[j * TG_HS + h] = (uint16_t)(j < m && h < H ? v2[u] : 0u);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int h = h0 + 16 * t + c16;
#pragma unroll
            for (int q = 0; q < DT; q++) w1[t][q] = *reinterpret_cast<const uint2 *>(s1 + h * XS + 16 * q + 4 * g);
#pragma unroll
            for (int q = 0; q < TG_M / 16; q++) {
                const uint16_t *c = s2 + (16 * q + 4 * g) * TG_HS + h;
                w2j[t][q].x = (uint32_t)c[0] | (uint32_t)c[TG_HS] << 16;
                w2j[t][q].y = (uint32_t)c[2 * TG_HS] | (uint32_t)c[3 * TG_HS] << 16;
            }
        }
#pragma unroll
        for (int q = 0; q < TG_H / 16; q++)
            w2k[q] = *reinterpret_cast<const uint2 *>(s2 + (16 * jt0 + c16) * TG_HS + 16 * q + 4 * g);
        __syncthreads();
    }
    float bias1[2];
#pragma unroll
    for (int t = 0; t < 2; t++) bias1[t] = h0 + 16 * t + c16 < H ? b1[h0 + 16 * t + c16] : 0.0f;
    const float bias2 = 16 * jt0 + c16 < m ? b2[16 * jt0 + c16] : 0.0f;

    f4 dw1[2][DT], dw2[TG_M / 16][2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int q = 0; q < DT; q++) dw1[t][q] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < TG_M / 16; q++) dw2[q][t] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    float db1[2] = {0.0f, 0.0f};
    f4 db2 = {0.0f, 0.0f, 0.0f, 0.0f};

    const int tiles = (R + TG_ROWS - 1) / TG_ROWS;
    float xr[DT];
    auto load_x = [&](int tile) {
#pragma unroll
        for (int u = 0; u < DT; u++) {
            const int e = tid + TG_THREADS * u;
            const int r = tile * TG_ROWS + e / (16 * DT), d = e % (16 * DT);
            xr[u] = (r < R && d < D) ? x[(size_t)r * D + d] : 0.0f;
        }
    };
    auto store_x = [&](float *to) {
#pragma unroll
        for (int u = 0; u < DT; u++) {
            const int e = tid + TG_THREADS * u;
            to[e / (16 * DT) * XS + e % (16 * DT)] = xr[u];
        }
    };
    load_x(blockIdx.x);
    store_x(xs);
    __syncthreads();
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int r0 = tile * TG_ROWS;
        const bool more = tile + (int)gridDim.x < tiles;
        if (more) load_x(tile + gridDim.x);
        const int row = r0 + (tid >> 4);   // this thread's row in step 3
        const int l0 = row < R ? lo[row] : 0, t = row < R ? target[row] : -1;
        // 1. h
        f4 h[2][2];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 2; t++) h[a][t] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < DT; q++) {
            f4 av[2], bv[2];
#pragma unroll
            for (int a = 0; a < 2; a++) av[a] = *reinterpret_cast<const f4 *>(xs + (16 * a + c16) * XS + 16 * q + 4 * g);
#pragma unroll
            for (int t = 0; t < 2; t++) bv[t] = unpack4(w1[t][q]);
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int t = 0; t < 2; t++) h[a][t] = TG_MFMA(av[a][c], bv[t][c], h[a][t]);
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int r = 16 * a + 4 * g + c;
                    float v = h[a][t][c] + bias1[t];
                    v = (v > 0.0f && r0 + r < R) ? v : 0.0f;
                    h[a][t][c] = v;
                    hs[r * TG_HS + h0 + 16 * t + c16] = v;
                }
        __syncthreads();
        if (more) store_x(xn);
        // 2. logits
        {
            f4 z[2] = {f4{0.0f, 0.0f, 0.0f, 0.0f}, f4{0.0f, 0.0f, 0.0f, 0.0f}};
            const float *hr = hs + (16 * rt + c16) * TG_HS + 4 * g;
            f4 ah[3] = {*reinterpret_cast<const f4 *>(hr), *reinterpret_cast<const f4 *>(hr + 16)};
#pragma unroll
            for (int q = 0; q < TG_H / 16; q++) {
                // two reads ahead of the products that use them
                if (q + 2 < TG_H / 16) ah[(q + 2) % 3] = *reinterpret_cast<const f4 *>(hr + 16 * (q + 2));
                __builtin_amdgcn_sched_barrier(0);
                const f4 av = ah[q % 3];
                const f4 bv = unpack4(w2k[q]);
#pragma unroll
                for (int c = 0; c < 4; c++) z[c & 1] = TG_MFMA(av[c], bv[c], z[c & 1]);
            }
#pragma unroll
            for (int c = 0; c < 4; c++)
                zs[(16 * rt + 4 * g + c) * TG_ZS + 16 * jt0 + c16] = z[0][c] + z[1][c] + bias2;
        }
        __syncthreads();
        // 3. masked softmax cross-entropy (ce_kernel's rules), 16 lanes per row
        {
            const int sub = tid & 15;
            float *zr = zs + (tid >> 4) * TG_ZS + 4 * sub;
            const f4 z = *reinterpret_cast<const f4 *>(zr);
            const bool ok = t >= l0 && t < m && l0 >= 0;
            float mx = -3.0e38f;
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (4 * sub + u >= l0 && 4 * sub + u < m) mx = fmaxf(mx, z[u]);
            mx = row_max(mx);
            float se = 0.0f;
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (4 * sub + u >= l0 && 4 * sub + u < m) se += __expf(z[u] - mx);
            const float lse = mx + __logf(row_sum(se));
            f4 dz;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int j = 4 * sub + u;
                const float p = (j >= l0 && j < m) ? __expf(z[u] - lse) : 0.0f;
                dz[u] = ok ? (p - (j == t ? 1.0f : 0.0f)) * scale : 0.0f;
                if (ok && j == t) loss[row] = lse - z[u];
            }
            if (!ok && row < R && sub == 0) loss[row] = __int_as_float(0x7f800000);
            *reinterpret_cast<f4 *>(zr) = dz;
            db2 += dz;
        }
        __syncthreads();
        // 4. dh
        f4 dh[2][2];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 2; t++) dh[a][t] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < TG_M / 16; q++) {
            f4 av[2], bv[2];
#pragma unroll
            for (int a = 0; a < 2; a++)
                av[a] = *reinterpret_cast<const f4 *>(zs + (16 * a + c16) * TG_ZS + 16 * q + 4 * g);
#pragma unroll
            for (int t = 0; t < 2; t++) bv[t] = unpack4(w2j[t][q]);
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int t = 0; t < 2; t++) dh[a][t] = TG_MFMA(av[a][c], bv[t][c], dh[a][t]);
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float v = h[a][t][c] > 0.0f ? dh[a][t][c] : 0.0f;
                    dh[a][t][c] = v;
                    db1[t] += v;
                }
        // 5. weight gradients
#pragma unroll
        for (int a = 0; a < 2; a++) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float *zr = zs + (16 * a + 4 * g + c) * TG_ZS + c16;
#pragma unroll
                for (int q = 0; q < TG_M / 16; q++) {
                    const float dz = zr[16 * q];
#pragma unroll
                    for (int t = 0; t < 2; t++) dw2[q][t] = TG_MFMA(dz, h[a][t][c], dw2[q][t]);
                }
                const float *xrow = xs + (16 * a + 4 * g + c) * XS + c16;
#pragma unroll
                for (int q = 0; q < DT; q++) {
                    const float xv = xrow[16 * q];
#pragma unroll
                    for (int t = 0; t < 2; t++) dw1[t][q] = TG_MFMA(dh[a][t][c], xv, dw1[t][q]);
                }
            }
        }
        float *sw = xs;
        xs = xn;
        xn = sw;
    }
    // this workgroup's partial, as its lanes hold it: 2 DT + 8 accumulators of
    // four, [accumulator][thread]; db1 (256) | db2 (64) after them
    f4 *P = reinterpret_cast<f4 *>(part) + (size_t)blockIdx.x * tg_part(DT);
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int q = 0; q < DT; q++) P[(t * DT + q) * TG_THREADS + tid] = dw1[t][q];
#pragma unroll
        for (int q = 0; q < TG_M / 16; q++) P[(2 * DT + 2 * q + t) * TG_THREADS + tid] = dw2[q][t];
    }
    float *bias = reinterpret_cast<float *>(P + (2 * DT + 8) * TG_THREADS);
#pragma unroll
    for (int t = 0; t < 2; t++) {
        float s = db1[t];
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
        if (g == 0) bias[h0 + 16 * t + c16] = s;
    }
    __syncthreads();
    *reinterpret_cast<f4 *>(zs + (tid >> 4) * TG_ZS + 4 * (tid & 15)) = db2;
    __syncthreads();
    if (tid < TG_M) {
        float s = 0.0f;
        for (int r = 0; r < TG_ROWS; r++) s += zs[r * TG_ZS + tid];
        bias[TG_H + tid] = s;
    }
}

// Sum of the partials: 16 f4 entries per workgroup, 32 groups of partials
// summed side by side and combined in order.
__global__ void __launch_bounds__(512) train_reduce_kernel(const f4 *__restrict__ part, int parts, int H, int D, int dt,
                                                           int m, float *__restrict__ dW1, float *__restrict__ db1,
                                                           float *__restrict__ dW2, float *__restrict__ db2)
{
    __shared__ f4 s_sum[32][16];
    const int P = tg_part(dt);
    const int col = threadIdx.x & 15, grp = threadIdx.x >> 4;
    const int e = blockIdx.x * 16 + col;
    f4 s = {0.0f, 0.0f, 0.0f, 0.0f};
    if (e < P)
#pragma unroll 8
        for (int k = grp; k < parts; k += 32) s += part[(size_t)k * P + e];
    s_sum[grp][col] = s;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int f = blockIdx.x * 64 + threadIdx.x, c = f & 3;   // entry f: component c of f4 f / 4
    if (f >= 4 * P) return;
    const float *p = reinterpret_cast<const float *>(s_sum) + threadIdx.x;
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; k++) v += p[64 * k];
    const int acc = f / (4 * TG_THREADS), tid = (f >> 2) % TG_THREADS;
    const int c16 = tid & 15, row = 4 * ((tid >> 4) & 3) + c, h0 = 32 * (tid >> 6);
    if (acc < 2 * dt) {
        const int h = h0 + 16 * (acc / dt) + row, d = 16 * (acc % dt) + c16;
        if (h < H && d < D) dW1[(size_t)h * D + d] = v;
    } else if (acc < 2 * dt + 8) {
        const int j = 16 * ((acc - 2 * dt) / 2) + row, h = h0 + 16 * (acc & 1) + c16;
        if (j < m && h < H) dW2[(size_t)j * H + h] = v;
    } else {
        const int i = f - 4 * TG_THREADS * (2 * dt + 8);
        if (i < TG_H) {
            if (i < H) db1[i] = v;
        } else if (i - TG_H < m) {
            db2[i - TG_H] = v;
        }
    }
}

// Adam on fp32 master weights; writes the bf16 copy used by the products.
// Up to four tensors in one launch (a network's weights and biases), tensor
// blockIdx.y: at 5 us a launch each cost more than its work.
constexpr int ADAM_TENSORS = 4;
struct AdamTensors {
    float *w[ADAM_TENSORS];
    const float *g[ADAM_TENSORS];
    float *m1[ADAM_TENSORS], *m2[ADAM_TENSORS];
    uint16_t *wb[ADAM_TENSORS];
    int64_t count[ADAM_TENSORS];
};

__global__ void adam_kernel(AdamTensors T, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = blockIdx.y;
    if (e >= T.count[k]) return;
    float *w = T.w[k], *m1 = T.m1[k], *m2 = T.m2[k];
    const float *g = T.g[k];
    uint16_t *wb = T.wb[k];
    const float gg = g[e];
    const float a = b1 * m1[e] + (1.0f - b1) * gg;
    const float b = b2 * m2[e] + (1.0f - b2) * gg * gg;
    m1[e] = a;
    m2[e] = b;
    const float v = w[e] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    w[e] = v;
    if (wb) wb[e] = f32_to_bf16(v);
}

__global__ void to_bf16_kernel(const float *__restrict__ w, uint16_t *__restrict__ wb, int64_t count)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < count) wb[e] = f32_to_bf16(w[e]);
}

// Features of step p for each sequence row b: x = [counts of seq[b][0..p-1] | onehot(p)],
// and the mask bound lo[b] = seq[b][p-1] (0 at p = 0).
__global__ void features_kernel(const int32_t *__restrict__ seq, int B, int n, int m, int p,
                                float *__restrict__ x, int32_t *__restrict__ lo)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const int D = m + n;
    float *xb = x + (size_t)b * D;
    for (int j = 0; j < D; j++) xb[j] = 0.0f;
    for (int q = 0; q < p; q++) {
        const int j = seq[(size_t)b * n + q];
        if (j >= 0 && j < m) xb[j] += 1.0f;
    }
    xb[m + p] = 1.0f;
    const int l = p > 0 ? seq[(size_t)b * n + p - 1] : 0;
    lo[b] = (l >= 0 && l < m) ? l : 0;
}

// Teacher-forcing features for all (row, step) pairs of a batch of sorted
// sequences: row b*n + p.  Also writes the targets seq[b][p].  A workgroup per
// sequence, a thread per feature that keeps its count over the steps: rows are
// written contiguously (a thread per row wrote 64 rows at once, 4 bytes each:
// 32 us for 2,048 sequences of 20 photons in 60 modes against 5.7).
constexpr int FA_THREADS = 128;

__global__ void __launch_bounds__(FA_THREADS) features_all_kernel(const int32_t *__restrict__ seq, int B, int n, int m,
                                                                  float *__restrict__ x, int32_t *__restrict__ lo,
                                                                  int32_t *__restrict__ target)
{
    const int D = m + n;
    for (int b = blockIdx.x; b < B; b += gridDim.x) {
        const int32_t *s = seq + (size_t)b * n;
        for (int d = threadIdx.x; d < D; d += FA_THREADS) {
            float *xd = x + (size_t)b * n * D + d;
            float count = 0.0f;
            for (int p = 0; p < n; p++) {
                xd[(size_t)p * D] = d < m ? count : (d - m == p ? 1.0f : 0.0f);
                if (s[p] == d) count += 1.0f;
            }
        }
        for (int p = threadIdx.x; p < n; p += FA_THREADS) {
            const int l = p > 0 ? s[p - 1] : 0;
            lo[(size_t)b * n + p] = (l >= 0 && l < m) ? l : 0;
            target[(size_t)b * n + p] = s[p];   // validated by ce_kernel
        }
    }
}

// Draw step p of every row from the masked softmax of its logits; the uniform
// is the counter-based stream (seed, first + b, p).  Accumulates log q.
__global__ void sample_step_kernel(const float *__restrict__ logits, int B, int m, int n, int p,
                                   const int32_t *__restrict__ lo, uint64_t seed, uint64_t first,
                                   int32_t *__restrict__ seq, double *__restrict__ logq)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const float *z = logits + (size_t)b * m;
    const int l0 = lo[b];
    float mx = -3.0e38f;
    for (int j = l0; j < m; j++) mx = fmaxf(mx, z[j]);
    double se = 0.0;
    for (int j = l0; j < m; j++) se += exp((double)(z[j] - mx));
    const double target = uniform01(seed, first + (uint64_t)b, (uint64_t)p) * se;
    double cum = 0.0;
    int pick = m - 1;
    for (int j = l0; j < m; j++) {
        cum += exp((double)(z[j] - mx));
        if (target < cum) { pick = j; break; }
    }
    seq[(size_t)b * n + p] = pick;
    const double lp = (double)(z[pick] - mx) - log(se);
    logq[b] = (p == 0 ? 0.0 : logq[b]) + lp;
}

// All n autoregressive steps of a tile of proposals in one launch.  The first
// layer's input is [counts of the modes drawn so far | one-hot of the step],
// so its pre-activation is updated in place: + W1[:, drawn mode], and the
// one-hot column moves from m+p to m+p+1 (no GEMM, no HBM round trip).  The
// second layer runs from LDS (relu(h)^T in fp32, W2^T in bf16), each thread
// computing a 4-sample x 2-logit tile.  The draw is the masked softmax of the
// logits with the uniform (seed, first + b, p), done by the sample's 8
// threads: group max, group sum of exp (double), ordered partial sums for the
// inverse CDF; log q accumulates (z_pick - max) - log(sum) from the same
// logits, so q is exactly the law of the draw.
constexpr int FS_TB = 16;            // proposals per workgroup
constexpr int FS_THREADS = 128;      // 8 per proposal
constexpr int FS_MW = 64;            // logits padded to 64 modes
constexpr int FS_MAX_H = 256;
constexpr int FS_HPT = FS_MAX_H / 8; // h_pre entries per thread

__global__ void __launch_bounds__(FS_THREADS) sample_fused_kernel(
    const uint16_t *__restrict__ W1, const float *__restrict__ b1, const uint16_t *__restrict__ W2,
    const float *__restrict__ b2, int B, int m, int n, int H, uint64_t seed, uint64_t first,
    int32_t *__restrict__ seq, double *__restrict__ logq)
{
    extern __shared__ float s_fs[];
    float *hT = s_fs;                                           // H x TB
    float *zs = hT + (size_t)H * FS_TB;                         // TB x 64
    uint16_t *W2T = reinterpret_cast<uint16_t *>(zs + FS_TB * FS_MW);   // H x 64
    const int tid = threadIdx.x;
    const int D = m + n;
    for (int e = tid; e < H * FS_MW; e += FS_THREADS) {
        const int h = e / FS_MW, j = e % FS_MW;
        W2T[e] = j < m ? W2[(size_t)j * H + h] : (uint16_t)0;
    }
    // ownership for h_pre and the draw: proposal s, sub-thread sub
    const int s = tid >> 3, sub = tid & 7;
    const int64_t b = (int64_t)blockIdx.x * FS_TB + s;
    const bool valid = b < B;
    const int hpt = H / 8;
    float hp[FS_HPT];
#pragma unroll
    for (int t = 0; t < FS_HPT; t++) {
        const int h = sub + 8 * t;
        hp[t] = (t < hpt) ? b1[h] + bf16_to_f32(W1[(size_t)h * D + m]) : 0.0f;
    }
    // z tile: proposals 4*sq .. 4*sq+3, logits 2*jp, 2*jp+1
    const int sq = tid & 3, jp = tid >> 2;
    int lo = 0;
    double lq = 0.0;
    __syncthreads();
    for (int p = 0; p < n; p++) {
#pragma unroll
        for (int t = 0; t < FS_HPT; t++)
            if (t < hpt) hT[(sub + 8 * t) * FS_TB + s] = hp[t] > 0.0f ? hp[t] : 0.0f;
        __syncthreads();
        float acc[4][2] = {};
        for (int h = 0; h < H; h++) {
            const float4 hv = *reinterpret_cast<const float4 *>(hT + h * FS_TB + 4 * sq);
            const uint32_t w2 = *reinterpret_cast<const uint32_t *>(W2T + h * FS_MW + 2 * jp);
            const float w0 = __uint_as_float(w2 << 16), w1 = __uint_as_float(w2 & 0xffff0000u);
            acc[0][0] = fmaf(hv.x, w0, acc[0][0]); acc[0][1] = fmaf(hv.x, w1, acc[0][1]);
            acc[1][0] = fmaf(hv.y, w0, acc[1][0]); acc[1][1] = fmaf(hv.y, w1, acc[1][1]);
            acc[2][0] = fmaf(hv.z, w0, acc[2][0]); acc[2][1] = fmaf(hv.z, w1, acc[2][1]);
            acc[3][0] = fmaf(hv.w, w0, acc[3][0]); acc[3][1] = fmaf(hv.w, w1, acc[3][1]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int j = 2 * jp + c;
                zs[(4 * sq + r) * FS_MW + j] = j < m ? acc[r][c] + b2[j] : 0.0f;
            }
        __syncthreads();
        // draw of proposal s by its 8 threads; thread sub owns modes 8*sub .. 8*sub+7
        const float *z = zs + s * FS_MW;
        float mx = -3.0e38f;
        for (int u = 0; u < 8; u++) {
            const int j = 8 * sub + u;
            if (j >= lo && j < m) mx = fmaxf(mx, z[j]);
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        double ev[8];   // this thread's exp(z_j - mx), reused by the draw below
        double part = 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = 8 * sub + u;
            ev[u] = (j >= lo && j < m) ? exp((double)(z[j] - mx)) : 0.0;
            if (j >= lo && j < m) part += ev[u];
        }
        double se = part;
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) se += __shfl_xor(se, o, 64);
        // exclusive prefix of the partial sums in sub order
        double base = 0.0;
        for (int v = 0; v < 7; v++) {
            const double pv = __shfl(part, (tid & ~7) + v, 64);
            if (v < sub) base += pv;
        }
        const double target = uniform01(seed, first + (uint64_t)(valid ? b : 0), (uint64_t)p) * se;
        int cand = -1;
        if (target >= base || sub == 0) {
            double cum = base;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int j = 8 * sub + u;
                if (cand < 0 && j >= lo && j < m) {
                    cum += ev[u];
                    if (target < cum) cand = j;
                }
            }
            if (target < base) cand = -1;   // belongs to an earlier thread
        }
        // the first thread (in sub order) that holds the target; none -> last mode
        int pick = m - 1;
        for (int v = 7; v >= 0; v--) {
            const int cv = __shfl(cand, (tid & ~7) + v, 64);
            if (cv >= 0) pick = cv;
        }
        lq += (double)(z[pick] - mx) - log(se);
        if (valid && sub == 0) seq[b * n + p] = pick;
        lo = pick;
        // next pre-activation: + W1[:, pick], one-hot m+p -> m+p+1
#pragma unroll
        for (int t = 0; t < FS_HPT; t++) {
            if (t < hpt) {
                const size_t row = (size_t)(sub + 8 * t) * D;
                float v = hp[t] + bf16_to_f32(W1[row + pick]) - bf16_to_f32(W1[row + m + p]);
                if (p + 1 < n) v += bf16_to_f32(W1[row + m + p + 1]);
                hp[t] = v;
            }
        }
        __syncthreads();   // zs and hT are rewritten by the next step
    }
    if (valid && sub == 0) logq[b] = lq;
}

} // namespace pcvl

using namespace pcvl;

static int grid1(int64_t count) { return (int)((count + 255) / 256); }

extern "C" int pcvl_mlp_gemm(const float *d_A, int64_t sai, int64_t sak, const void *d_B, int b_is_bf16,
                             int64_t sbk, int64_t sbj, float *d_Y, int64_t ldy, int M, int N, int K,
                             const float *d_bias, int relu, int accumulate, hipStream_t stream)
{
    PCVL_ARG_CHECK(M >= 0 && N >= 0 && K >= 0, "negative GEMM size");
    if (M == 0 || N == 0) return OK;
    PCVL_ARG_CHECK(d_A && d_B && d_Y, "null device buffer");
    dim3 grid((N + GT - 1) / GT, (M + GT - 1) / GT);
    if (b_is_bf16) {
        hipLaunchKernelGGL(gemm_kernel<uint16_t>, grid, dim3(256), 0, stream, d_A, sai, sak,
                           static_cast<const uint16_t *>(d_B), sbk, sbj, d_Y, ldy, M, N, K, d_bias, relu, accumulate);
    } else {
        hipLaunchKernelGGL(gemm_kernel<float>, grid, dim3(256), 0, stream, d_A, sai, sak,
                           static_cast<const float *>(d_B), sbk, sbj, d_Y, ldy, M, N, K, d_bias, relu, accumulate);
    }
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

static int wgrad_splits(int R)
{
    int s = R / 256;
    return s < 1 ? 1 : (s > 128 ? 128 : s);
}

extern "C" int pcvl_mlp_wgrad_workspace(int R, int Mo, int No, int64_t *floats)
{
    PCVL_ARG_CHECK(floats != nullptr, "null output pointer");
    PCVL_ARG_CHECK(R >= 0 && Mo >= 0 && No >= 0, "negative size");
    *floats = (int64_t)wgrad_splits(R) * Mo * (No + 1);
    return OK;
}

extern "C" int pcvl_mlp_wgrad(const float *d_dY, int64_t ldd, const float *d_X, int64_t ldx, int R, int Mo, int No,
                              float *d_dW, float *d_db, float *d_work, int64_t work_floats, hipStream_t stream)
{
    PCVL_ARG_CHECK(R >= 0 && Mo >= 0 && No >= 0, "negative size");
    if (Mo == 0) return OK;
    PCVL_ARG_CHECK(d_dY && d_work && (No == 0 || d_X), "null device buffer");
    PCVL_ARG_CHECK(ldd >= Mo && (No == 0 || ldx >= No), "leading dimension below the row length");
    const int splits = wgrad_splits(R);
    PCVL_ARG_CHECK(work_floats >= (int64_t)splits * Mo * (No + 1), "workspace too small");
    const int rows_per = R > 0 ? (R + splits - 1) / splits : 0;
    dim3 grid((No + 1 + GT - 1) / GT, (Mo + GT - 1) / GT, splits);
    hipLaunchKernelGGL(wgrad_partial_kernel, grid, dim3(256), 0, stream, d_dY, ldd, d_X, ldx, R, Mo, No, rows_per,
                       d_work);
    PCVL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(grid1((int64_t)Mo * (No + 1))), dim3(256), 0, stream, d_work, splits,
                       Mo, No, d_dW, d_db);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mlp_relu_bwd(float *d_dH, const float *d_H, int64_t count, hipStream_t stream)
{
    if (count <= 0) return OK;
    hipLaunchKernelGGL(relu_bwd_kernel, dim3(grid1(count)), dim3(256), 0, stream, d_dH, d_H, count);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mlp_colsum(const float *d_dY, int M, int N, float *d_db, hipStream_t stream)
{
    if (N <= 0) return OK;
    hipLaunchKernelGGL(colsum_kernel, dim3((N + 63) / 64), dim3(256), 0, stream, d_dY, M, N, d_db);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mlp_ce(const float *d_logits, int M, int m, const int32_t *d_target, const int32_t *d_lo,
                           float scale, float *d_loss, float *d_dlogits, hipStream_t stream)
{
    if (M <= 0) return OK;
    hipLaunchKernelGGL(ce_kernel, dim3(grid1(M)), dim3(256), 0, stream, d_logits, M, m, d_target, d_lo, scale, d_loss,
                       d_dlogits);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mis_grads_workspace(int R, int m, int n, int H, int64_t *floats)
{
    PCVL_ARG_CHECK(floats != nullptr, "null output pointer");
    PCVL_ARG_CHECK(R >= 0 && m >= 0 && n >= 0 && H >= 0, "negative size");
    *floats = 0;
    if (m < 1 || n < 1 || H < 1 || m > TG_M || H > TG_H || m + n > 16 * TG_DT) return OK;
    const int64_t tiles = ((int64_t)R + TG_ROWS - 1) / TG_ROWS;
    *floats = std::max<int64_t>(1, std::min<int64_t>(tiles, TG_BLOCKS)) *
              4 * tg_part((m + n + 15) / 16);
    return OK;
}

template <int DT>
static int launch_train_grads(int dt, int grid, hipStream_t st, const float *x, int R, int D, const uint16_t *W1,
                              const float *b1, int H, const uint16_t *W2, const float *b2, int m,
                              const int32_t *target, const int32_t *lo, float scale, float *loss, float *part)
{
    if constexpr (DT > TG_DT) {
        set_error("internal: input width out of range");
        return ERR_ARG;
    } else {
        if (dt != DT)
            return launch_train_grads<DT + 1>(dt, grid, st, x, R, D, W1, b1, H, W2, b2, m, target, lo, scale, loss, part);
        hipLaunchKernelGGL(train_grads_kernel<DT>, dim3(grid), dim3(TG_THREADS), tg_lds(DT), st, x, R, D, W1, b1, H, W2,
                           b2, m, target, lo, scale, loss, part);
        PCVL_HIP_CHECK(hipGetLastError());
        return OK;
    }
}

extern "C" int pcvl_mis_grads(const float *d_x, int R, int m, int n, int H, const uint16_t *d_W1, const float *d_b1,
                              const uint16_t *d_W2, const float *d_b2, const int32_t *d_target, const int32_t *d_lo,
                              float scale, float *d_loss, float *d_dW1, float *d_db1, float *d_dW2, float *d_db2,
                              float *d_work, int64_t work_floats, hipStream_t stream)
{
    int64_t need = 0;
    const int rc = pcvl_mis_grads_workspace(R, m, n, H, &need);
    if (rc != OK) return rc;
    PCVL_ARG_CHECK(need > 0, "network empty or larger than 64 modes, 96 inputs or 256 hidden units");
    PCVL_ARG_CHECK(d_W1 && d_b1 && d_W2 && d_b2 && d_dW1 && d_db1 && d_dW2 && d_db2, "null device buffer");
    PCVL_ARG_CHECK(R == 0 || (d_x && d_target && d_lo && d_loss), "null device buffer");
    PCVL_ARG_CHECK(d_work && work_floats >= need, "workspace too small");
    PCVL_ARG_CHECK(reinterpret_cast<uintptr_t>(d_work) % 16 == 0, "workspace not aligned to 16 bytes");
    const int D = m + n;
    const int grid = (int)std::min<int64_t>(((int64_t)R + TG_ROWS - 1) / TG_ROWS, TG_BLOCKS);
    if (grid > 0) {
        const int lrc = launch_train_grads<1>((D + 15) / 16, grid, stream, d_x, R, D, d_W1, d_b1, H, d_W2, d_b2, m,
                                              d_target, d_lo, scale, d_loss, d_work);
        if (lrc != OK) return lrc;
    }
    const int dt = (D + 15) / 16;
    hipLaunchKernelGGL(train_reduce_kernel, dim3((tg_part(dt) + 15) / 16), dim3(512), 0, stream,
                       reinterpret_cast<const f4 *>(d_work), grid, H, D, dt, m, d_dW1, d_db1, d_dW2, d_db2);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mlp_adam_multi(int tensors, float *const *d_w, const float *const *d_g, float *const *d_m1,
                                   float *const *d_m2, uint16_t *const *d_wbf16, const int64_t *counts, float lr,
                                   float beta1, float beta2, float eps, int step, hipStream_t stream)
{
    PCVL_ARG_CHECK(step >= 1, "Adam step counts from 1");
    PCVL_ARG_CHECK(tensors >= 0 && tensors <= ADAM_TENSORS, "more than four tensors");
    PCVL_ARG_CHECK(tensors == 0 || (d_w && d_g && d_m1 && d_m2 && d_wbf16 && counts), "null table");
    const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    AdamTensors T = {};
    int64_t most = 0;
    for (int k = 0; k < tensors; k++) {
        PCVL_ARG_CHECK(counts[k] <= 0 || (d_w[k] && d_g[k] && d_m1[k] && d_m2[k]), "null device buffer");
        T.w[k] = d_w[k];
        T.g[k] = d_g[k];
        T.m1[k] = d_m1[k];
        T.m2[k] = d_m2[k];
        T.wb[k] = d_wbf16[k];
        T.count[k] = counts[k];
        most = std::max(most, counts[k]);
    }
    if (most <= 0) return OK;
    hipLaunchKernelGGL(adam_kernel, dim3(grid1(most), tensors), dim3(256), 0, stream, T, lr, beta1, beta2, eps, c1, c2);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mlp_adam(float *d_w, const float *d_g, float *d_m1, float *d_m2, uint16_t *d_wbf16, int64_t count,
                             float lr, float beta1, float beta2, float eps, int step, hipStream_t stream)
{
    return pcvl_mlp_adam_multi(1, &d_w, &d_g, &d_m1, &d_m2, &d_wbf16, &count, lr, beta1, beta2, eps, step, stream);
}

extern "C" int pcvl_mlp_to_bf16(const float *d_w, uint16_t *d_wbf16, int64_t count, hipStream_t stream)
{
    if (count <= 0) return OK;
    hipLaunchKernelGGL(to_bf16_kernel, dim3(grid1(count)), dim3(256), 0, stream, d_w, d_wbf16, count);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mis_features(const int32_t *d_seq, int B, int n, int m, int p, float *d_x, int32_t *d_lo,
                                 hipStream_t stream)
{
    PCVL_ARG_CHECK(p >= 0 && p < n, "step outside [0, n)");
    if (B <= 0) return OK;
    hipLaunchKernelGGL(features_kernel, dim3(grid1(B)), dim3(256), 0, stream, d_seq, B, n, m, p, d_x, d_lo);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mis_features_all(const int32_t *d_seq, int B, int n, int m, float *d_x, int32_t *d_lo,
                                     int32_t *d_target, hipStream_t stream)
{
    if (B <= 0) return OK;
    hipLaunchKernelGGL(features_all_kernel, dim3(B < 65536 ? B : 65536), dim3(FA_THREADS), 0, stream, d_seq, B, n, m,
                       d_x, d_lo, d_target);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mis_sample_fused(const uint16_t *d_W1, const float *d_b1, const uint16_t *d_W2,
                                     const float *d_b2, int B, int m, int n, int H, uint64_t seed, uint64_t first,
                                     int32_t *d_seq, double *d_logq, hipStream_t stream)
{
    PCVL_ARG_CHECK(m >= 1 && m <= FS_MW && n >= 1 && H >= 8 && H <= FS_MAX_H && H % 8 == 0,
                   "fused sampler needs 1 <= m <= 64, n >= 1, 8 <= H <= 256, H % 8 == 0");
    if (B <= 0) return OK;
    PCVL_ARG_CHECK(d_W1 && d_b1 && d_W2 && d_b2 && d_seq && d_logq, "null device buffer");
    const size_t lds = sizeof(float) * ((size_t)H * FS_TB + FS_TB * FS_MW) + sizeof(uint16_t) * (size_t)H * FS_MW;
    const unsigned grid = (unsigned)(((int64_t)B + FS_TB - 1) / FS_TB);
    hipLaunchKernelGGL(sample_fused_kernel, dim3(grid), dim3(FS_THREADS), lds, stream, d_W1, d_b1, d_W2, d_b2, B, m, n,
                       H, seed, first, d_seq, d_logq);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mis_sample_step(const float *d_logits, int B, int m, int n, int p, const int32_t *d_lo,
                                    uint64_t seed, uint64_t first, int32_t *d_seq, double *d_logq, hipStream_t stream)
{
    PCVL_ARG_CHECK(p >= 0 && p < n, "step outside [0, n)");
    if (B <= 0) return OK;
    hipLaunchKernelGGL(sample_step_kernel, dim3(grid1(B)), dim3(256), 0, stream, d_logits, B, m, n, p, d_lo, seed,
                       first, d_seq, d_logq);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}
