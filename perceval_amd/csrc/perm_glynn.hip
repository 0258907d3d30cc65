// Batched complex permanents by Glynn's formula in Gray-code order.
//
// Replaces xq.permanent_cx as called from NaiveBackend._compute_permanent
// (perceval/backends/_naive.py:70-71).  Glynn (2010):
//     perm(A) = 2^{-(n-1)} sum_{delta in {+-1}^n, delta_0 = +1} (prod_i delta_i) prod_j sum_i delta_i a_ij
// Step t of the binary-reflected Gray code flips row 1 + ctz(t); the sign of
// term t is (-1)^t.
//
// Work decomposition (orders 11..28): the 2^{n-1} terms of a matrix are cut
// into lane chunks of 2^c terms; one wavefront takes 64 consecutive chunks.
// The lowest one or two rows after row 0 are the low rows: a block of 2 or 4
// terms takes every low sign pattern, and the Gray code runs over the high
// rows, one flip per block.  Because a chunk starts at a multiple of 2^c,
// every lane flips the same high row at the same block, so the constants of a
// flip are wave-uniform; only its direction differs between lanes and is
// applied as a per-lane +-1 FMA.  The running sums are rebuilt from scratch at
// each chunk start, which bounds their drift to 2^(c-2) or 2^(c-1) updates.
// One persistent launch drains a cost-sorted queue of wave items of mixed
// order (largest first), then a second kernel sums each matrix's wave partials
// in a fixed order (bit-reproducible).  Orders 0..5 take a thread per matrix,
// 6..10 16 lanes.
#include "common.h"
#include "glynn_blocks.h"
#include "../../include/pcvl_hip.h"

#include <algorithm>
#include <numeric>
#include <cstring>
#include <new>
#include <mutex>
#include <vector>

namespace pcvl {

constexpr int PERM_WAVE_MIN = 11;
constexpr int PERM_WAVE_MAX = 28;   // the mixed-order launch
// Orders 29..32 run in a launch of their own (their registers would lower the
// occupancy of the mixed launch), from their own part of the queue.
constexpr int PERM_BIG_MIN = PERM_WAVE_MAX + 1;
constexpr int PERM_BIG_MAX = 32;
constexpr int PERM_THREAD_MAX = 5;  // a thread per matrix
constexpr int PERM_SMALL_MAX = 10;  // 16 lanes per matrix

struct PermItem {
    int64_t mat_off;   // complex offset of the matrix in the packed array
    uint32_t chunk0;   // first lane chunk of this wave
    int32_t slot;      // partial-sum slot written by this wave
    int32_t n;         // order
    int32_t c;         // log2 of Gray-code steps per lane
};

// --------------------------------------------------------------- wave path

// Low rows of an order: two up to order 24, one above.  A pair's state is 16
// VGPRs with two (T, T', E_1, E_2) and 12 with one, and two waves per SIMD
// leave 256: 22..24 spill 12..56 bytes and gain all the same, above the spills
// are inside the block loop.  Two -> one: 1,024 of order 21 3.40 -> 3.80 ms, 256 of
// 23 3.62 -> 3.94, 128 of 24 3.69 -> 3.99, 64 of 25 4.22 -> 4.19, 32 of 26 5.83 ->
// 4.38, 8 of 28 9.40 -> 5.09.
constexpr int PERM_LOW2_MAX = 24;
constexpr int perm_low_rows(int n, bool one) { return (n <= PERM_LOW2_MAX && !one) ? 2 : 1; }

// One wave item: 64 lanes x 2^c terms of one order-N matrix, in the column
// pairs of glynn_blocks.h.  Bound by FP64 issue: 4,096 order-20 matrices take
// 5.82 ms (8.00 ms with one update and product per column and term), 1,000 of
// orders 12..24 3.99 ms (5.22 ms).  The sums are updated once per block, so
// they drift less: error against direct float64 sums 3.3e-14 (9.9e-14) at
// order 20.
//
// sA is this wave's LDS slice (N x N).  High rows of the pair columns are
// overwritten with H_1 | H_2 (H_1 | unused); the rows of A that a flip adds to
// T come through the scalar cache, so the two constant streams (2 x 16 bytes
// per column and flip) use different paths: LDS alone would need 93% of its
// 128 B/clk at order 20.
template <int N, int LOW>
__device__ __forceinline__ cd glynn_wave_item(const double *__restrict__ mats, const PermItem &it, cd *sA)
{
    static_assert(N >= PERM_WAVE_MIN && (LOW == 1 || LOW == 2), "unsupported order or low rows");
    constexpr int P = N / 2;
    constexpr bool ODD = (N & 1) != 0;
    const int lane = threadIdx.x & 63;
    const cd *A = reinterpret_cast<const cd *>(mats) + it.mat_off;
    for (int e = lane; e < N * N; e += 64) sA[e] = A[e];
    __syncthreads();

    const int c = it.c;
    const uint32_t blocks = 1u << (c - LOW);
    const uint64_t base = (uint64_t)(it.chunk0 + (uint32_t)lane) << (c - LOW);   // in blocks of 2^LOW terms
    const uint64_t g0 = base ^ (base >> 1);

    // Column sums at low signs +1 and the high signs of Gray(base).
    cd T[N];
#pragma unroll
    for (int j = 0; j < N; j++) {
        T[j] = cadd(sA[j], sA[N + j]);
        if constexpr (LOW == 2) T[j] = cadd(T[j], sA[2 * N + j]);
        if (j & 1) asm volatile("" ::: "memory");   // a few reads in flight, not all rows in VGPRs
    }
#pragma unroll 1
    for (int i = LOW + 1; i < N; i++) {
        const double d = ((g0 >> (i - LOW - 1)) & 1) ? -1.0 : 1.0;
        const cd *row = sA + i * N;
#pragma unroll
        for (int j = 0; j < N; j++) {
            T[j].r = fma(d, row[j].r, T[j].r);
            T[j].i = fma(d, row[j].i, T[j].i);
        }
    }
    // 2 (s a'_r + s' a_r), s = T - a_r
    auto deriv = [&](int p, int r) {
        const cd a = sA[r * N + 2 * p], b = sA[r * N + 2 * p + 1];
        const cd s = {T[2 * p].r - a.r, T[2 * p].i - a.i}, t = {T[2 * p + 1].r - b.r, T[2 * p + 1].i - b.i};
        cd e = cmul(s, b);
        cfma_acc(e, t, a);
        return cd{2.0 * e.r, 2.0 * e.i};
    };
    cd E1[P], E2[LOW == 2 ? P : 1];
#pragma unroll
    for (int p = 0; p < P; p++) {
        E1[p] = deriv(p, 1);
        // formed here, not sunk past the barriers with every row it reads live
        asm volatile("" : "+v"(E1[p].r), "+v"(E1[p].i) : : "memory");
        if constexpr (LOW == 2) {
            E2[p] = deriv(p, 2);
            asm volatile("" : "+v"(E2[p].r), "+v"(E2[p].i) : : "memory");
        }
    }
    __syncthreads();
    // In place: H_1, H_2 over the pair columns of the high rows; with two low
    // rows G goes over row 0, and rows 1, 2 stay (2 a of an odd last column).
    auto pair_const = [&](int q, int r, int p) {
        const cd aq = sA[q * N + 2 * p], bq = sA[q * N + 2 * p + 1];
        const cd ar = sA[r * N + 2 * p], br = sA[r * N + 2 * p + 1];
        cd h = cmul(aq, br);
        cfma_acc(h, bq, ar);
        return cd{4.0 * h.r, 4.0 * h.i};
    };
    for (int e = lane; e < (N - 1 - LOW) * P; e += 64) {
        const int q = LOW + 1 + e / P, p = e % P;
        const cd h1 = pair_const(q, 1, p);
        cd h2 = h1;
        if constexpr (LOW == 2) h2 = pair_const(q, 2, p);
        sA[q * N + 2 * p] = h1;
        sA[q * N + 2 * p + 1] = h2;
    }
    if constexpr (LOW == 2) {
        if (lane < P) sA[lane] = pair_const(2, 1, lane);
    }
    __syncthreads();
    cd o1 = {0.0, 0.0}, o2 = {0.0, 0.0};   // 2 a_1, 2 a_2 of an odd last column
    if constexpr (ODD) {
        o1 = {2.0 * sA[N + N - 1].r, 2.0 * sA[N + N - 1].i};
        if constexpr (LOW == 2) o2 = {2.0 * sA[2 * N + N - 1].r, 2.0 * sA[2 * N + N - 1].i};
    }

    const cd sum = glynn_blocks<N, LOW, N, 2, false>(T, E1, E2, o1, o2, sA + (LOW + 1) * N, sA, blocks, base, [&](int b) {
        return (scalar_row)(uintptr_t)(A + (size_t)(b + LOW + 1) * N);
    });
    __syncthreads();   // sA is reused by the next item of this wave
    return sum;
}

__device__ __forceinline__ cd wave_sum(cd v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        v.r += __shfl_xor(v.r, off, 64);
        v.i += __shfl_xor(v.i, off, 64);
    }
    return v;
}

template <int NLO, int NHI, bool ONE>
__device__ __forceinline__ cd dispatch_item(const double *__restrict__ mats, const PermItem &it, cd *sA)
{
    if constexpr (NLO > NHI) {
        return {0.0, 0.0};
    } else {
        if (it.n == NLO) return glynn_wave_item<NLO, perm_low_rows(NLO, ONE)>(mats, it, sA);
        return dispatch_item<NLO + 1, NHI, ONE>(mats, it, sA);
    }
}

// Persistent wave kernel: one wavefront per workgroup, items pulled from a
// cost-sorted queue with an atomic cursor.  The cursor is returned to zero by
// perm_finalize so the same plan can be replayed (also inside a HIP graph).
template <int NLO, int NHI, bool ONE = false>
__global__ void __launch_bounds__(64, 2) perm_wave_kernel(const double *__restrict__ mats,
                                                       const PermItem *__restrict__ items,
                                                       const uint32_t *__restrict__ groups, int64_t ngroups,
                                                       unsigned long long *cursor, cd *__restrict__ partials)
{
    __shared__ cd sA[NHI * NHI];
    // A wave can take at most ngroups groups, so the loop is bounded whatever
    // the cursor holds; items whose order or chunk size lies outside what
    // this instantiation handles are skipped (their slot is left untouched).
    // The first group of a wave is its own, the others come from the cursor.
    uint64_t g = blockIdx.x;
    for (int64_t iter = 0; iter < ngroups && g < (uint64_t)ngroups; iter++) {
        const uint32_t lo = __builtin_amdgcn_readfirstlane(groups[g]), hi = __builtin_amdgcn_readfirstlane(groups[g + 1]);
        for (uint32_t ku = lo; ku < hi; ku++) {
            PermItem it;
            {
                const PermItem raw = items[ku];
                it.mat_off = (int64_t)(((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)raw.mat_off >> 32)) << 32) |
                                       __builtin_amdgcn_readfirstlane((uint32_t)raw.mat_off));
                it.chunk0 = __builtin_amdgcn_readfirstlane(raw.chunk0);
                it.slot = __builtin_amdgcn_readfirstlane(raw.slot);
                it.n = __builtin_amdgcn_readfirstlane(raw.n);
                it.c = __builtin_amdgcn_readfirstlane(raw.c);
            }
            if (it.n < NLO || it.n > NHI || it.c < 2 || it.c > it.n - 7) continue;
            cd v = dispatch_item<NLO, NHI, ONE>(mats, it, sA);
            v = wave_sum(v);
            if (threadIdx.x == 0) partials[it.slot] = v;
        }
        unsigned long long k = 0;
        if (threadIdx.x == 0) k = atomicAdd(cursor, 1ull);
        k = __shfl(k, 0, 64);
        // The group index and every field of an item are wave-uniform; say so,
        // so that loop control and LDS row addresses live in SGPRs.
        const uint32_t k_lo = __builtin_amdgcn_readfirstlane((uint32_t)k);
        const uint32_t k_hi = __builtin_amdgcn_readfirstlane((uint32_t)(k >> 32));
        g = gridDim.x + (((uint64_t)k_hi << 32) | k_lo);
    }
}

// --------------------------------------------------------------- small path

// Orders up to PERM_THREAD_MAX, one thread per matrix.
template <int N>
__device__ __forceinline__ cd glynn_thread(const cd *__restrict__ A)
{
    if constexpr (N == 0) {
        return {1.0, 0.0};
    } else {
        cd cs[N];
#pragma unroll
        for (int j = 0; j < N; j++) {
            cs[j] = A[j];
#pragma unroll
            for (int i = 1; i < N; i++) cs[j] = cadd(cs[j], A[i * N + j]);
        }
        cd acc = {0.0, 0.0};
#pragma unroll
        for (uint32_t t = 0; t < (1u << (N - 1)); t++) {
            if (t) {
                const int b = __builtin_ctz(t);
                const double d = ((t >> (b + 1)) & 1) ? 2.0 : -2.0;   // Gray bit b goes back, or on
#pragma unroll
                for (int j = 0; j < N; j++) {
                    const cd a = A[(b + 1) * N + j];
                    cs[j].r = fma(d, a.r, cs[j].r);
                    cs[j].i = fma(d, a.i, cs[j].i);
                }
            }
            cd p = cs[0];
#pragma unroll
            for (int j = 1; j < N; j++) p = cmul(p, cs[j]);
            if (t & 1) { acc.r -= p.r; acc.i -= p.i; } else { acc.r += p.r; acc.i += p.i; }
        }
        constexpr double sc = 1.0 / (1 << (N - 1));
        return {acc.r * sc, acc.i * sc};
    }
}

template <int N>
__device__ __forceinline__ cd dispatch_thread(int n, const cd *A)
{
    if constexpr (N > PERM_THREAD_MAX) {
        return {0.0, 0.0};
    } else {
        if (n == N) return glynn_thread<N>(A);
        return dispatch_thread<N + 1>(n, A);
    }
}

// Orders above, to PERM_SMALL_MAX, 16 lanes per matrix, A in LDS: lane bits sign rows 1..4, the
// remaining rows run through their Gray code with the column sums in registers.
template <int N>
__device__ __forceinline__ cd glynn_row(const cd *A, int lane)
{
    static_assert(N >= 5, "all 16 lanes take terms");
    constexpr int LB = 4;
    // unrolled, orders 9 and 10 keep rows in registers ahead of their use and spill
    constexpr int R = N <= 8 ? N : 3, S = N <= 8 ? 8 : 2;
    cd cs[N];
#pragma unroll
    for (int j = 0; j < N; j++) cs[j] = A[j];
#pragma unroll R
    for (int i = 1; i < N; i++) {
        const double d = i <= LB && ((lane >> (i - 1)) & 1) ? -1.0 : 1.0;
#pragma unroll
        for (int j = 0; j < N; j++) {
            const cd a = A[i * N + j];
            cs[j].r = fma(d, a.r, cs[j].r);
            cs[j].i = fma(d, a.i, cs[j].i);
        }
    }
    cd acc = {0.0, 0.0};
#pragma unroll S
    for (uint32_t t = 0; t < (1u << (N - 1 - LB)); t++) {
        if (t) {
            const int b = __builtin_ctz(t);
            const double d = ((t >> (b + 1)) & 1) ? 2.0 : -2.0;   // Gray bit b goes back, or on
#pragma unroll
            for (int j = 0; j < N; j++) {
                const cd a = A[(LB + 1 + b) * N + j];
                cs[j].r = fma(d, a.r, cs[j].r);
                cs[j].i = fma(d, a.i, cs[j].i);
            }
        }
        cd p = cs[0];
#pragma unroll
        for (int j = 1; j < N; j++) p = cmul(p, cs[j]);
        if (t & 1) { acc.r -= p.r; acc.i -= p.i; } else { acc.r += p.r; acc.i += p.i; }
    }
    if (__popc(lane) & 1) acc = {-acc.r, -acc.i};
    constexpr double sc = 1.0 / (1 << (N - 1));
    return {row_sum(acc.r) * sc, row_sum(acc.i) * sc};
}

template <int N>
__device__ __forceinline__ cd dispatch_row(int n, const cd *A, int lane)
{
    if constexpr (N > PERM_SMALL_MAX) {
        return {0.0, 0.0};
    } else {
        if (n == N) return glynn_row<N>(A, lane);
        return dispatch_row<N + 1>(n, A, lane);
    }
}

// The plan lists its small matrices by order; nthread of them go a thread each
// (workgroups below `first`), the others 16 lanes each.  Bound by launch and
// load latency at everyday counts (7 us from the caller).  Measured, a thread
// per matrix -> 16 lanes: 12,376 of order 6 18.4 -> 6.9 us, of order 8 118 ->
// 7.5 (column sums and rows of one thread spilled to scratch, 194 waves for 256
// CUs).  Orders 9 and 10 took a wave and an item of the queue each: 12,376 of
// order 9 202 -> 13.8, of order 10 252 -> 24.7, one of order 10 10.2 -> 9.3.
// PERM_THREAD_MAX: 100,000 of order 5 take 14 us a thread each and 54 in 16
// lanes, of order 6 65 and 23.  PERM_SMALL_MAX: 20,000 of order 11 are 112 us in
// the queue, and 16 lanes would do 64 terms each, ten times order 8's work.
constexpr int PERM_ROWS = 16;
constexpr int64_t PERM_ROW_LAUNCH = int64_t(1) << 22;   // matrices of one launch, milliseconds of work
constexpr int PERM_ROW_LD = PERM_SMALL_MAX * PERM_SMALL_MAX + 1;   // the four matrices of a wave on different banks

// nthread: the first matrix of 16 lanes in this launch; the ones before take a
// thread each in the first launch (first > 0).
__global__ void __launch_bounds__(16 * PERM_ROWS, 4) perm_small_kernel(
    const double *__restrict__ mats, const int64_t *__restrict__ idx, const int64_t *__restrict__ offs,
    const int32_t *__restrict__ ns, int64_t count, int64_t nthread, unsigned first, cd *__restrict__ out)
{
    __shared__ cd s_mat[PERM_ROWS * PERM_ROW_LD];
    if (blockIdx.x < first) {
        const int64_t k = (int64_t)blockIdx.x * (16 * PERM_ROWS) + threadIdx.x;
        if (k < nthread) out[idx[k]] = dispatch_thread<0>(ns[k], reinterpret_cast<const cd *>(mats) + offs[k]);
        return;
    }
    const int lane = threadIdx.x & 15, row = threadIdx.x >> 4;
    const int64_t k = nthread + (int64_t)(blockIdx.x - first) * PERM_ROWS + row;
    const bool in = k < count;
    const int n = in ? ns[k] : 0;
    cd *A = s_mat + row * PERM_ROW_LD;
    if (in) {
        const cd *M = reinterpret_cast<const cd *>(mats) + offs[k];
        for (int e = lane; e < n * n; e += 16) A[e] = M[e];
    }
    __syncthreads();
    const cd v = dispatch_row<PERM_THREAD_MAX + 1>(n, A, lane);
    if (in && lane == 0) out[idx[k]] = v;
}

// Sum each wave-path matrix's partials in slot order, scale by 2^{-(n-1)},
// and return the queue cursor to zero for the next replay.
__global__ void perm_finalize_kernel(const int64_t *__restrict__ idx, const int32_t *__restrict__ slot0,
                                     const int32_t *__restrict__ nslot, const int32_t *__restrict__ ns,
                                     int64_t count, const cd *__restrict__ partials, cd *__restrict__ out,
                                     unsigned long long *cursor)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) { cursor[0] = 0ull; cursor[1] = 0ull; }
    if (k >= count) return;
    cd s = {0.0, 0.0};
    for (int q = 0; q < nslot[k]; q++) s = cadd(s, partials[slot0[k] + q]);
    double sc = ldexp(1.0, -(ns[k] - 1));
    out[idx[k]] = {s.r * sc, s.i * sc};
}

// ------------------------------------------------------------------- plans

struct PermPlanImpl {
    int64_t count = 0;
    int64_t nitems = 0, nwave_mats = 0, nsmall = 0;
    int64_t nthread = 0;       // small matrices of a thread each, first in their list
    int64_t ngroups = 0, nbig_groups = 0;   // the queue's parts, below d_groups
    int64_t nbig = 0;          // items of orders 29..32, after the nitems others in the queue
    int grid_big = 0;
    int single_n = 0;          // order shared by every wave item, or 0 if mixed
    int variant = 0;           // 0, 1, 3: low rows by order; 2, 4 (single-order plans): one low row
    int grid = 0;
    PermItem *d_items = nullptr;
    uint32_t *d_groups = nullptr;   // first item of each group and the end: the queue of orders <= 28, then 29..32
    unsigned long long *d_cursor = nullptr;   // [0]: the queue of orders <= 28, [1]: orders 29..32
    cd *d_partials = nullptr;
    int64_t *d_wave_idx = nullptr;
    int32_t *d_wave_slot0 = nullptr, *d_wave_nslot = nullptr, *d_wave_n = nullptr;
    int64_t *d_small_idx = nullptr, *d_small_off = nullptr;
    int32_t *d_small_n = nullptr;
    void *d_block = nullptr;   // one allocation backing every array above
};

static int pick_chunk_log2(int n, int max_c)
{
    // 2^{n-1} steps = 2^{n-7} lane chunks of 2^{n-7-w} steps per wave when a
    // matrix is split over 2^w waves; take the longest chunk up to 2^max_c.
    int c = n - 7;
    if (c > max_c) c = max_c;
    if (c < 2) c = 2;
    return c;
}

template <int NLO, int NHI, bool ONE>
static int launch_wave(const PermPlanImpl *p, const double *mats, hipStream_t st, const uint32_t *groups,
                       int64_t ngroups, unsigned long long *cursor, int grid)
{
    hipLaunchKernelGGL((perm_wave_kernel<NLO, NHI, ONE>), dim3(grid), dim3(64), 0, st, mats, p->d_items, groups,
                       ngroups, cursor, p->d_partials);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

template <int NLO, int NHI, bool ONE>
static int launch_wave(const PermPlanImpl *p, const double *mats, hipStream_t st)
{
    return launch_wave<NLO, NHI, ONE>(p, mats, st, p->d_groups, p->ngroups, p->d_cursor, p->grid);
}

static bool perm_one_low_row(int variant) { return variant == 2 || variant == 4; }

template <int N>
static int launch_single(PermPlanImpl *p, const double *mats, hipStream_t st)
{
    if constexpr (N > PERM_WAVE_MAX) {
        set_error("internal: order out of range");
        return ERR_ARG;
    } else {
        if (p->single_n == N) {
            if constexpr (N <= PERM_LOW2_MAX) {
                if (perm_one_low_row(p->variant)) return launch_wave<N, N, true>(p, mats, st);
            }
            return launch_wave<N, N, false>(p, mats, st);
        }
        return launch_single<N + 1>(p, mats, st);
    }
}

template <int N>
static const void *single_kernel_ptr(int n, int variant)
{
    if constexpr (N > PERM_WAVE_MAX) {
        return nullptr;
    } else {
        if (n == N) {
            if constexpr (N <= PERM_LOW2_MAX) {
                if (perm_one_low_row(variant)) return reinterpret_cast<const void *>(&perm_wave_kernel<N, N, true>);
            }
            return reinterpret_cast<const void *>(&perm_wave_kernel<N, N, false>);
        }
        return single_kernel_ptr<N + 1>(n, variant);
    }
}

static int resident_waves(const void *kernel, int *out)
{
    int dev = 0, cus = 0, per_cu = 0;
    PCVL_HIP_CHECK(hipGetDevice(&dev));
    PCVL_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0));
    if (per_cu < 1) per_cu = 1;
    *out = cus * per_cu;
    return OK;
}

} // namespace pcvl

using namespace pcvl;

struct pcvl_perm_plan_s {
    PermPlanImpl impl;
};

// Work items above this count are refused (24 bytes each on the host and the
// device); partial-sum slots are int32 on the device.
static constexpr int64_t PERM_MAX_ITEMS = int64_t(1) << 27;

// Device block of a plan: items | cursor | wave arrays | small arrays | groups |
// partials, at these byte offsets.
struct PermLayout {
    size_t o_items = 0, o_cursor = 0, o_part = 0, o_widx = 0, o_ws0 = 0, o_wns = 0, o_wn = 0, o_sidx = 0,
           o_soff = 0, o_sn = 0, o_groups = 0, total = 0;
    size_t image = 0;     // bytes that are uploaded: all but the partials, which the waves write
    size_t scratch = 0;   // bytes that count against the scratch of pcvl_perm_batch_noalloc: all but the groups
};

// Cuts items [i0, i1) of the sorted queue into the groups that a wave takes at
// once; appends their starts and the end.  One pull from the cursor is an
// atomic on one address for the whole chip, 12..20 ns each however many waves
// wait, so small items cannot each have one: 20,000 of order 11 395 -> 112 us,
// of order 14 599 -> 398, 4,000 of order 16 469 -> 327.  Where the pulls would take
// more than a quarter of the work's time (estimated from the instructions of an
// item), the first groups, one a wave and not pulled, hold 70% of the work (a
// slow CU takes 1.3 times the average), and the rest is cut into as many groups
// as pulls fit into the work's time.  Otherwise every item is a group.
//
// perm_cost: an item's seconds of one SIMD: blocks, and the sums and constants
// before them; total: of all items.
static double perm_cost(int n, int c)
{
    constexpr double ISSUE = 4.0 / 2.1e9;
    return ISSUE * (4.3 * n * std::ldexp(1.0, c) + 2.0 * n * n + 40.0 * n);
}

static int64_t perm_groups(const std::vector<PermItem> &items, int64_t i0, int64_t i1, int resident, double total,
                           std::vector<uint32_t> &starts)
{
    constexpr double PULL = 15e-9, SIMDS = 1024.0;
    const int64_t count = i1 - i0, first = (int64_t)starts.size();
    auto each_item = [&]() {
        starts.resize((size_t)(first + count + 1));
        std::iota(starts.begin() + first, starts.end(), (uint32_t)i0);
        return count;
    };
    if (count <= resident || (double)count * PULL * 4.0 * SIMDS <= total) return each_item();
    const double pulls = std::max(total / SIMDS / PULL, 1.0);
    const double own = 0.7 * total / std::max(resident, 1), pulled = 0.3 * total / pulls;
    double sum = 0.0;
    int n = -1, c = -1;
    double cost = 0.0;
    for (int64_t i = i0; i < i1; i++) {
        const PermItem &it = items[(size_t)i];
        if (it.n != n || it.c != c) cost = perm_cost(n = it.n, c = it.c);
        const double want = (int64_t)starts.size() - first <= resident ? own : pulled;
        if (i == i0 || sum + 0.5 * cost >= want) {
            starts.push_back((uint32_t)i);
            sum = 0.0;
        }
        sum += cost;
    }
    const int64_t groups = (int64_t)starts.size() - first;
    starts.push_back((uint32_t)i1);
    return groups;
}

// Builds a plan on the host: the scheduling fields of p, the layout of its
// device block and the block's contents (cursor zero).  No device call but
// occupancy queries.
static int perm_plan_build(const int32_t *h_n, const int64_t *h_offsets, int64_t count, int max_chunk_log2,
                           int variant, PermPlanImpl &p, PermLayout &L, std::vector<char> &host)
{
    PCVL_ARG_CHECK(variant >= 0 && variant <= 4, "variant outside [0, 4]");
    PCVL_ARG_CHECK(count >= 0, "count < 0");
    PCVL_ARG_CHECK(count == 0 || (h_n && h_offsets), "null order/offset array");
    if (max_chunk_log2 <= 0) max_chunk_log2 = 11;
    PCVL_ARG_CHECK(max_chunk_log2 >= 2 && max_chunk_log2 <= 24, "max_chunk_log2 outside [2, 24]");

    std::vector<PermItem> items;
    std::vector<int64_t> wave_idx;
    std::vector<int32_t> wave_slot0, wave_nslot, wave_n;
    int64_t small_at[PERM_SMALL_MAX + 2] = {};   // small matrices of each order, then the first of each
    std::vector<int> wave_c;
    int nmin = 1 << 30, nmax = -1;
    bool any_big = false;
    for (int64_t b = 0; b < count; b++) {
        int n = h_n[b];
        PCVL_ARG_CHECK(n >= 0 && n <= PERM_BIG_MAX, "matrix order outside [0, 32]");
        PCVL_ARG_CHECK(h_offsets[b] >= 0, "negative matrix offset");
        if (n <= PERM_SMALL_MAX) {
            small_at[n + 1]++;
            continue;
        }
        wave_idx.push_back(b);
        wave_n.push_back(n);
        wave_c.push_back(pick_chunk_log2(n, max_chunk_log2));
        if (n >= PERM_BIG_MIN) {
            any_big = true;
            continue;
        }
        nmin = std::min(nmin, n);
        nmax = std::max(nmax, n);
    }
    // the small ones by order, a thread each first
    for (int n = 0; n <= PERM_SMALL_MAX; n++) small_at[n + 1] += small_at[n];
    const size_t nsmall = (size_t)small_at[PERM_SMALL_MAX + 1];
    p.nthread = small_at[PERM_THREAD_MAX + 1];
    // orders <= 28: one launch, specialised when they share one order
    const int single_n = (nmax >= 0 && nmin == nmax) ? nmax : 0;
    const int kvariant = single_n ? variant : 0;
    int rw = 0, rwb = 0;
    if (nmax >= 0) {
        const void *kp = single_n ? single_kernel_ptr<PERM_WAVE_MIN>(single_n, kvariant)
                                  : reinterpret_cast<const void *>(&perm_wave_kernel<PERM_WAVE_MIN, PERM_WAVE_MAX, false>);
        int rc = resident_waves(kp, &rw);
        if (rc != OK) return rc;
    }
    if (any_big) {
        int rc = resident_waves(reinterpret_cast<const void *>(&perm_wave_kernel<PERM_BIG_MIN, PERM_BIG_MAX, false>), &rwb);
        if (rc != OK) return rc;
    }
    // Tail refinement, per launch: the matrices whose items form the last
    // round of its queue (the last `resident waves` items in cost order) use
    // chunks 4x shorter, so the waves that finish last wait for at most a
    // quarter item.
    for (int big = 0; big < 2; big++) {
        std::vector<size_t> order;
        for (size_t i = 0; i < wave_idx.size(); i++)
            if ((wave_n[i] >= PERM_BIG_MIN) == (big == 1)) order.push_back(i);
        std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) {
            return ((int64_t)wave_n[a] << wave_c[a]) > ((int64_t)wave_n[b] << wave_c[b]);
        });
        const int resident = big ? rwb : rw;
        int64_t tail = 0;
        for (size_t r = order.size(); r-- > 0 && tail < resident;) {
            const size_t i = order[r];
            tail += (int64_t)((1ull << (wave_n[i] - 1 - wave_c[i])) / 64);
            // not where an item would then be mostly sums and constants (1,000 of
            // order 11 46 us with it, 22 without; 89 before the groups below)
            if (wave_c[i] >= 4 && 4.3 * (1 << (wave_c[i] - 2)) >= 2.0 * wave_n[i] + 40.0) wave_c[i] -= 2;
        }
    }
    int64_t total_slots = 0;
    for (size_t i = 0; i < wave_idx.size(); i++)
        total_slots += (int64_t)((1ull << (wave_n[i] - 1 - wave_c[i])) / 64);
    if (total_slots > PERM_MAX_ITEMS) {
        set_error("permanent batch needs " + std::to_string(total_slots) + " work items, above the limit of " +
                  std::to_string(PERM_MAX_ITEMS) + " (use a longer chunk or split the batch)");
        return ERR_RANGE;
    }
    items.reserve((size_t)total_slots);
    std::vector<PermItem> big_items;
    double work[2] = {0.0, 0.0};   // of the queue's two parts
    int32_t slots = 0;
    for (size_t i = 0; i < wave_idx.size(); i++) {
        const int n = wave_n[i], c = wave_c[i];
        const int64_t waves = (int64_t)((1ull << (n - 1 - c)) / 64);
        wave_slot0.push_back(slots);
        wave_nslot.push_back((int32_t)waves);
        work[n >= PERM_BIG_MIN] += (double)waves * perm_cost(n, c);
        std::vector<PermItem> &dst = n >= PERM_BIG_MIN ? big_items : items;
        for (int64_t w = 0; w < waves; w++)
            dst.push_back(PermItem{h_offsets[wave_idx[i]], (uint32_t)(w * 64), slots + (int32_t)w, n, c});
        slots += (int32_t)waves;
    }
    // Largest items first: the atomic queue then gives a greedy
    // longest-processing-time schedule over the resident waves.  The queue
    // holds the items of orders <= 28, then those of orders 29..32.
    auto by_cost = [](const PermItem &a, const PermItem &b) {
        return ((int64_t)a.n << a.c) > ((int64_t)b.n << b.c);
    };
    std::stable_sort(items.begin(), items.end(), by_cost);
    std::stable_sort(big_items.begin(), big_items.end(), by_cost);
    const int64_t nregular = (int64_t)items.size();
    items.insert(items.end(), big_items.begin(), big_items.end());

    std::vector<uint32_t> groups;
    p.ngroups = perm_groups(items, 0, nregular, rw, work[0], groups);
    p.nbig_groups = perm_groups(items, nregular, (int64_t)items.size(), rwb, work[1], groups);

    p.count = count;
    p.nitems = nregular;
    p.nbig = (int64_t)big_items.size();
    p.grid_big = p.nbig > 0 ? (int)std::min<int64_t>(p.nbig_groups, (int64_t)rwb) : 0;
    p.nwave_mats = (int64_t)wave_idx.size();
    p.nsmall = (int64_t)nsmall;
    p.single_n = single_n;
    p.variant = kvariant;
    p.grid = p.nitems > 0 ? (int)std::min<int64_t>(p.ngroups, (int64_t)rw) : 0;

    auto align = [](size_t x) { return (x + 255) & ~size_t(255); };
    L.o_items = 0;
    L.o_cursor = align(L.o_items + sizeof(PermItem) * items.size());
    L.o_widx = align(L.o_cursor + 2 * sizeof(unsigned long long));
    L.o_ws0 = align(L.o_widx + sizeof(int64_t) * wave_idx.size());
    L.o_wns = align(L.o_ws0 + sizeof(int32_t) * wave_idx.size());
    L.o_wn = align(L.o_wns + sizeof(int32_t) * wave_idx.size());
    L.o_sidx = align(L.o_wn + sizeof(int32_t) * wave_idx.size());
    L.o_soff = align(L.o_sidx + sizeof(int64_t) * nsmall);
    L.o_sn = align(L.o_soff + sizeof(int64_t) * nsmall);
    L.o_groups = align(L.o_sn + sizeof(int32_t) * nsmall);
    L.o_part = align(L.o_groups + sizeof(uint32_t) * groups.size());
    L.total = align(L.o_part + sizeof(cd) * (size_t)slots);
    L.image = L.o_part;
    L.scratch = L.total - (L.o_part - L.o_groups);

    host.assign(L.image, 0);
    auto put = [&](size_t off, const void *src, size_t bytes) { if (bytes) std::memcpy(host.data() + off, src, bytes); };
    put(L.o_items, items.data(), sizeof(PermItem) * items.size());
    put(L.o_widx, wave_idx.data(), sizeof(int64_t) * wave_idx.size());
    put(L.o_ws0, wave_slot0.data(), sizeof(int32_t) * wave_idx.size());
    put(L.o_wns, wave_nslot.data(), sizeof(int32_t) * wave_idx.size());
    put(L.o_wn, wave_n.data(), sizeof(int32_t) * wave_idx.size());
    int64_t *small_idx = reinterpret_cast<int64_t *>(host.data() + L.o_sidx);
    int64_t *small_off = reinterpret_cast<int64_t *>(host.data() + L.o_soff);
    int32_t *small_n = reinterpret_cast<int32_t *>(host.data() + L.o_sn);
    for (int64_t b = 0; nsmall && b < count; b++) {
        const int n = h_n[b];
        if (n > PERM_SMALL_MAX) continue;
        const int64_t at = small_at[n]++;
        small_idx[at] = b;
        small_off[at] = h_offsets[b];
        small_n[at] = n;
    }
    put(L.o_groups, groups.data(), sizeof(uint32_t) * groups.size());
    return OK;
}

// Points the plan's device arrays into a block laid out as L.
static void perm_plan_bind(PermPlanImpl &p, const PermLayout &L, void *block)
{
    char *base = static_cast<char *>(block);
    p.d_items = reinterpret_cast<PermItem *>(base + L.o_items);
    p.d_cursor = reinterpret_cast<unsigned long long *>(base + L.o_cursor);
    p.d_partials = reinterpret_cast<cd *>(base + L.o_part);
    p.d_wave_idx = reinterpret_cast<int64_t *>(base + L.o_widx);
    p.d_wave_slot0 = reinterpret_cast<int32_t *>(base + L.o_ws0);
    p.d_wave_nslot = reinterpret_cast<int32_t *>(base + L.o_wns);
    p.d_wave_n = reinterpret_cast<int32_t *>(base + L.o_wn);
    p.d_small_idx = reinterpret_cast<int64_t *>(base + L.o_sidx);
    p.d_small_off = reinterpret_cast<int64_t *>(base + L.o_soff);
    p.d_small_n = reinterpret_cast<int32_t *>(base + L.o_sn);
    p.d_groups = reinterpret_cast<uint32_t *>(base + L.o_groups);
}

static int perm_plan_create_impl(const int32_t *h_n, const int64_t *h_offsets, int64_t count,
                                 int max_chunk_log2, int variant, pcvl_perm_plan *out)
{
    PCVL_ARG_CHECK(out != nullptr, "out plan pointer is null");
    *out = nullptr;
    auto *plan = new (std::nothrow) pcvl_perm_plan_s();
    if (!plan) { set_error("host allocation failed"); return ERR_ALLOC; }
    PermPlanImpl &p = plan->impl;
    PermLayout L;
    std::vector<char> host;
    int rc = perm_plan_build(h_n, h_offsets, count, max_chunk_log2, variant, p, L, host);
    if (rc != OK) { delete plan; return rc; }
    hipError_t e = hipMalloc(&p.d_block, L.total);
    if (e != hipSuccess) {
        set_error(std::string("hipMalloc(perm plan): ") + hipGetErrorString(e));
        delete plan;
        return ERR_ALLOC;
    }
    perm_plan_bind(p, L, p.d_block);
    e = hipMemcpy(p.d_block, host.data(), L.image, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        set_error(std::string("hipMemcpy(perm plan): ") + hipGetErrorString(e));
        (void)hipFree(p.d_block);
        delete plan;
        return ERR_HIP;
    }
    *out = plan;
    return OK;
}

extern "C" int pcvl_perm_plan_create_ex(const int32_t *h_n, const int64_t *h_offsets, int64_t count,
                                        int max_chunk_log2, int variant, pcvl_perm_plan *out)
{
    try {
        return perm_plan_create_impl(h_n, h_offsets, count, max_chunk_log2, variant, out);
    } catch (const std::bad_alloc &) {
        set_error("host allocation failed while building the permanent plan");
        return ERR_ALLOC;
    } catch (...) {
        set_error("unexpected exception while building the permanent plan");
        return ERR_ALLOC;
    }
}

extern "C" int pcvl_perm_plan_create(const int32_t *h_n, const int64_t *h_offsets, int64_t count,
                                     int max_chunk_log2, pcvl_perm_plan *out)
{
    return pcvl_perm_plan_create_ex(h_n, h_offsets, count, max_chunk_log2, 0, out);
}

extern "C" int pcvl_perm_plan_execute(pcvl_perm_plan plan, const double *d_mats, double *d_out, hipStream_t stream)
{
    PCVL_ARG_CHECK(plan != nullptr, "plan is null");
    PermPlanImpl &p = plan->impl;
    if (p.count == 0) return OK;
    PCVL_ARG_CHECK(d_mats && d_out, "null device buffer");
    cd *out = reinterpret_cast<cd *>(d_out);
    if (p.nsmall > 0) {
        unsigned first = (unsigned)((p.nthread + 16 * PERM_ROWS - 1) / (16 * PERM_ROWS));
        int64_t row0 = p.nthread;
        do {   // PERM_ROW_LAUNCH at a time: a grid holds fewer than 2^32 threads, 2^28 such matrices
            const int64_t end = std::min(p.nsmall, row0 + PERM_ROW_LAUNCH);
            const unsigned rows = (unsigned)((end - row0 + PERM_ROWS - 1) / PERM_ROWS);
            hipLaunchKernelGGL(perm_small_kernel, dim3(first + rows), dim3(16 * PERM_ROWS), 0, stream, d_mats,
                               p.d_small_idx, p.d_small_off, p.d_small_n, end, row0, first, out);
            PCVL_HIP_CHECK(hipGetLastError());
            first = 0;
            row0 = end;
        } while (row0 < p.nsmall);
    }
    if (p.nwave_mats > 0) {
        int rc = OK;
        if (p.nbig > 0)   // orders 29..32 first: the longest items
            rc = launch_wave<PERM_BIG_MIN, PERM_BIG_MAX, false>(&p, d_mats, stream, p.d_groups + p.ngroups + 1,
                                                                p.nbig_groups, p.d_cursor + 1, p.grid_big);
        if (rc == OK && p.nitems > 0)
            rc = p.single_n ? launch_single<PERM_WAVE_MIN>(&p, d_mats, stream)
                            : launch_wave<PERM_WAVE_MIN, PERM_WAVE_MAX, false>(&p, d_mats, stream);
        if (rc != OK) return rc;
        int blocks = (int)((p.nwave_mats + 255) / 256);
        hipLaunchKernelGGL(perm_finalize_kernel, dim3(blocks), dim3(256), 0, stream, p.d_wave_idx,
                           p.d_wave_slot0, p.d_wave_nslot, p.d_wave_n, p.nwave_mats, p.d_partials, out,
                           p.d_cursor);
        PCVL_HIP_CHECK(hipGetLastError());
    }
    return OK;
}

extern "C" int pcvl_perm_plan_destroy(pcvl_perm_plan plan)
{
    if (!plan) return OK;
    hipError_t e = hipSuccess;
    if (plan->impl.d_block) e = hipFree(plan->impl.d_block);
    delete plan;
    if (e != hipSuccess) {
        set_error(std::string("hipFree(perm plan): ") + hipGetErrorString(e));
        return ERR_HIP;
    }
    return OK;
}

extern "C" int pcvl_perm_plan_info(pcvl_perm_plan plan, int64_t *nitems, int *grid, int *single_n)
{
    PCVL_ARG_CHECK(plan != nullptr, "plan is null");
    if (nitems) *nitems = plan->impl.nitems + plan->impl.nbig;
    if (grid) *grid = plan->impl.grid;
    if (single_n) *single_n = plan->impl.single_n;
    return OK;
}

extern "C" int pcvl_perm_batch(const double *d_mats, const int32_t *h_n, const int64_t *h_offsets, int64_t count,
                               double *d_out, hipStream_t stream)
{
    pcvl_perm_plan plan = nullptr;
    int rc = pcvl_perm_plan_create(h_n, h_offsets, count, 0, &plan);
    if (rc != OK) return rc;
    rc = pcvl_perm_plan_execute(plan, d_mats, d_out, stream);
    hipError_t e = hipStreamSynchronize(stream);
    int rc2 = pcvl_perm_plan_destroy(plan);
    if (rc != OK) return rc;
    if (e != hipSuccess) { set_error(std::string("hipStreamSynchronize: ") + hipGetErrorString(e)); return ERR_HIP; }
    return rc2;
}

// ------------------------------------------------------- no allocation
//
// pcvl_perm_batch_noalloc: the same batch with no device allocation.  The
// plan's block (work items, queue cursor, partial sums, per-matrix arrays)
// goes into `scratch`, a file-scope device array that each GPU holds from
// module load until the process ends.  Host code never passes the array's
// name to a kernel: its device address is looked up once per device with
// hipGetSymbolAddress, on the entry point's first call on that device, and
// that pointer is used for the copy and the kernel arguments.  Every call on
// a GPU shares its array: calls that overlap on one GPU (several host threads
// or streams) race.  Each call rewrites the whole block it uses, the queue
// cursor included (zero), before its kernels read it.
constexpr size_t PERM_SCRATCH_BYTES = size_t(16) << 20;
// The groups of the queue come on top of the 16 MiB (at most 4 bytes per item of
// 40), so that the limit does not depend on them.
static __device__ __align__(256) char scratch[PERM_SCRATCH_BYTES + PERM_SCRATCH_BYTES / 8];

static std::mutex g_scratch_mu;
static void *g_scratch_ptr[64] = {};

static int scratch_ptr(void **out)
{
    int dev = 0;
    PCVL_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) { set_error("device index outside [0, 64)"); return ERR_ARG; }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return ERR_HIP;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return OK;
}

static int perm_batch_noalloc_impl(const double *d_mats, const int32_t *h_n, const int64_t *h_offsets, int64_t count,
                                   double *d_out, hipStream_t stream)
{
    pcvl_perm_plan_s plan;
    PermPlanImpl &p = plan.impl;
    PermLayout L;
    std::vector<char> host;
    int rc = perm_plan_build(h_n, h_offsets, count, 0, 0, p, L, host);
    if (rc != OK) return rc;
    if (L.scratch > PERM_SCRATCH_BYTES) {
        set_error("permanent batch needs " + std::to_string(L.scratch) + " bytes of plan scratch, above the " +
                  std::to_string(PERM_SCRATCH_BYTES) + " of pcvl_perm_batch_noalloc (split the batch or use "
                  "pcvl_perm_batch)");
        return ERR_RANGE;
    }
    if (count == 0) return OK;
    PCVL_ARG_CHECK(d_mats && d_out, "null device buffer");
    void *base = nullptr;
    rc = scratch_ptr(&base);
    if (rc != OK) return rc;
    perm_plan_bind(p, L, base);
    PCVL_HIP_CHECK(hipMemcpyAsync(base, host.data(), L.image, hipMemcpyHostToDevice, stream));
    rc = pcvl_perm_plan_execute(&plan, d_mats, d_out, stream);
    // the host image must outlive its copy, and results are ready on return
    hipError_t e = hipStreamSynchronize(stream);
    if (rc != OK) return rc;
    if (e != hipSuccess) { set_error(std::string("hipStreamSynchronize: ") + hipGetErrorString(e)); return ERR_HIP; }
    return OK;
}

extern "C" int pcvl_perm_batch_noalloc(const double *d_mats, const int32_t *h_n, const int64_t *h_offsets,
                                       int64_t count, double *d_out, hipStream_t stream)
{
    try {
        return perm_batch_noalloc_impl(d_mats, h_n, h_offsets, count, d_out, stream);
    } catch (const std::bad_alloc &) {
        set_error("host allocation failed while building the permanent plan");
        return ERR_ALLOC;
    } catch (...) {
        set_error("unexpected exception while building the permanent plan");
        return ERR_ALLOC;
    }
}

extern "C" size_t pcvl_perm_noalloc_max_bytes(void) { return PERM_SCRATCH_BYTES; }
