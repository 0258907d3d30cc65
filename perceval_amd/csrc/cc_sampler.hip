// Exact boson sampling: algorithm A of Clifford & Clifford (2017), batched
// over samples.  Replaces xq.Clifford2017.samples
// (perceval/backends/_clifford2017.py:52-57; docs/source/backends.rst:108-116).
//
// For an input with photons in modes cols[0..n-1] let A = U[:, cols] (m x n).
// A sample permutes the columns of A uniformly, then for k = 1..n draws the
// output mode r_k with probability proportional to
//     w_i = | sum_{l<k} A[i, perm[l]] * perm(B^{(-l)}) |^2,
//     B = A[r_1..r_{k-1}, perm[0..k-1]]  ((k-1) x k),
// where B^{(-l)} drops column l.  All k sub-permanents come from one Glynn
// pass over the rows of B: per Gray-code term, the k column sums c_l are
// shared and prod_{l' != l} c_l' is the product of a prefix and a suffix.
//
// Mapping: one launch for steps 1..9 of up to 64 modes (16 lanes a sample), then
// one launch per photon step k, specialised on k so that each step gets its own
// register allocation.  A wavefront owns one sample (persistent over samples) up
// to step 13 and, by the rule of cc_one_wave, in steps 14 and 15; above, one slice
// of a sample's terms.  The terms (2^{k-2}; fewer from step 10 on, or
// from 14 on above CC_MULTI_MODES modes, where repeated rows are summed by
// multiplicity) are split over the 32 lane pairs; partial sums of the k
// sub-permanents are reduced across the wave, then lane i computes the weight of
// candidate row i and a wave prefix sum draws r_k.  Per-sample state (permuted
// columns, drawn modes)
// lives in a caller-provided workspace.  Random numbers
// are the counter-based uniforms of common.h: stream = sample index, counters
// 0..n-2 for the column permutation (Fisher-Yates, i = n-1 down to 1) and
// n-1+k-1 for the k-th photon, so a run is fixed by its seed.
#include "common.h"
#include "slices.h"
#include "../../include/pcvl_hip.h"

#include <algorithm>
#include <vector>

namespace pcvl {

constexpr int CC_MAX_N = 30;
constexpr int CC_MAX_M = 256;   // multiple of 64

// Per-step shared state, sized for step K: the LDS a step takes (and with it
// the occupancy the compiler plans its registers for) does not grow with the
// largest photon count the library accepts.
template <int K>
struct CCShared {
    // The lanes of a pair read columns h = K / 2 apart: at h = 8 (steps 16 and
    // 17) the same banks, so a column's room lies between the halves there
    // (20,000 samples of 20 photons in 60 modes: 1.68
    // -> 1.30 ms and 3.19 -> 2.56, VALU busy 67% -> 87% and 74% -> 93%).
    static constexpr int GAP = K / 2 == 8 ? 1 : 0, LD = K + GAP;
    cd B[(K > 1 ? K - 1 : 1) * LD];      // B[i*LD + l] = 2 * U[r_i, cols[perm[l]]] (l + GAP from h on)
    cd sub[K];
    int pc[K];                           // cols[perm[l]]: input mode of permuted column l
    int r[K];
    // multiset steps: distinct output modes in the order fixed, unique, groups
    int mode[K], kg[K], w0[K];           // kg, w0: copies and first weight of each group
    uint32_t inv[K];                     // ceil(2^32 / (k_g + 1)), see subperm_units
    double w[2 * K];                     // (-1)^t C(k_g, t), t = 0..k_g
};

// Partial sums of the k sub-permanents over this lane pair's chunk of
// Gray-code terms (B holds 2*A rows; rows = k-1 >= 1).  The k columns are cut
// into halves L = [0, h) and H = [h, k) with h = k/2; the even lane of a pair
// owns L, the odd lane owns H, each padded to hmax = k - h columns (a padding
// column has column sum 1 and never flips).  Per term each lane forms the
// prefix products of its half and the half total T; the partners swap T, and
// prod_{l' != l} c_l' = prefix(l) * suffix(l) * T_partner comes out of one
// backward pass.  acc[j] is this lane's partial for column c0 + j. 
template <int K>
__device__ __forceinline__ void subperm_pair(const cd *__restrict__ B, int lane, cd *acc)
{
    constexpr int rows = K - 1;
    constexpr int h = K / 2;
    constexpr int hmax = K - h;
    constexpr int total_log2 = rows - 1;                   // 2^{rows-1} terms
    constexpr int c = total_log2 > 5 ? total_log2 - 5 : 0; // 32 pairs
    constexpr int active_pairs = total_log2 > 5 ? 32 : (1 << total_log2);
    const int half = lane & 1;
    const int pair = lane >> 1;
    const int c0 = half ? h : 0;
    const int ncol = half ? hmax : h;    // columns this lane really owns
#pragma unroll
    for (int j = 0; j < hmax; j++) acc[j] = {0.0, 0.0};
    if (pair >= active_pairs) return;
    const uint32_t steps = 1u << c;
    const uint32_t base = (uint32_t)pair << c;
    const uint32_t g0 = base ^ (base >> 1);

    // For odd K the even lane's last column is padding: it reads a valid
    // column of B (column h) but scales it by 0 and starts at 1, so the
    // code has no lane-divergent branches.
    const double pad = (hmax - 1 < ncol) ? 1.0 : 0.0;
    cd cs[hmax];
#pragma unroll
    for (int j = 0; j < hmax; j++) {
        const double f = (j == hmax - 1) ? pad : 1.0;
        const cd b = B[c0 + j];
        cs[j] = {fma(0.5 * f, b.r, 1.0 - f), 0.5 * f * b.i};
    }
    for (int i = 1; i < rows; i++) {
        const double d = ((g0 >> (i - 1)) & 1) ? -0.5 : 0.5;
#pragma unroll
        for (int j = 0; j < hmax; j++) {
            const double dj = (j == hmax - 1) ? d * pad : d;
            const cd b = B[i * K + c0 + j];
            cs[j].r = fma(dj, b.r, cs[j].r);
            cs[j].i = fma(dj, b.i, cs[j].i);
        }
    }
    for (uint32_t u = 0; u < steps; u++) {
        const uint32_t t = base + u;
        if (u) {
            const int b = __builtin_ctz(t);
            const double s = (((t >> b) ^ (t >> (b + 1))) & 1) ? -1.0 : 1.0;
            const double sl = s * pad;
            const cd *row = B + (b + 1) * K + c0;
#pragma unroll
            for (int j = 0; j < hmax; j++) {
                const cd a = row[j];
                const double sj = (j == hmax - 1) ? sl : s;
                cs[j].r = fma(sj, a.r, cs[j].r);
                cs[j].i = fma(sj, a.i, cs[j].i);
            }
        }
        cd P[hmax];
        P[0] = {1.0, 0.0};
        if constexpr (hmax > 1) P[1] = cs[0];
#pragma unroll
        for (int j = 2; j < hmax; j++) P[j] = cmul(P[j - 1], cs[j - 1]);
        const cd T = (hmax == 1) ? cs[0] : cmul(P[hmax - 1], cs[hmax - 1]);
        cd Tp;
        Tp.r = __shfl_xor(T.r, 1, 64);
        Tp.i = __shfl_xor(T.i, 1, 64);
        cd S = (t & 1) ? cd{-Tp.r, -Tp.i} : Tp;
#pragma unroll
        for (int j = hmax - 1; j >= 1; j--) {
            cfma_acc(acc[j], P[j], S);
            S = cmul(S, cs[j]);
        }
        acc[0].r += S.r;
        acc[0].i += S.i;
        // Keep the next column-sum update below this term's products (no
        // overlap of two generations of cs; see perm_glynn.hip).
#pragma unroll
        for (int j = 0; j < hmax; j++)
            asm volatile("" : "+v"(cs[j].r), "+v"(cs[j].i) : "v"(acc[0].r), "v"(acc[0].i));
    }
}

// ---- multiset terms ---------------------------------------------------------
//
// From step CC_MULTI on, rows of B that repeat (photons already drawn in one
// mode) are summed by multiplicity: k copies of a row enter the column sums
// only through their sign total k - 2t, with weight (-1)^t C(k, t), so a group
// of k copies takes k + 1 terms instead of 2^k.  At m = 60 the 19 rows of step
// 20 leave 0.27 of the 2^18 terms on average, and fewer the smaller m is.
// One row of weight 1 is the fixed row (delta = +1), the other unique rows are
// walked in Gray-code order, and the group digits t_g form an outer
// mixed-radix index o with weight W_o.  With half column sums h (a flip adds
// the row)
//     sub_l = 2 sum_o W_o sum_{t < 2^nu} (-1)^t prod_{l' != l} h_l'.
// The O 2^nu terms are cut into units of 2^c Gray steps, one unit per lane
// pair at a time.
constexpr int CC_MULTI = 10;     // below, the terms are one or two passes of the 32 pairs
// Above so many modes, steps 10..13 sum every row by itself: they repeat too
// rarely to pay for the plan of the terms (100 modes, 100 samples of 12 photons
// 139 us, 146 with multiplicities; 5,000 of 13 361 and 358).
constexpr int CC_MULTI_MODES = 64;
// From step 14 on, a sample's units are cut into slices (20,000 samples at
// m = 60: step 15 takes 0.86 ms against 0.98 with one wave per sample, step 13
// would lose the four extra launches).
constexpr int CC_SLICED = 14;
constexpr int CC_MAX_C = 8;
// Steps of two slices at most that one wave may run one after another, drawing at
// their end: one launch a step instead of five.  Step 14 gains up to 8,192 samples
// (100 modes, 100 samples 230 -> 218 us; 48 modes, one sample 178 -> 164).  Step 15
// gains where many samples fill the waves and few of them repeat rows (60 modes,
// 1,000 samples 314 -> 287 us, 2,000 410 -> 366; 100 modes, 5,000 856 -> 769); with
// few samples the second slice is waited for (30 modes, one sample 204 -> 219 us,
// 64 243 -> 270, 500 282 -> 306; 38 modes, 256 280 -> 303; 100 modes, one 254 ->
// 282, but 16 305 -> 301), with many up to 64 modes slices balance better (38
// modes, 8,000 874 -> 900).  Of 16 photons, step 16 in it would take 262 us instead
// of 244.
constexpr int CC_ONE_WAVE = 15;
constexpr int64_t CC_ONE_WAVE_COUNT = 8192;
constexpr bool cc_one_wave(int k, int m, int64_t count)
{
    if (k < CC_SLICED) return true;
    if (k > CC_ONE_WAVE || count > CC_ONE_WAVE_COUNT) return false;
    if (k < CC_ONE_WAVE) return true;
    return m > CC_MULTI_MODES ? count >= 4 : m > 32 && count >= 512 && count <= CC_ONE_WAVE_COUNT / 2;
}

// Most slices of a sample at step k: at most 2^13 terms each up to step 27
// (0.2 ms of one wave: the tail when the last slices drain), 4,096 slices
// above (their partial sums are added one after another by the draw).
constexpr int cc_slice_cap(int k) { return k < CC_SLICED ? 1 : k < 16 ? 2 : k <= 27 ? 1 << (k - 15) : 4096; }

struct CCPlan {
    int nu, ng, c, slices;
    uint32_t units;
};

// Plans the rows sh.r[0..K-2] of a sample, one wave: fills sh.mode, sh.kg,
// sh.w0, sh.w.  Every field of the result is wave-uniform.
template <int K>
__device__ __forceinline__ CCPlan cc_plan(CCShared<K> &sh, int lane)
{
    constexpr int rows = K - 1;
    const int r = lane < rows ? sh.r[lane] : -1 - lane;
    int cnt = 0, first = 64;
#pragma unroll
    for (int i = 0; i < rows; i++) {
        const bool same = __builtin_amdgcn_readlane(r, i) == r;
        cnt += same ? 1 : 0;
        if (same && first == 64) first = i;
    }
    const bool lead = lane < rows && first == lane;   // first photon of its mode
    const uint64_t um = __ballot(lead && cnt == 1), gm = __ballot(lead && cnt > 1);
    const uint64_t below = (1ull << lane) - 1;
    CCPlan p;
    p.ng = __builtin_popcountll(gm);
    p.nu = um ? __builtin_popcountll(um) - 1 : 0;
    // the fixed row: the first unique row, else one copy of the first group
    const int fixed = __builtin_ctzll(um ? um : gm);
    if (lane == fixed) sh.mode[0] = r;
    if (lead && cnt == 1 && lane != fixed) sh.mode[__builtin_popcountll(um & below)] = r;
    int k = 0;
    if (lead && cnt > 1) {
        k = cnt - (lane == fixed ? 1 : 0);
        const int g = __builtin_popcountll(gm & below);
        sh.mode[1 + p.nu + g] = r;
        sh.kg[g] = k;
    }
    uint32_t O = 1;   // outer terms: the product of k_g + 1, at most 2^(K-2)
    for (uint64_t left = gm; left != 0; left &= left - 1)
        O *= (uint32_t)__builtin_amdgcn_readlane(k, __builtin_ctzll(left)) + 1;
    __syncthreads();
    if (lane < p.ng) {
        int w0 = 0;
        for (int g = 0; g < lane; g++) w0 += sh.kg[g] + 1;
        sh.w0[lane] = w0;
        const int kk = sh.kg[lane];
        sh.inv[lane] = (uint32_t)((0x100000000ull + (uint32_t)kk) / (uint32_t)(kk + 1));
        double w = 1.0;   // every quotient is a whole number
        for (int t = 0; t <= kk; t++) {
            sh.w[w0 + t] = w;
            w = -w * (double)(kk - t) / (double)(t + 1);
        }
    }
    // Unit length 2^c: short units fill the lane pairs of the last pass, long
    // ones repeat the column-sum set-up less often.  The c of least estimated
    // time, in operations per lane: passes x (2^c terms + set-up) + the slice's
    // own cost (rows into LDS, reduction of K sums).
    const int cmax = p.nu < CC_MAX_C ? p.nu : CC_MAX_C;
    const uint32_t setup = (uint32_t)((K + 1) * (2 + p.nu + p.ng) + 24 * p.ng + 40);
    constexpr uint32_t cap = (uint32_t)cc_slice_cap(K);   // a power of two
    uint32_t best = 0xffffffffu;
    for (int c = cmax; c >= 0 && c >= cmax - 4; c--) {
        const uint32_t units = O << (p.nu - c);
        const uint32_t want = (units + 31) / 32;
        const uint32_t sl = want < cap ? want : cap;
        const uint32_t passes = want < cap ? want : ((units + cap - 1) / cap + 31) / 32 * cap;
        const float est = __builtin_fmaf((float)passes, (float)((7 * K + 24) * (1 << c) + (int)setup), 4000.0f * (float)sl);
        const uint32_t e = __float_as_uint(est);   // positive floats order as their bits
        if (e < best) {
            best = e;
            p.c = c;
            p.slices = (int)sl;
            p.units = units;
        }
    }
    __syncthreads();
    return p;
}

// The value of the other lane of the pair, as a DPP move (no LDS round trip).
__device__ __forceinline__ double pair_swap(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);   // quad_perm [1, 0, 3, 2]
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// Bound by FP64 issue (14 K + 16 operations per term over the pair).  20,000
// samples at m = 60, n = 20 take 34.3 ms; 106.7 ms with all 2^{k-2} terms, one
// wave per sample, the row of a flip read at its use and the pair's exchange
// through LDS (38.1 ms with multiplicities and slices alone).
//
// Partial sums of the K sub-permanents (before the factor 2) over units
// [u0, u1) of a planned sample; columns over the lane pair as in subperm_pair.
// A holds the 1 + nu + ng distinct rows.
template <int K>
__device__ __forceinline__ void subperm_units(const CCShared<K> &sh, const CCPlan &pl, uint32_t u0, uint32_t u1,
                                              int lane, cd *acc)
{
    constexpr int h = K / 2;
    constexpr int hmax = K - h;
    constexpr int LD = CCShared<K>::LD;
    const cd *A = sh.B;
    const int half = lane & 1;
    const int c0 = half ? h + CCShared<K>::GAP : 0;
    const int ncol = half ? hmax : h;
    const double pad = (hmax - 1 < ncol) ? 1.0 : 0.0;
#pragma unroll
    for (int j = 0; j < hmax; j++) acc[j] = {0.0, 0.0};
    for (uint32_t unit = u0 + (uint32_t)(lane >> 1); unit < u1; unit += 32) {
        uint32_t o = unit >> (pl.nu - pl.c);
        const uint32_t base = (unit & ((1u << (pl.nu - pl.c)) - 1)) << pl.c;
        const uint32_t g0 = base ^ (base >> 1);
        cd cs[hmax];
#pragma unroll
        for (int j = 0; j < hmax; j++) {
            const double f = (j == hmax - 1) ? pad : 1.0;
            const cd a = A[c0 + j];
            cs[j] = {fma(0.5 * f, a.r, 1.0 - f), 0.5 * f * a.i};
        }
        auto add_row = [&](int i, double d) {
            const double dl = d * pad;
#pragma unroll
            for (int j = 0; j < hmax; j++) {
                const double dj = (j == hmax - 1) ? dl : d;
                const cd a = A[i * LD + c0 + j];
                cs[j].r = fma(dj, a.r, cs[j].r);
                cs[j].i = fma(dj, a.i, cs[j].i);
            }
        };
#pragma unroll 1
        for (int i = 1; i <= pl.nu; i++) add_row(i, ((g0 >> (i - 1)) & 1) ? -0.5 : 0.5);
        double W = 1.0;
#pragma unroll 1
        for (int g = 0; g < pl.ng; g++) {
            const int k = sh.kg[g];
            // o / (k + 1): exact while o (k + 1) < 2^32, and o < 2^(K-2) where k < 16,
            // below (k + 1) 2^(K-2-k) else
            const uint32_t quot = __umulhi(o, sh.inv[g]);
            const int t = (int)(o - quot * (uint32_t)(k + 1));
            o = quot;
            W *= sh.w[sh.w0[g] + t];
            add_row(1 + pl.nu + g, 0.5 * (double)(k - 2 * t));
        }
        if (base & 1u) W = -W;   // units of one term (c = 0): the term's Gray sign
        const uint32_t steps = 1u << pl.c;
        for (uint32_t u = 0; u < steps; u++) {
            // the flip to the next term; after the last one (of row 0, say)
            // its result is discarded
            const uint32_t t = base + u + 1;
            const int b = __builtin_ctz(u + 1);   // base is a multiple of 2^c
            const double s = (((t >> b) ^ (t >> (b + 1))) & 1) ? -1.0 : 1.0;
            const cd *row = A + (b < pl.nu ? b + 1 : 0) * LD + c0;
            cd P[hmax];
            P[0] = {1.0, 0.0};
            if constexpr (hmax > 1) P[1] = cs[0];
#pragma unroll
            for (int j = 2; j < hmax; j++) P[j] = cmul(P[j - 1], cs[j - 1]);
            // The backward pass flips each column once it is through with it;
            // the row's entries are read AHEAD columns before.
            constexpr int AHEAD = 3;
            cd nv[hmax];
#pragma unroll
            for (int j = hmax - 1; j >= 0 && j > hmax - 1 - AHEAD; j--) nv[j] = row[j];
            __builtin_amdgcn_sched_barrier(0);
            const cd T = (hmax == 1) ? cs[0] : cmul(P[hmax - 1], cs[hmax - 1]);
            cd S;
            S.r = W * pair_swap(T.r);
            S.i = W * pair_swap(T.i);
            W = -W;
#pragma unroll
            for (int j = hmax - 1; j >= 0; j--) {
                if (j >= AHEAD) nv[j - AHEAD] = row[j - AHEAD];
                if (j >= 1) {
                    cfma_acc(acc[j], P[j], S);
                    S = cmul(S, cs[j]);
                } else {
                    acc[0].r += S.r;
                    acc[0].i += S.i;
                }
                const double sj = (j == hmax - 1) ? s * pad : s;
                // in place: behind the product that read the old sum
                asm("" : "+v"(cs[j].r), "+v"(cs[j].i) : "v"(S.r), "v"(S.i));
                cs[j].r = fma(sj, nv[j].r, cs[j].r);
                cs[j].i = fma(sj, nv[j].i, cs[j].i);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

__device__ __forceinline__ double wave_sum_d(double v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sum over the lanes of one parity (the 32 pairs).
__device__ __forceinline__ double pair_sum_d(double v)
{
#pragma unroll
    for (int off = 32; off >= 2; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <int K>
__device__ __forceinline__ void subperms(CCShared<K> &sh, int lane)
{
    constexpr int h = K / 2;
    constexpr int hmax = K - h;
    cd acc[hmax];
    subperm_pair<K>(sh.B, lane, acc);
    constexpr int rows = K - 1;
    const double scale = ldexp(1.0, -(rows - 1));
#pragma unroll
    for (int j = 0; j < hmax; j++) {
        const double re = pair_sum_d(acc[j].r), im = pair_sum_d(acc[j].i);
        if (lane == 0 && j < h) sh.sub[j] = {re * scale, im * scale};
        if (lane == 1) sh.sub[h + j] = {re * scale, im * scale};
    }
}

// The partial sums of units [u0, u1) to dst[0..K-1].
template <int K>
__device__ __forceinline__ void subperms_units(const CCShared<K> &sh, const CCPlan &pl, uint32_t u0, uint32_t u1,
                                               int lane, cd *dst)
{
    constexpr int h = K / 2;
    constexpr int hmax = K - h;
    cd acc[hmax];
    subperm_units<K>(sh, pl, u0, u1, lane, acc);
#pragma unroll
    for (int j = 0; j < hmax; j++) {
        const double re = pair_sum_d(acc[j].r), im = pair_sum_d(acc[j].i);
        if (lane == 0 && j < h) dst[j] = {2.0 * re, 2.0 * im};
        if (lane == 1) dst[h + j] = {2.0 * re, 2.0 * im};
    }
}

// Distinct rows of a planned sample into sh.B: A[mode, perm[0..K-1]].
template <int K>
__device__ __forceinline__ void load_rows(CCShared<K> &sh, const CCPlan &pl, const cd *__restrict__ U, int m, int lane)
{
    constexpr int LD = CCShared<K>::LD, GAP = CCShared<K>::GAP, h = K / 2;
    for (int e = lane; e < (1 + pl.nu + pl.ng) * LD; e += 64) {
        const int l = e % LD;
        if (GAP && l == h) sh.B[e] = {0.0, 0.0};   // read as the padding column of an odd K
        else sh.B[e] = U[(size_t)sh.mode[e / LD] * m + sh.pc[l < h ? l : l - GAP]];
    }
    __syncthreads();
}

// Column permutation of each sample (Fisher-Yates, counters 0..n-2):
// pc[s*n + l] = input mode of permuted column l.
__global__ void cc_init_kernel(const int32_t *__restrict__ cols, int n, int64_t count, uint64_t seed, uint64_t first,
                               int32_t *__restrict__ pc)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= count) return;
    int perm[CC_MAX_N];
    for (int l = 0; l < n; l++) perm[l] = l;
    uint64_t ctr = 0;
    for (int i = n - 1; i >= 1; i--) {
        const double u = uniform01(seed, first + (uint64_t)s, ctr++);
        int j = (int)(u * (i + 1));
        if (j > i) j = i;
        const int t = perm[i]; perm[i] = perm[j]; perm[j] = t;
    }
    for (int l = 0; l < n; l++) pc[s * n + l] = cols[perm[l]];
}

// Several input states with the same photon number: the batch holds
// start[g + 1] - start[g] samples of its g-th input, whose photon columns are
// cols[g * n ...] and whose first output row is row0[g].  Sample s of the batch
// is global sample gidx[s] (its output row and counter stream).
__global__ void cc_init_multi_kernel(const int32_t *__restrict__ cols, const int64_t *__restrict__ start,
                                     const int64_t *__restrict__ row0, int ninputs, int n, int64_t count,
                                     uint64_t seed, uint64_t first, int64_t *__restrict__ gidx,
                                     int32_t *__restrict__ pc)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= count) return;
    int g = 0, hi = ninputs - 1;   // the last input that starts at or before s
    while (g < hi) {
        const int mid = (g + hi + 1) >> 1;
        if (start[mid] <= s) g = mid;
        else hi = mid - 1;
    }
    const int64_t row = row0[g] + (s - start[g]);
    gidx[s] = row;
    const int32_t *c = cols + (size_t)g * n;
    int perm[CC_MAX_N];
    for (int l = 0; l < n; l++) perm[l] = l;
    uint64_t ctr = 0;
    const uint64_t stream = first + (uint64_t)row;
    for (int i = n - 1; i >= 1; i--) {
        const double u = uniform01(seed, stream, ctr++);
        int j = (int)(u * (i + 1));
        if (j > i) j = i;
        const int t = perm[i]; perm[i] = perm[j]; perm[j] = t;
    }
    for (int l = 0; l < n; l++) pc[s * n + l] = c[perm[l]];
}

// Output rows of a multi-input batch: sample s goes to row gidx[s].
__global__ void cc_finish_multi_kernel(const int32_t *__restrict__ r_all, const int64_t *__restrict__ gidx, int m,
                                       int n, int64_t count, int32_t *__restrict__ out)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count * m) return;
    const int64_t s = e / m;
    const int i = (int)(e % m);
    int v = 0;
    for (int k = 0; k < n; k++) v += (r_all[s * n + k] == i) ? 1 : 0;
    out[gidx[s] * m + i] = v;
}

// Draw of photon K of sample s from the sub-permanents in sh.sub: the weight
// of every candidate row i (lane i of each 64-row chunk), then an inclusive
// scan over rows in order picks r_k.
template <int K>
__device__ __forceinline__ void cc_draw(const CCShared<K> &sh, const cd *__restrict__ U, int m, int n, int64_t s,
                                        uint64_t seed, uint64_t stream, int lane, int32_t *__restrict__ r_all)
{
    constexpr int CH = CC_MAX_M / 64;
    double wv[CH];
    double total = 0.0;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = c * 64 + lane;
        double w = 0.0;
        if (c * 64 < m && i < m) {
            cd a = {0.0, 0.0};
#pragma unroll
            for (int l = 0; l < K; l++) cfma_acc(a, U[(size_t)i * m + sh.pc[l]], sh.sub[l]);
            w = a.r * a.r + a.i * a.i;
        }
        wv[c] = w;
        total += wave_sum_d(w);
    }
    const double target = uniform01(seed, stream, (uint64_t)(n - 1) + (uint64_t)(K - 1)) * total;
    int pick = m - 1;
    double base = 0.0;
    bool found = false;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        if (!found && c * 64 < m) {
            const int i = c * 64 + lane;
            double incl = wv[c];
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const double v = __shfl_up(incl, off, 64);
                if (lane >= off) incl += v;
            }
            const bool hit = (i < m) && (target < base + incl);
            const unsigned long long mask = __ballot(hit);
            if (mask) {
                pick = c * 64 + (int)__builtin_ctzll(mask);
                found = true;
            }
            base += __shfl(incl, 63, 64);
        }
    }
    if (lane == 0) r_all[s * n + (K - 1)] = pick;
}

// Step k (= K) of every sample: one wavefront per sample, persistent.
// r[s*n + i] holds the output mode of photon i (i < k-1 already drawn).
// MULTI: repeated rows by multiplicity.
template <int K, bool MULTI>
__global__ void __launch_bounds__(64) cc_step_kernel(const cd *__restrict__ U, int m, int n, int64_t count,
                                                     uint64_t seed, uint64_t first, const int32_t *__restrict__ pc_all,
                                                     int32_t *__restrict__ r_all, const int64_t *__restrict__ gidx)
{
    __shared__ CCShared<K> sh;
    const int lane = threadIdx.x;
    for (int64_t s = blockIdx.x; s < count; s += gridDim.x) {
        const uint64_t stream = first + (uint64_t)(gidx ? gidx[s] : s);
        if (lane < K) sh.pc[lane] = pc_all[s * n + lane];
        if (lane < K - 1) sh.r[lane] = r_all[s * n + lane];
        __syncthreads();
        if constexpr (K == 1) {
            if (lane == 0) sh.sub[0] = {1.0, 0.0};
        } else {
            static_assert(MULTI || K < CC_SLICED, "slices are of multiset terms");
            if constexpr (K >= CC_SLICED) {
                // the slices of the sample one after another, summed in order
                // as by cc_slice_draw_kernel: the same bits
                __shared__ cd s_part[K];
                const CCPlan pl = cc_plan<K>(sh, lane);
                load_rows<K>(sh, pl, U, m, lane);
                const uint32_t per = (pl.units + (uint32_t)pl.slices - 1) / (uint32_t)pl.slices;
                cd v = {0.0, 0.0};
                for (uint32_t u0 = 0; u0 < pl.units; u0 += per) {
                    subperms_units<K>(sh, pl, u0, u0 + per < pl.units ? u0 + per : pl.units, lane, s_part);
                    __syncthreads();
                    if (lane < K) v = cadd(v, s_part[lane]);
                    __syncthreads();
                }
                if (lane < K) sh.sub[lane] = v;
            } else if constexpr (MULTI) {
                const CCPlan pl = cc_plan<K>(sh, lane);
                load_rows<K>(sh, pl, U, m, lane);
                subperms_units<K>(sh, pl, 0, pl.units, lane, sh.sub);
            } else {
                // B = 2 * A[r_1..r_{k-1}, perm[0..k-1]] with A = U[:, cols]
                for (int e = lane; e < (K - 1) * K; e += 64) {
                    const int i = e / K, l = e % K;
                    const cd a = U[(size_t)sh.r[i] * m + sh.pc[l]];
                    sh.B[e] = {2.0 * a.r, 2.0 * a.i};
                }
                __syncthreads();
                subperms<K>(sh, lane);
            }
        }
        __syncthreads();
        cc_draw<K>(sh, U, m, n, s, seed, stream, lane, r_all);
        __syncthreads();
    }
}

// ---- the first steps in one launch --------------------------------------------
//
// Steps 1..CC_FIRST of a sample are a few dozen terms each; with a launch and a
// wave per step their time goes to gathers, barriers and launches.  Here 16
// lanes take a sample through all of them: U sits in LDS, the sample's modes and
// columns in registers, sums and scans go through DPP moves within the 16
// lanes, and no barrier is needed.  With CC_FIRST photons or fewer the kernel
// writes the output rows, else the drawn modes for the steps that follow.
// What bounds it now: the chain of LDS reads and FP64 sums of a sample, with
// one or two waves per SIMD from 7 photons on (256 registers hold the columns).
// Measured, a launch per step -> one launch: 20 modes, 37 inputs of 6..8
// photons x 2,000 samples, 991 -> 180 us (26 launches of 21..49 us -> 3 of 14,
// 26 and 58 us); 9 photons x 50,000, 20 modes 875 -> 227 us, 64 modes 892 ->
// 310 us; 9 photons x 16, 64 modes 93 -> 56 us; 2 photons x 16, 39 -> 32 us.
// CC_FIRST: the steps below CC_MULTI, which sum without multiplicities.
// CC_FIRST_MODES: U and its padding take 65 KiB of LDS there, two workgroups a
// CU; above, one launch per step from step 1.
constexpr int CC_FIRST = CC_MULTI - 1;
constexpr int CC_FIRST_MODES = 64;

// Inclusive sums over the 16 lanes of a row (row_shr 1, 2, 4, 8; zeros enter).
__device__ __forceinline__ double row_scan(double v)
{
    v += row_dpp<0x111>(v);
    v += row_dpp<0x112>(v);
    v += row_dpp<0x114>(v);
    v += row_dpp<0x118>(v);
    return v;
}

// Photon K of a sample: row = output modes so far (16-byte offsets of their
// rows of U in LDS), pc = 16-byte offsets of its columns.  Returns the mode.
template <int K, int CH>
__device__ __forceinline__ int cc_first_step(const char *sU, int m, int ldu, const int (&row)[CC_FIRST],
                                             const int (&pc)[CC_FIRST], int lane, int shift, double u)
{
    auto at = [&](int r, int c) { return *reinterpret_cast<const cd *>(sU + r + c); };
    cd sub[K];
    if constexpr (K == 1) {
        sub[0] = {1.0, 0.0};
    } else {
        // 2^(K-2) terms, 2^CL per lane, Gray-code order; half column sums
        constexpr int TL = K - 2, CL = TL > 4 ? TL - 4 : 0;
        constexpr int active = TL > 4 ? 16 : 1 << TL;
        const uint32_t base = (uint32_t)lane << CL;
        const uint32_t g0 = base ^ (base >> 1);
        cd cs[K];
#pragma unroll
        for (int l = 0; l < K; l++) {
            const cd a = at(row[0], pc[l]);
            cs[l] = {0.5 * a.r, 0.5 * a.i};
        }
#pragma unroll
        for (int i = 1; i < K - 1; i++) {
            const double d = ((g0 >> (i - 1)) & 1) ? -0.5 : 0.5;
#pragma unroll
            for (int l = 0; l < K; l++) {
                const cd a = at(row[i], pc[l]);
                cs[l].r = fma(d, a.r, cs[l].r);
                cs[l].i = fma(d, a.i, cs[l].i);
            }
        }
#pragma unroll
        for (int l = 0; l < K; l++) sub[l] = {0.0, 0.0};
        double sign = CL == 0 && (base & 1) ? -1.0 : 1.0;
        if (active < 16 && lane >= active) sign = 0.0;
#pragma unroll
        for (int q = 0; q < (1 << CL); q++) {
            if (q) {
                const int b = __builtin_ctz(q);
                const uint32_t t = base + q;
                const double s = (((t >> b) ^ (t >> (b + 1))) & 1) ? -1.0 : 1.0;
#pragma unroll
                for (int l = 0; l < K; l++) {
                    const cd a = at(row[b + 1], pc[l]);
                    cs[l].r = fma(s, a.r, cs[l].r);
                    cs[l].i = fma(s, a.i, cs[l].i);
                }
            }
            cd P[K];
            P[0] = {1.0, 0.0};
            P[1] = cs[0];
#pragma unroll
            for (int l = 2; l < K; l++) P[l] = cmul(P[l - 1], cs[l - 1]);
            const double sg = (q & 1) ? -sign : sign;
            cd S = {sg, 0.0};
#pragma unroll
            for (int l = K - 1; l >= 1; l--) {
                if (l == K - 1) {
                    sub[l].r = fma(sg, P[l].r, sub[l].r);
                    sub[l].i = fma(sg, P[l].i, sub[l].i);
                    S = {sg * cs[l].r, sg * cs[l].i};
                } else {
                    cfma_acc(sub[l], P[l], S);
                    S = cmul(S, cs[l]);
                }
            }
            sub[0].r += S.r;
            sub[0].i += S.i;
        }
#pragma unroll
        for (int l = 0; l < K; l++) sub[l] = {row_sum(sub[l].r), row_sum(sub[l].i)};
    }
    // weights of candidate rows c * 16 + lane, then the draw as in cc_draw
    double wv[CH], total = 0.0;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int i = c * 16 + lane;
        wv[c] = 0.0;
        if (i < m) {
            cd a = {0.0, 0.0};
#pragma unroll
            for (int l = 0; l < K; l++) cfma_acc(a, at(i * ldu * 16, pc[l]), sub[l]);
            wv[c] = a.r * a.r + a.i * a.i;
        }
        total += row_sum(wv[c]);
    }
    const double target = u * total;
    int pick = m - 1;
    double below = 0.0;
    bool found = false;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const double incl = row_scan(wv[c]);
        const bool hit = c * 16 + lane < m && target < below + incl;
        const uint32_t mask = (uint32_t)(__ballot(hit) >> shift) & 0xFFFFu;
        if (!found && mask) {
            pick = c * 16 + (int)__builtin_ctz(mask);
            found = true;
        }
        below += row_sum(wv[c]);
    }
    return pick;
}

template <int K, int KMAX, int CH>
__device__ __forceinline__ void cc_first_steps(const char *sU, int m, int ldu, int (&row)[CC_FIRST],
                                               const int (&pc)[CC_FIRST], int (&r)[CC_FIRST], int lane, int shift,
                                               double my_u)
{
    if constexpr (K <= KMAX) {
        const double u = __shfl(my_u, K - 1, 16);
        r[K - 1] = cc_first_step<K, CH>(sU, m, ldu, row, pc, lane, shift, u);
        row[K - 1] = r[K - 1] * ldu * 16;
        cc_first_steps<K + 1, KMAX, CH>(sU, m, ldu, row, pc, r, lane, shift, my_u);
    }
}

// Photons 1..KMAX of every sample (KMAX = min(n, CC_FIRST)); rows of U up to
// 16 CH.  out: the occupation rows when n == KMAX, else unused.
template <int KMAX, int CH>
__global__ void __launch_bounds__(256) cc_first_kernel(const cd *__restrict__ U, int m, int n, int64_t count,
                                                       uint64_t seed, uint64_t first,
                                                       const int32_t *__restrict__ pc_all, int32_t *__restrict__ r_all,
                                                       const int64_t *__restrict__ gidx, int32_t *__restrict__ out)
{
    extern __shared__ cd s_u[];
    const int ldu = m | 1;   // no bank conflicts down a column
    for (int e = threadIdx.x; e < m * m; e += 256) s_u[(e / m) * ldu + e % m] = U[e];
    __syncthreads();
    const int lane = threadIdx.x & 15, shift = threadIdx.x & 48;
    // the 16 lanes of a sample run together; a wave's samples past the end repeat the last one
    for (int64_t s0 = (int64_t)blockIdx.x * 16; s0 < count; s0 += (int64_t)gridDim.x * 16) {
        const int64_t mine = s0 + (threadIdx.x >> 4);
        const int64_t s = mine < count ? mine : count - 1;
        const int64_t global = gidx ? gidx[s] : s;
        int pc[CC_FIRST], row[CC_FIRST], r[CC_FIRST];
#pragma unroll
        for (int l = 0; l < KMAX; l++) pc[l] = pc_all[s * n + l] * 16;
        const double my_u = uniform01(seed, first + (uint64_t)global, (uint64_t)(n - 1 + lane));   // photon lane + 1
        cc_first_steps<1, KMAX, CH>(reinterpret_cast<const char *>(s_u), m, ldu, row, pc, r, lane, shift, my_u);
        if (mine < count) {
            if (n == KMAX) {
                int32_t *o = out + global * m;
#pragma unroll
                for (int c = 0; c < CH; c++) {
                    const int i = c * 16 + lane;
                    int v = 0;
#pragma unroll
                    for (int k = 0; k < KMAX; k++) v += r[k] == i ? 1 : 0;
                    if (i < m) o[i] = v;
                }
            } else {
#pragma unroll
                for (int k = 0; k < KMAX; k++)
                    if (lane == k) r_all[s * n + k] = r[k];
            }
        }
    }
}

template <int KMAX>
static int launch_first(int kmax, const cd *U, int m, int n, int64_t count, uint64_t seed, uint64_t first,
                        const int32_t *pc, int32_t *r, const int64_t *gidx, int32_t *out, int cus, hipStream_t st)
{
    if constexpr (KMAX > CC_FIRST) {
        set_error("internal: first steps out of range");
        return ERR_ARG;
    } else {
        if (kmax != KMAX) return launch_first<KMAX + 1>(kmax, U, m, n, count, seed, first, pc, r, gidx, out, cus, st);
        auto kp = m <= 32 ? cc_first_kernel<KMAX, 2> : cc_first_kernel<KMAX, 4>;
        const size_t lds = sizeof(cd) * (size_t)m * (m | 1);
        int per_cu = 0;
        PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kp), 256, lds));
        const int grid = (int)std::min<int64_t>((count + 15) / 16, (int64_t)cus * std::max(per_cu, 1));
        hipLaunchKernelGGL(kp, dim3(grid), dim3(256), lds, st, U, m, n, count, seed, first, pc, r, gidx, out);
        PCVL_HIP_CHECK(hipGetLastError());
        return OK;
    }
}

// Steps from CC_SLICED on: a sample's units are cut into slices (at most
// cc_slice_cap(K), by its own rows only, so that its draws do not depend on how
// many samples a call holds).  cc_count_kernel plans the slices of every
// sample, launch_slice_owners lists them, cc_slice_kernel runs them from one
// cursor (so that samples of very different cost, and a single one, balance
// over the device) and writes each slice's partial sub-permanents, and
// cc_slice_draw_kernel sums a sample's slices in order and draws.
constexpr size_t CC_PART_BYTES = size_t(256) << 20;   // slices of one chunk of samples

// Samples of one chunk [s0, s0 + nchunk).
template <int K>
__global__ void __launch_bounds__(64) cc_count_kernel(int n, int64_t s0, int64_t nchunk,
                                                      const int32_t *__restrict__ r_all, int32_t *__restrict__ nslices,
                                                      unsigned long long *__restrict__ cursor)
{
    __shared__ CCShared<K> sh;
    const int lane = threadIdx.x;
    if (blockIdx.x == 0 && lane == 0) *cursor = 0ull;
    for (int64_t t = blockIdx.x; t < nchunk; t += gridDim.x) {
        if (lane < K - 1) sh.r[lane] = r_all[(s0 + t) * n + lane];
        __syncthreads();
        const CCPlan pl = cc_plan<K>(sh, lane);
        if (lane == 0) nslices[t] = pl.slices;
        __syncthreads();
    }
}

template <int K>
__global__ void __launch_bounds__(64, K <= 20 ? 3 : 2) cc_slice_kernel(const cd *__restrict__ U, int m, int n, int64_t s0,
                                                      int64_t nchunk, const int32_t *__restrict__ pc_all,
                                                      const int32_t *__restrict__ r_all,
                                                      const int64_t *__restrict__ slice0,
                                                      const uint64_t *__restrict__ owner,
                                                      unsigned long long *__restrict__ cursor, cd *__restrict__ partials)
{
    __shared__ CCShared<K> sh;
    const int lane = threadIdx.x;
    __shared__ SliceQueue::State squeue;
    SliceQueue queue(squeue, slice0[nchunk]);
    int64_t last = -1;   // sample in LDS
    CCPlan pl = {};
    for (int64_t g; (g = queue.next(cursor)) >= 0;) {
        int64_t t;
        int slice;
        slice_owner(owner[g], t, slice);
        if (t != last) {
            last = t;
            const int64_t s = s0 + t;
            if (lane < K) sh.pc[lane] = pc_all[s * n + lane];
            if (lane < K - 1) sh.r[lane] = r_all[s * n + lane];
            __syncthreads();
            pl = cc_plan<K>(sh, lane);
            load_rows<K>(sh, pl, U, m, lane);
        }
        const uint32_t per = (pl.units + (uint32_t)pl.slices - 1) / (uint32_t)pl.slices;
        const uint32_t u0 = (uint32_t)slice * per;
        const uint32_t u1 = u0 + per < pl.units ? u0 + per : pl.units;
        subperms_units<K>(sh, pl, u0, u1, lane, partials + g * K);
        __syncthreads();
    }
}

template <int K>
__global__ void __launch_bounds__(64) cc_slice_draw_kernel(const cd *__restrict__ U, int m, int n, int64_t s0,
                                                           int64_t nchunk, uint64_t seed, uint64_t first,
                                                           const int32_t *__restrict__ pc_all,
                                                           int32_t *__restrict__ r_all,
                                                           const int64_t *__restrict__ gidx,
                                                           const int64_t *__restrict__ slice0,
                                                           const cd *__restrict__ partials)
{
    __shared__ CCShared<K> sh;
    const int lane = threadIdx.x;
    for (int64_t t = blockIdx.x; t < nchunk; t += gridDim.x) {
        const int64_t s = s0 + t;
        const uint64_t stream = first + (uint64_t)(gidx ? gidx[s] : s);
        if (lane < K) {
            sh.pc[lane] = pc_all[s * n + lane];
            cd v = {0.0, 0.0};
            const int64_t g1 = slice0[t + 1];
            for (int64_t g = slice0[t]; g < g1; g++) {   // in slice order
                const cd x = partials[g * K + lane];
                v.r += x.r;
                v.i += x.i;
            }
            sh.sub[lane] = v;
        }
        __syncthreads();
        cc_draw<K>(sh, U, m, n, s, seed, stream, lane, r_all);
        __syncthreads();
    }
}

// Occupation vector of each sample from its drawn modes.
__global__ void cc_finish_kernel(const int32_t *__restrict__ r_all, int m, int n, int64_t count,
                                 int32_t *__restrict__ out)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count * m) return;
    const int64_t s = e / m;
    const int i = (int)(e % m);
    int v = 0;
    for (int k = 0; k < n; k++) v += (r_all[s * n + k] == i) ? 1 : 0;
    out[e] = v;
}

// Workspace of the sliced steps, for chunks of samples sized by the largest
// step of the call: slice counts | slice offsets | cursor | owners | partial sums.
struct CCSliceWork {
    int64_t chunk = 0;
    size_t o_s0 = 0, o_cur = 0, o_own = 0, o_part = 0, total = 0;
};

static CCSliceWork cc_slice_layout(int n, int64_t chunk)
{
    CCSliceWork w;
    if (n < CC_SLICED || chunk <= 0) return w;
    const size_t cap = (size_t)cc_slice_cap(n);
    w.chunk = chunk;
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    const size_t c = (size_t)chunk;
    w.o_s0 = al(sizeof(int32_t) * c);
    w.o_cur = w.o_s0 + al(sizeof(int64_t) * (c + 1));
    w.o_own = w.o_cur + 256;
    w.o_part = w.o_own + al(sizeof(uint64_t) * c * cap);
    w.total = w.o_part + al(sizeof(cd) * c * cap * (size_t)n);
    return w;
}

// The chunks that `room` bytes hold, CC_PART_BYTES of slices at most and one
// sample at least.
static CCSliceWork cc_slice_work(int n, int64_t count, size_t room = SIZE_MAX)
{
    if (n < CC_ONE_WAVE && count <= CC_ONE_WAVE_COUNT) return {};   // every step in one wave per sample
    const size_t per_sample = (size_t)cc_slice_cap(n) * ((size_t)n * sizeof(cd) + sizeof(uint64_t));
    int64_t lo = std::min<int64_t>(count, 1);
    int64_t hi = std::min(count, std::max<int64_t>(1, (int64_t)(CC_PART_BYTES / std::max<size_t>(per_sample, 1))));
    if (cc_slice_layout(n, hi).total <= room) lo = hi;
    while (lo + 1 < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (cc_slice_layout(n, mid).total <= room) lo = mid;
        else hi = mid;
    }
    return cc_slice_layout(n, lo);
}

template <int K>
static int launch_step(int k, const cd *U, int m, int n, int64_t count, uint64_t seed, uint64_t first,
                       const int32_t *pc, int32_t *r, const CCSliceWork &w, char *work, int cus, hipStream_t st,
                       const int64_t *gidx = nullptr)
{
    if constexpr (K > CC_MAX_N) {
        set_error("internal: photon step out of range");
        return ERR_ARG;
    } else {
        if (k != K) return launch_step<K + 1>(k, U, m, n, count, seed, first, pc, r, w, work, cus, st, gidx);
        if (cc_one_wave(K, m, count)) {
            constexpr int KS = K <= CC_ONE_WAVE ? K : 1;   // the others have no such kernel
            auto kp = cc_step_kernel<KS, (KS >= CC_MULTI)>;
            if constexpr (KS >= CC_MULTI && KS < CC_SLICED) {
                if (m > CC_MULTI_MODES) kp = cc_step_kernel<KS, false>;
            }
            int per_cu = 0;
            PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kp), 64, 0));
            if (per_cu < 1) per_cu = 1;
            const int grid = (int)std::min<int64_t>(count, (int64_t)cus * per_cu);
            hipLaunchKernelGGL(kp, dim3(grid), dim3(64), 0, st, U, m, n, count, seed, first, pc, r, gidx);
            PCVL_HIP_CHECK(hipGetLastError());
        } else if constexpr (K >= CC_SLICED) {
            int per_cu_s = 0, per_cu_d = 0;
            PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu_s, reinterpret_cast<const void *>(&cc_slice_kernel<K>), 64, 0));
            PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu_d, reinterpret_cast<const void *>(&cc_slice_draw_kernel<K>), 64, 0));
            per_cu_s = std::max(per_cu_s, 1);
            per_cu_d = std::max(per_cu_d, 1);
            int32_t *ns = reinterpret_cast<int32_t *>(work);
            int64_t *slice0 = reinterpret_cast<int64_t *>(work + w.o_s0);
            unsigned long long *cursor = reinterpret_cast<unsigned long long *>(work + w.o_cur);
            uint64_t *owner = reinterpret_cast<uint64_t *>(work + w.o_own);
            cd *partials = reinterpret_cast<cd *>(work + w.o_part);
            for (int64_t s0 = 0; s0 < count; s0 += w.chunk) {
                const int64_t nchunk = std::min(w.chunk, count - s0);
                const int gd = (int)std::min<int64_t>(nchunk, (int64_t)cus * per_cu_d);
                hipLaunchKernelGGL((cc_count_kernel<K>), dim3((unsigned)std::min<int64_t>(nchunk, (int64_t)cus * 16)),
                                   dim3(64), 0, st, n, s0, nchunk, r, ns, cursor);
                PCVL_HIP_CHECK(hipGetLastError());
                int rc = launch_slice_owners(ns, nchunk, slice0, owner, st);
                if (rc != OK) return rc;
                const int gs = (int)std::min<int64_t>(nchunk * cc_slice_cap(K), (int64_t)cus * per_cu_s);
                hipLaunchKernelGGL((cc_slice_kernel<K>), dim3(gs), dim3(64), 0, st, U, m, n, s0, nchunk, pc, r, slice0,
                                   owner, cursor, partials);
                PCVL_HIP_CHECK(hipGetLastError());
                hipLaunchKernelGGL((cc_slice_draw_kernel<K>), dim3(gd), dim3(64), 0, st, U, m, n, s0, nchunk, seed,
                                   first, pc, r, gidx, slice0, partials);
                PCVL_HIP_CHECK(hipGetLastError());
            }
        }
        return OK;
    }
}

// Every photon of `count` samples whose columns are in pc, and their output
// rows (row gidx[s], or s): the first steps, the steps after them, the rows.
static int cc_run(const cd *U, int m, int n, int64_t count, uint64_t seed, uint64_t first, const int32_t *pc,
                  int32_t *r, const CCSliceWork &w, char *work, const int64_t *gidx, int32_t *out, int cus, hipStream_t st)
{
    int k = 1;
    if (m <= CC_FIRST_MODES) {
        const int kmax = std::min(n, CC_FIRST);
        const int rc = launch_first<1>(kmax, U, m, n, count, seed, first, pc, r, gidx, out, cus, st);
        if (rc != OK || n == kmax) return rc;
        k = kmax + 1;
    }
    for (; k <= n; k++) {
        const int rc = launch_step<1>(k, U, m, n, count, seed, first, pc, r, w, work, cus, st, gidx);
        if (rc != OK) return rc;
    }
    const int64_t tot = count * m;
    if (gidx)
        hipLaunchKernelGGL(cc_finish_multi_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, r, gidx, m, n,
                           count, out);
    else
        hipLaunchKernelGGL(cc_finish_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, r, m, n, count, out);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

} // namespace pcvl

using namespace pcvl;

// pc (count*n) | r (count*n) | cols (CC_MAX_N)
static size_t cc_head_bytes(int n, int64_t count)
{
    return sizeof(int32_t) * ((size_t)2 * (size_t)count * (size_t)std::max(n, 1) + (size_t)CC_MAX_N);
}

// The head, then from a 256-byte boundary the slices of the sliced steps (14
// photons and more).
static size_t cc_work_bytes(int n, int64_t count, size_t slices)
{
    const size_t head = cc_head_bytes(n, count);
    return slices ? ((head + 255) & ~size_t(255)) + slices : head;
}

extern "C" int pcvl_cc_workspace_bytes(int n, int64_t count, size_t *bytes)
{
    PCVL_ARG_CHECK(bytes != nullptr, "bytes is null");
    PCVL_ARG_CHECK(n >= 0 && n <= CC_MAX_N && count >= 0, "n outside [0, 30] or count < 0");
    *bytes = cc_work_bytes(n, count, cc_slice_work(n, count).total);
    return OK;
}

extern "C" int pcvl_cc_workspace_least_bytes(int n, int64_t count, size_t *bytes)
{
    PCVL_ARG_CHECK(bytes != nullptr, "bytes is null");
    PCVL_ARG_CHECK(n >= 0 && n <= CC_MAX_N && count >= 0, "n outside [0, 30] or count < 0");
    *bytes = cc_work_bytes(n, count, cc_slice_work(n, count, 0).total);
    return OK;
}

extern "C" int pcvl_cc_samples(const double *d_U, int m, const int32_t *h_in_occ, int64_t count, uint64_t seed,
                               uint64_t first_sample, int32_t *d_out, void *d_work, size_t work_bytes,
                               hipStream_t stream)
{
    PCVL_ARG_CHECK(m >= 1 && m <= CC_MAX_M, "mode count outside [1, 256]");
    PCVL_ARG_CHECK(h_in_occ != nullptr, "input state is null");
    PCVL_ARG_CHECK(count >= 0, "count < 0");
    std::vector<int32_t> cols;
    for (int i = 0; i < m; i++) {
        PCVL_ARG_CHECK(h_in_occ[i] >= 0, "negative occupation");
        for (int v = 0; v < h_in_occ[i]; v++) cols.push_back(i);
    }
    PCVL_ARG_CHECK((int)cols.size() <= CC_MAX_N, "more than 30 photons");
    if (count == 0) return OK;
    PCVL_ARG_CHECK(d_U && d_out, "null device buffer");
    const int n = (int)cols.size();
    size_t need = 0;
    pcvl_cc_workspace_least_bytes(n, count, &need);
    PCVL_ARG_CHECK(d_work != nullptr && work_bytes >= need, "workspace missing or smaller than pcvl_cc_workspace_least_bytes");
    if (n == 0) {
        const int64_t tot = count * m;
        hipLaunchKernelGGL(cc_finish_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, stream,
                           static_cast<const int32_t *>(d_work), m, 0, count, d_out);
        PCVL_HIP_CHECK(hipGetLastError());
        return OK;
    }
    // workspace: pc (count*n) | r (count*n) | cols (CC_MAX_N) | slices
    int32_t *pc = static_cast<int32_t *>(d_work);
    int32_t *r = pc + (size_t)count * n;
    int32_t *d_cols = r + (size_t)count * n;
    const size_t head = (cc_head_bytes(n, count) + 255) & ~size_t(255);
    char *slices = static_cast<char *>(d_work) + head;
    const CCSliceWork work = cc_slice_work(n, count, work_bytes > head ? work_bytes - head : 0);
    PCVL_HIP_CHECK(hipMemcpyAsync(d_cols, cols.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, stream));
    const cd *U = reinterpret_cast<const cd *>(d_U);
    int dev = 0, cus = 0;
    PCVL_HIP_CHECK(hipGetDevice(&dev));
    PCVL_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    hipLaunchKernelGGL(cc_init_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, d_cols, n, count,
                       seed, first_sample, pc);
    PCVL_HIP_CHECK(hipGetLastError());
    const int rc = cc_run(U, m, n, count, seed, first_sample, pc, r, work, slices, nullptr, d_out, cus, stream);
    if (rc != OK) return rc;
    // the host column list copied above must outlive the copy
    PCVL_HIP_CHECK(hipStreamSynchronize(stream));
    return OK;
}

extern "C" int pcvl_cc_samples_multi(const double *d_U, int m, const int32_t *h_inputs, const int64_t *h_counts,
                                     int ninputs, uint64_t seed, uint64_t first_sample, int32_t *d_out,
                                     hipStream_t stream)
{
    PCVL_ARG_CHECK(m >= 1 && m <= CC_MAX_M, "mode count outside [1, 256]");
    PCVL_ARG_CHECK(ninputs >= 0 && (ninputs == 0 || (h_inputs && h_counts)), "null input table");
    // photon columns of each input, its photon number and its first output row
    std::vector<std::vector<int32_t>> cols((size_t)ninputs);
    std::vector<int64_t> row0((size_t)ninputs + 1, 0);
    for (int i = 0; i < ninputs; i++) {
        PCVL_ARG_CHECK(h_counts[i] >= 0, "negative sample count");
        for (int q = 0; q < m; q++) {
            const int32_t v = h_inputs[(size_t)i * m + q];
            PCVL_ARG_CHECK(v >= 0, "negative occupation");
            for (int t = 0; t < v; t++) cols[(size_t)i].push_back(q);
        }
        PCVL_ARG_CHECK(cols[(size_t)i].size() <= (size_t)CC_MAX_N, "more than 30 photons");
        row0[(size_t)i + 1] = row0[(size_t)i] + h_counts[i];
    }
    const int64_t total = row0[(size_t)ninputs];
    if (total == 0) return OK;
    PCVL_ARG_CHECK(d_U && d_out, "null device buffer");
    // group the inputs by photon number; each group runs one launch sequence.
    // The tables of all groups (first sample and output row of each input, its
    // photon columns) go to the device in one copy.
    struct Group { int n; int64_t count = 0; std::vector<int> inputs; size_t o_start = 0, o_row = 0, o_cols = 0; };
    std::vector<Group> groups;
    for (int i = 0; i < ninputs; i++) {
        if (h_counts[i] == 0) continue;
        const int n = (int)cols[(size_t)i].size();
        size_t g = 0;
        while (g < groups.size() && groups[g].n != n) g++;
        if (g == groups.size()) { groups.emplace_back(); groups[g].n = n; }
        groups[g].inputs.push_back(i);
        groups[g].count += h_counts[i];
    }
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    std::vector<char> tab;
    int64_t gmax = 0;
    int nmax = 1;
    size_t b_part = 0;
    for (Group &g : groups) {
        const size_t ni = g.inputs.size();
        g.o_start = al(tab.size());
        g.o_row = g.o_start + al(sizeof(int64_t) * ni);
        g.o_cols = g.o_row + al(sizeof(int64_t) * ni);
        tab.resize(g.o_cols + al(sizeof(int32_t) * ni * (size_t)std::max(g.n, 1)), 0);
        int64_t at = 0;
        for (size_t q = 0; q < ni; q++) {
            const int i = g.inputs[q];
            reinterpret_cast<int64_t *>(tab.data() + g.o_start)[q] = at;
            reinterpret_cast<int64_t *>(tab.data() + g.o_row)[q] = row0[(size_t)i];
            for (int l = 0; l < g.n; l++)
                reinterpret_cast<int32_t *>(tab.data() + g.o_cols)[q * (size_t)g.n + l] = cols[(size_t)i][(size_t)l];
            at += h_counts[i];
        }
        gmax = std::max(gmax, g.count);
        nmax = std::max(nmax, g.n);
    }
    size_t least = 0;   // where the device is nearly full
    for (const Group &g : groups) {
        b_part = std::max(b_part, cc_slice_work(g.n, g.count).total);
        least = std::max(least, cc_slice_work(g.n, g.count, 0).total);
    }
    // device block: pc | r (gmax * nmax each) | gidx (gmax) | tables | slices
    const size_t b_pr = al(sizeof(int32_t) * (size_t)gmax * nmax);
    const size_t b_gidx = al(sizeof(int64_t) * (size_t)gmax);
    const size_t b_head = 2 * b_pr + b_gidx + al(tab.size());
    char *blk = nullptr;
    hipError_t e = ws_alloc(reinterpret_cast<void **>(&blk), b_head + al(b_part), stream);
    while (e == hipErrorOutOfMemory && least < b_part) {
        (void)hipGetLastError();
        b_part = std::max(least, b_part / 4);
        e = ws_alloc(reinterpret_cast<void **>(&blk), b_head + al(b_part), stream);
    }
    PCVL_HIP_CHECK(e);
    int32_t *pc = reinterpret_cast<int32_t *>(blk);
    int32_t *r = reinterpret_cast<int32_t *>(blk + b_pr);
    int64_t *d_gidx = reinterpret_cast<int64_t *>(blk + 2 * b_pr);
    char *d_tab = blk + 2 * b_pr + b_gidx;
    char *slices = d_tab + al(tab.size());
    const cd *U = reinterpret_cast<const cd *>(d_U);
    int dev = 0, cus = 0;
    int rc = OK;
    e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipMemcpyAsync(d_tab, tab.data(), tab.size(), hipMemcpyHostToDevice, stream);
    if (e != hipSuccess) { set_error(std::string("cc multi tables: ") + hipGetErrorString(e)); rc = ERR_HIP; }
    for (const Group &g : groups) {
        if (rc != OK) break;
        const unsigned blocks = (unsigned)((g.count + 255) / 256);
        hipLaunchKernelGGL(cc_init_multi_kernel, dim3(blocks), dim3(256), 0, stream,
                           reinterpret_cast<const int32_t *>(d_tab + g.o_cols),
                           reinterpret_cast<const int64_t *>(d_tab + g.o_start),
                           reinterpret_cast<const int64_t *>(d_tab + g.o_row), (int)g.inputs.size(), g.n, g.count, seed,
                           first_sample, d_gidx, pc);
        e = hipGetLastError();
        if (e != hipSuccess) { set_error(std::string("cc_init_multi: ") + hipGetErrorString(e)); rc = ERR_HIP; break; }
        if (g.n > 0) {
            rc = cc_run(U, m, g.n, g.count, seed, first_sample, pc, r, cc_slice_work(g.n, g.count, b_part), slices, d_gidx,
                        d_out, cus, stream);
        } else {
            hipLaunchKernelGGL(cc_finish_multi_kernel, dim3((unsigned)((g.count * m + 255) / 256)), dim3(256), 0,
                               stream, r, d_gidx, m, 0, g.count, d_out);
            e = hipGetLastError();
            if (e != hipSuccess) { set_error(std::string("cc_finish_multi: ") + hipGetErrorString(e)); rc = ERR_HIP; }
        }
    }
    // the host tables must outlive their copy, and results are ready on return
    hipError_t se = hipStreamSynchronize(stream);
    hipError_t fe = hipFreeAsync(blk, stream);
    if (rc == OK && se != hipSuccess) { set_error(std::string("cc multi: ") + hipGetErrorString(se)); rc = ERR_HIP; }
    if (rc == OK && fe != hipSuccess) { set_error(std::string("hipFreeAsync(cc multi): ") + hipGetErrorString(fe)); rc = ERR_HIP; }
    return rc;
}
