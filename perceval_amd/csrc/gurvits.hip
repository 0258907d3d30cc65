// Gurvits' randomised permanent estimate, batched.
//
// Replaces xq.estimate_permanent_cx(M, iterations) as called from
// NaiveApproxBackend._compute_permanent and prob_amplitude_with_error
// (perceval/backends/_naive_approx.py:52-62; the estimator is Gurvits &
// Samorodnitsky 2002, docs/source/references.bib:1135).  For x uniform in
// {+1,-1}^n,
//     X(x) = (prod_j x_j) prod_i (sum_j a_ij x_j),   E[X] = perm(A),
// since every term of the expanded product that is not a permutation carries
// an odd power of some x_j.  The estimate is the mean of `iters` samples; its
// 99% error bound is the normal one, 2.5758 * sqrt((E|X|^2 - |mean|^2) / iters).
//
// Sample s of matrix b takes its signs from the 64 bits rand64(seed,
// stream0 + b, s) (bit j -> x_j = -1), so the oracle draws the same samples
// and a batch can be split across calls.  A matrix's samples are split into
// parts so that a small batch still fills the device; one wavefront per
// (matrix, part) stages A in LDS (zero-padded to NP x NP), lane l takes
// samples l, l + 64, ... of the part, forms y_i = sum_j x_j a_ij row by row
// (2 FMAs per broadcast LDS read) and multiplies the y_i into four chains by
// i mod 4; a finalize pass sums each matrix's parts in order.
#include "common.h"
#include "../../include/pcvl_hip.h"

#include <algorithm>
#include <vector>

namespace pcvl {

constexpr int GURVITS_MAX_N = 48;
constexpr int GURVITS_WAVES = 4;   // waves per workgroup of the matrix-core kernel

struct GurvitsItem {
    int64_t off;   // complex offset of the matrix
    int32_t n;
    int32_t pad;
};

// Scale of a matrix that keeps the FP64 products (see gurvits_int8_kernel).
constexpr int32_t GURVITS_FP64 = INT32_MIN;

template <int NP>
__device__ __forceinline__ cd gurvits_prod(const cd *y)
{
    cd p0 = y[0], p1 = y[1], p2 = y[2], p3 = y[3];
#pragma unroll
    for (int i = 4; i < NP; i++) {
        if ((i & 3) == 0) p0 = cmul(p0, y[i]);
        else if ((i & 3) == 1) p1 = cmul(p1, y[i]);
        else if ((i & 3) == 2) p2 = cmul(p2, y[i]);
        else p3 = cmul(p3, y[i]);
    }
    return cmul(cmul(p0, p1), cmul(p2, p3));
}

// One wavefront per (matrix, part): part q of a matrix takes samples
// [q * per, min(iters, (q + 1) * per)), lane l of them l, l + 64, ...; it
// writes (sum Re X, sum Im X, sum |X|^2) to its slot, and the finalize kernel
// sums a matrix's parts in order (deterministic for a given split).
template <int NP>
__global__ void __launch_bounds__(64) gurvits_kernel(const cd *__restrict__ mats, const GurvitsItem *__restrict__ items,
                                                     int64_t count, int parts, int64_t iters, int64_t per,
                                                     uint64_t seed, uint64_t stream0, double *__restrict__ partial)
{
    __shared__ cd sA[NP * NP];
    const int lane = threadIdx.x;
    const int64_t nwork = count * parts;
    for (int64_t wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
        const int64_t b = wi / parts;
        const int64_t q = wi % parts;
        const int n = __builtin_amdgcn_readfirstlane(items[b].n);
        const int64_t off = items[b].off;
        for (int e = lane; e < NP * NP; e += 64) {
            const int i = e / NP, j = e % NP;
            sA[e] = (i < n && j < n) ? mats[off + (int64_t)i * n + j] : cd{0.0, 0.0};
        }
        __syncthreads();
        const uint64_t mask = n >= 64 ? ~0ull : ((1ull << n) - 1);
        const int64_t s_lo = q * per;
        const int64_t s_hi = (s_lo + per < iters) ? s_lo + per : iters;
        cd sum = {0.0, 0.0};
        double sq = 0.0;
        for (int64_t s = s_lo + lane; s < s_hi; s += 64) {
            const uint64_t bits = rand64(seed, stream0 + (uint64_t)b, (uint64_t)s);
            double x[NP];
#pragma unroll
            for (int j = 0; j < NP; j++) x[j] = ((bits >> j) & 1) ? -1.0 : 1.0;
            cd p0 = {1.0, 0.0}, p1 = {1.0, 0.0}, p2 = {1.0, 0.0}, p3 = {1.0, 0.0};
            for (int i = 0; i < n; i++) {
                const cd *row = sA + i * NP;
                cd y = {0.0, 0.0};
#pragma unroll
                for (int j = 0; j < NP; j++) {   // zero padding beyond n adds nothing
                    const cd a = row[j];
                    y.r = fma(x[j], a.r, y.r);
                    y.i = fma(x[j], a.i, y.i);
                }
                const int c = i & 3;
                if (c == 0) p0 = cmul(p0, y);
                else if (c == 1) p1 = cmul(p1, y);
                else if (c == 2) p2 = cmul(p2, y);
                else p3 = cmul(p3, y);
            }
            cd X = cmul(cmul(p0, p1), cmul(p2, p3));
            if (__builtin_popcountll(bits & mask) & 1) X = {-X.r, -X.i};
            sum.r += X.r;
            sum.i += X.i;
            sq = fma(X.r, X.r, fma(X.i, X.i, sq));
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            sum.r += __shfl_xor(sum.r, o, 64);
            sum.i += __shfl_xor(sum.i, o, 64);
            sq += __shfl_xor(sq, o, 64);
        }
        if (lane == 0) {
            partial[3 * wi] = sum.r;
            partial[3 * wi + 1] = sum.i;
            partial[3 * wi + 2] = sq;
        }
        __syncthreads();
    }
}

// The same estimate with y = A x formed on the FP64 matrix cores, 16 samples
// at a time: Y (NP x 16) = A (NP x NP) X (NP x 16, entries +-1), real and
// imaginary parts as two products, by v_mfma_f64_16x16x4f64 over 16-row
// blocks rb and 4-column blocks kb.  Operand layouts of that instruction
// (checked on the device): lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]
// of the 16 x 4 and 4 x 16 operands, and D[l / 16 + 4 v][l % 16] in register v
// of the 16 x 16 result.  So lane l works on sample s0 + l % 16, takes
// x_j = bit j of that sample's signs for j = 4 kb + l / 16, and ends holding
// rows l / 16 + 4 v of every row block of y; the product over i < n is taken
// over those rows, then across the four lanes of the sample (lane ^ 16,
// lane ^ 32).  Lanes 0-15 accumulate.  A's fragments stay in registers up to
// NP = 32 and are read from LDS above.
typedef double gv_d4 __attribute__((ext_vector_type(4)));

template <int NP>
__global__ void __launch_bounds__(64 * GURVITS_WAVES, NP <= 32 ? 3 : 1) gurvits_mfma_kernel(const cd *__restrict__ mats,
                                                          const GurvitsItem *__restrict__ items, int64_t count,
                                                          int parts, int64_t iters, int64_t per, uint64_t seed,
                                                          uint64_t stream0, double *__restrict__ partial,
                                                          const int32_t *__restrict__ scale)
{
    constexpr int RB = NP / 16, KB = NP / 4;
    // A is read from LDS at each product: the registers it would take cost a
    // wave per SIMD, and the GURVITS_WAVES waves of a workgroup share one copy
    constexpr bool AREG = false;
    __shared__ cd sA[NP * NP];
    __shared__ double sred[GURVITS_WAVES][3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, quad = lane >> 4;
    const int64_t nwork = count * parts;
    for (int64_t wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
        const int64_t b = wi / parts;
        const int64_t q = wi % parts;
        if (scale && scale[b] != GURVITS_FP64) continue;   // taken by gurvits_int8_kernel
        const int n = __builtin_amdgcn_readfirstlane(items[b].n);
        const int64_t off = items[b].off;
        for (int e = threadIdx.x; e < NP * NP; e += 64 * GURVITS_WAVES) {
            const int i = e / NP, j = e % NP;
            sA[e] = (i < n && j < n) ? mats[off + (int64_t)i * n + j] : cd{0.0, 0.0};
        }
        __syncthreads();
        double ar[AREG ? RB * KB : 1], ai[AREG ? RB * KB : 1];
        if constexpr (AREG) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int kb = 0; kb < KB; kb++) {
                    const cd v = sA[(16 * rb + col) * NP + 4 * kb + quad];
                    ar[rb * KB + kb] = v.r;
                    ai[rb * KB + kb] = v.i;
                }
        }
        const uint64_t mask = n >= 64 ? ~0ull : ((1ull << n) - 1);
        const int64_t s_lo = q * per;
        const int64_t s_hi = (s_lo + per < iters) ? s_lo + per : iters;
        cd sum = {0.0, 0.0};
        double sq = 0.0;
        for (int64_t s0 = s_lo + 16 * wave; s0 < s_hi; s0 += 16 * GURVITS_WAVES) {
            const int64_t s = s0 + col;
            const bool valid = s < s_hi;
            const uint64_t bits = valid ? rand64(seed, stream0 + (uint64_t)b, (uint64_t)s) : 0ull;
            gv_d4 yr[RB], yi[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                yr[rb] = gv_d4{0.0, 0.0, 0.0, 0.0};
                yi[rb] = gv_d4{0.0, 0.0, 0.0, 0.0};
            }
#pragma unroll
            for (int kb = 0; kb < KB; kb++) {
                const double x = ((bits >> (4 * kb + quad)) & 1) ? -1.0 : 1.0;   // columns j >= n are zero in A
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    double a_r, a_i;
                    if constexpr (AREG) {
                        a_r = ar[rb * KB + kb];
                        a_i = ai[rb * KB + kb];
                    } else {
                        const cd v = sA[(16 * rb + col) * NP + 4 * kb + quad];
                        a_r = v.r;
                        a_i = v.i;
                    }
                    yr[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a_r, x, yr[rb], 0, 0, 0);
                    yi[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a_i, x, yi[rb], 0, 0, 0);
                }
            }
            // this lane's rows quad + 4 v of each block, then the sample's four lanes
            cd p = {1.0, 0.0};
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (16 * rb + quad + 4 * v < n) p = cmul(p, cd{yr[rb][v], yi[rb][v]});
            cd o = {__shfl_xor(p.r, 16, 64), __shfl_xor(p.i, 16, 64)};
            p = cmul(p, o);
            o = {__shfl_xor(p.r, 32, 64), __shfl_xor(p.i, 32, 64)};
            p = cmul(p, o);
            if (__builtin_popcountll(bits & mask) & 1) p = {-p.r, -p.i};
            if (valid && quad == 0) {
                sum.r += p.r;
                sum.i += p.i;
                sq = fma(p.r, p.r, fma(p.i, p.i, sq));
            }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            sum.r += __shfl_xor(sum.r, o, 64);
            sum.i += __shfl_xor(sum.i, o, 64);
            sq += __shfl_xor(sq, o, 64);
        }
        if (lane == 0) {
            sred[wave][0] = sum.r;
            sred[wave][1] = sum.i;
            sred[wave][2] = sq;
        }
        __syncthreads();
        if (threadIdx.x == 0) {   // the waves' sums in wave order
            double r = 0.0, im = 0.0, q2 = 0.0;
            for (int w = 0; w < GURVITS_WAVES; w++) {
                r += sred[w][0];
                im += sred[w][1];
                q2 += sred[w][2];
            }
            partial[3 * wi] = r;
            partial[3 * wi + 1] = im;
            partial[3 * wi + 2] = q2;
        }
        __syncthreads();
    }
}

// ---- y = A x in integers -----------------------------------------------------
//
// The signs are whole numbers, so y = A x can be formed exactly from the digits
// of a fixed-point A on the int8 matrix cores, 64 times the rate of the FP64
// ones.  Row i is scaled by a power of two to components below 1, and every
// component is exactly a 2^77 = sum_s d_s 2^(13 s) with six balanced digits
// d_s; d_s = lo + 64 hi splits a digit into two int8: one
// v_mfma_i32_16x16x64_i8 per digit takes the lo parts against x = +-1 in its
// first 32 products and the hi parts against +-64 in the other 32.  |sum d_s x|
// <= 2^17, so two digits share an int32, and three conversions and FMAs make a
// component of y: its last bit or two is all that is rounded, also where large
// entries of a row cancel.  Matrices with a component below 2^-24 of its row's
// largest (its 53 bits would not fit 2^-77 of it), or one that is not finite,
// keep the FP64 products.
// Error of the means against long double sums over the same draws (8 Haar
// submatrices, 65,536 draws, relative to the mean size of a draw's product):
// 9.8e-18, 9.4e-18, 1.5e-17 at orders 30, 21, 12, where the FP64 products give
// 3.1e-17, 1.8e-17, 1.8e-17.
// Operand slots: lane l and byte j of its 16 hold row (A) or sample (B) l % 16
// and slot 16 (l / 16) + j; A and B pair equal slots, whatever k the
// instruction gives them.  Slot t is column t % 32, lo part for t < 32, hi
// above.  The result's register v of lane l is row 4 (l / 16) + v of the row
// block and sample l % 16.  A padding row (i >= n) is 1 in column n, whose sign
// is always +1, so that it multiplies by y = 1.
typedef int gv_i4 __attribute__((ext_vector_type(4)));
constexpr int GURVITS_DIGITS = 6;   // of 13 bits: 2^77 a, |a| < 1
constexpr int GURVITS_SPAN = 24;    // 2^-77 is the last bit of components down to 2^-24 of the row's largest
// Rounds of waves that a call is cut into: each part is dispatched as its own
// workgroup (64 matrices of order 30, 10^6 samples, at five digits: 2.03 ms; 2.21
// ms with four rounds on resident waves, whose compute units do not run at one
// speed).
constexpr int GURVITS_ROUNDS = 8;
// Fragments kept at a time (10,922 matrices of orders up to 16, 5,461 above): a
// call's workspace does not grow with its matrices beyond this.
constexpr size_t GURVITS_CHUNK_BYTES = size_t(128) << 20;
// The integer products pay for their two more launches (about 30 us) and for a
// matrix's digits and fragments from so many samples of a call and of a matrix
// on.  FP64 -> integer products, us, at orders 17..32: 64 matrices, 2^20 samples
// in all 126 -> 105, 2^21 201 -> 133; 20,000 matrices of 209 samples 532 -> 614,
// of 419 825 -> 770, of 838 1,442 -> 1,081.  At orders 9..16: 64 matrices, 2^21
// samples 104 -> 106, 2^22 164 -> 148; 20,000 matrices of 419 samples 351 -> 390,
// of 838 566 -> 558; 2,000 of 2,097 174 -> 171.
constexpr bool gurvits_int8_pays(int nmax, int64_t count, int64_t iters)
{
    return nmax <= 16 ? iters >= 1024 && (double)count * (double)iters >= 0x1p22
                      : iters >= 512 && (double)count * (double)iters >= 0x1p21;
}

// Fragments of one matrix: [row block][component][digit][lane].
constexpr int gurvits_frags(int np) { return np / 16 * 2 * GURVITS_DIGITS * 64; }

template <int NP>
__global__ void __launch_bounds__(256) gurvits_digits_kernel(const cd *__restrict__ mats,
                                                             const GurvitsItem *__restrict__ items, int64_t count,
                                                             int split, gv_i4 *__restrict__ frags,
                                                             int32_t *__restrict__ scale)
{
    __shared__ cd sA[NP * NP];
    __shared__ int sexp[NP];
    __shared__ int sbad;
    const int tid = threadIdx.x;
    constexpr int RC = NP / 16 * 2, PER = gurvits_frags(NP) / RC;   // row blocks x components
    for (int64_t w = blockIdx.x; w < count * split; w += gridDim.x) {
        const int64_t b = w / split;
        const int rc0 = (int)(w % split);
        const int n = items[b].n;
        const int64_t off = items[b].off;
        if (tid == 0) sbad = 0;
        for (int e = tid; e < NP * NP; e += 256) {
            const int i = e / NP, j = e % NP;
            cd v = {0.0, 0.0};
            if (i < n && j < n) v = mats[off + (int64_t)i * n + j];
            else if (i >= n && j == n) v.r = 1.0;   // n < NP here
            sA[e] = v;
        }
        __syncthreads();
        for (int i = tid >> 3; i < NP; i += 32) {   // eight lanes per row
            double mx = 0.0, mn = INFINITY;        // largest and smallest nonzero component
            bool bad = false;
            for (int j = tid & 7; j < NP; j += 8) {
                const cd v = sA[i * NP + j];
                const double x = fabs(v.r), y = fabs(v.i);
                bad |= !(x < INFINITY) || !(y < INFINITY);
                mx = fmax(mx, fmax(x, y));
                mn = fmin(mn, fmin(x > 0.0 ? x : INFINITY, y > 0.0 ? y : INFINITY));
            }
#pragma unroll
            for (int o = 4; o >= 1; o >>= 1) {
                mx = fmax(mx, __shfl_xor(mx, o, 64));
                mn = fmin(mn, __shfl_xor(mn, o, 64));
                bad |= __shfl_xor((int)bad, o, 64) != 0;
            }
            bad |= mn < ldexp(mx, -GURVITS_SPAN);
            if ((tid & 7) == 0) {
                sexp[i] = bad || mx == 0.0 ? 0 : ilogb(mx) + 1;   // |components| 2^-e < 1
                if (bad) sbad = 1;
            }
        }
        __syncthreads();
        if (tid == 0 && rc0 == 0) {
            int E = 0;
            for (int i = 0; i < n; i++) E += sexp[i];
            for (int i = n; i < NP; i++) E += sexp[i];   // padding rows: 2^-1 each against an exponent of 1
            scale[b] = sbad ? GURVITS_FP64 : E;
        }
        if (!sbad) {
            // thread: dword d4 of lane f's 16 bytes, every digit of its four columns
            const int f = tid >> 2, d4 = tid & 3, g = f >> 4;
            for (int rc = rc0; rc < RC; rc += split) {
                const int comp = rc & 1, row = 16 * (rc >> 1) + (f & 15), e = sexp[row];
                uint32_t word[GURVITS_DIGITS] = {};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int col = (16 * g + 4 * d4 + j) & 31;
                    if (col >= NP) continue;
                    const cd a = sA[row * NP + col];
                    // a 2^(77 - e) = f 2^53 2^(ex + 24 - e), f's 53 bits shifted by 0..24 places
                    int ex;
                    const double fr = frexp(comp ? a.i : a.r, &ex);
                    const int64_t mant = (int64_t)ldexp(fr, 53);
                    __int128 v = mant == 0 ? (__int128)0 : (__int128)mant << (ex + GURVITS_SPAN - e);
#pragma unroll
                    for (int k = 0; k < GURVITS_DIGITS; k++) {   // balanced digits from the low end
                        const int d = k < GURVITS_DIGITS - 1 ? (int)(((int64_t)v & 8191) ^ 4096) - 4096 : (int)v;
                        v = (v - d) >> 13;
                        const int hi = (d + 32) >> 6;
                        word[k] |= (uint32_t)(uint8_t)(g >= 2 ? hi : d - 64 * hi) << (8 * j);
                    }
                }
                uint32_t *dst = reinterpret_cast<uint32_t *>(frags + (b * RC + rc) * PER);
#pragma unroll
                for (int k = 0; k < GURVITS_DIGITS; k++) dst[(k * 64 + f) * 4 + d4] = word[k];
            }
        }
        __syncthreads();
    }
}

// One wave per (matrix, part), 64 samples' signs at a time, 16 samples per
// product.  A's fragments stay in VGPRs.  Bound by the vector ALU (busy 88%;
// the matrix cores 30%): the conversions and FMAs of each y component and the
// product over rows.  64 matrices of order 30, 10^6 samples each, take 2.13 ms
// (4.79 ms on the FP64 matrix cores).
template <int NP>
__global__ void __launch_bounds__(64, NP <= 16 ? 4 : 3) gurvits_int8_kernel(const gv_i4 *__restrict__ frags,
                                                                             const GurvitsItem *__restrict__ items,
                                                                             int64_t count, int parts, int64_t iters,
                                                                             int64_t per, uint64_t seed,
                                                                             uint64_t stream0,
                                                                             double *__restrict__ partial,
                                                                             const int32_t *__restrict__ scale)
{
    constexpr int RB = NP / 16, ND = GURVITS_DIGITS;
    const int lane = threadIdx.x;
    const int col = lane & 15, quad = lane >> 4;
    const int64_t nwork = count * parts;
    // signs to bytes: x = base ^ (byte mask & flip): +-1 in the lo slots, +-64 in the hi ones
    const uint32_t xbase = quad < 2 ? 0x01010101u : 0x40404040u;
    const uint32_t xflip = quad < 2 ? 0xFEFEFEFEu : 0x80808080u;
    for (int64_t wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
        const int64_t b = wi / parts;
        const int64_t q = wi % parts;
        if (scale[b] == GURVITS_FP64) continue;
        const int n = __builtin_amdgcn_readfirstlane(items[b].n);
        gv_i4 a[RB][2][ND];
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int s = 0; s < ND; s++)
                    a[rb][c][s] = frags[b * gurvits_frags(NP) + ((rb * 2 + c) * ND + s) * 64 + lane];
        const uint32_t mask = n >= 32 ? ~0u : ((1u << n) - 1);
        const int64_t s_lo = q * per;
        const int64_t s_hi = (s_lo + per < iters) ? s_lo + per : iters;
        cd sum = {0.0, 0.0};
        double sq = 0.0;
        for (int64_t s0 = s_lo; s0 < s_hi; s0 += 64) {
            // signs of sample s0 + lane; the columns from n on keep +1
            const uint32_t mine = (uint32_t)rand64(seed, stream0 + (uint64_t)b, (uint64_t)(s0 + lane)) & mask;
#pragma unroll 1
            for (int sub = 0; sub < 4; sub++) {
                if (s0 + 16 * sub >= s_hi) break;
                const uint32_t bits = (uint32_t)__shfl((int)mine, 16 * sub + col, 64);
                const uint32_t half = bits >> (16 * (quad & 1));
                gv_i4 x;
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    const uint32_t nib = (half >> (4 * w)) & 15u;
                    const uint32_t one = __umul24(nib, 0x204081u) & 0x01010101u;   // bit k to byte k
                    uint32_t up = one << 8;
                    asm("" : "+v"(up));   // or the byte mask becomes a quarter-rate multiplication by 255
                    x[w] = (int)(((up - one) & xflip) ^ xbase);
                }
                // y comes out as 2^25 times the scaled row's sum, four or eight
                // rows to a lane; the sign is prod_j x_j, in one of the
                // sample's four lanes
                const double start = RB == 2 ? 0x1p-200 : 0x1p-100;
                cd p = {quad == 0 && (__builtin_popcount(bits) & 1) ? -start : start, 0.0};
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    double y[2][4];
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        // a pair of digits at a time, the high one first
#pragma unroll
                        for (int s = ND - 2; s >= 0; s -= 2) {
                            const gv_i4 lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[rb][c][s], x, gv_i4{0, 0, 0, 0}, 0, 0, 0);
                            const gv_i4 hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[rb][c][s + 1], x, gv_i4{0, 0, 0, 0}, 0, 0, 0);
                            const double unit = s == 4 ? 1.0 : s == 2 ? 0x1p-26 : 0x1p-52;
#pragma unroll
                            for (int v = 0; v < 4; v++) {
                                const double t = (double)((hi[v] << 13) + lo[v]);
                                y[c][v] = s == ND - 2 ? t : fma(t, unit, y[c][v]);
                            }
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 4; v++) p = cmul(p, cd{y[0][v], y[1][v]});
                }
                // this lane's rows, then the sample's four lanes
                cd o = {__shfl_xor(p.r, 16, 64), __shfl_xor(p.i, 16, 64)};
                p = cmul(p, o);
                o = {__shfl_xor(p.r, 32, 64), __shfl_xor(p.i, 32, 64)};
                p = cmul(p, o);
                // all four lanes hold the product: each adds one group of 16 in four
                if (quad == sub && s0 + 16 * sub + col < s_hi) {
                    sum.r += p.r;
                    sum.i += p.i;
                    sq = fma(p.r, p.r, fma(p.i, p.i, sq));
                }
            }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            sum.r += __shfl_xor(sum.r, o, 64);
            sum.i += __shfl_xor(sum.i, o, 64);
            sq += __shfl_xor(sq, o, 64);
        }
        if (lane == 0) {
            partial[3 * wi] = sum.r;
            partial[3 * wi + 1] = sum.i;
            partial[3 * wi + 2] = sq;
        }
    }
}

// scale: powers of two of the matrices' rows that the sums leave out (NULL or
// GURVITS_FP64: none).
// LANES: 64 a matrix, or one where it has few parts (200,000 matrices of order 12
// and one part: 1,021 -> 956 us a call).
template <int LANES>
__global__ void gurvits_finalize_kernel(const double *__restrict__ partial, int64_t count, int parts, int64_t iters,
                                        const int32_t *__restrict__ scale, cd *__restrict__ est,
                                        double *__restrict__ err)
{
    const int64_t b = (int64_t)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
    const int lane = threadIdx.x % LANES;
    if (b >= count) return;
    double sr = 0.0, si = 0.0, sq = 0.0;
    for (int q = lane; q < parts; q += LANES) {
        const double *pp = partial + 3 * (b * parts + q);
        sr += pp[0];
        si += pp[1];
        sq += pp[2];
    }
#pragma unroll
    for (int o = LANES / 2; o >= 1; o >>= 1) {
        sr += __shfl_xor(sr, o, 64);
        si += __shfl_xor(si, o, 64);
        sq += __shfl_xor(sq, o, 64);
    }
    if (lane != 0) return;
    const double inv = 1.0 / (double)iters;
    const cd mean = {sr * inv, si * inv};
    const double var = sq * inv - (mean.r * mean.r + mean.i * mean.i);
    const int E = scale && scale[b] != GURVITS_FP64 ? scale[b] : 0;
    est[b] = {ldexp(mean.r, E), ldexp(mean.i, E)};
    err[b] = ldexp(2.5758293035489004 * sqrt((var > 0.0 ? var : 0.0) * inv), E);
}

template <int NP>
static int launch_gurvits(const cd *mats, const GurvitsItem *items, int64_t count, int parts, int64_t iters,
                          int64_t per, uint64_t seed, uint64_t stream0, double *partial, const int32_t *scale,
                          hipStream_t st)
{
    int dev = 0, cus = 0, per_cu = 0;
    PCVL_HIP_CHECK(hipGetDevice(&dev));
    PCVL_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    // orders above 8: y = A x on the matrix cores (NP a multiple of 16)
    constexpr bool MF = NP >= 16 && NP % 16 == 0;
    const void *kp = MF ? reinterpret_cast<const void *>(&gurvits_mfma_kernel<MF ? NP : 16>)
                        : reinterpret_cast<const void *>(&gurvits_kernel<NP>);
    const int threads = MF ? 64 * GURVITS_WAVES : 64;
    PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kp, threads, 0));
    if (per_cu < 1) per_cu = 1;
    const int grid = (int)std::min<int64_t>(count * parts, (int64_t)cus * per_cu);
    if constexpr (MF)
        hipLaunchKernelGGL((gurvits_mfma_kernel<NP>), dim3(grid), dim3(threads), 0, st, mats, items, count, parts,
                           iters, per, seed, stream0, partial, scale);
    else
        hipLaunchKernelGGL((gurvits_kernel<NP>), dim3(grid), dim3(64), 0, st, mats, items, count, parts, iters, per,
                           seed, stream0, partial);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

// Integer products of a chunk of matrices: their digits, the int8 kernel, and
// the FP64 kernel for those that keep it (usually none: its waves leave at
// once).
template <int NP>
static int launch_gurvits_int8(const cd *mats, const GurvitsItem *items, int64_t count, int parts, int64_t iters,
                               int64_t per, uint64_t seed, uint64_t stream0, double *partial, gv_i4 *frags,
                               int32_t *scale, int cus, hipStream_t st)
{
    // a workgroup per row block and component while matrices alone are few
    const int split = count < 4 * (int64_t)cus ? NP / 8 : 1;
    hipLaunchKernelGGL((gurvits_digits_kernel<NP>), dim3((unsigned)std::min<int64_t>(count * split, (int64_t)cus * 8)),
                       dim3(256), 0, st, mats, items, count, split, frags, scale);
    PCVL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL((gurvits_int8_kernel<NP>), dim3((unsigned)(count * parts)), dim3(64), 0, st, frags, items, count,
                       parts, iters, per, seed, stream0, partial, scale);
    PCVL_HIP_CHECK(hipGetLastError());
    return launch_gurvits<NP>(mats, items, count, parts, iters, per, seed, stream0, partial, scale, st);
}

// The same for a call's matrices, GURVITS_CHUNK_BYTES of fragments at a time.
template <int NP>
static int launch_gurvits_chunks(const cd *mats, const GurvitsItem *items, int64_t count, int parts, int64_t iters,
                                 int64_t per, uint64_t seed, uint64_t stream0, double *partial, gv_i4 *frags,
                                 int32_t *scale, int64_t chunk, int cus, hipStream_t st)
{
    for (int64_t c0 = 0; c0 < count; c0 += chunk) {
        const int rc = launch_gurvits_int8<NP>(mats, items + c0, std::min(chunk, count - c0), parts, iters, per, seed,
                                               stream0 + (uint64_t)c0, partial + 3 * c0 * parts, frags, scale + c0, cus,
                                               st);
        if (rc != OK) return rc;
    }
    return OK;
}

// Parts of a matrix for the integer kernel: equal rounds of the resident
// waves, each part at least 1,024 samples.
template <int NP>
static int gurvits_int8_parts(int64_t count, int64_t iters, int cus, int *parts)
{
    int per_cu = 0;
    PCVL_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, reinterpret_cast<const void *>(&gurvits_int8_kernel<NP>), 64, 0));
    *parts = (int)std::max<int64_t>(1, std::min<int64_t>(GURVITS_ROUNDS * (int64_t)cus * std::max(per_cu, 1) / count, iters / 1024));
    return OK;
}

} // namespace pcvl

using namespace pcvl;

extern "C" int pcvl_gurvits_batch(const double *d_mats, const int32_t *h_n, const int64_t *h_offsets, int64_t count,
                                  int64_t iters, uint64_t seed, uint64_t stream0, double *d_est, double *d_err,
                                  hipStream_t stream)
{
    PCVL_ARG_CHECK(count >= 0 && iters >= 1, "count < 0 or iterations < 1");
    if (count == 0) return OK;
    PCVL_ARG_CHECK(d_mats && h_n && h_offsets && d_est && d_err, "null buffer");
    std::vector<GurvitsItem> items((size_t)count);
    int nmax = 0;
    for (int64_t b = 0; b < count; b++) {
        PCVL_ARG_CHECK(h_n[b] >= 0 && h_n[b] <= GURVITS_MAX_N, "matrix order outside [0, 48]");
        PCVL_ARG_CHECK(h_offsets[b] >= 0, "negative matrix offset");
        items[(size_t)b] = GurvitsItem{h_offsets[b], h_n[b], 0};
        nmax = std::max(nmax, (int)h_n[b]);
    }
    int dev = 0, cus = 0;
    PCVL_HIP_CHECK(hipGetDevice(&dev));
    PCVL_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    // Integer products for orders 9..32 (orders up to 8 take the vector kernel,
    // above 32 a digit's two halves do not fit the 64 products of an instruction)
    const bool int8 = nmax > 8 && nmax <= 32 && count <= INT32_MAX && gurvits_int8_pays(nmax, count, iters);
    // samples of a matrix are split into parts of at least 64 * 16 samples so
    // that the batch fills the device (4 waves per SIMD of 256 CUs)
    int parts = (int)std::max<int64_t>(1, std::min<int64_t>((4096 + count - 1) / count, iters / 1024));
    const size_t frag = sizeof(gv_i4) * (size_t)gurvits_frags(nmax <= 16 ? 16 : 32);
    const int64_t chunk = std::min<int64_t>(count, (int64_t)(GURVITS_CHUNK_BYTES / frag));
    if (int8) {
        int rc = nmax <= 16 ? gurvits_int8_parts<16>(chunk, iters, cus, &parts)
                            : gurvits_int8_parts<32>(chunk, iters, cus, &parts);
        if (rc != OK) return rc;
    }
    const int64_t per = (iters + parts - 1) / parts;
    parts = (int)((iters + per - 1) / per);
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    const size_t b_items = al(sizeof(GurvitsItem) * items.size());
    const size_t b_part = al(sizeof(double) * 3 * (size_t)count * parts);
    const size_t b_scale = int8 ? al(sizeof(int32_t) * (size_t)count) : 0;
    const size_t b_frag = int8 ? frag * (size_t)chunk : 0;
    char *blk = nullptr;
    PCVL_HIP_CHECK(ws_alloc(reinterpret_cast<void **>(&blk), b_items + b_part + b_scale + b_frag, stream));
    GurvitsItem *d_items = reinterpret_cast<GurvitsItem *>(blk);
    double *d_part = reinterpret_cast<double *>(blk + b_items);
    int32_t *d_scale = int8 ? reinterpret_cast<int32_t *>(blk + b_items + b_part) : nullptr;
    gv_i4 *d_frag = reinterpret_cast<gv_i4 *>(blk + b_items + b_part + b_scale);
    hipError_t e = hipMemcpyAsync(d_items, items.data(), sizeof(GurvitsItem) * items.size(), hipMemcpyHostToDevice,
                                  stream);
    int rc = OK;
    if (e != hipSuccess) {
        set_error(std::string("hipMemcpyAsync(gurvits items): ") + hipGetErrorString(e));
        rc = ERR_HIP;
    } else {
        const cd *mats = reinterpret_cast<const cd *>(d_mats);
        if (int8 && nmax <= 16)
            rc = launch_gurvits_chunks<16>(mats, d_items, count, parts, iters, per, seed, stream0, d_part, d_frag, d_scale, chunk, cus, stream);
        else if (int8)
            rc = launch_gurvits_chunks<32>(mats, d_items, count, parts, iters, per, seed, stream0, d_part, d_frag, d_scale, chunk, cus, stream);
        else if (nmax <= 8)
            rc = launch_gurvits<8>(mats, d_items, count, parts, iters, per, seed, stream0, d_part, nullptr, stream);
        else if (nmax <= 16)
            rc = launch_gurvits<16>(mats, d_items, count, parts, iters, per, seed, stream0, d_part, nullptr, stream);
        else if (nmax <= 32)
            rc = launch_gurvits<32>(mats, d_items, count, parts, iters, per, seed, stream0, d_part, nullptr, stream);
        else
            rc = launch_gurvits<48>(mats, d_items, count, parts, iters, per, seed, stream0, d_part, nullptr, stream);
        if (rc == OK) {
            const int lanes = parts < 16 ? 1 : 64;
            hipLaunchKernelGGL(lanes == 1 ? gurvits_finalize_kernel<1> : gurvits_finalize_kernel<64>,
                               dim3((unsigned)((count * lanes + 255) / 256)), dim3(256), 0, stream, d_part, count, parts,
                               iters, d_scale, reinterpret_cast<cd *>(d_est), d_err);
            e = hipGetLastError();
            if (e != hipSuccess) { set_error(std::string("gurvits finalize: ") + hipGetErrorString(e)); rc = ERR_HIP; }
        }
    }
    // the table must outlive the kernel: wait for it, then release it
    hipError_t se = hipStreamSynchronize(stream);
    hipError_t fe = hipFreeAsync(blk, stream);
    if (rc == OK && se != hipSuccess) { set_error(std::string("gurvits: ") + hipGetErrorString(se)); rc = ERR_HIP; }
    if (rc == OK && fe != hipSuccess) { set_error(std::string("hipFree(gurvits items): ") + hipGetErrorString(fe)); rc = ERR_HIP; }
    return rc;
}
