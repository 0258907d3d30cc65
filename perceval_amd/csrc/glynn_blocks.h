// The inner loop of Glynn sums over blocks of low-row sign patterns, shared by
// the permanent kernel and the multiset permanents of the learned sampler.
#pragma once

#include "common.h"

namespace pcvl {

// Returns v, made to look dependent on dep: keeps LDS reads at an offset of v
// inside the loop that dep counts (they would otherwise be hoisted as loop
// invariant, holding them in VGPRs).
__device__ __forceinline__ int glynn_loop_variant(int v, uint32_t dep)
{
    asm("" : "+s"(v) : "s"(dep));
    return v;
}

// Entries of a row, read through the scalar data path (wave-uniform address).
typedef const __attribute__((address_space(4))) double *scalar_row;

// Sum over `blocks` blocks of 2^LOW Glynn terms of an order-N matrix by one
// lane, the blocks in Gray-code order from block `base` on.
//
// The term's product over columns is taken in column pairs.  With T the column
// sums at low-row signs +1, a pair's product is V = T T', and flipping low row
// r to -1 takes V to V - E_r, E_r = (s a'_r + s' a_r) times the row's change
// (s: the sums without row r).  E_r is linear in the sums, so a flip of high
// row q to sign x adds x H_r[q] to it, H_r[q] = a_q a'_r + a'_q a_r times the
// two changes, a constant of the matrix; and E_2 with low row 1 flipped is
// E_2 - G, G = H_2[1].  Per pair and 2^LOW terms that is 4 operations for T T',
// 4 to flip T and T', 2 per E_r and 2 per further term (8 with the E_2 - G of
// two low rows): 20 for 4 terms (LOW = 2), 12 for 2 (LOW = 1), where updating
// and multiplying the two column sums of each term takes 8.  An order-N term
// costs 2.5 N (3 N) + 4 (N/2 - 1) FP64 operations instead of 6 N - 4: 86
// instead of 116 at order 20.
//
// The rows that a flip adds to T (row(b): the b-th high row) come through the
// scalar cache and H, G from LDS: 2 x 16 bytes per column and flip on each of
// the two paths; LDS alone would need 93% of its 128 B/clk at order 20.
//
// T, E: state at block `base` (E2 unused with LOW = 1); o1, o2: change of an
// odd last column by the low rows.  H: HS complex per high row, pair p's H_1,
// H_2 at HP p.  HALF: T holds half column sums (a flip adds the row, not twice
// the row).  After the last block the constants of one further flip are read:
// H needs one row, and row() a readable address, beyond the log2(blocks) high
// rows that flip (two rows when blocks == 1).
template <int N, int LOW, int HS, int HP, bool HALF, class Row>
__device__ __forceinline__ cd glynn_blocks(cd (&T)[N], cd (&E1)[N / 2], cd (&E2)[LOW == 2 ? N / 2 : 1], cd o1, cd o2,
                                           const cd *H, const cd *G, uint32_t blocks, uint64_t base, Row row)
{
    static_assert(N >= 4 && (LOW == 1 || LOW == 2), "unsupported order or low rows");
    constexpr int P = N / 2;
    constexpr bool ODD = (N & 1) != 0;
    // Above order 22, H_2 and G are read in their own turn instead of one pair
    // ahead: 8 VGPRs less (256 matrices of order 24: 6.80 ms, 7.34 ms ahead
    // with spills; 512 of order 22: 3.10 ms, 3.23 ms with G in its own turn).
    constexpr bool AHEAD = N <= 22;
    struct PairConst {
        cd h1, h2, g;
        double a[4];
    };
    auto load_pair = [&](PairConst &k, int b, scalar_row arow, int p, uint32_t v) {
        k.h1 = H[b * HS + HP * p];
        if constexpr (LOW == 2 && AHEAD) {
            k.h2 = H[b * HS + HP * p + 1];
            k.g = (G + glynn_loop_variant(0, v))[p];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) k.a[i] = arow[4 * p + i];
    };
    // Blocks alternate in sign (the parity of the high Gray bits): instead of
    // a sign, each block starts its sums from the negated sums so far.
    cd accp = {0.0, 0.0}, accm = {0.0, 0.0};   // terms of even / odd low parity
    scalar_row arow = row(0);
    PairConst kc, kn;
    load_pair(kn, 0, arow, 0, 0);
    for (uint32_t v = 0; v < blocks; v++) {
        // the flip that follows, of high row b; after the last block it is
        // taken and its result discarded
        const int b = __builtin_ctz(v + 1), bnext = __builtin_ctz(v + 2);
        const scalar_row anext = row(bnext);
        const uint64_t t = base + v + 1;
        const double s1 = (((t >> b) ^ (t >> (b + 1))) & 1) ? -1.0 : 1.0;
        const double s2 = HALF ? s1 : s1 + s1;
        cd q[1 << LOW];
#pragma unroll
        for (int p = 0; p < P; p++) {
            // A pair's constants are read while the pair before it is worked
            // on: wait for this pair's, start the next one's, then compute.
            // The scheduling barriers keep that order (and the values of one
            // pair at a time in VGPRs); without them a read sits 2-4
            // instructions before its use, 30 times per block (4,096 matrices
            // of order 20: 6.50 ms against 5.82 ms).
            kc = kn;
            asm volatile("" : "+v"(kc.h1.r), "+v"(kc.h1.i), "+s"(kc.a[0]), "+s"(kc.a[1]), "+s"(kc.a[2]), "+s"(kc.a[3]));
            if constexpr (LOW == 2) {
                if constexpr (AHEAD) {
                    asm volatile("" : "+v"(kc.h2.r), "+v"(kc.h2.i), "+v"(kc.g.r), "+v"(kc.g.i));
                } else {
                    kc.g = (G + glynn_loop_variant(0, v))[p];
                    kc.h2 = H[b * HS + HP * p + 1];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (p + 1 < P) load_pair(kn, b, arow, p + 1, v);
            else load_pair(kn, bnext, anext, 0, v);
            double oa[2];
            if constexpr (ODD) {
                if (p == P - 1) {
                    oa[0] = arow[2 * (N - 1)];
                    oa[1] = arow[2 * (N - 1) + 1];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            cd &x = T[2 * p], &y = T[2 * p + 1];
            cd V[1 << LOW];   // signs of the low rows: ++, -+, (+-, --)
            V[0] = cmul(x, y);
            V[1] = {V[0].r - E1[p].r, V[0].i - E1[p].i};
            if constexpr (LOW == 2) {
                const cd e = {E2[p].r - kc.g.r, E2[p].i - kc.g.i};
                V[2] = {V[0].r - E2[p].r, V[0].i - E2[p].i};
                V[3] = {V[1].r - e.r, V[1].i - e.i};
            }
            // T and E of the pair are free once its values are formed: flip
            // them to the next block (the empty asm keeps the flips behind
            // the values, so that they happen in place)
            constexpr int last = (1 << LOW) - 1;
            asm("" : "+v"(x.r), "+v"(x.i), "+v"(y.r), "+v"(y.i), "+v"(E1[p].r), "+v"(E1[p].i)
                : "v"(V[1].r), "v"(V[1].i), "v"(V[last].r), "v"(V[last].i));
            if constexpr (LOW == 2) asm("" : "+v"(E2[p].r), "+v"(E2[p].i) : "v"(V[2].r), "v"(V[2].i), "v"(V[3].r), "v"(V[3].i));
            x.r = fma(s2, kc.a[0], x.r);
            x.i = fma(s2, kc.a[1], x.i);
            y.r = fma(s2, kc.a[2], y.r);
            y.i = fma(s2, kc.a[3], y.i);
            E1[p].r = fma(s1, kc.h1.r, E1[p].r);
            E1[p].i = fma(s1, kc.h1.i, E1[p].i);
            if constexpr (LOW == 2) {
                E2[p].r = fma(s1, kc.h2.r, E2[p].r);
                E2[p].i = fma(s1, kc.h2.i, E2[p].i);
            }
            if (p == 0) {
#pragma unroll
                for (int k = 0; k < (1 << LOW); k++) q[k] = V[k];
            } else if (p < P - 1 || ODD) {
#pragma unroll
                for (int k = 0; k < (1 << LOW); k++) q[k] = cmul(q[k], V[k]);
            } else {
                accp = {-accp.r, -accp.i};
                accm = {-accm.r, -accm.i};
                cfma_acc(accp, q[0], V[0]);
                cfma_acc(accm, q[1], V[1]);
                if constexpr (LOW == 2) {
                    cfma_acc(accm, q[2], V[2]);
                    cfma_acc(accp, q[3], V[3]);
                }
            }
            if constexpr (ODD) {
                if (p == P - 1) {
                    cd &z = T[N - 1];
                    const cd m1 = {z.r - o1.r, z.i - o1.i};
                    accp = {-accp.r, -accp.i};
                    accm = {-accm.r, -accm.i};
                    cfma_acc(accp, q[0], z);
                    cfma_acc(accm, q[1], m1);
                    if constexpr (LOW == 2) {
                        cfma_acc(accm, q[2], cd{z.r - o2.r, z.i - o2.i});
                        cfma_acc(accp, q[3], cd{m1.r - o2.r, m1.i - o2.i});
                    }
                    asm("" : "+v"(z.r), "+v"(z.i) : "v"(accp.r), "v"(accp.i), "v"(accm.r), "v"(accm.i));
                    z.r = fma(s2, oa[0], z.r);
                    z.i = fma(s2, oa[1], z.i);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        arow = anext;
    }
    const double sg = (blocks & 1) ? 1.0 : -1.0;   // the last block's sign (base is even unless it is the only one)
    const double sb = (blocks == 1 && (base & 1)) ? -sg : sg;
    return {sb * (accp.r - accm.r), sb * (accp.i - accm.i)};
}

} // namespace pcvl
