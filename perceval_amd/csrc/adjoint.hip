// Gradients of output probabilities with respect to circuit phases.
//
// The reference has no analytic gradient: its QML loop differentiates
// numerically (benchmark/benchmark_QML-DE-solver.py:140-142) through repeated
// SLOSBackend.set_circuit/all_prob calls (perceval/backends/_slos.py:130-141).
// This kernel returns, for a batch of phase vectors of one mesh, the loss
//     L(phi) = sum_{s in targets} P(s),  P(s) = |perm(U[s, in])|^2 / (prod s! prod t!)
// and dL/dphi for every phase, in one pass per parameter set.  The host cuts
// the mesh program (phase shifters and fixed 2x2 blocks, circuit order as
// perceval/components/linear_circuit.py:487-503) into cells: runs of ops on one
// pair of modes with nothing between them, e.g. a whole MZI.
//   1. every cell's 2x2 matrix, and U(phi) = C_K ... C_1;
//   2. per target, the amplitude A_s and all n*n cofactor permanents
//      d perm / d a_rc by one Glynn pass (2^{n-1} terms; per term the column
//      sums, prod_{c' != c} by prefix/suffix, and delta_r); they accumulate
//      G_ij = sum_s conj(A_s) dA_s/dU_ij;
//   3. with W = U G^T, one backward sweep W <- C^H W C over the cells.  A phase
//      phi on mode q contributes dL/dphi = -2 Im W_qq at its place in the
//      program, which depends on W's 2x2 block on the cell's modes alone: the
//      sweep keeps each cell's block, and the phases of all cells follow from
//      their blocks side by side.
// One workgroup per parameter set; all arithmetic complex FP64.
#include "common.h"
#include "../../include/pcvl_hip.h"

#include <algorithm>
#include <cmath>
#include <new>
#include <string>
#include <vector>

namespace pcvl {

constexpr int ADJ_MAX_M = 32;
constexpr int ADJ_MAX_N = 8;
constexpr int ADJ_MAX_TARGETS = 512;     // targets of one plan (its LDS decides what fits)
constexpr int ADJ_THREADS = 512;
constexpr int ADJ_GROUP_ITEMS = 256;     // (target, row) pairs from which a thread takes a target's rows together

struct MeshOp {
    int32_t kind;    // 0: phase shifter on mode q; 1: fixed 2x2 block on (q, q+1)
    int32_t q;
    int32_t param;   // phase index (kind 0), -1 for a constant phase
    int32_t grad;    // 0: no phase of its own; 1: the only op of its phase; 2: one of several
    double c[8];     // kind 0: c[0] = constant phase; kind 1: 2x2 block row-major (re, im)
};

__device__ __forceinline__ cd cexpi(double ph) { return {cos(ph), sin(ph)}; }
__device__ __forceinline__ cd cconj(cd a) { return {a.r, -a.i}; }

// Sum over the 64 lanes of a wave, every lane receiving it (butterfly: a
// fixed order, so the result does not depend on timing).
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Glynn with derivatives for RH target rows r0, r0 + 1, ... of M = U[rows,
// cols] (n = N; U in LDS, leading dimension ld, rows the target's modes, cols
// the input's): dr[q][c] = nrm * d perm / d M[r0 + q][c] and perm = nrm *
// perm(M).  The matrix is read from LDS as the Gray walk flips its rows, so no
// N x N copy sits in registers.
template <int N, int RH>
__device__ __forceinline__ void glynn_with_row_derivs(const cd *U, int ld, const int32_t *rows, const int32_t *cols,
                                                      int r0, double nrm, cd (&dr)[RH][N], cd &perm)
{
    int col[N];
#pragma unroll
    for (int c = 0; c < N; c++) col[c] = cols[c];
    cd cs[N];
#pragma unroll
    for (int c = 0; c < N; c++) cs[c] = {0.0, 0.0};
    for (int i = 0; i < N; i++) {
        const cd *row = U + rows[i] * ld;
#pragma unroll
        for (int c = 0; c < N; c++) cs[c] = cadd(cs[c], row[col[c]]);
    }
    perm = {0.0, 0.0};
#pragma unroll
    for (int q = 0; q < RH; q++)
#pragma unroll
        for (int c = 0; c < N; c++) dr[q][c] = {0.0, 0.0};
    uint32_t g = 0;
#pragma unroll 1
    for (uint32_t t = 0; t < (1u << (N - 1)); t++) {
        if (t) {
            const int b = __builtin_ctz(t);
            g ^= 1u << b;
            const double sgn = ((g >> b) & 1) ? -2.0 : 2.0;
            const cd *row = U + rows[b + 1] * ld;
#pragma unroll
            for (int c = 0; c < N; c++) {
                const cd v = row[col[c]];
                cs[c].r = fma(sgn, v.r, cs[c].r);
                cs[c].i = fma(sgn, v.i, cs[c].i);
            }
        }
        const double sign = (t & 1) ? -1.0 : 1.0;
        // delta_r of this term (row 0 always +1)
        double dr_sign[RH];
#pragma unroll
        for (int q = 0; q < RH; q++) dr_sign[q] = (((g << 1) >> (r0 + q)) & 1) ? -1.0 : 1.0;
        cd P[N];
        P[0] = {1.0, 0.0};
        if constexpr (N > 1) P[1] = cs[0];
#pragma unroll
        for (int c = 2; c < N; c++) P[c] = cmul(P[c - 1], cs[c - 1]);
        cd S = {sign, 0.0};
#pragma unroll
        for (int c = N - 1; c >= 0; c--) {
            // sign * prod_{c' != c} cs_c'
            cd ex;
            if (c == N - 1) ex = {sign * P[c].r, sign * P[c].i};
            else if (c == 0) ex = S;
            else ex = cmul(P[c], S);
#pragma unroll
            for (int q = 0; q < RH; q++) {
                dr[q][c].r = fma(dr_sign[q], ex.r, dr[q][c].r);
                dr[q][c].i = fma(dr_sign[q], ex.i, dr[q][c].i);
            }
            if (c == N - 1) S = {sign * cs[c].r, sign * cs[c].i};
            else S = cmul(S, cs[c]);
        }
        perm = cadd(perm, S);                 // S = sign * prod_c cs_c
    }
    const double sc = ldexp(1.0, -(N - 1)) * nrm;
#pragma unroll
    for (int q = 0; q < RH; q++)
#pragma unroll
        for (int c = 0; c < N; c++) dr[q][c] = {dr[q][c].r * sc, dr[q][c].i * sc};
    perm = {perm.r * sc, perm.i * sc};
}

// Rows of a target per thread when every target's rows are not worth a thread
// each: all of them up to 6 photons, 4 above (VGPRs).
constexpr int adj_rows(int n) { return n <= 6 ? n : 4; }

// Targets whose amplitudes one pass of the threads forms.
constexpr int adj_pass(int n, int rows) { return ADJ_THREADS / ((n + rows - 1) / rows); }

// Index tables of one call, one int32 array (offsets in entries):
//   cell[ncells+1]   first op of each cell (ops are stored cell by cell) << 6 |
//                    single << 5 | first mode; cells are in level order: a
//                    level's cells act on disjoint modes, so they commute and
//                    may run side by side
//   lstart[nlev+1]   first cell of each level
//   rstart[subs*(m+1)], rlist[targets*n]   per sub-block of targets and mode i,
//                    the (s*n + r) with rows_s[r] = i
//   cstart[m+1], clist[n]           per mode j, the c with in[c] = j
//   jlist[m]         the modes j with an input photon
//   tm[targets*n], in[n]            target modes, input modes
struct AdjIdx {
    int cell, lstart, rstart, rlist, cstart, clist, jlist, tm, in, total;
    int nlev, ncells, nj;
    int glog;   // lanes per cell slot in the sweeps: 2^glog >= m
    int sub;    // targets of a sub-block
    int ld;     // leading dimension of U and W: m | 1 (no bank conflicts down a column), m where LDS is short
    int nparts; // partial sums of G: threads (part, j, i)
    int pass;   // targets per pass (a multiple of sub, or all of them)
    int block;  // targets whose cofactors are in LDS at once (a multiple of sub)
    int nshared; // phases that several ops use
};

// Dynamic LDS of the kernel, in order (byte offsets rounded to 16): the mesh
// program (when staged), e^{i phi} of the set's phases, cell matrices and their
// W blocks (when kept), U and W (m x ld),
// amplitudes of a pass's targets, cofactors (n x n) of a block of them (reused
// for the partial sums of G), target norms and weights, a reduction buffer, the index
// tables.
struct AdjLds {
    size_t ops, zph, cells, U, W, amp, cof, tn, tw, red, idx, bytes;
};

__host__ __device__ inline size_t adj_al16(size_t b) { return (b + 15) & ~(size_t)15; }

__host__ __device__ inline AdjLds adj_lds(int nops, int nparams, int ncells, int m, int ld, int n, int ntargets,
                                          int pass, int block, int ngsum, int nidx)
{
    AdjLds L;
    size_t o = 0;
    L.ops = o; o = adj_al16(o + sizeof(MeshOp) * (size_t)nops);
    L.zph = o; o = adj_al16(o + sizeof(cd) * (size_t)(nparams > 0 ? nparams : 1));
    L.cells = o; o = adj_al16(o + 8 * sizeof(cd) * (size_t)ncells);
    L.U = o; o = adj_al16(o + sizeof(cd) * (size_t)m * ld);
    L.W = o; o = adj_al16(o + sizeof(cd) * (size_t)m * ld);
    L.amp = o; o = adj_al16(o + sizeof(cd) * (size_t)pass);
    const size_t cof = sizeof(cd) * (size_t)block * n * n, parts = sizeof(cd) * (size_t)ngsum;
    L.cof = o; o = adj_al16(o + (cof > parts ? cof : parts));
    L.tn = o; o = adj_al16(o + sizeof(double) * (size_t)ntargets);
    L.tw = o; o = adj_al16(o + sizeof(double) * (size_t)ntargets);
    L.red = o; o = adj_al16(o + sizeof(double) * (ADJ_THREADS / 64));
    L.idx = o; o = adj_al16(o + sizeof(int32_t) * (size_t)nidx);
    L.bytes = o;
    return L;
}

// 2x2 matrix of cell c: its ops' product, first op rightmost.
__device__ __forceinline__ void adj_cell_matrix(const MeshOp *ops, const int32_t *cell, const cd *zph, int c, cd (&M)[4])
{
    const int e0 = cell[c] >> 6, e1 = cell[c + 1] >> 6, q = cell[c] & 31;
    M[0] = {1.0, 0.0}; M[1] = {0.0, 0.0}; M[2] = {0.0, 0.0}; M[3] = {1.0, 0.0};
    for (int e = e0; e < e1; e++) {
        const MeshOp &op = ops[e];
        if (op.kind == 0) {
            const cd z = op.param >= 0 ? zph[op.param] : cexpi(op.c[0]);
            if (op.q == q) { M[0] = cmul(z, M[0]); M[1] = cmul(z, M[1]); }
            else { M[2] = cmul(z, M[2]); M[3] = cmul(z, M[3]); }
        } else {
            const cd a = {op.c[0], op.c[1]}, b = {op.c[2], op.c[3]}, d = {op.c[4], op.c[5]}, f = {op.c[6], op.c[7]};
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const cd x = M[k], y = M[2 + k];
                M[k] = cadd(cmul(a, x), cmul(b, y));
                M[2 + k] = cadd(cmul(d, x), cmul(f, y));
            }
        }
    }
}

// Gradients of cell c's phases from W's block B (rows and columns of the
// cell's modes) after the cell: through the ops in reverse, a phase shifter's is
// -2 Im B_aa on its mode a (to sink, with its op), and B <- L^H B L.  A phase's
// gradient is the sum over its shifters.
template <class Sink>
__device__ __forceinline__ void adj_cell_grads(const MeshOp *ops, const int32_t *cell, const cd *zph, int c, cd (&B)[4],
                                               Sink sink)
{
    const int e0 = cell[c] >> 6, e1 = cell[c + 1] >> 6, q = cell[c] & 31;
    for (int e = e1 - 1; e >= e0; e--) {
        const MeshOp &op = ops[e];
        if (op.kind == 0) {
            const bool first = op.q == q;
            if (op.grad) sink(op, -2.0 * (first ? B[0].i : B[3].i));
            const cd z = op.param >= 0 ? zph[op.param] : cexpi(op.c[0]);
            if (first) { B[1] = cmul(cconj(z), B[1]); B[2] = cmul(B[2], z); }
            else { B[1] = cmul(B[1], z); B[2] = cmul(cconj(z), B[2]); }
        } else {
            const cd l[4] = {{op.c[0], op.c[1]}, {op.c[2], op.c[3]}, {op.c[4], op.c[5]}, {op.c[6], op.c[7]}};
            cd T[4];
#pragma unroll
            for (int k = 0; k < 2; k++) {   // L^H B
                T[k] = cadd(cmul(cconj(l[0]), B[k]), cmul(cconj(l[2]), B[2 + k]));
                T[2 + k] = cadd(cmul(cconj(l[1]), B[k]), cmul(cconj(l[3]), B[2 + k]));
            }
#pragma unroll
            for (int k = 0; k < 4; k += 2) {   // (L^H B) L
                B[k] = cadd(cmul(T[k], l[0]), cmul(T[k + 1], l[2]));
                B[k + 1] = cadd(cmul(T[k], l[1]), cmul(T[k + 1], l[3]));
            }
        }
    }
}

// LDS writes of the wave's lanes before, its reads after (one wave: in order).
__device__ __forceinline__ void adj_wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Stage 2 of a set.  Threads take (target, row group) items, X.pass targets at a
// time; the cofactors stay in their registers and go to LDS a block of targets
// at a time, where thread (part, j, i) adds sub-blocks part, part + nparts, ...
// of the block to its share of G.  A thread takes a whole target (its Gray walk
// shared by the target's rows) once one thread per row would take more than
// half the threads: 462 targets of 6 photons take 45 us where one thread per
// row, 64 targets at a time, took 360.
//     G[i][j] = sum over (s, r) with rows_s[r] = i (increasing s, r) of
//               w_s conj(A_s) sum over c with in[c] = j of cof[s][r][c].
template <int N, int RH>
__device__ __forceinline__ void adj_targets(const AdjIdx &X, int m, int ntargets, const cd *U, const int32_t *idx,
                                            const double *tn, const double *tw, cd *amp, cd *cof, double *probs,
                                            double &lacc, cd &gacc)
{
    constexpr int H = (N + RH - 1) / RH;
    const int tid = threadIdx.x;
    const int npairs = X.nj * m;
    const int part = tid / npairs, pr = tid - part * npairs;
    const int gj = pr / m, gi = pr - gj * m;
    const int32_t *rlist = idx + X.rlist, *clist = idx + X.clist;
    for (int p0 = 0; p0 < ntargets; p0 += X.pass) {
        const int np = ntargets - p0 < X.pass ? ntargets - p0 : X.pass;
        const int sl = tid / H, r0 = (tid - sl * H) * RH;   // the pass's target sl, rows r0...
        const bool active = sl < np;
        cd dr[RH][N], perm;
        if (active) {
            glynn_with_row_derivs<N, RH>(U, X.ld, idx + X.tm + (p0 + sl) * N, idx + X.in, r0, tn[p0 + sl], dr, perm);
            if (r0 == 0) {
                const double p = perm.r * perm.r + perm.i * perm.i, w = tw[p0 + sl];
                if (probs) probs[p0 + sl] = p;
                lacc = fma(w, p, lacc);
                amp[sl] = {w * perm.r, -(w * perm.i)};
            }
        }
        for (int b0 = 0; b0 < np; b0 += X.block) {
            const int nb = np - b0 < X.block ? np - b0 : X.block;
            if (active && sl >= b0 && sl < b0 + nb) {
                cd *dst = cof + ((size_t)(sl - b0) * N + r0) * N;
#pragma unroll
                for (int q = 0; q < RH; q++)
                    if (N % RH == 0 || r0 + q < N)
#pragma unroll
                        for (int c = 0; c < N; c++) dst[q * N + c] = dr[q][c];
            }
            __syncthreads();
            if (part < X.nparts) {
                const int j = idx[X.jlist + gj], c0 = idx[X.cstart + j], c1 = idx[X.cstart + j + 1];
                const int first = (p0 + b0) / X.sub, last = (p0 + b0 + nb + X.sub - 1) / X.sub;
                for (int b = first + part; b < last; b += X.nparts) {
                    const int32_t *rs = idx + X.rstart + b * (m + 1);
                    const int u1 = rs[gi + 1];
#pragma unroll 4
                    for (int u = rs[gi]; u < u1; u++) {
                        const int sr = rlist[u] - (p0 + b0) * N;   // (s, r) within the block
                        const cd ca = amp[b0 + sr / N];
                        for (int v = c0; v < c1; v++) cfma_acc(gacc, ca, cof[(size_t)sr * N + clist[v]]);
                    }
                }
            }
            __syncthreads();   // amp and cof are rewritten
        }
    }
}

// One workgroup per parameter set (grid-stride).  The products over cells run
// in wave 0, level by level: the wave holds 64 >> glog cell slots of 2^glog
// lanes, lane `col` of a slot owning column col (forward, and C^H W) or row col
// (W C).  Everything else runs over all threads.  The chain of dependent steps
// is what bounds a set: at 12 modes (132 phases, 264 ops in 66 cells) the sweeps
// take 12 levels of a cell each way, where one op per level, its record read
// through a generic pointer, took 98 levels of about 1 us.  256 sets: 12 modes,
// 6 photons, 32 targets 48 us (130 us before); 6 modes, 462 targets 80 us (395 us).
//
// STAGE: the program is in LDS.  KEEP: so are the cell matrices, formed by all
// threads before the sweeps; else every slot forms its cell's (programs of so
// many cells that they do not fit).
template <int N, bool STAGE, bool KEEP>
__global__ void __launch_bounds__(ADJ_THREADS) mesh_adjoint_kernel(
    const MeshOp *__restrict__ ops_g, int nops, int m, const double *__restrict__ phases, int nparams, int nsets,
    const int32_t *__restrict__ idx_g, AdjIdx X, const int32_t *__restrict__ shared_g,
    const double *__restrict__ tn_g, const double *__restrict__ tw_g, int ntargets, int grouped, double *__restrict__ loss_out, double *__restrict__ grad_out,
    double *__restrict__ probs_out)
{
    extern __shared__ uint64_t s_adj[];
    const AdjLds L = adj_lds(STAGE ? nops : 0, nparams, KEEP ? X.ncells : 0, m, X.ld, N, ntargets, X.pass,
                             X.block, X.nj * m * X.nparts, X.total);
    char *base = reinterpret_cast<char *>(s_adj);
    cd *zph = reinterpret_cast<cd *>(base + L.zph);
    MeshOp *ops_l = reinterpret_cast<MeshOp *>(base + L.ops);
    cd *cells = reinterpret_cast<cd *>(base + L.cells);
    cd *U = reinterpret_cast<cd *>(base + L.U);
    cd *W = reinterpret_cast<cd *>(base + L.W);
    cd *amp = reinterpret_cast<cd *>(base + L.amp);
    cd *cof = reinterpret_cast<cd *>(base + L.cof);
    double *tn = reinterpret_cast<double *>(base + L.tn);
    double *tw = reinterpret_cast<double *>(base + L.tw);
    double *red = reinterpret_cast<double *>(base + L.red);
    int32_t *idx = reinterpret_cast<int32_t *>(base + L.idx);
    const int32_t *cell = idx + X.cell, *lstart = idx + X.lstart, *jlist = idx + X.jlist;
    const int tid = threadIdx.x, ld = X.ld;
    // the program and index tables, once per workgroup
    if constexpr (STAGE)
        for (int e = tid; e < nops * (int)(sizeof(MeshOp) / 8); e += ADJ_THREADS)
            reinterpret_cast<uint64_t *>(ops_l)[e] = reinterpret_cast<const uint64_t *>(ops_g)[e];
    for (int e = tid; e < X.total; e += ADJ_THREADS) idx[e] = idx_g[e];
    for (int e = tid; e < ntargets; e += ADJ_THREADS) {
        tn[e] = tn_g[e];
        tw[e] = tw_g[e];
    }
    __syncthreads();
    auto ops = [&]() { if constexpr (STAGE) return (const MeshOp *)ops_l; else return ops_g; };
    const bool w0 = tid < 64;
    const int glog = X.glog, slots = 64 >> glog;
    const int slot = tid >> glog, col = tid & ((1 << glog) - 1);   // in wave 0
    const int npairs = X.nj * m, nparts = X.nparts;   // nj m <= 256, nj m nparts <= ADJ_THREADS
    for (int set = blockIdx.x; set < nsets; set += gridDim.x) {
        const double *ph = phases + (size_t)set * nparams;
        double *grad = grad_out + (size_t)set * nparams;
        for (int e = tid; e < nparams; e += ADJ_THREADS) {
            zph[e] = cexpi(ph[e]);
            grad[e] = 0.0;   // a phase that no op uses
        }
        for (int e = tid; e < m * m; e += ADJ_THREADS) U[(e / m) * ld + e % m] = {e / m == e % m ? 1.0 : 0.0, 0.0};
        __syncthreads();
        if constexpr (KEEP) {
            for (int c = tid; c < X.ncells; c += ADJ_THREADS) {
                cd M[4];
                adj_cell_matrix(ops(), cell, zph, c, M);
#pragma unroll
                for (int k = 0; k < 4; k++) cells[4 * c + k] = M[k];
            }
            __syncthreads();
        }
        // 1. U = C_K ... C_1, the levels in circuit order
        if (w0) {
            for (int lv = 0; lv < X.nlev; lv++) {
                const int e1 = lstart[lv + 1];
                for (int c = lstart[lv] + slot; c < e1; c += slots) {
                    cd M[4];
                    if constexpr (KEEP) {
#pragma unroll
                        for (int k = 0; k < 4; k++) M[k] = cells[4 * c + k];
                    } else {
                        adj_cell_matrix(ops(), cell, zph, c, M);
                    }
                    const int q = cell[c] & 31;
                    const bool two = !((cell[c] >> 5) & 1);
                    if (col < m) {
                        cd *u = U + q * ld + col;
                        const cd x = u[0], y = two ? u[ld] : cd{0.0, 0.0};
                        u[0] = cadd(cmul(M[0], x), cmul(M[1], y));
                        if (two) u[ld] = cadd(cmul(M[2], x), cmul(M[3], y));
                    }
                }
                adj_wave_order();   // the next level's cells may read them from other slots
            }
        }
        __syncthreads();
        // 2. amplitudes, cofactors, the loss and G
        double lacc = 0.0;
        cd gacc = {0.0, 0.0};
        const int part = tid / npairs;
        double *probs = probs_out ? probs_out + (size_t)set * ntargets : nullptr;
        if (grouped)
            adj_targets<N, adj_rows(N)>(X, m, ntargets, U, idx, tn, tw, amp, cof, probs, lacc, gacc);
        else
            adj_targets<N, 1>(X, m, ntargets, U, idx, tn, tw, amp, cof, probs, lacc, gacc);
        if (part < nparts) cof[tid] = gacc;
        lacc = wave_sum(lacc);
        if ((tid & 63) == 0) red[tid >> 6] = lacc;
        __syncthreads();
        if (tid == 0) {
            double l = 0.0;
            for (int w = 0; w < ADJ_THREADS / 64; w++) l += red[w];
            loss_out[set] = l;
        }
        // G in place of the first part, then W = U G^T: W[a][b] = sum_j U[a][j] G[b][j]
        if (tid < npairs) {
            cd g = cof[tid];
            for (int q = 1; q < nparts; q++) g = cadd(g, cof[q * npairs + tid]);
            cof[tid] = g;
        }
        __syncthreads();
        for (int e = tid; e < m * m; e += ADJ_THREADS) {
            const int a = e / m, b = e - a * m;
            cd w = {0.0, 0.0};
            for (int q = 0; q < X.nj; q++) cfma_acc(w, U[a * ld + jlist[q]], cof[q * m + b]);
            W[a * ld + b] = w;
        }
        __syncthreads();
        // 3. backward sweep, levels in reverse: keep the cell's block, W <- C^H W, W <- W C
        if (w0) {
            for (int lv = X.nlev - 1; lv >= 0; lv--) {
                const int e0 = lstart[lv], e1 = lstart[lv + 1];
                for (int half = 0; half < 2; half++) {
                    for (int c = e0 + slot; c < e1; c += slots) {
                        cd M[4];
                        if constexpr (KEEP) {
#pragma unroll
                            for (int k = 0; k < 4; k++) M[k] = cells[4 * c + k];
                        } else {
                            adj_cell_matrix(ops(), cell, zph, c, M);
                        }
                        const int q = cell[c] & 31;
                        const bool two = !((cell[c] >> 5) & 1);
                        if (half == 0) {
                            if constexpr (!KEEP) {   // the cell's gradients at once
                                if (col == 0) {
                                    cd B[4] = {W[q * ld + q], {0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
                                    if (two) {
                                        B[1] = W[q * ld + q + 1];
                                        B[2] = W[(q + 1) * ld + q];
                                        B[3] = W[(q + 1) * ld + q + 1];
                                    }
                                    adj_cell_grads(ops(), cell, zph, c, B, [&](const MeshOp &op, double v) {
                                        if (op.grad == 1) grad[op.param] = v;
                                    });
                                }
                                // phases of several shifters: one cell after another
                                for (int s = 0; X.nshared && s < slots; s++) {
                                    if (slot == s && col == 0) {
                                        cd B[4] = {W[q * ld + q], {0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
                                        if (two) {
                                            B[1] = W[q * ld + q + 1];
                                            B[2] = W[(q + 1) * ld + q];
                                            B[3] = W[(q + 1) * ld + q + 1];
                                        }
                                        adj_cell_grads(ops(), cell, zph, c, B, [&](const MeshOp &op, double v) {
                                            if (op.grad == 2) grad[op.param] += v;
                                        });
                                    }
                                    __threadfence_block();
                                }
                            }
                            cd b0 = {0.0, 0.0}, b1 = {0.0, 0.0};
                            if (col < m) {
                                cd *w = W + q * ld + col;
                                const cd x = w[0], y = two ? w[ld] : cd{0.0, 0.0};
                                b0 = x;
                                b1 = y;
                                w[0] = cadd(cmul(cconj(M[0]), x), cmul(cconj(M[2]), y));
                                if (two) w[ld] = cadd(cmul(cconj(M[1]), x), cmul(cconj(M[3]), y));
                            }
                            if constexpr (KEEP) {
                                // lanes q, q + 1 hold the block's columns; the matrix of a level's
                                // cell is still needed for the other half, so the block waits there
                                if (col == q) { cells[4 * (X.ncells + c)] = b0; cells[4 * (X.ncells + c) + 2] = b1; }
                                if (two && col == q + 1) { cells[4 * (X.ncells + c) + 1] = b0; cells[4 * (X.ncells + c) + 3] = b1; }
                            }
                        } else if (col < m) {
                            cd *w = W + col * ld + q;
                            const cd x = w[0], y = two ? w[1] : cd{0.0, 0.0};
                            w[0] = cadd(cmul(x, M[0]), cmul(y, M[2]));
                            if (two) w[1] = cadd(cmul(x, M[1]), cmul(y, M[3]));
                        }
                    }
                    adj_wave_order();
                }
            }
        }
        __syncthreads();
        if constexpr (KEEP) {
            for (int c = tid; c < X.ncells; c += ADJ_THREADS) {
                cd B[4];
#pragma unroll
                for (int k = 0; k < 4; k++) B[k] = cells[4 * (X.ncells + c) + k];
                adj_cell_grads(ops(), cell, zph, c, B, [&](const MeshOp &op, double v) {
                    if (op.grad == 1) grad[op.param] = v;
                });
            }
            // phases of several shifters, a thread each over the cells that hold
            // them: start[nshared + 1] | phase[nshared] | cells
            for (int s = tid; s < X.nshared; s += ADJ_THREADS) {
                const int32_t prm = shared_g[X.nshared + 1 + s];
                double sum = 0.0;
                for (int u = shared_g[s]; u < shared_g[s + 1]; u++) {
                    const int c = shared_g[u];
                    cd B[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) B[k] = cells[4 * (X.ncells + c) + k];
                    adj_cell_grads(ops(), cell, zph, c, B, [&](const MeshOp &op, double v) {
                        if (op.param == prm) sum += v;
                    });
                }
                grad[prm] = sum;
            }
        }
        __syncthreads();   // U, W, zph and the cells are rewritten by the next set
    }
}

} // namespace pcvl

using namespace pcvl;

struct pcvl_mesh_plan_s {
    int m = 0, n = 0, nops = 0, nparams = 0, ntargets = 0;
    AdjIdx X{};
    bool stage_ops = false, keep_cells = false, grouped = false;
    size_t lds = 0;
    char *d_blk = nullptr;            // program, index tables, target norms and weights, shared phases
    const MeshOp *d_ops = nullptr;
    const int32_t *d_idx = nullptr;
    const int32_t *d_shared = nullptr;   // phases of several shifters
    const double *d_tn = nullptr;
    double *d_tw = nullptr;           // per-target weights of the loss (ones unless set)
    int grid_cap = 0;
};

extern "C" int pcvl_mesh_plan_create(const int32_t *h_kind, const int32_t *h_mode, const int32_t *h_param,
                                     const double *h_const, int nops, int m, int nparams, const int32_t *h_in_occ,
                                     const int32_t *h_targets, int ntargets, pcvl_mesh_plan *out)
{
    PCVL_ARG_CHECK(out != nullptr, "out plan pointer is null");
    *out = nullptr;
    PCVL_ARG_CHECK(m >= 1 && m <= ADJ_MAX_M, "mode count outside [1, 32]");
    PCVL_ARG_CHECK(nops >= 0 && (nops == 0 || (h_kind && h_mode && h_param && h_const)), "bad mesh program");
    PCVL_ARG_CHECK(nparams >= 0, "negative sizes");
    PCVL_ARG_CHECK(ntargets >= 1 && ntargets <= ADJ_MAX_TARGETS, "target count outside [1, 512]");
    PCVL_ARG_CHECK(h_in_occ && h_targets, "null input/target states");
    std::vector<MeshOp> ops(nops);
    for (int p = 0; p < nops; p++) {
        MeshOp &o = ops[p];
        o.kind = h_kind[p];
        o.q = h_mode[p];
        o.param = h_param[p];
        o.grad = 0;
        for (int k = 0; k < 8; k++) o.c[k] = h_const[p * 8 + k];
        PCVL_ARG_CHECK(o.kind == 0 || o.kind == 1, "op kind must be 0 (phase) or 1 (2x2 block)");
        PCVL_ARG_CHECK(o.q >= 0 && o.q + (o.kind == 1 ? 1 : 0) < m, "op mode out of range");
        PCVL_ARG_CHECK(o.kind == 1 ? o.param == -1 : (o.param >= -1 && o.param < nparams), "op parameter out of range");
    }
    std::vector<int32_t> in_modes, tmodes;
    double pin = 1.0;
    for (int i = 0; i < m; i++) {
        PCVL_ARG_CHECK(h_in_occ[i] >= 0, "negative occupation");
        for (int v = 0; v < h_in_occ[i]; v++) in_modes.push_back(i);
        for (int v = 2; v <= h_in_occ[i]; v++) pin *= v;
    }
    const int n = (int)in_modes.size();
    PCVL_ARG_CHECK(n >= 1 && n <= ADJ_MAX_N, "photon count outside [1, 8]");
    std::vector<double> tnorm(ntargets);
    for (int s = 0; s < ntargets; s++) {
        int ns = 0;
        double ps = 1.0;
        for (int i = 0; i < m; i++) {
            const int v = h_targets[s * m + i];
            PCVL_ARG_CHECK(v >= 0, "negative target occupation");
            ns += v;
            for (int k = 0; k < v; k++) tmodes.push_back(i);
            for (int k = 2; k <= v; k++) ps *= k;
        }
        PCVL_ARG_CHECK(ns == n, "target photon number differs from the input's");
        tnorm[s] = 1.0 / sqrt(ps * pin);
    }
    std::vector<int> uses((size_t)nparams, 0);   // shifters of each phase
    for (const MeshOp &o : ops)
        if (o.kind == 0 && o.param >= 0) uses[(size_t)o.param]++;
    for (MeshOp &o : ops)
        if (o.kind == 0 && o.param >= 0) o.grad = uses[(size_t)o.param] == 1 ? 1 : 2;
    int oplev = 0;   // levels of single ops: one above the last op on any of its modes
    {
        std::vector<int> on((size_t)m, 0);
        for (const MeshOp &o : ops) {
            const int q2 = o.kind == 1 ? o.q + 1 : o.q;
            const int lv = std::max(on[(size_t)o.q], on[(size_t)q2]) + 1;
            on[(size_t)o.q] = on[(size_t)q2] = lv;
            oplev = std::max(oplev, lv);
        }
    }
    // The size that a plan may have: U and Z, every phase, 64 targets'
    // cofactors, one entry per op and the target tables within 160 KiB (what
    // the kernel takes is less, see adj_lds).
    constexpr size_t LDS_MAX = 160 * 1024;
    {
        const size_t nb = (size_t)std::min(ntargets, 64), nblk = (size_t)(ntargets + 63) / 64;
        const size_t entries = (size_t)nops + oplev + 1 + nblk * (m + 1) + 2 * (size_t)ntargets * n + m + 1 + 2 * n;
        const size_t need = sizeof(cd) * (std::max(nparams, 1) + 2 * (size_t)m * m + nb * (1 + (size_t)n * n)) +
                            2 * adj_al16(sizeof(double) * ntargets) + sizeof(double) * ADJ_THREADS +
                            adj_al16(sizeof(int32_t) * entries);
        if (need > LDS_MAX) {   // a caller may split the targets over several plans
            set_error("too many phases or targets for the kernel's LDS (" + std::to_string(need) + " bytes)");
            return ERR_RANGE;
        }
    }
    // cells: an op joins the cell that last touched its modes; a phase on a
    // mode that no cell has touched joins the first one that does, or has the
    // mode to itself
    struct Cell { int32_t q, level, ops; bool single; };
    std::vector<Cell> cells;
    std::vector<int32_t> last((size_t)m, -1), first((size_t)m, -1), cell_of((size_t)nops, -1);
    int nlev = 0;
    for (int p = 0; p < nops; p++) {
        const int q = ops[p].q;
        int32_t c = last[q];
        if (ops[p].kind == 1 && (c < 0 || c != last[q + 1])) {   // only a cell of this pair touches both
            Cell cell{q, 0, 0, false};
            c = (int32_t)cells.size();
            for (int x : {q, q + 1}) {
                if (last[x] >= 0) cell.level = std::max(cell.level, cells[(size_t)last[x]].level + 1);
                else first[x] = c;
                last[x] = c;
            }
            cells.push_back(cell);
        }
        cell_of[(size_t)p] = c;
    }
    for (int p = 0; p < nops; p++) {
        int32_t &c = cell_of[(size_t)p];
        if (c < 0) {
            const int q = ops[p].q;
            if (first[q] < 0) {
                first[q] = (int32_t)cells.size();
                cells.push_back(Cell{q, 0, 0, true});
            }
            c = first[q];
        }
        cells[(size_t)c].ops++;
    }
    for (const Cell &c : cells) nlev = std::max(nlev, c.level + 1);
    AdjIdx X;
    X.nlev = nlev;
    X.ncells = (int)cells.size();
    X.glog = 0;
    while ((1 << X.glog) < m) X.glog++;
    // in level order, and the program cell by cell
    std::vector<int32_t> lstart((size_t)nlev + 1, 0), at((size_t)X.ncells), order((size_t)X.ncells);
    for (const Cell &c : cells) lstart[(size_t)c.level + 1]++;
    for (int lv = 0; lv < nlev; lv++) lstart[(size_t)lv + 1] += lstart[(size_t)lv];
    {
        std::vector<int32_t> next(lstart);
        for (int c = 0; c < X.ncells; c++) order[(size_t)next[(size_t)cells[(size_t)c].level]++] = c;
    }
    std::vector<int32_t> idx;
    idx.reserve((size_t)X.ncells + 1);
    X.cell = (int)idx.size();   // 0
    int32_t nsorted = 0;
    for (int32_t c : order) {
        at[(size_t)c] = nsorted;
        idx.push_back((nsorted << 6) | (cells[(size_t)c].single ? 32 : 0) | cells[(size_t)c].q);
        nsorted += cells[(size_t)c].ops;
    }
    idx.push_back(nsorted << 6);
    std::vector<MeshOp> sorted(ops.size());
    for (int p = 0; p < nops; p++) sorted[(size_t)at[(size_t)cell_of[(size_t)p]]++] = ops[(size_t)p];
    ops.swap(sorted);
    // phases of several shifters and the cells that hold them, in order
    std::vector<int32_t> shared;
    {
        std::vector<int32_t> prms, at((size_t)nparams, -1);
        for (int prm = 0; prm < nparams; prm++)
            if (uses[(size_t)prm] > 1) {
                at[(size_t)prm] = (int32_t)prms.size();
                prms.push_back(prm);
            }
        std::vector<std::vector<int32_t>> held(prms.size());
        for (int c = 0; c < X.ncells; c++)
            for (int e = idx[(size_t)c] >> 6; e < idx[(size_t)c + 1] >> 6; e++) {
                if (ops[(size_t)e].grad != 2) continue;
                std::vector<int32_t> &h = held[(size_t)at[(size_t)ops[(size_t)e].param]];
                if (h.empty() || h.back() != c) h.push_back(c);
            }
        X.nshared = (int)prms.size();
        int32_t first = 2 * X.nshared + 1;
        for (const auto &h : held) {
            shared.push_back(first);
            first += (int32_t)h.size();
        }
        shared.push_back(first);
        shared.insert(shared.end(), prms.begin(), prms.end());
        for (const auto &h : held) shared.insert(shared.end(), h.begin(), h.end());
    }
    X.lstart = (int)idx.size();
    idx.insert(idx.end(), lstart.begin(), lstart.end());
    const int common = (int)idx.size();
    // per mode j the c whose input column is j
    std::vector<int32_t> cstart(m + 1, 0), clist, jlist;
    for (int j = 0; j < m; j++) {
        cstart[j] = (int32_t)clist.size();
        for (int c = 0; c < n; c++)
            if (in_modes[(size_t)c] == j) clist.push_back(c);
        if ((int32_t)clist.size() > cstart[j]) jlist.push_back(j);
    }
    cstart[m] = (int32_t)clist.size();
    X.nj = (int)jlist.size();
    // one thread per (target, row) while that takes at most half the threads,
    // else one per target, which walks the Gray code once for all its rows
    const bool grouped = ntargets * n > ADJ_GROUP_ITEMS;
    auto nidx = [&](int sub) {
        return common + (ntargets + sub - 1) / sub * (m + 1) + ntargets * n * 2 + (m + 1) + n + X.nj + n;
    };
    auto bytes = [&](bool stage, bool keep) {
        return adj_lds(stage ? nops : 0, nparams, keep ? X.ncells : 0, m, X.ld, n, ntargets, X.pass, X.block,
                       X.nj * m * X.nparts, nidx(X.sub)).bytes;
    };
    // Sub-blocks of 16 targets (several per part of G), passes of all threads;
    // the cell matrices, then the program go to LDS if they fit beside them,
    // and blocks take the rest.  Where even one sub-block does not fit, LDS is
    // spared step by step.
    X.ld = m | 1;
    X.nparts = ADJ_THREADS / (X.nj * m);
    X.sub = 16;
    X.pass = std::min(ntargets, adj_pass(n, grouped ? adj_rows(n) : 1));
    X.block = std::min(X.sub, ntargets);
    bool keep = bytes(false, true) <= LDS_MAX;
    if (bytes(false, keep) > LDS_MAX) {
        X.pass = std::min(X.pass, 64);
        X.nparts = 1;
        X.ld = m;
        if (bytes(false, keep) > LDS_MAX) {
            X.sub = 64;
            X.block = std::min(X.sub, ntargets);
        }
    }
    const bool stage_ops = bytes(true, keep) <= LDS_MAX;
    while (X.block < X.pass) {
        X.block += X.sub;
        if (bytes(stage_ops, keep) > LDS_MAX) {
            X.block -= X.sub;
            break;
        }
    }
    const int sub = X.sub;
    // per sub-block and mode i the (s, r) whose target row is i (rstart[b * (m + 1) + i])
    X.rstart = (int)idx.size();
    const int nsub = (ntargets + sub - 1) / sub;
    std::vector<int32_t> rstart((size_t)nsub * (m + 1), 0), rlist((size_t)ntargets * n), next((size_t)m);
    for (int b = 0; b < nsub; b++) {
        const int e0 = b * sub * n, e1 = std::min(ntargets, (b + 1) * sub) * n;
        int32_t *rs = rstart.data() + (size_t)b * (m + 1);
        rs[0] = e0;
        for (int e = e0; e < e1; e++) rs[tmodes[(size_t)e] + 1]++;
        for (int i = 0; i < m; i++) rs[i + 1] += rs[i];
        std::copy(rs, rs + m, next.begin());
        for (int e = e0; e < e1; e++) rlist[(size_t)next[(size_t)tmodes[(size_t)e]]++] = e;
    }
    idx.insert(idx.end(), rstart.begin(), rstart.end());
    X.rlist = (int)idx.size();
    idx.insert(idx.end(), rlist.begin(), rlist.end());
    X.cstart = (int)idx.size();
    idx.insert(idx.end(), cstart.begin(), cstart.end());
    X.clist = (int)idx.size();
    idx.insert(idx.end(), clist.begin(), clist.end());
    X.jlist = (int)idx.size();
    idx.insert(idx.end(), jlist.begin(), jlist.end());
    X.tm = (int)idx.size();
    idx.insert(idx.end(), tmodes.begin(), tmodes.end());
    X.in = (int)idx.size();
    idx.insert(idx.end(), in_modes.begin(), in_modes.end());
    X.total = (int)idx.size();
    const AdjLds L = adj_lds(stage_ops ? nops : 0, nparams, keep ? X.ncells : 0, m, X.ld, n, ntargets, X.pass,
                             X.block, X.nj * m * X.nparts, X.total);
    if (L.bytes > LDS_MAX) {
        set_error("internal: mesh plan takes " + std::to_string(L.bytes) + " bytes of LDS");
        return ERR_RANGE;
    }
    auto *plan = new (std::nothrow) pcvl_mesh_plan_s();
    if (!plan) { set_error("host allocation failed"); return ERR_ALLOC; }
    plan->m = m; plan->n = n; plan->nops = nops; plan->nparams = nparams; plan->ntargets = ntargets;
    plan->X = X;
    plan->stage_ops = stage_ops;
    plan->keep_cells = keep;
    plan->grouped = grouped;
    plan->lds = L.bytes;
    // one device block: program, index tables, norms
    const size_t b_ops = adj_al16(sizeof(MeshOp) * std::max(1, nops));
    const size_t b_idx = adj_al16(sizeof(int32_t) * idx.size()), b_n = adj_al16(sizeof(double) * ntargets);
    const size_t b_shared = X.nshared ? adj_al16(sizeof(int32_t) * shared.size()) : 0;
    hipError_t e = hipMalloc((void **)&plan->d_blk, b_ops + b_idx + 2 * b_n + b_shared);
    if (e != hipSuccess) {
        delete plan;
        set_error(std::string("hipMalloc(mesh plan): ") + hipGetErrorString(e));
        return ERR_ALLOC;
    }
    plan->d_ops = reinterpret_cast<const MeshOp *>(plan->d_blk);
    plan->d_idx = reinterpret_cast<const int32_t *>(plan->d_blk + b_ops);
    plan->d_tn = reinterpret_cast<const double *>(plan->d_blk + b_ops + b_idx);
    plan->d_tw = reinterpret_cast<double *>(plan->d_blk + b_ops + b_idx + b_n);
    plan->d_shared = reinterpret_cast<const int32_t *>(plan->d_blk + b_ops + b_idx + 2 * b_n);
    const std::vector<double> ones((size_t)ntargets, 1.0);
    if (nops) e = hipMemcpy(plan->d_blk, ops.data(), sizeof(MeshOp) * nops, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(plan->d_blk + b_ops, idx.data(), sizeof(int32_t) * idx.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(plan->d_blk + b_ops + b_idx, tnorm.data(), sizeof(double) * ntargets,
                                       hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(plan->d_tw, ones.data(), sizeof(double) * ntargets, hipMemcpyHostToDevice);
    if (e == hipSuccess && b_shared)
        e = hipMemcpy(plan->d_blk + b_ops + b_idx + 2 * b_n, shared.data(), sizeof(int32_t) * shared.size(),
                      hipMemcpyHostToDevice);
    int dev = 0, cus = 0;
    if (e == hipSuccess) e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) {
        (void)hipFree(plan->d_blk);
        delete plan;
        set_error(std::string("mesh plan upload: ") + hipGetErrorString(e));
        return ERR_HIP;
    }
    plan->grid_cap = cus * 4;
    *out = plan;
    return OK;
}

template <int N>
static int launch_mesh(const pcvl_mesh_plan_s &P, const double *d_phases, int nsets, double *d_loss, double *d_grad,
                       double *d_probs, hipStream_t stream)
{
    if constexpr (N > ADJ_MAX_N) {
        set_error("internal: photon count out of range");
        return ERR_ARG;
    } else {
        if (P.n != N) return launch_mesh<N + 1>(P, d_phases, nsets, d_loss, d_grad, d_probs, stream);
        auto kp = P.stage_ops ? (P.keep_cells ? mesh_adjoint_kernel<N, true, true> : mesh_adjoint_kernel<N, true, false>)
                              : (P.keep_cells ? mesh_adjoint_kernel<N, false, true> : mesh_adjoint_kernel<N, false, false>);
        hipLaunchKernelGGL(kp, dim3(std::min(nsets, P.grid_cap)), dim3(ADJ_THREADS), P.lds, stream, P.d_ops, P.nops,
                           P.m, d_phases, P.nparams, nsets, P.d_idx, P.X, P.d_shared, P.d_tn, P.d_tw, P.ntargets,
                           P.grouped ? 1 : 0, d_loss, d_grad, d_probs);
        PCVL_HIP_CHECK(hipGetLastError());
        return OK;
    }
}

extern "C" int pcvl_mesh_plan_execute(pcvl_mesh_plan plan, const double *d_phases, int nsets, double *d_loss,
                                      double *d_grad, double *d_probs, hipStream_t stream)
{
    PCVL_ARG_CHECK(plan != nullptr, "plan is null");
    PCVL_ARG_CHECK(nsets >= 0, "negative set count");
    if (nsets == 0) return OK;
    PCVL_ARG_CHECK(d_phases && d_loss && d_grad, "null device buffer");
    const pcvl_mesh_plan_s &P = *plan;
    const int rc = launch_mesh<1>(P, d_phases, nsets, d_loss, d_grad, d_probs, stream);
    if (rc != OK) return rc;
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

extern "C" int pcvl_mesh_plan_set_weights(pcvl_mesh_plan plan, const double *h_weights)
{
    PCVL_ARG_CHECK(plan != nullptr, "plan is null");
    std::vector<double> w((size_t)plan->ntargets, 1.0);
    if (h_weights)
        for (int s = 0; s < plan->ntargets; s++) {
            PCVL_ARG_CHECK(std::isfinite(h_weights[s]), "target weights must be finite");
            w[(size_t)s] = h_weights[s];
        }
    PCVL_HIP_CHECK(hipMemcpy(plan->d_tw, w.data(), sizeof(double) * w.size(), hipMemcpyHostToDevice));
    return OK;
}

extern "C" int pcvl_mesh_plan_destroy(pcvl_mesh_plan plan)
{
    if (!plan) return OK;
    hipError_t e = plan->d_blk ? hipFree(plan->d_blk) : hipSuccess;
    delete plan;
    if (e != hipSuccess) {
        set_error(std::string("hipFree(mesh plan): ") + hipGetErrorString(e));
        return ERR_HIP;
    }
    return OK;
}

extern "C" int pcvl_mesh_adjoint(const int32_t *h_kind, const int32_t *h_mode, const int32_t *h_param,
                                 const double *h_const, int nops, int m, const double *d_phases, int nparams,
                                 int nsets, const int32_t *h_in_occ, const int32_t *h_targets, int ntargets,
                                 double *d_loss, double *d_grad, double *d_probs, hipStream_t stream)
{
    PCVL_ARG_CHECK(nsets >= 0 && nparams >= 0, "negative sizes");
    pcvl_mesh_plan plan = nullptr;
    int rc = pcvl_mesh_plan_create(h_kind, h_mode, h_param, h_const, nops, m, nparams, h_in_occ, h_targets, ntargets,
                                   &plan);
    if (rc != OK) return rc;
    rc = pcvl_mesh_plan_execute(plan, d_phases, nsets, d_loss, d_grad, d_probs, stream);
    if (rc == OK) {
        const hipError_t e = hipStreamSynchronize(stream);
        if (e != hipSuccess) {
            set_error(std::string("hipStreamSynchronize: ") + hipGetErrorString(e));
            rc = ERR_HIP;
        }
    }
    const int rc2 = pcvl_mesh_plan_destroy(plan);
    return rc != OK ? rc : rc2;
}
