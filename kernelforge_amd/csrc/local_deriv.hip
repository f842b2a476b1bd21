// local_deriv.hip -- energy+force forms of the element-matched local Gaussian
// kernel on gfx950: Jacobian (dK/dR2), transposed Jacobian (-dK/dR1), Hessian and
// the full [[EE, EF], [FE, FF]] kernel, dense or symmetric RFP (TRANSR='N', UPLO='U').
//
// For a molecule pair (a, b) and every label-matched atom pair m = (i, j):
//   d_m = x_ai - x_bj,  e_m = exp(-|d_m|^2 / 2 s^2),  c_m = e_m / s^2,  w_m = e_m / s^4
//   EE = sum_m e_m
//   FE = -sum_m c_m J_ai^T d_m                       (dK/dR_a, 3 n_a)
//   EF = +sum_m c_m J_bj^T d_m                       (dK/dR_b, 3 n_b)
//   FF = sum_i J_ai^T T_i - sum_m w_m v_m u_m^T      (3 n_a x 3 n_b)
//        T_i = sum_{j matched to i} c_m J_bj,  v_m = J_ai^T d_m,  u_m = J_bj^T d_m
// which is the reference's per-pair DGEMV/DGER + S_sum DGEMM scheme
// (src/local_kernels.cpp:1171-1419 derivation, 2511-2815 full RFP) regrouped so
// that the dominant term is one long contraction over K = (feature, atom).
//
// Two kernels per batch of molecule pairs, one 256-thread work-group per pair:
//  * deriv_prep_kernel (FP64 VALU): the matched list, e_m, and the projections of
//    J onto difference vectors streamed over the features (v_m, u_m for the
//    Hessian forms; s_i = sum_j c_m d_m and t_j = sum_i c_m d_m for the E-only
//    Jacobian forms).  Writes EE / EF / FE, and e_m, v_m, u_m to a per-pair slot.
//  * deriv_ff_kernel (FP64 MFMA 16x16x4): per feature f, T_f = C J_b[:,f,:] and
//    FF += J_a[:,f,:]^T T_f, both on MFMA with operands streamed from HBM into
//    registers (T_f's accumulators are the B operands of the second product; blocks that
//    ff_blocks_kernel found zero left out), then the rank-1 sum as a second MFMA pass over
//    the slot; writes FF.
// Every output entry belongs to exactly one molecule pair, so no atomics are used
// and results are deterministic.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>
#include <vector>

#include "feature_compact.hpp"
#include "kf_common.hpp"
#include "local_plan.hpp"

namespace kf {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int NT = 256;            // threads per work-group (4 waves)
constexpr int MAXA = 32;           // atoms per molecule supported here (3*MAXA <= 96 columns)
constexpr int MAXM = MAXA * MAXA;  // matched atom pairs per molecule pair
constexpr int VCH = 12;            // difference vectors per projection pass
constexpr int FCH = 128;           // features per staged projection chunk

enum DerivMode {
    M_JAC = 0,         // (nm1, naq2)        EF
    M_JAC_T,           // (naq1, nm2)        -FE
    M_HESS,            // (naq1, naq2)       FF
    M_FULL,            // (nm1+naq1, nm2+naq2)
    M_HESS_SYMM,       // (naq, naq) dense, pairs a <= b mirrored
    M_HESS_SYMM_RFP,   // RFP of order naq
    M_FULL_SYMM,       // (nm+naq)^2 dense
    M_FULL_SYMM_RFP,   // RFP of order nm+naq
    M_DIAG_BLOCKS,     // per molecule b: the (E_b, F_b) diagonal block, bs x bs, bs = 1 + 3 ma
};
__host__ __device__ constexpr bool has_ff(int m) { return m >= M_HESS; }
__host__ __device__ constexpr bool has_ee(int m) {
    return m == M_FULL || m == M_FULL_SYMM || m == M_FULL_SYMM_RFP || m == M_DIAG_BLOCKS;
}
__host__ __device__ constexpr bool has_ef(int m) { return m == M_JAC || has_ee(m); }
__host__ __device__ constexpr bool has_fe(int m) { return m == M_JAC_T || has_ee(m); }
__host__ __device__ constexpr bool is_symm(int m) { return m >= M_HESS_SYMM && m != M_DIAG_BLOCKS; }
__host__ __device__ constexpr bool is_rfp(int m) {
    return m == M_HESS_SYMM_RFP || m == M_FULL_SYMM_RFP;
}

// The order in which a molecule's atoms are taken by deriv_ff_kernel.
struct FfOrder {
    signed char row[MAXA];  // atom in row r, -1 for none
    signed char col[MAXA];  // atom of force columns 3r .. 3r+2, -1 past the last
};

struct DerivArgs {
    const double *x1, *dx1, *x2, *dx2;
    const int *q1, *q2, *n1, *n2;
    const int *offs1, *offs2;  // 3 * prefix sums of clamped atom counts
    const int2 *pairs;         // (a, b) per work-group
    int ma1, ma2, rep;
    double cexp, inv_s2, inv_s4;
    double *out;
    size_t ld;     // dense row stride, or the RFP order
    int ebase1;    // energy rows preceding the force rows (nm1 for the full forms)
    int ebase2;    // energy columns preceding the force columns
    double *slot;  // per-pair scratch: e[maxm] | V[maxm][ldv] | U[maxm][ldu]
    size_t slot_len;
    int maxm, ldv, ldu;
    const FfOrder *order1, *order2;  // a row per molecule (Hessian forms over kFfDense atoms)
    const uint2 *blocks1, *blocks2;  // ff_blocks_kernel: a word per (molecule, feature), as well
};

__device__ inline int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Work-group -> pair index.  Consecutive pairs share their first molecule; the
// hardware deals work-groups round-robin over the 8 XCDs, so this keeps runs of
// consecutive pairs (and their J_a) on one XCD's L2.
__device__ inline int pair_slot() {
    const int g = blockIdx.x, G = gridDim.x;
    return (G % 8 == 0) ? (g % 8) * (G / 8) + g / 8 : g;
}

// ---------------------------------------------------------------------------
// Output addressing per form.  (a, b) is the pair, oa/ob the force offsets.
// ---------------------------------------------------------------------------
template <int MODE>
struct Out {
    double *o;
    size_t ld;
    int a, b, oa, ob, e1, e2;
    __device__ void put(size_t r, size_t c, double v) const {
        if (MODE == M_DIAG_BLOCKS)
            o[((size_t)a * ld + r) * ld + c] = v;  // block a, local (r, c)
        else if (is_rfp(MODE))
            o[rfp_upper(ld, r, c)] = v;  // caller guarantees r <= c
        else
            o[r * ld + c] = v;
    }
    __device__ void ee(double v) const {
        if (MODE == M_DIAG_BLOCKS) put(0, 0, v);
        if (MODE == M_FULL) put(a, b, v);
        if (MODE == M_FULL_SYMM) { put(a, b, v); put(b, a, v); }
        if (MODE == M_FULL_SYMM_RFP) put(a, b, v);
    }
    // EF[r] = dK/dR_b; row a, force column ob + r.
    __device__ void ef(int r, double v) const {
        const size_t col = (size_t)e2 + ob + r;
        if (MODE == M_DIAG_BLOCKS) put(0, 1 + r, v);
        if (MODE == M_JAC || MODE == M_FULL || MODE == M_FULL_SYMM_RFP) put(a, col, v);
        if (MODE == M_FULL_SYMM) {
            put(a, col, v);
            if (a != b) put(col, a, v);
        }
    }
    // FE[r] = dK/dR_a; force row oa + r, column b.
    __device__ void fe(int r, double v) const {
        const size_t row = (size_t)e1 + oa + r;
        if (MODE == M_DIAG_BLOCKS) put(1 + r, 0, v);
        if (MODE == M_JAC_T) put(oa + r, b, -v);
        if (MODE == M_FULL) put(row, b, v);
        if (MODE == M_FULL_SYMM) {
            put(row, b, v);
            if (a != b) put(b, row, v);
        }
        if (MODE == M_FULL_SYMM_RFP && a != b) put(b, row, v);
    }
    __device__ void ff(int r, int t, double v) const {
        const size_t row = (size_t)e1 + oa + r, col = (size_t)e2 + ob + t;
        if (MODE == M_DIAG_BLOCKS) put(1 + r, 1 + t, v);
        if (MODE == M_HESS || MODE == M_FULL) put(row, col, v);
        if (MODE == M_HESS_SYMM || MODE == M_FULL_SYMM) {
            put(row, col, v);
            if (a != b) put(col, row, v);
        }
        if (MODE == M_HESS_SYMM_RFP || MODE == M_FULL_SYMM_RFP) {
            if (a != b || r <= t) put(row, col, v);
        }
    }
};

// Matched list of one pair, built by thread 0 in i-major order (m -> (i, j)),
// with per-i ranges and a j-major permutation.
struct PairLists {
    int ml[MAXM];        // (i << 8) | j
    int ist[MAXA + 1];   // i-major ranges
    int jst[MAXA + 1];   // j-major ranges into jl
    int jl[MAXM];        // m indices grouped by j (ascending i inside a group)
    int qa[MAXA], qb[MAXA];
    int cj[MAXA];        // per-j fill cursors
    int np;
};

__device__ void build_lists(PairLists &L, const int *q1, const int *q2, int a, int b, int ma1,
                            int ma2, int na, int nb) {
    const int tid = threadIdx.x;
    if (tid < na) L.qa[tid] = q1[(size_t)a * ma1 + tid];
    if (tid < nb) L.qb[tid] = q2[(size_t)b * ma2 + tid];
    __syncthreads();
    if (tid == 0) {
        int cnt = 0;
        int *cj = L.cj;
        for (int j = 0; j < nb; ++j) cj[j] = 0;
        for (int i = 0; i < na; ++i) {
            L.ist[i] = cnt;
            const int qi = L.qa[i];
            for (int j = 0; j < nb; ++j)
                if (L.qb[j] == qi) { L.ml[cnt++] = (i << 8) | j; cj[j]++; }
        }
        L.ist[na] = cnt;
        int acc = 0;
        for (int j = 0; j < nb; ++j) { L.jst[j] = acc; acc += cj[j]; cj[j] = L.jst[j]; }
        L.jst[nb] = acc;
        for (int m = 0; m < cnt; ++m) L.jl[cj[L.ml[m] & 255]++] = m;
        L.np = cnt;
    }
    __syncthreads();
}

// acc[v] (for this thread's column p and feature slice) += sum_f J[f, p] vec_v[f],
// vectors produced chunk-wise by mk(v, f); emit(v, p, pb, value) after the
// cross-slice reduction.  J rows have stride ldj; ncol columns are live.
template <int NV, class MakeVec, class Emit>
__device__ void project(const double *J, int ldj, int ncol, int rep, int nv, MakeVec mk,
                        Emit emit, double (*dv)[VCH], double (*red)[VCH][64]) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    for (int pb = 0; pb * 64 < ncol; ++pb) {
        const int p = pb * 64 + lane;
        double acc[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = 0.0;
        for (int f0 = 0; f0 < rep; f0 += FCH) {
            const int fn = min(FCH, rep - f0);
            __syncthreads();
            for (int e = tid; e < nv * FCH; e += NT) {
                const int v = e / FCH, f = e - v * FCH;
                dv[f][v] = f < fn ? mk(v, f0 + f) : 0.0;
            }
            __syncthreads();
            if (p < ncol) {
                // four independent row loads in flight per thread
                const double *jp = J + (size_t)f0 * ldj + p;
                int f = wv;
                for (; f + 12 < fn; f += 16) {
                    const double j0 = jp[(size_t)f * ldj], j1 = jp[(size_t)(f + 4) * ldj],
                                 j2 = jp[(size_t)(f + 8) * ldj], j3 = jp[(size_t)(f + 12) * ldj];
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        double t = fma(j0, dv[f][v], acc[v]);
                        t = fma(j1, dv[f + 4][v], t);
                        t = fma(j2, dv[f + 8][v], t);
                        acc[v] = fma(j3, dv[f + 12][v], t);
                    }
                }
                for (; f < fn; f += 4) {
                    const double jv = jp[(size_t)f * ldj];
#pragma unroll
                    for (int v = 0; v < NV; ++v) acc[v] = fma(jv, dv[f][v], acc[v]);
                }
            }
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) red[wv][v][lane] = acc[v];
        __syncthreads();
        for (int v = wv; v < nv; v += 4)
            if (p < ncol)
                emit(v, p, pb, red[0][v][lane] + red[1][v][lane] + red[2][v][lane] +
                                   red[3][v][lane]);
        __syncthreads();
    }
}

template <int MODE>
__global__ __launch_bounds__(NT) void deriv_prep_kernel(DerivArgs A, int pair0) {
    __shared__ PairLists L;
    __shared__ double em[MAXM];
    __shared__ __align__(16) double dv[FCH][VCH];  // feature-major: one row per feature
    __shared__ double red[4][VCH][64];
    __shared__ double part[4][2 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int t = pair0 + pair_slot();
    const int a = A.pairs[t].x, b = A.pairs[t].y;
    const int na = clampi(A.n1[a], 0, A.ma1), nb = clampi(A.n2[b], 0, A.ma2);
    const int rep = A.rep, nca = 3 * na, ncb = 3 * nb;
    build_lists(L, A.q1, A.q2, a, b, A.ma1, A.ma2, na, nb);
    const int np = L.np;
    const double *xa0 = A.x1 + (size_t)a * A.ma1 * rep;
    const double *xb0 = A.x2 + (size_t)b * A.ma2 * rep;

    // e_m from the exact squared distance (one wave per matched pair).
    for (int m = wv; m < np; m += 4) {
        const double *xa = xa0 + (size_t)(L.ml[m] >> 8) * rep;
        const double *xb = xb0 + (size_t)(L.ml[m] & 255) * rep;
        double s = 0.0;
        for (int f = lane; f < rep; f += 64) {
            const double d = xa[f] - xb[f];
            s = fma(d, d, s);
        }
        s = wave_sum(s);
        if (lane == 0) em[m] = exp(s * A.cexp);
    }
    __syncthreads();

    Out<MODE> out{A.out, A.ld, a, b, A.offs1[a], A.offs2[b], A.ebase1, A.ebase2};
    double *slot = has_ff(MODE) ? A.slot + (size_t)(t - pair0) * A.slot_len : nullptr;
    if (has_ff(MODE))
        for (int m = tid; m < np; m += NT) slot[m] = em[m];
    if (has_ee(MODE) && tid == 0) {
        double s = 0.0;
        for (int m = 0; m < np; ++m) s += em[m];
        out.ee(s);
    }
    const double inv_s2 = A.inv_s2;
    // Per-thread partial sums of FE (pb 0/1 for column pb*64+lane).
    double fe_acc[2] = {0.0, 0.0};
    double ef_acc[2] = {0.0, 0.0};

    // ---------------- A side: J_ai projections ----------------
    if (has_fe(MODE) || has_ff(MODE)) {
        const size_t lda = 3 * (size_t)A.ma1;
        for (int i = 0; i < na; ++i) {
            const int m0 = L.ist[i], m1 = L.ist[i + 1];
            if (m1 == m0) continue;
            const double *J = A.dx1 + ((size_t)a * A.ma1 + i) * rep * lda;
            const double *xa = xa0 + (size_t)i * rep;
            if (has_ff(MODE)) {
                double *V = slot + A.maxm;
                for (int c0 = m0; c0 < m1; c0 += VCH) {
                    const int nv = min(VCH, m1 - c0);
                    project<VCH>(
                        J, (int)lda, nca, rep, nv,
                        [&](int v, int f) {
                            return xa[f] - xb0[(size_t)(L.ml[c0 + v] & 255) * rep + f];
                        },
                        [&](int v, int p, int pb, double val) {
                            V[(size_t)(c0 + v) * A.ldv + p] = val;
                            const double c = em[c0 + v] * inv_s2 * val;
                            if (pb == 0) fe_acc[0] -= c; else fe_acc[1] -= c;
                        },
                        dv, red);
                }
            } else {
                project<1>(
                    J, (int)lda, nca, rep, 1,
                    [&](int, int f) {
                        double s = 0.0;
                        for (int m = m0; m < m1; ++m)
                            s += em[m] * (xa[f] - xb0[(size_t)(L.ml[m] & 255) * rep + f]);
                        return s * inv_s2;
                    },
                    [&](int, int, int pb, double val) {
                        if (pb == 0) fe_acc[0] -= val; else fe_acc[1] -= val;
                    },
                    dv, red);
            }
        }
    }
    // ---------------- B side: J_bj projections ----------------
    if (has_ff(MODE) || has_ef(MODE)) {
        const size_t ldb = 3 * (size_t)A.ma2;
        for (int j = 0; j < nb; ++j) {
            const int g0 = L.jst[j], g1 = L.jst[j + 1];
            if (g1 == g0) continue;
            const double *J = A.dx2 + ((size_t)b * A.ma2 + j) * rep * ldb;
            const double *xb = xb0 + (size_t)j * rep;
            if (has_ff(MODE)) {
                double *U = slot + A.maxm + (size_t)A.maxm * A.ldv;
                for (int c0 = g0; c0 < g1; c0 += VCH) {
                    const int nv = min(VCH, g1 - c0);
                    project<VCH>(
                        J, (int)ldb, ncb, rep, nv,
                        [&](int v, int f) {
                            return xa0[(size_t)(L.ml[L.jl[c0 + v]] >> 8) * rep + f] - xb[f];
                        },
                        [&](int v, int p, int pb, double val) {
                            const int m = L.jl[c0 + v];
                            U[(size_t)m * A.ldu + p] = val;
                            const double c = em[m] * inv_s2 * val;
                            if (pb == 0) ef_acc[0] += c; else ef_acc[1] += c;
                        },
                        dv, red);
                }
            } else {
                project<1>(
                    J, (int)ldb, ncb, rep, 1,
                    [&](int, int f) {
                        double s = 0.0;
                        for (int g = g0; g < g1; ++g) {
                            const int m = L.jl[g];
                            s += em[m] * (xa0[(size_t)(L.ml[m] >> 8) * rep + f] - xb[f]);
                        }
                        return s * inv_s2;
                    },
                    [&](int, int, int pb, double val) {
                        if (pb == 0) ef_acc[0] += val; else ef_acc[1] += val;
                    },
                    dv, red);
            }
        }
    }
    // ---------------- reduce the partial FE / EF and write ----------------
    if (has_fe(MODE)) {
        part[wv][lane] = fe_acc[0];
        part[wv][64 + lane] = fe_acc[1];
        __syncthreads();
        for (int r = tid; r < nca; r += NT)
            out.fe(r, part[0][r] + part[1][r] + part[2][r] + part[3][r]);
        __syncthreads();
    }
    if (has_ef(MODE)) {
        part[wv][lane] = ef_acc[0];
        part[wv][64 + lane] = ef_acc[1];
        __syncthreads();
        for (int r = tid; r < ncb; r += NT)
            out.ef(r, part[0][r] + part[1][r] + part[2][r] + part[3][r]);
    }
}

// ---------------------------------------------------------------------------
// Projections for the Hessian forms on FP64 MFMA, pairs grouped by a shared molecule.
//   v_m = J_ai^T d_m,  u_m = J_bj^T d_m,  d_m = x_ai - x_bj   (63-vectors for 21 atoms)
// u of pair (a, b) at (i, j) is -v of the ordered pair (b, a) at (j, i), so one kernel
// computes v for ordered pairs (x, y): a group is a molecule x and up to PG partners
// y_k.  Side 0 groups the stored pairs (x, y) by their first molecule and writes V (and
// e_m); side 1 groups them by their second molecule (x = b, y = a) and writes U = -v.
// For one atom i of x the columns are every label-matched (k, j) of the group:
//   V_i (3 n_x x ncol) = J_xi^T (3 n_x x rep) * D (rep x ncol),  D[f][c] = x_xi[f] - x_yj[f]
// which streams each J_xi row once for the whole group (the one-pair form streamed it
// once per pair).  The columns depend only on the label of atom i, so they are listed
// once per label of x, and the (atom, pair of 16-column fragments) items are dealt over the
// waves of the group's work-groups; A operands (J rows, shared by the two fragments) and B
// operands (differences, formed in registers) come straight from HBM, 16 features ahead.
// Held to 256 registers: at the 347 it takes otherwise one wave fits a SIMD, and 200
// conformers of 21 atoms take 10.3 ms instead of 8.8 (16-byte loads of the descriptor rows
// with the summation index permuted spill more than they save: 13.8).
// ---------------------------------------------------------------------------
constexpr int PG = 8;  // partners per group

struct ProjGroup {
    int x, n, side, pad;
    int y[PG];     // partner molecules
    int slot[PG];  // batch-local slot of the stored pair
};

template <int NPF>
__global__ __launch_bounds__(NT, 2) void deriv_vproj_kernel(DerivArgs A, const ProjGroup *groups) {
    __shared__ int qx[MAXA], qy[PG][MAXA], ny[PG], ist[PG][MAXA], rnk[PG][MAXA], rx[MAXA];
    __shared__ int cols[PG * MAXA], wbase[5], gy[PG], gslot[PG], xl[MAXA], s_nl;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, col = lane & 15, kr = lane >> 4;
    const ProjGroup *gp = groups + blockIdx.x;
    const bool s0 = gp->side == 0;
    // side 0: x from set 1, partners from set 2; side 1 the other way round
    const double *Xx = s0 ? A.x1 : A.x2, *Xy = s0 ? A.x2 : A.x1;
    const double *Jx = s0 ? A.dx1 : A.dx2;
    const int *Qx = s0 ? A.q1 : A.q2, *Qy = s0 ? A.q2 : A.q1;
    const int *Nx = s0 ? A.n1 : A.n2, *Ny = s0 ? A.n2 : A.n1;
    const int max_ = s0 ? A.ma1 : A.ma2, may = s0 ? A.ma2 : A.ma1;
    const int rep = A.rep, x = gp->x, n = gp->n;
    const int nx = clampi(Nx[x], 0, max_), ncx = 3 * nx;
    const int lda = 3 * max_;
    if (tid < MAXA) qx[tid] = tid < nx ? Qx[(size_t)x * max_ + tid] : 0;
    if (tid < PG) {
        gy[tid] = tid < n ? gp->y[tid] : 0;
        gslot[tid] = tid < n ? gp->slot[tid] : 0;
        ny[tid] = tid < n ? clampi(Ny[gp->y[tid]], 0, may) : 0;
    }
    __syncthreads();
    {
        const int k = tid >> 5, j = tid & 31;  // 8 x 32 = NT
        qy[k][j] = j < ny[k] ? Qy[(size_t)gy[k] * may + j] : 0;
    }
    __syncthreads();
    {
        // m-offset tables.  Side 0, pair (x, y): m(i, j) = ist[k][i] + rnk[k][j], with
        // ist = sum over atoms i' < i of x of the partner's count of label q(i') and rnk =
        // rank of j among the partner's atoms of its label.  Side 1, pair (y, x):
        // m(j, i) = ist[k][j] + rx[i], ist summing x's counts over the partner's atoms j' < j.
        const int k = tid >> 5, t = tid & 31;
        if (k < n) {
            int s = 0;
            if (s0) {
                for (int i2 = 0; i2 < t && i2 < nx; ++i2)
                    for (int j2 = 0; j2 < ny[k]; ++j2) s += qy[k][j2] == qx[i2];
            } else {
                for (int j2 = 0; j2 < t && j2 < ny[k]; ++j2)
                    for (int i2 = 0; i2 < nx; ++i2) s += qx[i2] == qy[k][j2];
            }
            ist[k][t] = s;
            int r = 0;
            for (int j2 = 0; j2 < t; ++j2) r += qy[k][j2] == qy[k][t];
            rnk[k][t] = r;
        }
        if (tid < MAXA) {
            int r = 0;
            for (int i2 = 0; i2 < tid; ++i2) r += qx[i2] == qx[tid];
            rx[tid] = r;
        }
    }
    const double *xx0 = Xx + (size_t)x * max_ * rep;
    const double *Jx0 = Jx + (size_t)x * max_ * rep * lda;
    int pofs[NPF];
#pragma unroll
    for (int y = 0; y < NPF; ++y) pofs[y] = min(16 * y + col, max(ncx, 1) - 1);

    // one pass per label of x (taken at its first atom, rx == 0): the columns are every
    // label-matched (k, j) of the group, the same for all atoms of x with that label, and
    // the (atom, column fragment) items of all labels are dealt over the waves of the
    // group's gridDim.y work-groups
    const int nw = 4 * gridDim.y;
    int turn = 4 * blockIdx.y + wv;  // items until this wave's next
    __syncthreads();  // tables ready (rx decides the passes below, uniformly)
    for (int i0 = 0; i0 < nx; ++i0) {
        if (rx[i0] != 0) continue;  // not the first atom of its label (uniform)
        __syncthreads();  // the previous label's columns and atoms consumed
        const int l = qx[i0];
        {
            // columns: every (k, j) with q_y[k][j] == l, k-major (j < ny[k]: a label may have any
            // value, so none can stand for the places past the atoms; ny is 0 past the partners)
            const int k = tid >> 5, j = tid & 31;
            const bool v = (j < ny[k]) & (qy[k][j] == l);
            const unsigned long long bal = __ballot(v);
            const int pre = __popcll(bal & ((1ull << lane) - 1));
            if (lane == 0) wbase[wv + 1] = __popcll(bal);
            // atoms of x with label l, in order (rx is the rank among them)
            if (tid < MAXA && tid < nx && qx[tid] == l) xl[rx[tid]] = tid;
            if (wv == 0) {
                const unsigned long long bx = __ballot(tid < MAXA && tid < nx && qx[tid] == l);
                if (lane == 0) s_nl = __popcll(bx);
            }
            __syncthreads();
            if (tid == 0) {
                wbase[0] = 0;
                for (int w = 1; w <= 4; ++w) wbase[w] += wbase[w - 1];
            }
            __syncthreads();
            if (v) cols[wbase[wv] + pre] = (k << 5) | j;
            __syncthreads();
        }
        const int ncol = wbase[4];
        const int ncf = (ncol + 15) >> 4;
        // items: an atom i of the label and a pair of column fragments (2 zp, 2 zp + 1); the
        // two fragments share the streamed J_xi rows (eight MFMAs per k-step on one load of
        // the A operands).  A second fragment past the last is computed on clamped columns
        // and not stored.
        const int npf2 = (ncf + 1) >> 1;
        const int nitems = s_nl * npf2;
        int it = turn;
        for (; it < nitems; it += nw) {
            const int i = xl[it / npf2], zp = it % npf2;
            const double *xi = xx0 + (size_t)i * rep;
            const double *Ji = Jx0 + (size_t)i * rep * lda;
            const double *xj[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int c = min(16 * (2 * zp + h) + col, ncol - 1);
                const int kc = cols[c] >> 5, jc = cols[c] & 31;
                xj[h] = Xy + ((size_t)gy[kc] * may + jc) * rep;
            }
            v4d acc[2][NPF];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int y = 0; y < NPF; ++y) acc[h][y] = (v4d){0.0, 0.0, 0.0, 0.0};
            double d2[2] = {0.0, 0.0};
            // 16 features (4 k-steps) per block; the next block is loaded during this one
            double ja[2][4][NPF], da[2][4], db[2][2][4];
#define KF_VP_LOAD(S, F0)                                                                      \
    do {                                                                                       \
        _Pragma("unroll") for (int u = 0; u < 4; ++u) {                                        \
            const int f_ = min((F0) + 4 * u + kr, rep - 1);                                    \
            da[S][u] = xi[f_];                                                                 \
            db[S][0][u] = xj[0][f_];                                                           \
            db[S][1][u] = xj[1][f_];                                                           \
            _Pragma("unroll") for (int y = 0; y < NPF; ++y)                                    \
                ja[S][u][y] = Ji[(size_t)f_ * lda + pofs[y]];                                  \
        }                                                                                      \
    } while (0)
#define KF_VP_MMA(S, F0)                                                                       \
    do {                                                                                       \
        _Pragma("unroll") for (int u = 0; u < 4; ++u) {                                        \
            const bool in_ = (F0) + 4 * u + kr < rep;                                          \
            _Pragma("unroll") for (int h = 0; h < 2; ++h) {                                    \
                const double d_ = in_ ? da[S][u] - db[S][h][u] : 0.0;                          \
                d2[h] = fma(d_, d_, d2[h]);                                                    \
                _Pragma("unroll") for (int y = 0; y < NPF; ++y)                                \
                    acc[h][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ja[S][u][y], d_, acc[h][y], 0, 0, 0); \
            }                                                                                  \
        }                                                                                      \
    } while (0)
            KF_VP_LOAD(0, 0);
            for (int f0 = 0; f0 < rep; f0 += 32) {
                KF_VP_LOAD(1, f0 + 16);
                KF_VP_MMA(0, f0);
                if (f0 + 16 >= rep) break;
                KF_VP_LOAD(0, f0 + 32);
                KF_VP_MMA(1, f0 + 16);
            }
#undef KF_VP_LOAD
#undef KF_VP_MMA
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // |d|^2 of column c: the four lanes kr = 0..3 hold quarter sums
                double q2 = d2[h];
                q2 += __shfl_xor(q2, 16, 64);
                q2 += __shfl_xor(q2, 32, 64);
                const int cc = 16 * (2 * zp + h) + col;
                if (cc >= ncol) continue;
                const int k = cols[cc] >> 5, j = cols[cc] & 31;
                double *slot = A.slot + (size_t)gslot[k] * A.slot_len;
                if (s0) {
                    const int m = ist[k][i] + rnk[k][j];
                    double *V = slot + A.maxm + (size_t)m * A.ldv;
                    if (kr == 0) slot[m] = exp(q2 * A.cexp);
                    // acc[h][y][v] is row p = 16y + 4v + kr of column cc
#pragma unroll
                    for (int y = 0; y < NPF; ++y)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int p = 16 * y + 4 * v + kr;
                            if (p < ncx) V[p] = acc[h][y][v];
                        }
                } else {
                    const int m = ist[k][j] + rx[i];
                    double *U = slot + A.maxm + (size_t)A.maxm * A.ldv + (size_t)m * A.ldu;
#pragma unroll
                    for (int y = 0; y < NPF; ++y)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int p = 16 * y + 4 * v + kr;
                            if (p < ncx) U[p] = -acc[h][y][v];
                        }
                }
            }
        }
        turn = it - nitems;
    }
}

// ---------------------------------------------------------------------------
// FF = sum_f J_a[:,f,:]^T (C J_b[:,f,:])  -  sum_m w_m v_m u_m^T   on FP64 MFMA,
// C[i][j] = c_ij for label-matched atoms (0 otherwise).  Per feature f both factors
// are MFMA products:
//   T_f = C x J_b[:,f,q-block]      (A = C from LDS, B = J_b rows straight from HBM)
//   FF += J_a[:,f,:]^T x T_f        (A = J_a[:,f,:] staged in LDS, B = T_f)
// The f64 16x16x4 accumulator layout (register v of lane l = row 4v + l/16, column
// l%16) is exactly the B-operand layout of k-step v (lane l supplies row 4v + l/16,
// column l%16), so T_f's accumulators feed the second product without a shuffle.
// Wave w owns q-block w (16 force columns of b) and all p-blocks of a.  J_a[:,f,:] is
// shared by the four waves: it is staged through two LDS buffers (one barrier per
// feature); T for f+1 is formed after the product of f, whose loads have then come in,
// and the operands of f+2 are loaded during f.  Every global load is unconditional.
//
// The matrix cores bound it, and most of what they would multiply is zero: C joins atoms of
// one label, and a feature that belongs to some labels (an FCHL19 channel) changes only with
// the positions of atoms of those labels and of its own centre.  So a molecule's atoms are
// taken in an order that puts atoms of one label next to each other (rows: 4*NK places,
// labels starting at multiples of 4 where they fit; force columns: the same order without
// gaps, 16*NP), ff_blocks_kernel notes per feature which 4-row by 16-column blocks of the
// Jacobian hold anything, and a wave leaves out the MFMAs of empty blocks: for 21 atoms of 3
// labels 20 of 36 remain (the busiest wave's q-block 23), and 20,100 pairs of such molecules
// take 26.5 ms instead of 34.6, 703 pairs of 5-23 mixed atoms 2.0 instead of 3.4; what is
// lost against the count is the waves' wait for one another at each feature's barrier.  Exact
// zeros alone are left out, so the sums are the same.  Where
// 0 * x would not be 0 (a feature or a coefficient that is not finite) all blocks are taken.
// Rows past the atoms of a molecule are rows of C that are zero.
// Pairs of up to kFfDense atoms take every block, atoms in their own order: they have one or
// two of the four q-blocks, each step is then a chain of loads and waits rather than of MFMAs,
// and the words add to it (45,150 pairs of 5 atoms 9.9 ms with them, 7.4 without; 20,100 of 10
// atoms 8.3 and 7.3; of 12 atoms 9.5 and 11.3).
// ---------------------------------------------------------------------------
// blocks[m][f]: bit 8 y + s set when rows 4s .. 4s+3, columns 16y .. 16y+15 of feature f hold
// a value that is not zero; bit 63 when one is not finite.  A wave takes a feature at a
// time, its lanes the force columns.  Bound by the read of the Jacobians.
constexpr int kBlkRun = 32;   // features per work-group
constexpr int kFfDense = 10;  // atoms up to which every block is taken
__global__ __launch_bounds__(NT) void ff_blocks_kernel(const double *__restrict__ dx,
                                                       const int *__restrict__ N,
                                                       const FfOrder *__restrict__ order, int ma,
                                                       int rep, uint2 *__restrict__ blocks) {
    __shared__ int row[MAXA], blk[3 * MAXA];
    const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, n = clampi(N[m], 0, ma);
    const int ld = 3 * ma, nc = 3 * n;
    if (tid < MAXA) {
        const int r = order[m].row[tid], c = order[m].col[tid];
        if (r >= 0) row[r] = tid >> 2;
        if (c >= 0)
            for (int d = 0; d < 3; ++d) blk[3 * c + d] = (3 * tid + d) >> 4;
    }
    __syncthreads();
    const int c0 = min(lane, max(nc - 1, 0)), c1 = min(lane + 64, max(nc - 1, 0));
    // 32-bit words and shifts: a 64-bit shift by a VGPR has been seen to use another register's
    // value where the amount is in the last VGPR that the kernel allocates
    const int y0 = n ? blk[c0] : 0, y1 = n ? blk[c1] : 0;
    const int f1 = min(rep, (int)(blockIdx.y + 1) * kBlkRun);
    for (int f = blockIdx.y * kBlkRun + (tid >> 6); f < f1; f += NT / 64) {
        unsigned w0 = 0, w1 = 0, bad = 0;  // of the lane's columns; any value not finite
        const double *p = dx + ((size_t)m * ma * rep + f) * ld;
        for (int i0 = 0; i0 < n; i0 += 4) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double *pi = p + (size_t)min(i0 + u, n - 1) * rep * ld;
                v[u] = pi[c0];
                v[u + 4] = pi[c1];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned bit = 1u << row[min(i0 + u, n - 1)];
                w0 |= v[u] != 0.0 ? bit : 0u;
                w1 |= v[u + 4] != 0.0 ? bit : 0u;
                bad |= (!(fabs(v[u]) <= DBL_MAX) | !(fabs(v[u + 4]) <= DBL_MAX)) ? 1u : 0u;
            }
        }
        w0 <<= 8 * (y0 & 3);
        w1 <<= 8 * (y1 & 3);
        unsigned lo = (y0 < 4 ? w0 : 0u) | (y1 < 4 ? w1 : 0u);
        unsigned hi = (y0 < 4 ? 0u : w0) | (y1 < 4 ? 0u : w1) | bad << 31;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            lo |= (unsigned)__shfl_xor((int)lo, o, 64);
            hi |= (unsigned)__shfl_xor((int)hi, o, 64);
        }
        if (lane == 0) blocks[(size_t)m * rep + f] = make_uint2(lo, hi);
    }
}

// What a pair's work-group keeps in LDS.
struct FfPair {
    double Cm[32 * 33];                  // C by rows of a and b
    int ra[MAXA], rb[MAXA];              // atom in a row (a valid one where there is none)
    int pa[3 * MAXA], pb[3 * MAXA];      // force column of the molecule at place c
    int cg[8];                           // bit s: row groups (this, s) of a and b share a label
    int full;                            // C holds values that are not finite
};

__device__ inline unsigned long long ff_uniform(uint2 v) {
    return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)v.y) << 32 |
           (unsigned)__builtin_amdgcn_readfirstlane((int)v.x);
}

// fn(0) ... fn(N - 1), each with its index as a constant: the operands below then stay in
// registers of their own (left to loop unrolling, conditional MFMAs move them about).
template <int N, int I = 0, typename Fn>
__device__ __forceinline__ void static_for(Fn &&fn) {
    if constexpr (I < N) {
        fn(std::integral_constant<int, I>{});
        static_for<N, I + 1>(fn);
    }
}

// One feature's operands: J_b (column operands), T, the row groups of T that hold anything
// and the block word of J_a.
template <int NK, int NX>
struct FfOperand {
    double jb[NK];
    v4d t[NX];
    int rows;
    unsigned long long blocks;
};

template <int MODE, int NK, int NP>
__device__ __forceinline__ void ff_pair(const DerivArgs &A, int a, int b, int na, int nb,
                                        const FfPair &L, double *Jbuf, int np,
                                        const double *mc, const double *slot, int f0, int fe,
                                        double *part) {
    typedef unsigned long long u64;
    constexpr int NX = (NK + 3) / 4;         // 16-row fragments of C / T (atoms of a)
    constexpr int FFR = 4 * NK, FFP = 16 * NP;  // staged J_a feature: rows x columns
    constexpr int NEL = FFR * FFP, NST = (NEL + NT - 1) / NT;  // elements, per thread
    constexpr int ALL = (1 << NK) - 1;
    constexpr bool SPARSE = NP >= 3;  // more than kFfDense atoms
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kr = lane >> 4,
              wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rep = A.rep, nca = 3 * na, ncb = 3 * nb;
    const int nqb = (ncb + 15) >> 4;
    const int lda = 3 * A.ma1, ldb = 3 * A.ma2;
    const double *dxa = A.dx1 + (size_t)a * A.ma1 * rep * lda;
    const double *dxb = A.dx2 + (size_t)b * A.ma2 * rep * ldb;
    // staging map: element e = tid + NT*u of a feature -> row e / FFP, column e % FFP
    int soff[NST];
#pragma unroll
    for (int u = 0; u < NST; ++u) {
        const int e = min(tid + NT * u, NEL - 1), r = e / FFP, c = e % FFP;
        soff[u] = L.ra[r] * rep * lda + L.pa[min(c, nca - 1)];
    }
    int rb[NK], cg[NK], cx[NX], full = __builtin_amdgcn_readfirstlane(L.full);
#pragma unroll
    for (int s = 0; s < NK; ++s) rb[s] = L.rb[4 * s + kr] * rep * ldb;
#pragma unroll
    for (int x = 0; x < NX; ++x) cx[x] = 0;
#pragma unroll
    for (int s = 0; s < NK; ++s) {
        cg[s] = __builtin_amdgcn_readfirstlane(L.cg[s]);
        cx[s / 4] |= cg[s];
    }
    double c[NX * NK];  // A operands of T
    static_for<NX * NK>([&](auto e) { c[e] = L.Cm[(16 * (e / NK) + col) * 33 + 4 * (e % NK) + kr]; });
    const uint2 *wa = A.blocks1 + (size_t)a * rep, *wb = A.blocks2 + (size_t)b * rep;
    Out<MODE> out{A.out, A.ld, a, b, A.offs1[a], A.offs2[b], A.ebase1, A.ebase2};
    // rounds of four q-blocks (more than one only past 21 atoms of b)
    for (int qr = 0; 4 * qr < nqb; ++qr) {
    const int qb = 4 * qr + wv;
    const bool busy = qb < nqb;
    const int q = L.pb[min(16 * qb + col, ncb - 1)];

    v4d acc[NP];
#pragma unroll
    for (int y = 0; y < NP; ++y) acc[y] = (v4d){0.0, 0.0, 0.0, 0.0};
    double st[NST];
    FfOperand<NK, NX> o0, o1;
    uint2 la, lb;  // the words of the next feature
    auto stage_load = [&](int f) {
        const double *p = dxa + (size_t)f * lda;
        static_for<NST>([&](auto u) { st[u] = p[soff[u]]; });
    };
    auto stage_store = [&](double *buf) {
        static_for<NST>([&](auto u) {
            if (NEL % NT == 0 || tid + NT * u < NEL) buf[tid + NT * u] = st[u];
        });
    };
    // the words of a feature and its column operands
    auto load_b = [&](FfOperand<NK, NX> &o, int f) {
        if (SPARSE) la = wa[f], lb = wb[f];
        const double *p = dxb + (size_t)f * ldb + q;
        static_for<NK>([&](auto s) { o.jb[s] = p[rb[s]]; });
    };
    // T of the feature whose words were loaded last
    auto form_t = [&](FfOperand<NK, NX> &o) {
        const u64 a_ = SPARSE ? ff_uniform(la) : 0, b_ = SPARSE ? ff_uniform(lb) : 0;
        const bool all = !SPARSE || (full | (((a_ | b_) >> 63) != 0));
        const int m = all ? ALL : int(b_ >> (8 * qb)) & ALL;
        o.blocks = all ? ~0ull : a_;
        int act = all ? ALL : 0;
        static_for<NK>([&](auto s) { act |= (cg[s] & m) ? 1 << s : 0; });
        o.rows = act;
        static_for<NX>([&](auto x) {
            const int mx = all ? ALL : cx[x] & m;
            v4d t = {0.0, 0.0, 0.0, 0.0};
            static_for<NK>([&](auto s) {
                if (!SPARSE || (mx >> s & 1))
                    t = __builtin_amdgcn_mfma_f64_16x16x4f64(c[x * NK + s], o.jb[s], t, 0, 0, 0);
            });
            o.t[x] = t;
        });
    };
    // J_a's rows of a group are read from LDS while the group before is multiplied
    double av[2][NP];
    auto load_a = [&](const double *buf, auto s) {
        static_for<NP>([&](auto y) { av[s % 2][y] = buf[(4 * s + kr) * FFP + 16 * y + col]; });
    };
    auto add_product = [&](const FfOperand<NK, NX> &o, const double *buf) {
        static_for<NK>([&](auto s) {
            if constexpr (s + 1 < NK) load_a(buf, std::integral_constant<int, s + 1>{});
            if (!SPARSE || __builtin_expect(o.rows >> s & 1, 1))
                static_for<NP>([&](auto y) {
                    if (!SPARSE || (o.blocks >> (8 * y + s) & 1))
                        acc[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            av[s % 2][y], o.t[s / 4][s % 4], acc[y], 0, 0, 0);
                });
        });
    };
    // prologue: J_a(0) in buffer 0, J_a(1) in registers, T(0), J_b(1)
    double *const J0 = Jbuf, *const J1 = Jbuf + NEL;
    stage_load(f0);
    stage_store(J0);
    stage_load(min(f0 + 1, fe - 1));
    load_b(o0, f0);
    form_t(o0);
    load_b(o1, min(f0 + 1, fe - 1));
    __syncthreads();
    for (int f = f0; f < fe; f += 2) {
        // feature f: buffer J0, T in o0; prepare f+1 (J1, T in o1) and loads for f+2
        stage_store(J1);
        stage_load(min(f + 2, fe - 1));
        if (busy) {
            load_a(J0, std::integral_constant<int, 0>{});
            add_product(o0, J0);
            form_t(o1);
        }
        load_b(o0, min(f + 2, fe - 1));
        __syncthreads();
        if (f + 1 >= fe) break;
        // feature f+1: buffer J1, T in o1; prepare f+2 (J0, T in o0) and loads for f+3
        stage_store(J0);
        stage_load(min(f + 3, fe - 1));
        if (busy) {
            load_a(J1, std::integral_constant<int, 0>{});
            add_product(o1, J1);
            form_t(o0);
        }
        load_b(o1, min(f + 3, fe - 1));
        __syncthreads();
    }
    if (!busy) continue;
    // rank-1 part (of the first run of features): acc -= sum_m (w_m v_m) u_m^T, K = matched pairs
    if (f0 == 0) {
        const double *V = slot + A.maxm, *U = V + (size_t)A.maxm * A.ldv;
        // loads of clamped (valid) entries, unconditional, masked by selects on '&'
        // conditions ('&&' turns into a branch around each load, which is then waited
        // for before the next one); np >= 1 and nca, ncb >= 1 inside the loop
        for (int m0 = 0; m0 < np; m0 += 4) {
            const int m = m0 + kr;
            const bool ok = m < np;
            const int mm = min(m, np - 1);
            const double w = ok ? -mc[mm] * A.inv_s2 : 0.0;  // -e/s^4
            const double u = U[(size_t)mm * A.ldu + q];
            const double bv = (ok & (16 * qb + col < ncb)) ? u : 0.0;
            double vv[NP];
#pragma unroll
            for (int y = 0; y < NP; ++y)
                vv[y] = V[(size_t)mm * A.ldv + L.pa[min(16 * y + col, nca - 1)]];
#pragma unroll
            for (int y = 0; y < NP; ++y) {
                const int p = 16 * y + col;
                const double av = (ok & (p < nca)) ? w * vv[y] : 0.0;
                acc[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[y], 0, 0, 0);
            }
        }
    }
    const int tc = 16 * qb + col;
#pragma unroll
    for (int y = 0; y < NP; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * y + mfma16_row_f64(lane, v);
            if (r < nca && tc < ncb) {
                if (part) part[(size_t)L.pa[r] * A.ldu + q] = acc[y][v];
                else out.ff(L.pa[r], q, acc[y][v]);
            }
        }
    }
}

// Shape buckets by m = max(atoms of a, atoms of b): (NK, NP) and the LDS they stage.
inline void ff_bucket(int m, int &nk, int &np) {
    if (m <= 5) { nk = 2; np = 1; }
    else if (m <= 10) { nk = 3; np = 2; }
    else if (m <= 16) { nk = 4; np = 3; }
    else if (m <= 21) { nk = 6; np = 4; }
    else if (m <= 24) { nk = 6; np = 5; }
    else { nk = 8; np = 6; }
}
inline size_t ff_lds_bytes(int ma1, int ma2) {
    int nk, np;
    ff_bucket(ma1 > ma2 ? ma1 : ma2, nk, np);
    return 2 * sizeof(double) * (size_t)(4 * nk) * (16 * np);
}

// Shape buckets by m = max(atoms of a, atoms of b): NK k-steps of 4 atoms, NP 16-column
// force blocks (3 m columns).
// SMALL: a set of up to kFfDense atoms per molecule, whose kernel holds no larger bucket: those
// set the registers of all (256; 100 without them), and with two work-groups on a CU a pair of
// a few atoms is a chain of waits.  E+F kernels of 800 molecules of 5 atoms of one element
// 23.5 ms (31.9 in the kernel of all sizes), 1,500 of 3 atoms 68 (91), 400 of 10 atoms 28 (41).
template <int MODE, bool SMALL>
__global__ __launch_bounds__(NT, SMALL ? 4 : 2) void deriv_ff_kernel(DerivArgs A, int pair0,
                                                                     double *__restrict__ parts) {
    constexpr int MM = SMALL ? kFfDense * kFfDense : MAXM;
    __shared__ FfPair L;
    extern __shared__ double Jbuf[];  // two staged J_a features of the largest bucket
    __shared__ int qa[MAXA], qb_[MAXA], ia[MAXA], ib[MAXA], ist[MAXA + 1], mi[MM], mj[MM];
    __shared__ double mc[MM];
    __shared__ int s_np;
    const int tid = threadIdx.x;
    const int t = pair0 + pair_slot();
    const int a = A.pairs[t].x, b = A.pairs[t].y;
    const int na = clampi(A.n1[a], 0, A.ma1), nb = clampi(A.n2[b], 0, A.ma2);
    const int mx = na > nb ? na : nb;
    const bool sparse = !SMALL && mx > kFfDense;
    // a molecule without atoms still gets its zero EE / FE / EF entries written
    const double *slot = A.slot + (size_t)(t - pair0) * A.slot_len;
    if (tid < na) qa[tid] = A.q1[(size_t)a * A.ma1 + tid];
    if (tid < nb) qb_[tid] = A.q2[(size_t)b * A.ma2 + tid];
    for (int e = tid; e < 32 * 33; e += NT) L.Cm[e] = 0.0;
    if (tid < 8) L.cg[tid] = 0;
    if (tid == 0) L.full = 0;
    if (tid >= 64 && tid < 64 + 2 * MAXA) {  // the orders of both molecules
        const int r = (tid - 64) % MAXA, second = (tid - 64) / MAXA;
        int at = r < (second ? nb : na) ? r : -1, c = at;
        if (sparse) {
            const FfOrder &o = second ? A.order2[b] : A.order1[a];
            at = o.row[r], c = o.col[r];
        }
        (second ? L.rb : L.ra)[r] = max(at, 0);
        if (at >= 0) (second ? ib : ia)[at] = r;
        for (int d = 0; d < 3; ++d) (second ? L.pb : L.pa)[3 * r + d] = 3 * max(c, 0) + d;
    }
    __syncthreads();
    if (tid == 0) {  // matched list, i-major: the order of the slot entries
        int cnt = 0;
        for (int i = 0; i < na; ++i) {
            ist[i] = cnt;
            for (int j = 0; j < nb; ++j)
                if (qb_[j] == qa[i]) { mi[cnt] = i; mj[cnt] = j; ++cnt; }
        }
        ist[na] = cnt;
        s_np = cnt;
    }
    __syncthreads();
    const int np = s_np;
    for (int m = tid; m < np; m += NT) {
        const double c = slot[m] * A.inv_s2;
        mc[m] = c;
        const int r = ia[mi[m]], k = ib[mj[m]];
        L.Cm[r * 33 + k] = c;
        if (sparse) {
            atomicOr(&L.cg[r >> 2], 1 << (k >> 2));
            if (!(fabs(c) <= DBL_MAX)) L.full = 1;
        }
    }
    __syncthreads();
    if (blockIdx.y == 0) {
        // EE = sum_m e_m, FE = -sum_m c_m v_m, EF = sum_m c_m u_m from the slot
        Out<MODE> out{A.out, A.ld, a, b, A.offs1[a], A.offs2[b], A.ebase1, A.ebase2};
        const double *V = slot + A.maxm, *U = V + (size_t)A.maxm * A.ldv;
        if (has_ee(MODE) && tid == 0) {
            double e = 0.0;
            for (int m = 0; m < np; ++m) e += slot[m];
            out.ee(e);
        }
        if (has_fe(MODE) && tid < 3 * na) {
            double sfe = 0.0;
            for (int m = 0; m < np; ++m) sfe -= mc[m] * V[(size_t)m * A.ldv + tid];
            out.fe(tid, sfe);
        }
        if (has_ef(MODE) && tid >= 128 && tid - 128 < 3 * nb) {
            double sef = 0.0;
            for (int m = 0; m < np; ++m) sef += mc[m] * U[(size_t)m * A.ldu + tid - 128];
            out.ef(tid - 128, sef);
        }
    }
    if (na == 0 || nb == 0) return;
    // this work-group's run of features, and where its part of FF goes if there are several
    const int run = (A.rep + gridDim.y - 1) / gridDim.y, f0 = blockIdx.y * run,
              fe = min(f0 + run, A.rep);
    double *part = gridDim.y > 1 ? parts + ((size_t)(t - pair0) * gridDim.y + blockIdx.y) *
                                               A.ldv * A.ldu
                                 : nullptr;
    if constexpr (SMALL) {
        if (mx <= 5) ff_pair<MODE, 2, 1>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
        else ff_pair<MODE, 3, 2>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
    } else {
        if (mx <= 5) ff_pair<MODE, 2, 1>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
        else if (mx <= 10) ff_pair<MODE, 3, 2>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
        else if (mx <= 16) ff_pair<MODE, 4, 3>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
        else if (mx <= 21) ff_pair<MODE, 6, 4>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
        else if (mx <= 24) ff_pair<MODE, 6, 5>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
        else ff_pair<MODE, 8, 6>(A, a, b, na, nb, L, Jbuf, np, mc, slot, f0, fe, part);
    }
}

// FF of a pair from the parts of its runs of features, in order.
template <int MODE>
__global__ __launch_bounds__(NT) void ff_sum_kernel(DerivArgs A, int pair0, int runs,
                                                    const double *__restrict__ parts) {
    const int t = pair0 + blockIdx.x;
    const int a = A.pairs[t].x, b = A.pairs[t].y;
    const int nca = 3 * clampi(A.n1[a], 0, A.ma1), ncb = 3 * clampi(A.n2[b], 0, A.ma2);
    Out<MODE> out{A.out, A.ld, a, b, A.offs1[a], A.offs2[b], A.ebase1, A.ebase2};
    const size_t len = (size_t)A.ldv * A.ldu;
    const double *p = parts + (size_t)blockIdx.x * runs * len;
    for (int e = threadIdx.x; e < nca * ncb; e += NT) {
        const int r = e / ncb, c = e - r * ncb;
        double s = 0.0;
        for (int k = 0; k < runs; ++k) s += p[k * len + (size_t)r * A.ldu + c];
        out.ff(r, c, s);
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct SideMeta {
    std::vector<int> q, n, offs;  // offs: nm + 1
    std::vector<int> hist;        // per molecule label histogram over `labels`
    int naq = 0;
};

void side_meta(const std::vector<int> &hQ, const std::vector<int> &hN, int nm, int ma,
               const std::vector<int> &labels, SideMeta &s) {
    s.q = hQ;
    s.n = hN;
    s.offs.assign(nm + 1, 0);
    const int L = (int)labels.size();
    s.hist.assign((size_t)nm * L, 0);
    int acc = 0;
    for (int m = 0; m < nm; ++m) {
        const int na = std::min(std::max(hN[m], 0), ma);
        s.offs[m] = acc;
        acc += 3 * na;
        for (int i = 0; i < na; ++i) {
            const int l = int(std::lower_bound(labels.begin(), labels.end(), hQ[(size_t)m * ma + i]) -
                              labels.begin());
            if (l < L && labels[l] == hQ[(size_t)m * ma + i]) s.hist[(size_t)m * L + l]++;
        }
    }
    s.offs[nm] = acc;
    s.naq = acc;
}

// Atoms by label: labels start at multiples of 4 rows where the 4 * nk rows of the molecule's
// bucket allow it, and 16 rows are filled with labels that fit whole as far as possible.
FfOrder ff_order(const int *q, int n) {
    FfOrder o;
    std::fill(o.row, o.row + MAXA, (signed char)-1);
    std::fill(o.col, o.col + MAXA, (signed char)-1);
    int nk, np;
    ff_bucket(n, nk, np);
    std::vector<std::vector<int>> sets;  // atoms of each label, the largest set first
    for (int i = 0; i < n; ++i) {
        size_t k = 0;
        while (k < sets.size() && q[sets[k][0]] != q[i]) ++k;
        if (k == sets.size()) sets.emplace_back();
        sets[k].push_back(i);
    }
    std::stable_sort(sets.begin(), sets.end(), [](const std::vector<int> &u, const std::vector<int> &v) {
        return u.size() > v.size();
    });
    int groups = 0, r = 0, c = 0;
    for (const auto &s : sets) groups += ((int)s.size() + 3) / 4;
    const bool aligned = groups <= nk;
    while (!sets.empty()) {
        size_t k = 0;
        if (aligned)
            while (k < sets.size() && (int)(sets[k].size() + 3) / 4 > 4 - r / 4 % 4) ++k;
        if (k == sets.size()) k = 0;
        for (int at : sets[k]) {
            o.row[r++] = (signed char)at;
            o.col[c++] = (signed char)at;
        }
        if (aligned) r = (r + 3) / 4 * 4;
        sets.erase(sets.begin() + k);
    }
    return o;
}

template <int MODE>
int deriv_launch(DerivArgs A, const std::vector<int2> &pairs, const SideMeta &s1,
                 const SideMeta &s2, int nlab, hipStream_t stream) {
    const size_t npairs = pairs.size();
    if (npairs == 0) return KF_OK;
    // offsets + pair list to the device (one staging copy)
    const size_t n_off = s1.offs.size() + s2.offs.size();
    const size_t pair_off = (sizeof(int) * n_off + 15) / 16 * 16;
    const bool one_set = is_symm(MODE) || MODE == M_DIAG_BLOCKS;
    const size_t order_off = pair_off + sizeof(int2) * npairs, nm1 = s1.n.size(),
                 nm2 = one_set ? 0 : s2.n.size();
    // (up to kFfDense atoms no block is left out, and the atoms keep their own order)
    const bool sparse = has_ff(MODE) && std::max(A.ma1, A.ma2) > kFfDense;
    const size_t bytes = order_off + (sparse ? sizeof(FfOrder) * (nm1 + nm2) : 0);
    char *dev = static_cast<char *>(workspace(WS_PLAN, bytes, stream));
    char *stage = static_cast<char *>(host_staging(WS_PLAN, bytes));
    KF_REQUIRE(dev && stage, KF_ERR_NOMEM, "workspace allocation failed (%zu B)", bytes);
    if (sparse) {
        FfOrder *o = reinterpret_cast<FfOrder *>(stage + order_off);
        for (size_t m = 0; m < nm1; ++m)
            o[m] = ff_order(s1.q.data() + m * A.ma1, (s1.offs[m + 1] - s1.offs[m]) / 3);
        for (size_t m = 0; m < nm2; ++m)
            o[nm1 + m] = ff_order(s2.q.data() + m * A.ma2, (s2.offs[m + 1] - s2.offs[m]) / 3);
    }
    std::copy(s1.offs.begin(), s1.offs.end(), reinterpret_cast<int *>(stage));
    std::copy(s2.offs.begin(), s2.offs.end(), reinterpret_cast<int *>(stage) + s1.offs.size());
    std::copy(pairs.begin(), pairs.end(), reinterpret_cast<int2 *>(stage + pair_off));
    KF_HIP_TRY(hipMemcpyAsync(dev, stage, bytes, hipMemcpyHostToDevice, stream));
    A.offs1 = reinterpret_cast<int *>(dev);
    A.offs2 = A.offs1 + s1.offs.size();
    A.pairs = reinterpret_cast<const int2 *>(dev + pair_off);

    size_t batch = npairs;
    if (has_ff(MODE)) {
        if (sparse) {  // which blocks of the Jacobians are not zero
            A.order1 = reinterpret_cast<const FfOrder *>(dev + order_off);
            A.order2 = A.order1 + (one_set ? 0 : nm1);
            uint2 *w = static_cast<uint2 *>(
                workspace(WS_PLAN2, sizeof(uint2) * (nm1 + nm2) * A.rep, stream));
            KF_REQUIRE(w, KF_ERR_NOMEM, "workspace allocation failed");
            A.blocks1 = w;
            A.blocks2 = one_set ? w : w + nm1 * A.rep;
            const unsigned nrun = (A.rep + kBlkRun - 1) / kBlkRun;
            for (int set = 0; set < (one_set ? 1 : 2); ++set) {
                const int ma = set ? A.ma2 : A.ma1;
                const int rc = for_groups(set ? nm2 : nm1, [&](size_t first, unsigned n) {
                    hipLaunchKernelGGL(ff_blocks_kernel, dim3(n, nrun), dim3(NT), 0, stream,
                                       (set ? A.dx2 : A.dx1) + first * ma * A.rep * 3 * ma,
                                       (set ? A.n2 : A.n1) + first,
                                       (set ? A.order2 : A.order1) + first, ma, A.rep,
                                       w + ((set ? nm1 : 0) + first) * A.rep);
                });
                if (rc) return rc;
            }
        }
        // slot layout and the largest matched count over the pairs
        int maxm = 1;
        for (const int2 &p : pairs) {
            int c = 0;
            for (int l = 0; l < nlab; ++l)
                c += s1.hist[(size_t)p.x * nlab + l] * s2.hist[(size_t)p.y * nlab + l];
            maxm = std::max(maxm, c);
        }
        A.maxm = maxm;
        A.ldv = (3 * A.ma1 + 15) / 16 * 16;
        A.ldu = (3 * A.ma2 + 15) / 16 * 16;
        A.slot_len = (size_t)maxm * (1 + A.ldv + A.ldu);
        const size_t budget = size_t(1) << 30;
        batch = std::max<size_t>(1, std::min(npairs, budget / (A.slot_len * sizeof(double))));
        A.slot = static_cast<double *>(
            workspace(WS_AUX2, batch * A.slot_len * sizeof(double), stream));
        KF_REQUIRE(A.slot, KF_ERR_NOMEM, "scratch allocation failed");
    } else {
        batch = std::min<size_t>(npairs, size_t(1) << 20);
    }
    // Hessian forms: the projection groups of every batch, built once and uploaded once
    // (side 0: runs of stored pairs with the same first molecule; side 1: the same pairs
    // grouped by their second molecule)
    std::vector<size_t> gstart;
    const ProjGroup *dgroups = nullptr;
    if (has_ff(MODE)) {
        std::vector<ProjGroup> groups;
        std::vector<std::pair<int, int>> byb;
        for (size_t p0 = 0; p0 < npairs; p0 += batch) {
            const int nbat = (int)std::min(batch, npairs - p0);
            gstart.push_back(groups.size());
            for (int k = 0; k < nbat;) {
                ProjGroup g{};
                g.x = pairs[p0 + k].x;
                g.side = 0;
                while (k < nbat && pairs[p0 + k].x == g.x && g.n < PG) {
                    g.y[g.n] = pairs[p0 + k].y;
                    g.slot[g.n++] = k++;
                }
                groups.push_back(g);
            }
            byb.clear();
            for (int k = 0; k < nbat; ++k) byb.emplace_back(pairs[p0 + k].y, k);
            std::stable_sort(byb.begin(), byb.end(),
                             [](const std::pair<int, int> &u, const std::pair<int, int> &v) {
                                 return u.first < v.first;
                             });
            for (size_t k = 0; k < byb.size();) {
                ProjGroup g{};
                g.x = byb[k].first;
                g.side = 1;
                while (k < byb.size() && byb[k].first == g.x && g.n < PG) {
                    g.y[g.n] = pairs[p0 + byb[k].second].x;
                    g.slot[g.n++] = byb[k].second;
                    ++k;
                }
                groups.push_back(g);
            }
        }
        gstart.push_back(groups.size());
        const size_t gb = sizeof(ProjGroup) * groups.size();
        ProjGroup *dg = static_cast<ProjGroup *>(workspace(WS_AUX3, gb, stream));
        ProjGroup *hg = static_cast<ProjGroup *>(host_staging(WS_AUX3, gb));
        KF_REQUIRE(dg && hg, KF_ERR_NOMEM, "workspace allocation failed (%zu B)", gb);
        std::copy(groups.begin(), groups.end(), hg);
        KF_HIP_TRY(hipMemcpyAsync(dg, hg, gb, hipMemcpyHostToDevice, stream));
        dgroups = dg;
    }
    const int npf = (3 * std::max(A.ma1, A.ma2) + 15) / 16;
    size_t bi = 0;
    for (size_t p0 = 0; p0 < npairs; p0 += batch, ++bi) {
        const unsigned nb = (unsigned)std::min(batch, npairs - p0);
        if (!has_ff(MODE)) {
            hipLaunchKernelGGL(deriv_prep_kernel<MODE>, dim3(nb), dim3(NT), 0, stream, A, (int)p0);
            KF_HIP_TRY(hipGetLastError());
        }
        if (has_ff(MODE)) {
            const unsigned ng = (unsigned)(gstart[bi + 1] - gstart[bi]);
            const ProjGroup *gp = dgroups + gstart[bi];
            // Few groups: up to eight work-groups share the items of one, whose longest chain
            // (a 23-atom molecule's some 50 items over four waves) else bounds the launch: 370
            // groups of mixed molecules 0.76 ms, 1.29 with one each
            const dim3 vg(ng, std::max(1u, std::min(8u, 2048u / ng)));
            switch (npf) {
                case 1: hipLaunchKernelGGL(deriv_vproj_kernel<1>, vg, dim3(NT), 0, stream, A, gp); break;
                case 2: hipLaunchKernelGGL(deriv_vproj_kernel<2>, vg, dim3(NT), 0, stream, A, gp); break;
                case 3: hipLaunchKernelGGL(deriv_vproj_kernel<3>, vg, dim3(NT), 0, stream, A, gp); break;
                case 4: hipLaunchKernelGGL(deriv_vproj_kernel<4>, vg, dim3(NT), 0, stream, A, gp); break;
                case 5: hipLaunchKernelGGL(deriv_vproj_kernel<5>, vg, dim3(NT), 0, stream, A, gp); break;
                default: hipLaunchKernelGGL(deriv_vproj_kernel<6>, vg, dim3(NT), 0, stream, A, gp); break;
            }
            KF_HIP_TRY(hipGetLastError());
            // Few pairs: each pair's features in several runs (of 32 and more), so that there
            // are about 2,048 work-groups, four per slot of the GPU (512): 703 pairs of mixed
            // molecules of 5-23 atoms 3.5 ms, 4.5 with one run each (every block taken)
            // (not two runs of a few atoms: 465 pairs of 3 atoms, 64 features, 165 us, 135 with one)
            int runs = std::max(1, std::min((int)(2048 / nb), A.rep / 32));
            if (!sparse && A.rep < 128) runs = 1;
            const int run = (A.rep + runs - 1) / runs;
            runs = (A.rep + run - 1) / run;  // none of them empty
            double *parts = nullptr;
            if (runs > 1) {
                const size_t bytes = sizeof(double) * nb * runs * (size_t)A.ldv * A.ldu;
                parts = static_cast<double *>(workspace(WS_AUX0, bytes, stream));
                if (!parts) runs = 1;  // (up to 150 MB that the one-run form does without)
            }
            auto ff = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(nb, runs), dim3(NT), ff_lds_bytes(A.ma1, A.ma2),
                                   stream, A, (int)p0, parts);
            };
            if (sparse) ff(deriv_ff_kernel<MODE, false>);
            else ff(deriv_ff_kernel<MODE, true>);
            KF_HIP_TRY(hipGetLastError());
            if (runs > 1) {
                hipLaunchKernelGGL(ff_sum_kernel<MODE>, dim3(nb), dim3(NT), 0, stream, A, (int)p0,
                                   runs, parts);
                KF_HIP_TRY(hipGetLastError());
            }
        }
    }
    return KF_OK;
}

// ---------------------------------------------------------------------------
// Any molecule size: the derivative forms for sets with more than MAXA atoms per molecule.
// One work-group per molecule pair, every pair-size-dependent list in global scratch:
//   matched list (i, j) of equal labels, i-major; e_m = exp(-|d_m|^2 / 2 s^2),
//   d_m = x_ai - x_bj;  v_m = J_ai^T d_m (3 na), u_m = J_bj^T d_m (3 nb);
//   EE = sum e_m, FE = -sum c_m v_m, EF = sum c_m u_m (c = e / s^2), and
//   FF = sum_f J_a[:, f, :]^T T_f - sum_m (e_m / s^4) v_m u_m^T with
//   T_f[i, :] = sum_{m in row i} c_m J_b[j_m, f, :],
// FF in 64 x 64 output tiles, T_f staged in LDS per (feature, 64-row block of i).  The
// blocks land through the same Out<MODE> addressing as the fixed-size kernels.  VALU
// FP64: it carries the sizes the MFMA kernels above do not take, not their speed.
// ---------------------------------------------------------------------------
constexpr int GT = 64;  // output tile edge / staged i-rows

template <int MODE>
__global__ __launch_bounds__(NT) void deriv_generic_kernel(DerivArgs A, int pair0,
                                                           int *__restrict__ iscr,
                                                           size_t iscr_len) {
    __shared__ double T[GT][GT + 1];
    __shared__ int s_np;
    const int tid = threadIdx.x;
    const int t = pair0 + blockIdx.x;
    const int a = A.pairs[t].x, b = A.pairs[t].y;
    const int na = clampi(A.n1[a], 0, A.ma1), nb = clampi(A.n2[b], 0, A.ma2);
    const int ld1 = 3 * A.ma1, ld2 = 3 * A.ma2, rep = A.rep;
    double *slot = A.slot + (size_t)blockIdx.x * A.slot_len;
    double *em = slot, *V = slot + A.maxm, *U = V + (size_t)A.maxm * A.ldv;
    int *mi = iscr + (size_t)blockIdx.x * iscr_len, *mj = mi + A.maxm, *ist = mj + A.maxm;
    if (tid == 0) {  // matched list, i-major
        int cnt = 0;
        for (int i = 0; i < na; ++i) {
            ist[i] = cnt;
            const int qi = A.q1[(size_t)a * A.ma1 + i];
            for (int j = 0; j < nb; ++j)
                if (A.q2[(size_t)b * A.ma2 + j] == qi) { mi[cnt] = i; mj[cnt] = j; ++cnt; }
        }
        ist[na] = cnt;
        s_np = cnt;
    }
    __syncthreads();
    const int np = s_np;
    const double *x1 = A.x1 + (size_t)a * A.ma1 * rep, *x2 = A.x2 + (size_t)b * A.ma2 * rep;
    for (int m = tid; m < np; m += NT) {
        const double *p = x1 + (size_t)mi[m] * rep, *q = x2 + (size_t)mj[m] * rep;
        double s2 = 0.0;
        for (int f = 0; f < rep; ++f) {
            const double d = p[f] - q[f];
            s2 = fma(d, d, s2);
        }
        em[m] = exp(A.cexp * s2);
    }
    const bool want_v = has_fe(MODE) || has_ff(MODE), want_u = has_ef(MODE) || has_ff(MODE);
    if (want_v)
        for (long idx = tid; idx < (long)np * 3 * na; idx += NT) {
            const int m = (int)(idx / (3 * na)), r = (int)(idx - (long)m * 3 * na);
            const double *p = x1 + (size_t)mi[m] * rep, *q = x2 + (size_t)mj[m] * rep;
            const double *J = A.dx1 + ((size_t)a * A.ma1 + mi[m]) * rep * ld1 + r;
            double s = 0.0;
            for (int f = 0; f < rep; ++f) s = fma(J[(size_t)f * ld1], p[f] - q[f], s);
            V[(size_t)m * A.ldv + r] = s;
        }
    if (want_u)
        for (long idx = tid; idx < (long)np * 3 * nb; idx += NT) {
            const int m = (int)(idx / (3 * nb)), c = (int)(idx - (long)m * 3 * nb);
            const double *p = x1 + (size_t)mi[m] * rep, *q = x2 + (size_t)mj[m] * rep;
            const double *J = A.dx2 + ((size_t)b * A.ma2 + mj[m]) * rep * ld2 + c;
            double s = 0.0;
            for (int f = 0; f < rep; ++f) s = fma(J[(size_t)f * ld2], p[f] - q[f], s);
            U[(size_t)m * A.ldu + c] = s;
        }
    __syncthreads();
    Out<MODE> out{A.out, A.ld, a, b, A.offs1[a], A.offs2[b], A.ebase1, A.ebase2};
    if (has_ee(MODE) && tid == 0) {
        double e = 0.0;
        for (int m = 0; m < np; ++m) e += em[m];
        out.ee(e);
    }
    if (has_fe(MODE))
        for (int r = tid; r < 3 * na; r += NT) {
            double s = 0.0;
            for (int m = 0; m < np; ++m) s -= em[m] * A.inv_s2 * V[(size_t)m * A.ldv + r];
            out.fe(r, s);
        }
    if (has_ef(MODE))
        for (int c = tid; c < 3 * nb; c += NT) {
            double s = 0.0;
            for (int m = 0; m < np; ++m) s += em[m] * A.inv_s2 * U[(size_t)m * A.ldu + c];
            out.ef(c, s);
        }
    if (!has_ff(MODE) || na == 0 || nb == 0) return;
    const int tr = tid >> 4, tc = tid & 15;
    const double *J1 = A.dx1 + (size_t)a * A.ma1 * rep * ld1;
    const double *J2 = A.dx2 + (size_t)b * A.ma2 * rep * ld2;
    for (int r0 = 0; r0 < 3 * na; r0 += GT)
        for (int c0 = 0; c0 < 3 * nb; c0 += GT) {
            double acc[4][4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int w = 0; w < 4; ++w) acc[u][w] = 0.0;
            for (int f = 0; f < rep; ++f)
                for (int i0 = 0; i0 < na; i0 += GT) {
                    __syncthreads();  // the previous T tile is no longer read
                    for (int e = tid; e < GT * GT; e += NT) {
                        const int ii = e / GT, cc = e - ii * GT;
                        const int i = i0 + ii, c = c0 + cc;
                        double s = 0.0;
                        if (i < na && c < 3 * nb)
                            for (int m = ist[i]; m < ist[i + 1]; ++m)
                                s = fma(em[m] * A.inv_s2,
                                        J2[((size_t)mj[m] * rep + f) * ld2 + c], s);
                        T[ii][cc] = s;
                    }
                    __syncthreads();
                    const int iend = min(GT, na - i0);
                    for (int ii = 0; ii < iend; ++ii) {
                        const double *jr = J1 + ((size_t)(i0 + ii) * rep + f) * ld1;
                        double jv[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int r = r0 + tr + 16 * u;
                            jv[u] = r < 3 * na ? jr[r] : 0.0;
                        }
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            const double tv = T[ii][tc + 16 * w];
#pragma unroll
                            for (int u = 0; u < 4; ++u) acc[u][w] = fma(jv[u], tv, acc[u][w]);
                        }
                    }
                }
            // rank-one terms, then write the tile
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int r = r0 + tr + 16 * u, c = c0 + tc + 16 * w;
                    if (r >= 3 * na || c >= 3 * nb) continue;
                    double s = acc[u][w];
                    for (int m = 0; m < np; ++m)
                        s -= em[m] * A.inv_s4 * V[(size_t)m * A.ldv + r] * U[(size_t)m * A.ldu + c];
                    out.ff(r, c, s);
                }
        }
}

template <int MODE>
int deriv_launch_generic(DerivArgs A, const std::vector<int2> &pairs, const SideMeta &s1,
                         const SideMeta &s2, int nlab, hipStream_t stream) {
    const size_t npairs = pairs.size();
    if (npairs == 0) return KF_OK;
    const size_t n_off = s1.offs.size() + s2.offs.size();
    const size_t pair_off = (sizeof(int) * n_off + 15) / 16 * 16;
    const size_t bytes = pair_off + sizeof(int2) * npairs;
    char *dev = static_cast<char *>(workspace(WS_PLAN, bytes, stream));
    char *stage = static_cast<char *>(host_staging(WS_PLAN, bytes));
    KF_REQUIRE(dev && stage, KF_ERR_NOMEM, "workspace allocation failed (%zu B)", bytes);
    std::copy(s1.offs.begin(), s1.offs.end(), reinterpret_cast<int *>(stage));
    std::copy(s2.offs.begin(), s2.offs.end(), reinterpret_cast<int *>(stage) + s1.offs.size());
    std::copy(pairs.begin(), pairs.end(), reinterpret_cast<int2 *>(stage + pair_off));
    KF_HIP_TRY(hipMemcpyAsync(dev, stage, bytes, hipMemcpyHostToDevice, stream));
    A.offs1 = reinterpret_cast<int *>(dev);
    A.offs2 = A.offs1 + s1.offs.size();
    A.pairs = reinterpret_cast<const int2 *>(dev + pair_off);
    int maxm = 1;
    for (const int2 &p : pairs) {
        int c = 0;
        for (int l = 0; l < nlab; ++l)
            c += s1.hist[(size_t)p.x * nlab + l] * s2.hist[(size_t)p.y * nlab + l];
        maxm = std::max(maxm, c);
    }
    A.maxm = maxm;
    A.ldv = 3 * A.ma1;
    A.ldu = 3 * A.ma2;
    A.slot_len = (size_t)maxm * (1 + A.ldv + A.ldu);
    const size_t iscr_len = 2 * (size_t)maxm + A.ma1 + 1;
    const size_t per_pair = A.slot_len * sizeof(double) + iscr_len * sizeof(int);
    const size_t budget = size_t(1) << 30;
    const size_t batch = std::max<size_t>(1, std::min(npairs, budget / per_pair));
    char *ws = static_cast<char *>(workspace(WS_AUX2, batch * per_pair + 256, stream));
    KF_REQUIRE(ws, KF_ERR_NOMEM, "scratch allocation failed");
    A.slot = reinterpret_cast<double *>(ws);
    int *iscr = reinterpret_cast<int *>(ws + batch * A.slot_len * sizeof(double));
    for (size_t p0 = 0; p0 < npairs; p0 += batch) {
        const unsigned nb = (unsigned)std::min(batch, npairs - p0);
        hipLaunchKernelGGL(deriv_generic_kernel<MODE>, dim3(nb), dim3(NT), 0, stream, A, (int)p0,
                           iscr, iscr_len);
        KF_HIP_TRY(hipGetLastError());
    }
    return KF_OK;
}

// Drop the descriptor columns that are zero for every atom of both sets (in X and in the
// Jacobians the mode reads): A then points at compacted copies.
int compact_features(DerivArgs &A, const int *N1, const int *N2, int nm1, int nm2,
                     hipStream_t stream) {
    CompactSets c;
    c.x1 = A.x1; c.dx1 = A.dx1; c.n1 = N1; c.nm1 = nm1; c.ma1 = A.ma1;
    c.x2 = A.x2; c.dx2 = A.dx2; c.n2 = N2; c.nm2 = nm2; c.ma2 = A.ma2;
    int nf = A.rep;
    const int rc = compact_columns(c, A.rep, WS_PACK, WS_PACK2, stream, &nf);
    if (rc) return rc;
    A.x1 = c.x1; A.dx1 = c.dx1; A.x2 = c.x2; A.dx2 = c.dx2;
    A.rep = nf;
    return KF_OK;
}

template <int MODE>
int deriv_impl(const double *X1, const double *dX1, const double *X2, const double *dX2,
               const int *Q1, const int *Q2, const int *N1, const int *N2, int nm1, int nm2,
               int ma1, int ma2, int rep, double sigma, double *out, hipStream_t stream) {
    KF_REQUIRE(std::isfinite(sigma) && sigma > 0.0, KF_ERR_SIGMA, "sigma must be > 0");
    KF_REQUIRE(nm1 >= 0 && nm2 >= 0 && ma1 >= 0 && ma2 >= 0 && rep >= 1, KF_ERR_ARG,
               "bad dimensions");
    // more than MAXA atoms per molecule: the size-general kernel
    const bool general = ma1 > MAXA || ma2 > MAXA;
    if (nm1 == 0 || nm2 == 0) return KF_OK;
    KF_REQUIRE(X1 && X2 && Q1 && Q2 && N1 && N2 && out, KF_ERR_ARG, "null pointer");
    const bool need1 = has_fe(MODE) || has_ff(MODE), need2 = has_ef(MODE) || has_ff(MODE);
    KF_REQUIRE((!need1 || dX1) && (!need2 || dX2), KF_ERR_ARG, "null Jacobian pointer");
    std::vector<int> q1, n1, q2, n2;
    int rc;
    if ((rc = read_metadata(Q1, N1, nm1, ma1, q1, n1, stream, WS_AUX0))) return rc;
    if (is_symm(MODE) || MODE == M_DIAG_BLOCKS) {
        q2 = q1;
        n2 = n1;
    } else if ((rc = read_metadata(Q2, N2, nm2, ma2, q2, n2, stream, WS_AUX1))) {
        return rc;
    }
    std::vector<int> labels;
    {
        std::vector<int> l1 = distinct_labels(q1.data(), n1.data(), nm1, ma1),
                         l2 = distinct_labels(q2.data(), n2.data(), nm2, ma2);
        labels.resize(l1.size() + l2.size());
        labels.erase(std::set_union(l1.begin(), l1.end(), l2.begin(), l2.end(), labels.begin()),
                     labels.end());
    }
    SideMeta s1, s2;
    side_meta(q1, n1, nm1, ma1, labels, s1);
    side_meta(q2, n2, nm2, ma2, labels, s2);

    DerivArgs A{};
    // a Jacobian the mode does not use is not read (nor compacted)
    A.x1 = X1; A.dx1 = need1 ? dX1 : nullptr; A.x2 = X2; A.dx2 = need2 ? dX2 : nullptr;
    A.q1 = Q1; A.q2 = Q2; A.n1 = N1; A.n2 = N2;
    A.ma1 = ma1; A.ma2 = ma2; A.rep = rep;
    A.cexp = -1.0 / (2.0 * sigma * sigma);
    A.inv_s2 = 1.0 / (sigma * sigma);
    A.inv_s4 = A.inv_s2 * A.inv_s2;
    A.out = out;
    switch (MODE) {
        case M_JAC: A.ld = s2.naq; break;
        case M_JAC_T: A.ld = nm2; break;
        case M_HESS: A.ld = s2.naq; break;
        case M_FULL: A.ld = (size_t)nm2 + s2.naq; A.ebase1 = nm1; A.ebase2 = nm2; break;
        case M_HESS_SYMM:
        case M_HESS_SYMM_RFP: A.ld = s1.naq; break;
        case M_DIAG_BLOCKS: A.ld = 1 + 3 * (size_t)ma1; break;
        default: A.ld = (size_t)nm1 + s1.naq; A.ebase1 = nm1; A.ebase2 = nm1; break;
    }
    std::vector<int2> pairs;
    if (MODE == M_DIAG_BLOCKS) {
        pairs.reserve(nm1);
        for (int a = 0; a < nm1; ++a) pairs.push_back(make_int2(a, a));
    } else if (is_symm(MODE)) {
        pairs.reserve((size_t)nm1 * (nm1 + 1) / 2);
        for (int a = 0; a < nm1; ++a)
            for (int b = a; b < nm1; ++b) pairs.push_back(make_int2(a, b));
    } else {
        pairs.reserve((size_t)nm1 * nm2);
        for (int a = 0; a < nm1; ++a)
            for (int b = 0; b < nm2; ++b) pairs.push_back(make_int2(a, b));
    }
    // the Hessian forms of zero-size sets have nothing to write
    if ((MODE == M_HESS || MODE == M_HESS_SYMM || MODE == M_HESS_SYMM_RFP) &&
        (s1.naq == 0 || s2.naq == 0))
        return KF_OK;
    if ((rc = compact_features(A, N1, N2, nm1, nm2, stream))) return rc;
    ScopedTimer timer(TM_FULL, stream);
    if (general) return deriv_launch_generic<MODE>(A, pairs, s1, s2, (int)labels.size(), stream);
    return deriv_launch<MODE>(A, pairs, s1, s2, (int)labels.size(), stream);
}

}  // namespace
}  // namespace kf

using namespace kf;

extern "C" int kf_local_kernel_jacobian(const double *X1, const double *X2, const double *dX2,
                                        const int *Q1, const int *Q2, const int *N1,
                                        const int *N2, int nm1, int nm2, int max_atoms1,
                                        int max_atoms2, int rep, double sigma, double *K,
                                        void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_JAC>(X1, nullptr, X2, dX2, Q1, Q2, N1, N2, nm1, nm2, max_atoms1,
                             max_atoms2, rep, sigma, K, as_stream(stream));
}

extern "C" int kf_local_kernel_jacobian_t(const double *X1, const double *X2, const double *dX1,
                                          const int *Q1, const int *Q2, const int *N1,
                                          const int *N2, int nm1, int nm2, int max_atoms1,
                                          int max_atoms2, int rep, double sigma, double *K,
                                          void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_JAC_T>(X1, dX1, X2, nullptr, Q1, Q2, N1, N2, nm1, nm2, max_atoms1,
                               max_atoms2, rep, sigma, K, as_stream(stream));
}

extern "C" int kf_local_kernel_hessian(const double *X1, const double *X2, const double *dX1,
                                       const double *dX2, const int *Q1, const int *Q2,
                                       const int *N1, const int *N2, int nm1, int nm2,
                                       int max_atoms1, int max_atoms2, int rep, double sigma,
                                       double *K, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_HESS>(X1, dX1, X2, dX2, Q1, Q2, N1, N2, nm1, nm2, max_atoms1, max_atoms2,
                              rep, sigma, K, as_stream(stream));
}

extern "C" int kf_local_kernel_full(const double *X1, const double *X2, const double *dX1,
                                    const double *dX2, const int *Q1, const int *Q2,
                                    const int *N1, const int *N2, int nm1, int nm2,
                                    int max_atoms1, int max_atoms2, int rep, double sigma,
                                    double *K, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_FULL>(X1, dX1, X2, dX2, Q1, Q2, N1, N2, nm1, nm2, max_atoms1, max_atoms2,
                              rep, sigma, K, as_stream(stream));
}

extern "C" int kf_local_kernel_hessian_symm(const double *X, const double *dX, const int *Q,
                                            const int *N, int nm, int max_atoms, int rep,
                                            double sigma, double *K, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_HESS_SYMM>(X, dX, X, dX, Q, Q, N, N, nm, nm, max_atoms, max_atoms, rep,
                                   sigma, K, as_stream(stream));
}

extern "C" int kf_local_kernel_hessian_symm_rfp(const double *X, const double *dX, const int *Q,
                                                const int *N, int nm, int max_atoms, int rep,
                                                double sigma, double *arf, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_HESS_SYMM_RFP>(X, dX, X, dX, Q, Q, N, N, nm, nm, max_atoms, max_atoms,
                                       rep, sigma, arf, as_stream(stream));
}

extern "C" int kf_local_kernel_full_symm(const double *X, const double *dX, const int *Q,
                                         const int *N, int nm, int max_atoms, int rep,
                                         double sigma, double *K, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_FULL_SYMM>(X, dX, X, dX, Q, Q, N, N, nm, nm, max_atoms, max_atoms, rep,
                                   sigma, K, as_stream(stream));
}

extern "C" int kf_local_kernel_full_symm_rfp(const double *X, const double *dX, const int *Q,
                                             const int *N, int nm, int max_atoms, int rep,
                                             double sigma, double *arf, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return deriv_impl<M_FULL_SYMM_RFP>(X, dX, X, dX, Q, Q, N, N, nm, nm, max_atoms, max_atoms,
                                       rep, sigma, arf, as_stream(stream));
}

extern "C" int kf_local_full_diag_blocks(const double *X, const double *dX, const int *Q,
                                         const int *N, int nm, int max_atoms, int rep,
                                         double sigma, double *blocks, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    // entries beyond a molecule's 1 + 3 N[b] live rows/columns are not written
    return deriv_impl<M_DIAG_BLOCKS>(X, dX, X, dX, Q, Q, N, N, nm, nm, max_atoms, max_atoms, rep,
                                     sigma, blocks, as_stream(stream));
}
