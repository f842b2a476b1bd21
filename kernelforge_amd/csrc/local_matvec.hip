// local_matvec.hip -- matrix-free products with the energy+force local kernel:
// alpha_desc, the Jacobian-transposed (energy) matvec, the Hessian (force) matvec and
// the full [E; F] matvec that drives PCG on the energy+force system.
//
// With alpha_desc[b,j,:] = J_bj alpha_F[b] (kf_local_alpha_desc) and, for every
// query atom (a,i) and label-matched train atom (b,j):
//   d = x_ai - x_bj,  e = exp(-|d|^2/2s^2),  c = e/s^2,  inner = d . alpha_desc[b,j]
//   E[a]  += e alpha_E[b] + c inner
//   G_ai  += c alpha_desc[b,j] - (e/s^4) inner d + c alpha_E[b] x_bj - c alpha_E[b] x_ai
//   F[a]  += J_ai^T G_ai
// (src/local_kernels.cpp:2895-3425).  Collecting terms per label, with
//   beta_ij = (e/s^4) inner_ij + c_ij alpha_E[b(j)]
//   G = C * ALPHA_DESC + B * X2 - diag(B 1) * X1
// so each label is two FP64 MFMA products over packed rows:
//   [S | P] = X1 [X2; ALPHA_DESC]^T, turned into T = [B | C] in registers
//   G = T [X2; ALPHA_DESC]
// then one pass over dX1 forms J_ai^T (G_ai - w_ai x_ai) per query atom, and per-
// molecule sums in a fixed order (deterministic, no atomics).
//
// The products run over the descriptor columns that are non-zero in the training side
// (X2 or ALPHA_DESC): the others add exact zeros to S, P and G whatever the query holds
// (C9H8O4 conformers use 312 of 720).  All labels share each launch: the packed rows of a
// label start at a multiple of 16 and are padded with zero rows to one, and a list of
// segments (label, query rows) tells a wave which tile it has.  Operands go from global
// memory straight into registers: the 16 values of a row that four MFMA steps need are two
// 16-byte loads per lane when the summation index of a step is permuted the same way in
// both operands (lane group g holds k = 2 g, 2 g + 1, 2 g + 8, 2 g + 9), so no LDS tile and no
// barrier is needed, and a product with a handful of query rows runs at the speed its
// training rows can be read.
//
// Measured (whole calls on 21-atom C/H/O conformers, with the descriptors): one molecule
// against 200 in a plan 81 us (2,110 before: one wave per atom for the back-projection,
// 64-row tiles without splits for the products); 100 against 1,000, float32 in and out,
// 1.7 ms (8.5), of which the two products 0.5 ms each at 36 TFLOP/s.
#include <algorithm>
#include <new>
#include <cmath>
#include <vector>

#include "kf_common.hpp"
#include "local_plan.hpp"
#include "reg_pipeline.hpp"

namespace kf {
namespace {

constexpr int NT = 256;
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// alpha_desc[b,j,f] = sum_c dX[b,j,f,c] alpha[offs[b] + c] for j < N[b]; 0 otherwise.
// One wave per (molecule, atom), lanes over Jacobian columns, wave sum per feature.
__global__ __launch_bounds__(NT) void alpha_desc_kernel(const double *__restrict__ dX,
                                                        const int *__restrict__ N,
                                                        const int *__restrict__ offs, int nm,
                                                        int ma, int rep,
                                                        const double *__restrict__ alpha,
                                                        double *__restrict__ out) {
    const int lane = threadIdx.x & 63;
    const long atom = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (atom >= (long)nm * ma) return;
    const int b = (int)(atom / ma), j = (int)(atom - (long)b * ma);
    const int nb = min(max(N[b], 0), ma);
    double *o = out + atom * rep;
    if (j >= nb) {
        for (int f = lane; f < rep; f += 64) o[f] = 0.0;
        return;
    }
    const int ld = 3 * ma, nc = 3 * nb;
    const double *J = dX + atom * rep * ld;
    // Jacobian columns in groups of 128 (two per lane); one group for up to 42 atoms
    for (int c0 = 0; c0 < nc; c0 += 128) {
        const double a0 = c0 + lane < nc ? alpha[offs[b] + c0 + lane] : 0.0;
        const double a1 = c0 + lane + 64 < nc ? alpha[offs[b] + c0 + lane + 64] : 0.0;
        for (int f = 0; f < rep; ++f) {
            const double *row = J + (size_t)f * ld + c0;
            double s = c0 + lane < nc ? row[lane] * a0 : 0.0;
            if (c0 + lane + 64 < nc) s = fma(row[lane + 64], a1, s);
            s = wave_sum(s);
            if (lane == 0) o[f] = c0 == 0 ? s : o[f] + s;
        }
    }
}

// One segment: a run of packed query rows of one label against the label's training rows.
struct MvSeg {
    int q0, R1;           // first packed query row, rows (q0 a multiple of 16)
    int r2, R2, R2p;      // first packed training row, rows, rows padded to 16
    int nsplit;           // splits of the summation over the training rows in G = T [X2; AD]
    int it1, it2;         // first item of the segment in the two products' launches
    size_t toff, goff, eoff;  // offsets into T, the partial G and the partial row sums
};

// Segment of item / row `x`: the last one whose start (by `at`) is not beyond it.
template <class At>
__device__ inline int find_seg(const MvSeg *segs, int nseg, int x, At at) {
    int s = 0;
    while (s + 1 < nseg && at(segs[s + 1]) <= x) ++s;
    return s;
}

// flag[f] = 1 when column f is non-zero in X2 or AD for an atom of the training set.  A
// work-group takes `per` molecules and its threads a column each, leaving a column at its
// first non-zero value.
template <typename T>
__global__ __launch_bounds__(NT) void train_cols_kernel(const T *__restrict__ X2,
                                                        const T *__restrict__ AD,
                                                        const int *__restrict__ N, int nm, int ma,
                                                        int rep, int per, int *__restrict__ flag) {
    const int b0 = blockIdx.x * per, b1 = min(b0 + per, nm);
    for (int f = threadIdx.x; f < rep; f += NT) {
        bool nz = false;
        for (int b = b0; b < b1 && !nz; ++b) {
            const int nb = min(max(N[b], 0), ma);
            const size_t base = (size_t)b * ma * rep + f;
            for (int i = 0; i < nb && !nz; i += 4) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const size_t at = base + (size_t)min(i + u, nb - 1) * rep;
                    nz |= (X2[at] != T(0)) | (AD[at] != T(0));
                }
            }
        }
        if (nz) flag[f] = 1;
    }
}

// Packed row r < rows takes source row src[r] (-1: a zero row) on the columns with
// inv[f] >= 0 (its place in the packed row of nfp columns, the rest zero).  For a training
// set (src2) row r goes to the stacked block of its segment, X2 rows first, then AD rows,
// with |x|^2, x . ad and the molecule's alpha_E; for a query set to row r with |x|^2, NaN where
// a column left out is not finite.
template <typename T>
__global__ __launch_bounds__(NT) void pack_rows_kernel(const T *__restrict__ src,
                                                       const T *__restrict__ src2,
                                                       const int *__restrict__ idx, int rows,
                                                       size_t first, int ma, int rep,
                                                       const int *__restrict__ inv, int nf, int nfp,
                                                       const MvSeg *__restrict__ segs, int nseg,
                                                       const T *__restrict__ aE,
                                                       double *__restrict__ dst,
                                                       double *__restrict__ n2,
                                                       double *__restrict__ dot,
                                                       double *__restrict__ aEr) {
    const int lane = threadIdx.x & 63;
    const int r = (int)(first + blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int at = idx[r];
    double *d = dst + (size_t)r * nfp, *da = nullptr;
    if (src2) {
        const MvSeg &S = segs[find_seg(segs, nseg, r, [](const MvSeg &t) { return t.r2; })];
        d = dst + (size_t)(S.r2 + r) * nfp;
        da = d + (size_t)S.R2p * nfp;
    }
    for (int f = nf + lane; f < nfp; f += 64) {
        d[f] = 0.0;
        if (da) da[f] = 0.0;
    }
    double nn = 0.0, dd = 0.0;
    for (int f = lane; f < rep; f += 64) {
        const int c = inv[f];
        const double v = at >= 0 ? (double)src[(size_t)at * rep + f] : 0.0;
        if (c >= 0) d[c] = v;
        nn = fma(v, v, nn);
        if (src2) {
            const double w = at >= 0 ? (double)src2[(size_t)at * rep + f] : 0.0;
            if (c >= 0) da[c] = w;
            dd = fma(v, w, dd);
        } else if (c < 0) {
            dd = fma(v, 0.0, dd);
        }
    }
    nn = wave_sum(nn);
    dd = wave_sum(dd);
    if (lane == 0) {
        n2[r] = src2 ? nn : nn + dd;
        if (dot) dot[r] = dd;
        if (aEr) aEr[r] = (aE && at >= 0) ? (double)aE[at / ma] : 0.0;
    }
}

// Work-group -> tile index, consecutive tiles on one XCD (work-groups are dealt round-robin
// over eight of them) so that the waves that share an operand share an L2.
__device__ inline int xcd_tile() {
    const int g = blockIdx.x, G = gridDim.x;
    return (G % 8 == 0) ? (g % 8) * (G / 8) + g / 8 : g;
}

// The four summation steps of 16 columns: k = 2 g, 2 g + 1, 2 g + 8, 2 g + 9 for lane group
// g, so that a load takes 64 contiguous bytes of 16 rows.
__device__ inline void load4(const double *p, double (&v)[4]) {
    const v2d a = *reinterpret_cast<const v2d *>(p), b = *reinterpret_cast<const v2d *>(p + 8);
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}

// T = [B | C] of a tile of 16 MF query rows x 16 NFT training rows per wave (KW = 1) or per
// work-group with its four waves each taking a quarter of the columns (KW = 4, for launches
// with too few tiles to fill the GPU: one molecule against 200 conformers is 263 tiles).
//   d2 = n1 + n2 - 2 S, e = exp(cexp d2), c = e / s^2, inner = P - rdot
//   B = (e / s^4) inner + c aE,  C = c
// and per 16 training rows the row sums of e aE + c inner (ep) and of B (wp).
template <int MF, int NFT, int KW>
__global__ __launch_bounds__(NT, 2) void coef_kernel(
    const MvSeg *__restrict__ segs, int nseg, int items, const double *__restrict__ Xq, int row0,
    int qrows,
    const double *__restrict__ nq, const double *__restrict__ P2, const double *__restrict__ n2,
    const double *__restrict__ rdot, const double *__restrict__ aE, int nfp, double cexp,
    double inv_s2, double *__restrict__ T, double *__restrict__ ep, double *__restrict__ wp) {
    __shared__ double red[KW > 1 ? KW : 1][KW > 1 ? MF * NFT * 8 : 1][64];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int item = KW == 1 ? xcd_tile() * 4 + wv : xcd_tile();
    if (item >= items) return;
    const MvSeg S = segs[find_seg(segs, nseg, item, [](const MvSeg &t) { return t.it1; })];
    const int mt = (S.R1 + 16 * MF - 1) / (16 * MF), q0 = S.q0 - row0;
    const int loc = item - S.it1, m0 = (loc % mt) * 16 * MF, n0 = (loc / mt) * 16 * NFT;
    const double *pa[MF], *pb[NFT], *pd[NFT];
#pragma unroll
    for (int m = 0; m < MF; ++m)
        pa[m] = Xq + (size_t)min(q0 + m0 + 16 * m + r, qrows - 1) * nfp + 2 * g;
#pragma unroll
    for (int n = 0; n < NFT; ++n) {
        pb[n] = P2 + (size_t)(2 * S.r2 + min(n0 + 16 * n + r, S.R2p - 1)) * nfp + 2 * g;
        pd[n] = pb[n] + (size_t)S.R2p * nfp;
    }
    v4d s[MF][NFT], p[MF][NFT];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int n = 0; n < NFT; ++n) s[m][n] = p[m][n] = (v4d){0.0, 0.0, 0.0, 0.0};
    double a[2][MF][4], b[2][NFT][4], d[2][NFT][4];
    auto load = [&](int buf, int k) {
#pragma unroll
        for (int m = 0; m < MF; ++m) load4(pa[m] + k, a[buf][m]);
#pragma unroll
        for (int n = 0; n < NFT; ++n) {
            load4(pb[n] + k, b[buf][n]);
            load4(pd[n] + k, d[buf][n]);
        }
    };
    auto mul = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int m = 0; m < MF; ++m)
#pragma unroll
                for (int n = 0; n < NFT; ++n) {
                    s[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[buf][m][u], b[buf][n][u],
                                                                   s[m][n], 0, 0, 0);
                    p[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[buf][m][u], d[buf][n][u],
                                                                   p[m][n], 0, 0, 0);
                }
    };
    const int kb = KW == 1 ? 0 : 16 * wv;
    reg_pipeline((nfp - kb + 16 * KW - 1) / (16 * KW),
                 [&](int buf, int i) { load(buf, kb + i * 16 * KW); }, mul);
    if (KW > 1) {
#pragma unroll
        for (int m = 0; m < MF; ++m)
#pragma unroll
            for (int n = 0; n < NFT; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    red[wv][(m * NFT + n) * 8 + v][lane] = s[m][n][v];
                    red[wv][(m * NFT + n) * 8 + 4 + v][lane] = p[m][n][v];
                }
        __syncthreads();
    }
    const int nfr = S.R2p >> 4;
    const size_t ldt = 2 * (size_t)S.R2p;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int n = 0; n < NFT; ++n) {
            if (KW > 1 && ((m * NFT + n) & 3) != wv) continue;
            const int t = n0 + 16 * n + r;
            if (n0 + 16 * n >= S.R2p) continue;
            const bool live = t < S.R2;
            const double nt = n2[S.r2 + t], rd = rdot[S.r2 + t], ae = aE[S.r2 + t];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = m0 + 16 * m + mfma16_row_f64(lane, v);
                double sv = s[m][n][v], pv = p[m][n][v];
                if (KW > 1) {
                    sv = pv = 0.0;
#pragma unroll
                    for (int w = 0; w < KW; ++w) {
                        sv += red[w][(m * NFT + n) * 8 + v][lane];
                        pv += red[w][(m * NFT + n) * 8 + 4 + v][lane];
                    }
                }
                const double q = nq[min(q0 + row, qrows - 1)];
                const double d2 = fmax(q + nt - 2.0 * sv, 0.0);
                const double e = live ? exp(cexp * d2) : 0.0, c = e * inv_s2;
                // a query row with an infinity or a NaN in a column that the training side
                // lacks still gives NaN; an infinite norm alone is a row far away
                const double inner = q != q ? q : pv - rd;
                double bco = c * inv_s2 * inner + c * ae;
                double es = e * ae + c * inner;
                if (!live) bco = es = 0.0;
                if (row < S.R1 && T) {
                    T[S.toff + row * ldt + t] = bco;
                    T[S.toff + row * ldt + S.R2p + t] = c;
                }
#pragma unroll
                for (int o = 1; o < 16; o <<= 1) {
                    es += __shfl_xor(es, o, 64);
                    bco += __shfl_xor(bco, o, 64);
                }
                if (r == 0 && row < S.R1) {
                    ep[S.eoff + (size_t)row * nfr + (n0 >> 4) + n] = es;
                    wp[S.eoff + (size_t)row * nfr + (n0 >> 4) + n] = bco;
                }
            }
        }
}

// Partial G = T [X2; AD] over `ks` of the 2 R2p summed rows: a wave has 16 MF query rows x
// 64 columns of one split.  Without splits the product of a few query rows has as many
// tiles as columns / 64: 12 work-groups for one 21-atom molecule.
template <int MF>
__global__ __launch_bounds__(NT, 2) void weighted_rows_kernel(const MvSeg *__restrict__ segs, int nseg,
                                                           int items, int ks,
                                                           const double *__restrict__ T,
                                                           const double *__restrict__ P2, int nfp,
                                                           double *__restrict__ G) {
    constexpr int NF = 4;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int item = xcd_tile() * 4 + wv;
    if (item >= items) return;
    const MvSeg S = segs[find_seg(segs, nseg, item, [](const MvSeg &t) { return t.it2; })];
    const int mt = (S.R1 + 16 * MF - 1) / (16 * MF), nt = (nfp + 63) / 64;
    const int loc = item - S.it2, n0 = (loc % nt) * 64, m0 = (loc / nt % mt) * 16 * MF,
              split = loc / (nt * mt);
    const int kb = split * ks, ke = min(kb + ks, 2 * S.R2p);
    const double *pa[MF], *pb[NF];
#pragma unroll
    for (int m = 0; m < MF; ++m)
        pa[m] = T + S.toff + (size_t)min(m0 + 16 * m + r, S.R1 - 1) * (2 * S.R2p) + 2 * g;
#pragma unroll
    for (int n = 0; n < NF; ++n)
        pb[n] = P2 + (size_t)(2 * S.r2 + 2 * g) * nfp + min(n0 + 16 * n + r, nfp - 1);
    v4d c[MF][NF];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int n = 0; n < NF; ++n) c[m][n] = (v4d){0.0, 0.0, 0.0, 0.0};
    double a[2][MF][4], b[2][NF][4];
    auto load = [&](int buf, int k) {
#pragma unroll
        for (int m = 0; m < MF; ++m) load4(pa[m] + k, a[buf][m]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int n = 0; n < NF; ++n) b[buf][n][u] = pb[n][(size_t)(k + (u < 2 ? u : u + 6)) * nfp];
    };
    auto mul = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int m = 0; m < MF; ++m)
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    c[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[buf][m][u], b[buf][n][u],
                                                                   c[m][n], 0, 0, 0);
    };
    reg_pipeline((ke - kb) / 16, [&](int buf, int i) { load(buf, kb + i * 16); }, mul);
    double *out = G + S.goff + (size_t)split * S.R1 * nfp;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int n = 0; n < NF; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = m0 + 16 * m + mfma16_row_f64(lane, v), col = n0 + 16 * n + r;
                if (row < S.R1 && col < nfp) out[(size_t)row * nfp + col] = c[m][n][v];
            }
}

// One packed query row and one run of features per work-group:
//   Fat[part][src, c] = sum over the run of dX1[src, f, c] (G[f] - w X1[src, f])
// with G summed over its splits and w, E over the partial row sums, in a fixed order.
// The rows of dX1 are contiguous, so the threads take nrow rows of nc columns at a time.
// Bound by the read of dX1; the runs (`parts`, at most 16) give a batch of a few molecules
// enough work-groups to draw on the whole memory system.
template <typename T>
__global__ __launch_bounds__(NT) void backproj_kernel(const MvSeg *__restrict__ segs, int nseg,
                                                      int row0, const double *__restrict__ G,
                                                      const double *__restrict__ ep,
                                                      const double *__restrict__ wp,
                                                      const T *__restrict__ X1,
                                                      const T *__restrict__ dX1,
                                                      const int *__restrict__ idx,
                                                      const int *__restrict__ inv,
                                                      const int *__restrict__ offs, int ma,
                                                      int rep, int nfp, int natoms,
                                                      double *__restrict__ erow,
                                                      double *__restrict__ Fat) {
    extern __shared__ double lds[];  // the run's features, then a partial sum per thread
    __shared__ double part_e[4], part_w[4];
    const int row = row0 + blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int src = idx[row];
    if (src < 0) return;
    const MvSeg S = segs[find_seg(segs, nseg, row, [](const MvSeg &t) { return t.q0; })];
    const int loc = row - S.q0, nfr = S.R2p >> 4;
    double es = 0.0, w = 0.0;
    for (int t = tid; t < nfr; t += NT) {
        es += ep[S.eoff + (size_t)loc * nfr + t];
        w += wp[S.eoff + (size_t)loc * nfr + t];
    }
    es = wave_sum(es);
    w = wave_sum(w);
    if (lane == 0) {
        part_e[wv] = es;
        part_w[wv] = w;
    }
    __syncthreads();
    w = part_w[0] + part_w[1] + part_w[2] + part_w[3];
    if (erow && blockIdx.y == 0 && tid == 0)
        erow[src] = part_e[0] + part_e[1] + part_e[2] + part_e[3];
    if (!Fat) return;
    const int run = (rep + gridDim.y - 1) / gridDim.y;
    const int f0 = blockIdx.y * run, fn = min(run, rep - f0);
    for (int t = tid; t < fn; t += NT) {
        const int c = inv[f0 + t];
        double gv = 0.0;
        if (c >= 0) {
            const double *gp = G + S.goff + (size_t)loc * nfp + c;
            const size_t st = (size_t)S.R1 * nfp;
            int k = 0;
            for (; k + 4 <= S.nsplit; k += 4) {
                const double g0 = gp[k * st], g1 = gp[(k + 1) * st], g2 = gp[(k + 2) * st],
                             g3 = gp[(k + 3) * st];
                gv = (((gv + g0) + g1) + g2) + g3;
            }
            for (; k < S.nsplit; ++k) gv += gp[k * st];
        }
        lds[t] = gv - w * (double)X1[(size_t)src * rep + f0 + t];
    }
    __syncthreads();
    double *red = lds + run;
    const int a = src / ma, ld = 3 * ma, nc = offs[a + 1] - offs[a];
    const T *J = dX1 + ((size_t)src * rep + f0) * ld;
    double *o = Fat + ((size_t)blockIdx.y * natoms + src) * ld;
    // columns in groups of NT (one for up to 85 atoms)
    for (int c0 = 0; c0 < nc; c0 += NT) {
        const int cn = min(nc - c0, NT), nrow = NT / cn, rr = tid / cn, c = c0 + tid - rr * cn;
        double s = 0.0;
        if (rr < nrow) {
            int f = rr;
            for (; f + 7 * nrow < fn; f += 8 * nrow) {
                T j[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) j[u] = J[(size_t)(f + u * nrow) * ld + c];
#pragma unroll
                for (int u = 0; u < 8; ++u) s = fma((double)j[u], lds[f + u * nrow], s);
            }
            for (; f < fn; f += nrow) s = fma((double)J[(size_t)f * ld + c], lds[f], s);
        }
        red[tid] = s;
        __syncthreads();
        if (tid < cn) {
            for (int x = 1; x < nrow; ++x) s += red[x * cn + tid];
            o[c0 + tid] = s;
        }
        __syncthreads();
    }
}

// erow and the Fat rows of the atoms in idx are zero: atoms whose label the training side
// lacks, which the products leave out (0 times what they hold would make NaN of a value that
// is not finite).
__global__ __launch_bounds__(64) void zero_rows_kernel(const int *__restrict__ idx, int ld,
                                                       int parts, int natoms,
                                                       double *__restrict__ erow,
                                                       double *__restrict__ Fat) {
    const int src = idx[blockIdx.x];
    if (threadIdx.x == 0) erow[src] = 0.0;
    if (!Fat) return;
    for (int t = threadIdx.x; t < parts * ld; t += 64)
        Fat[((size_t)(t / ld) * natoms + src) * ld + t % ld] = 0.0;
}

// E[a] = sum_i erow[a*ma+i]; F[offs[a] + c] = sum over the parts and the atoms of
// Fat[part][a*ma+i, c] (fixed order).  Atom counts come from the force offsets.  The
// (part, atom) rows are dealt over the groups of nc threads: one molecule of 21 atoms in 16
// parts is 336 rows, a 30 us chain for one thread per column.
constexpr int kReduceThreads = 512;
__global__ __launch_bounds__(kReduceThreads) void reduce_mol_kernel(
    const double *__restrict__ erow, const double *__restrict__ Fat, int parts,
    const int *__restrict__ offs, int natoms, int ma, size_t first, double *__restrict__ E,
    double *__restrict__ F) {
    __shared__ double red[kReduceThreads];
    const int a = (int)(first + blockIdx.x), tid = threadIdx.x;
    const int nc = offs[a + 1] - offs[a], na = nc / 3, ld = 3 * ma;
    if (E && tid < 64) {
        double s = 0.0;
        for (int i = tid; i < na; i += 64) s += erow[(size_t)a * ma + i];
        s = wave_sum(s);
        if (tid == 0) E[a] = s;
    }
    if (!F) return;
    for (int c0 = 0; c0 < nc; c0 += kReduceThreads) {
        const int cn = min(nc - c0, kReduceThreads), nrow = kReduceThreads / cn, rr = tid / cn;
        const double *q = Fat + (size_t)a * ma * ld + c0 + tid - rr * cn;
        double s = 0.0;
        if (rr < nrow) {
#pragma unroll 4
            for (int t = rr; t < parts * na; t += nrow)
                s += q[((size_t)(t / na) * natoms + t % na) * ld];
        }
        red[tid] = s;
        __syncthreads();
        if (tid < cn) {
            for (int x = 1; x < nrow; ++x) s += red[x * cn + tid];
            F[offs[a] + c0 + tid] = s;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Host side: the layout of one matvec (packed rows, segments, rounds) and its launches.
// ---------------------------------------------------------------------------
struct MvRound {
    int seg0, nseg;    // segments of the round
    int row0, rows;    // packed query rows they cover
    int items1, items2, ks;
    bool wide, split_k;  // 32-row tiles; KW = 4
};

struct MvLayout {
    int nm1 = 0, ma1 = 0, rep = 0, nf = 0, nfp = 0, parts = 1;
    int q_rows = 0, t_rows = 0;             // packed rows, padding included: of the longest
                                            // round, of the training set
    std::vector<int> offs, src1, src2, inv;  // force offsets, packed rows' sources, columns
    std::vector<int> src0;                   // query atoms without a partner
    std::vector<MvSeg> segs;
    std::vector<MvRound> rounds;
    size_t T_len = 0, G_len = 0, e_len = 0;  // per round, the largest
    // one device block of ints: segments first (8-byte aligned), then the vectors
    size_t meta_bytes() const {
        return sizeof(MvSeg) * segs.size() +
               sizeof(int) * (offs.size() + src1.size() + src2.size() + inv.size() + src0.size());
    }
    void write_meta(char *p) const {
        auto put = [&](const void *v, size_t n) { std::copy((const char *)v, (const char *)v + n, p); p += n; };
        put(segs.data(), sizeof(MvSeg) * segs.size());
        put(offs.data(), sizeof(int) * offs.size());
        put(src1.data(), sizeof(int) * src1.size());
        put(src2.data(), sizeof(int) * src2.size());
        put(inv.data(), sizeof(int) * inv.size());
        put(src0.data(), sizeof(int) * src0.size());
    }
    size_t train_doubles() const { return (size_t)2 * t_rows * nfp + 3 * (size_t)t_rows; }
    size_t query_doubles() const {
        return (size_t)q_rows * nfp + q_rows + T_len + G_len + 2 * e_len;
    }
    size_t acc_doubles(bool forces) const {
        const size_t natom = (size_t)nm1 * ma1;
        return natom + (forces ? (size_t)parts * natom * 3 * ma1 : 0);
    }
};
// device addresses of a layout's pieces
struct MvDev {
    const MvSeg *segs;
    const int *offs, *src1, *src2, *inv, *src0;
    double *P2, *n2, *rdot, *aE;
    double *Xq, *nq, *T, *G, *ep, *wp;
    double *erow, *Fat;
};

int round_up16(int n) { return (n + 15) & ~15; }

// The packed query rows of one round with their parts of T and G stay within this many doubles
// (1 GiB), whatever the query set's size.
constexpr size_t kTBudget = (size_t(1) << 30) / sizeof(double);

// The layout of all labels of the query set, or of its `only`th (with `parts` runs of features
// then); returns how many there are.
int mv_layout(const std::vector<int> &q1, const std::vector<int> &n1, int nm1, int ma1,
               const std::vector<int> &q2, const std::vector<int> &n2, int nm2, int ma2, int rep,
               const int *flag, bool forces, MvLayout &L, int only = -1, int parts = 0) {
    L.nm1 = nm1;
    L.ma1 = ma1;
    L.rep = rep;
    const std::vector<int> labels = distinct_labels(q1.data(), n1.data(), nm1, ma1);
    LocalPlan p1, p2;
    build_plan(q1.data(), n1.data(), nm1, ma1, labels, p1);
    if (nm2 > 0) build_plan(q2.data(), n2.data(), nm2, ma2, labels, p2);
    L.offs.assign(nm1 + 1, 0);
    for (int a = 0; a < nm1; ++a) L.offs[a + 1] = L.offs[a] + 3 * clamp_atoms(n1[a], ma1);
    L.inv.assign(rep, -1);
    for (int f = 0; f < rep; ++f)
        if (flag[f]) L.inv[f] = L.nf++;
    L.nfp = std::max(16, round_up16(L.nf));
    const int nt2 = (L.nfp + 63) / 64;
    int q0 = 0, r2 = 0;
    MvRound R{};
    size_t T = 0, G = 0, E = 0;
    auto close = [&]() {  // choose the round's variants and lay its segments out
        if (R.nseg == 0) return;
        int maxR1 = 0;
        for (int s = R.seg0; s < R.seg0 + R.nseg; ++s) maxR1 = std::max(maxR1, L.segs[s].R1);
        // 32-row tiles read the training rows once for two row fragments; up to 16 query
        // rows of a label (one molecule) would leave half of such a tile empty
        R.wide = maxR1 > 16;
        const int mf = R.wide ? 32 : 16;
        long tiles = 0, work = 0;
        for (int s = R.seg0; s < R.seg0 + R.nseg; ++s) {
            const MvSeg &g = L.segs[s];
            const long mt = (g.R1 + mf - 1) / mf;
            tiles += mt * ((g.R2p + 31) / 32);
            work += mt * nt2 * 2 * g.R2p;
        }
        R.split_k = !R.wide || tiles < 2048;
        // rows summed per split: about 2,048 waves (two per SIMD) over all tiles, in whole
        // groups of 16, at least 64 so that a wave's start-up does not dominate
        R.ks = (int)std::max<long>(64, (work / 2048 + 15) & ~15L);
        const int nft = R.wide && !R.split_k ? 32 : 16;
        for (int s = R.seg0; s < R.seg0 + R.nseg; ++s) {
            MvSeg &g = L.segs[s];
            const int mt = (g.R1 + mf - 1) / mf;
            g.nsplit = (2 * g.R2p + R.ks - 1) / R.ks;
            g.it1 = R.items1;
            g.it2 = R.items2;
            R.items1 += mt * ((g.R2p + nft - 1) / nft);
            R.items2 += mt * nt2 * g.nsplit;
            g.toff = T;
            g.goff = G;
            g.eoff = E;
            T += (size_t)g.R1 * 2 * g.R2p;
            G += (size_t)g.nsplit * g.R1 * L.nfp;
            E += (size_t)g.R1 * (g.R2p / 16);
        }
        L.T_len = std::max(L.T_len, forces ? T + (T & 1) : 0);
        L.G_len = std::max(L.G_len, forces ? G : 0);
        L.e_len = std::max(L.e_len, E);
        L.q_rows = std::max(L.q_rows, R.rows);
        L.rounds.push_back(R);
        T = G = E = 0;
        R = MvRound{};
    };
    size_t held = 0;
    for (int l = only < 0 ? 0 : only; l < (only < 0 ? p1.nlabels : only + 1); ++l) {
        const int *m1 = &p1.mol_row[(size_t)l * (nm1 + 1)];
        const int R1 = m1[nm1] - m1[0];
        int R2 = 0, b2 = 0;
        if (nm2 > 0) {
            const int *m2 = &p2.mol_row[(size_t)l * (nm2 + 1)];
            b2 = m2[0];
            R2 = m2[nm2] - b2;
        }
        if (R2 == 0) {
            L.src0.insert(L.src0.end(), p1.src.begin() + m1[0], p1.src.begin() + m1[nm1]);
            continue;
        }
        if (R1 == 0) continue;
        const int R2p = round_up16(R2);
        L.src2.insert(L.src2.end(), p2.src.begin() + b2, p2.src.begin() + b2 + R2);
        L.src2.insert(L.src2.end(), R2p - R2, -1);
        const size_t per_row = 2 * ((size_t)R2p + L.nfp);
        const int qb = std::max<int>(
            64, (int)std::min<size_t>((size_t)round_up16(R1), kTBudget / per_row / 64 * 64));
        for (int x = 0; x < R1; x += qb) {
            const int n = std::min(qb, R1 - x), np = round_up16(n);
            const size_t need = n * per_row;
            if (R.nseg > 0 && held + need > kTBudget) {
                close();
                held = 0;
            }
            if (R.nseg == 0) {
                R.seg0 = (int)L.segs.size();
                R.row0 = q0;
            }
            held += need;
            L.segs.push_back({q0, n, r2, R2, R2p, 0, 0, 0, 0, 0, 0});
            ++R.nseg;
            R.rows += np;
            L.src1.insert(L.src1.end(), p1.src.begin() + m1[0] + x, p1.src.begin() + m1[0] + x + n);
            L.src1.insert(L.src1.end(), np - n, -1);
            q0 += np;
        }
        r2 += R2p;
    }
    close();
    L.t_rows = r2;
    // runs of features per query row in the back-projection: 2,048 work-groups, at most 16;
    // a run is held in LDS, 4,096 features (32 KB) at most
    const int least = (rep + 4095) / 4096;
    L.parts = parts > 0 ? std::max(parts, least)
              : q0 == 0 ? 1
                        : std::max(least, std::min({16, 2048 / q0, (rep + 31) / 32}));
    return p1.nlabels;
}

MvDev mv_place(const MvLayout &L, char *meta, double *train, double *query, double *acc) {
    MvDev D{};
    D.segs = reinterpret_cast<const MvSeg *>(meta);
    D.offs = reinterpret_cast<const int *>(meta + sizeof(MvSeg) * L.segs.size());
    D.src1 = D.offs + L.offs.size();
    D.src2 = D.src1 + L.src1.size();
    D.inv = D.src2 + L.src2.size();
    D.src0 = D.inv + L.inv.size();
    D.P2 = train;
    D.n2 = D.P2 + (size_t)2 * L.t_rows * L.nfp;
    D.rdot = D.n2 + L.t_rows;
    D.aE = D.rdot + L.t_rows;
    D.Xq = query;
    D.nq = D.Xq + (size_t)L.q_rows * L.nfp;
    D.T = D.nq + L.q_rows;
    D.G = D.T + L.T_len;
    D.ep = D.G + L.G_len;
    D.wp = D.ep + L.e_len;
    D.erow = acc;
    D.Fat = acc + (size_t)L.nm1 * L.ma1;
    return D;
}

template <typename T>
int mv_pack_train(const MvLayout &L, const MvDev &D, const T *X2, const T *ad, const T *aE,
                  int ma2, hipStream_t stream) {
    if (L.t_rows == 0) return KF_OK;
    return for_groups((L.t_rows + 3) / 4, [&](size_t first, unsigned n) {
        hipLaunchKernelGGL(pack_rows_kernel<T>, dim3(n), dim3(NT), 0, stream, X2, ad, D.src2,
                           L.t_rows, first, ma2, L.rep, D.inv, L.nf, L.nfp, D.segs,
                           (int)L.segs.size(), aE, D.P2, D.n2, D.rdot, D.aE);
    });
}

int mv_zero_unmatched(const MvLayout &L, const MvDev &D, bool forces, hipStream_t stream) {
    if (L.src0.empty()) return KF_OK;
    return for_groups(L.src0.size(), [&](size_t first, unsigned n) {
        hipLaunchKernelGGL(zero_rows_kernel, dim3(n), dim3(64), 0, stream, D.src0 + first,
                           3 * L.ma1, L.parts, L.nm1 * L.ma1, D.erow,
                           forces ? D.Fat : (double *)nullptr);
    });
}

// The per-atom energies (mode bit 1) and back-projections (bit 2) of the layout's labels.
template <typename T>
int mv_run(const MvLayout &L, const MvDev &D, const T *X1, const T *dX1, double sigma, int mode,
           hipStream_t stream) {
    const double cexp = -1.0 / (2.0 * sigma * sigma), inv_s2 = 1.0 / (sigma * sigma);
    const int natoms = L.nm1 * L.ma1;
    const bool forces = mode & 2;
    for (const MvRound &R : L.rounds) {
        const MvSeg *segs = D.segs + R.seg0;
        const int rc = for_groups((R.rows + 3) / 4, [&](size_t first, unsigned n) {
            hipLaunchKernelGGL(pack_rows_kernel<T>, dim3(n), dim3(NT), 0, stream, X1,
                               (const T *)nullptr, D.src1 + R.row0, R.rows, first, L.ma1, L.rep,
                               D.inv, L.nf, L.nfp, segs, R.nseg, (const T *)nullptr, D.Xq, D.nq,
                               (double *)nullptr, (double *)nullptr);
        });
        if (rc) return rc;
        if (R.items1 > 0) {
            auto coef = [&](auto kern, int per) {
                hipLaunchKernelGGL(kern, dim3((R.items1 + per - 1) / per), dim3(NT), 0, stream,
                                   segs, R.nseg, R.items1, D.Xq, R.row0, R.rows, D.nq, D.P2, D.n2,
                                   D.rdot, D.aE, L.nfp, cexp, inv_s2,
                                   forces ? D.T : (double *)nullptr, D.ep, D.wp);
            };
            if (!R.wide) coef(coef_kernel<1, 1, 4>, 1);
            else if (R.split_k) coef(coef_kernel<2, 1, 4>, 1);
            else coef(coef_kernel<2, 2, 1>, 4);
            KF_HIP_TRY(hipGetLastError());
        }
        if (forces && R.items2 > 0) {
            hipLaunchKernelGGL(R.wide ? weighted_rows_kernel<2> : weighted_rows_kernel<1>,
                               dim3((R.items2 + 3) / 4), dim3(NT), 0, stream, segs, R.nseg,
                               R.items2, R.ks, D.T, D.P2, L.nfp, D.G);
            KF_HIP_TRY(hipGetLastError());
        }
        const size_t lds = sizeof(double) * ((L.rep + L.parts - 1) / L.parts + NT);
        hipLaunchKernelGGL(backproj_kernel<T>, dim3(R.rows, forces ? L.parts : 1), dim3(NT), lds,
                           stream, segs, R.nseg, R.row0, D.G, D.ep, D.wp, X1, dX1, D.src1, D.inv,
                           D.offs, L.ma1, L.rep, L.nfp, natoms,
                           (mode & 1) ? D.erow : (double *)nullptr,
                           forces ? D.Fat : (double *)nullptr);
        KF_HIP_TRY(hipGetLastError());
    }
    return KF_OK;
}

// E and F from the per-atom sums of mv_run
int mv_reduce(const MvLayout &L, const MvDev &D, double *E, double *F, int mode,
              hipStream_t stream) {
    return for_groups(L.nm1, [&](size_t first, unsigned n) {
        hipLaunchKernelGGL(reduce_mol_kernel, dim3(n), dim3(kReduceThreads), 0, stream, D.erow,
                           D.Fat, L.parts, D.offs, L.nm1 * L.ma1, L.ma1, first,
                           (mode & 1) ? E : (double *)nullptr,
                           (mode & 2) ? F : (double *)nullptr);
    });
}

// Labels and counts of both sets and the training side's used columns on the host, with one
// synchronisation.
template <typename T>
int mv_read(const int *Q1, const int *N1, int nm1, int ma1, const T *X2, const T *ad,
            const int *Q2, const int *N2, int nm2, int ma2, int rep, std::vector<int> &q1,
            std::vector<int> &n1, std::vector<int> &q2, std::vector<int> &n2,
            std::vector<int> &flag, hipStream_t stream) {
    flag.assign(rep, 0);
    int *dflag = nullptr, *hflag = nullptr;
    if (nm2 > 0 && ma2 > 0) {
        dflag = static_cast<int *>(workspace(WS_AUX1, sizeof(int) * rep, stream));
        hflag = static_cast<int *>(host_staging(WS_AUX3, sizeof(int) * rep));
        KF_REQUIRE(dflag && hflag, KF_ERR_NOMEM, "workspace allocation failed");
        KF_HIP_TRY(hipMemsetAsync(dflag, 0, sizeof(int) * rep, stream));
        const int per = std::max(1, (nm2 + 1023) / 1024);
        hipLaunchKernelGGL(train_cols_kernel<T>, dim3((nm2 + per - 1) / per), dim3(NT), 0, stream,
                           X2, ad, N2, nm2, ma2, rep, per, dflag);
        KF_HIP_TRY(hipGetLastError());
        KF_HIP_TRY(hipMemcpyAsync(hflag, dflag, sizeof(int) * rep, hipMemcpyDeviceToHost, stream));
    }
    int rc;
    if (nm2 > 0) {
        const size_t nq = (size_t)nm2 * ma2;
        int *stage = static_cast<int *>(host_staging(WS_AUX1, sizeof(int) * (nq + nm2)));
        KF_REQUIRE(stage, KF_ERR_NOMEM, "pinned staging allocation failed");
        if (nq)
            KF_HIP_TRY(hipMemcpyAsync(stage, Q2, sizeof(int) * nq, hipMemcpyDeviceToHost, stream));
        KF_HIP_TRY(hipMemcpyAsync(stage + nq, N2, sizeof(int) * nm2, hipMemcpyDeviceToHost, stream));
        if ((rc = read_metadata(Q1, N1, nm1, ma1, q1, n1, stream, WS_AUX0))) return rc;
        q2.assign(stage, stage + nq);
        n2.assign(stage + nq, stage + nq + nm2);
    } else if ((rc = read_metadata(Q1, N1, nm1, ma1, q1, n1, stream, WS_AUX0))) {
        return rc;
    }
    if (hflag) std::copy(hflag, hflag + rep, flag.begin());
    return KF_OK;
}

// modes: bit 1 E, bit 2 F, bit 4 alpha_E terms
template <typename T>
int matvec_impl(const T *X1, const T *dX1, const T *X2, const T *ad, const T *aE, const int *Q1,
                const int *Q2, const int *N1, const int *N2, int nm1, int nm2, int ma1, int ma2,
                int rep, double sigma, double *E, double *F, int mode, hipStream_t stream) {
    KF_REQUIRE(std::isfinite(sigma) && sigma > 0.0, KF_ERR_SIGMA, "sigma must be > 0");
    KF_REQUIRE(nm1 >= 0 && nm2 >= 0 && ma1 >= 0 && ma2 >= 0 && rep >= 1, KF_ERR_ARG,
               "bad dimensions");
    if (nm1 == 0) return KF_OK;
    KF_REQUIRE(X1 && Q1 && N1 && (nm2 == 0 || (X2 && ad && Q2 && N2)), KF_ERR_ARG,
               "null pointer");
    KF_REQUIRE(!(mode & 2) || dX1, KF_ERR_ARG, "null dX1");  // F may be null when naq1 == 0
    KF_REQUIRE(!(mode & 1) || E, KF_ERR_ARG, "null E");
    KF_REQUIRE(!(mode & 4) || nm2 == 0 || aE, KF_ERR_ARG, "null alpha_E");
    std::vector<int> q1, n1, q2, n2, flag;
    int rc;
    if ((rc = mv_read(Q1, N1, nm1, ma1, X2, ad, Q2, N2, nm2, ma2, rep, q1, n1, q2, n2, flag,
                      stream)))
        return rc;
    // All labels in one layout; where its scratch is refused, one label after another, each
    // with the scratch of its own rows alone (and one run of features).
    int nlabels = 1;
    for (int only = -1; only < nlabels; ++only) {
        MvLayout L;
        nlabels = mv_layout(q1, n1, nm1, ma1, q2, n2, nm2, ma2, rep, flag.data(), mode & 2, L,
                            only, only < 0 ? 0 : 1);
        if (only >= nlabels) break;  // no atoms at all
        if (only > 0) KF_HIP_TRY(hipStreamSynchronize(stream));  // the staging is still read
        char *meta = static_cast<char *>(workspace(WS_PLAN, L.meta_bytes(), stream));
        char *stage = static_cast<char *>(host_staging(WS_PLAN, L.meta_bytes()));
        const size_t qb = sizeof(double) * L.query_doubles();
        // (not in WS_PACK or WS_PACK2: the matrix-free solver keeps its operands there)
        const size_t tpad = (L.train_doubles() + 31) & ~size_t(31);
        double *train = static_cast<double *>(workspace(WS_AUX2, sizeof(double) * tpad + qb, stream));
        double *acc = static_cast<double *>(
            workspace(WS_AUX3, sizeof(double) * L.acc_doubles(mode & 2), stream));
        if (only < 0 && nlabels > 0 && !(meta && stage && train && acc)) continue;
        KF_REQUIRE(meta && stage && train && acc, KF_ERR_NOMEM,
                   "workspace allocation failed (%zu B)", sizeof(double) * tpad + qb);
        L.write_meta(stage);
        KF_HIP_TRY(hipMemcpyAsync(meta, stage, L.meta_bytes(), hipMemcpyHostToDevice, stream));
        const MvDev D = mv_place(L, meta, train, train + tpad, acc);
        ScopedTimer timer(TM_MATVEC, stream);
        if ((rc = mv_pack_train(L, D, X2, ad, (mode & 4) ? aE : (const T *)nullptr, ma2, stream)) ||
            (rc = mv_zero_unmatched(L, D, mode & 2, stream)) ||
            (rc = mv_run(L, D, X1, dX1, sigma, mode, stream)))
            return rc;
        if (only < 0 || only + 1 == nlabels) return mv_reduce(L, D, E, F, mode, stream);
    }
    return KF_OK;
}

}  // namespace
}  // namespace kf

// A full matvec planned once for fixed labels of the query set and a fixed training side
// (descriptors, alpha_desc, alpha_E): the layout, the packed training rows of every label
// with their norms and dot products, and the query workspace all live in device memory
// owned by the plan, so an execution neither reads anything back nor allocates.
struct kf_matvec_plan {
    int device = 0;
    double sigma = 1.0;
    kf::MvLayout layout;
    kf::MvDev dev{};
    char *meta = nullptr;
    double *train = nullptr, *query = nullptr, *acc = nullptr;
    ~kf_matvec_plan() {
        (void)hipFree(meta);
        (void)hipFree(train);
        (void)hipFree(query);
        (void)hipFree(acc);
    }
};

namespace kf {
namespace {

int plan_alloc(void **p, size_t bytes) {
    if (hipMalloc(p, bytes ? bytes : 256) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        set_last_error("hipMalloc of %zu bytes for a matvec plan failed", bytes);
        return KF_ERR_NOMEM;
    }
    return KF_OK;
}

int plan_create(const int *Q1, const int *N1, int nm1, int ma1, const double *X2,
                const double *ad, const double *aE, const int *Q2, const int *N2, int nm2,
                int ma2, int rep, double sigma, kf_matvec_plan *P, hipStream_t stream) {
    KF_REQUIRE(std::isfinite(sigma) && sigma > 0.0, KF_ERR_SIGMA, "sigma must be > 0");
    KF_REQUIRE(nm1 >= 1 && nm2 >= 0 && ma1 >= 1 && ma2 >= 0 && rep >= 1, KF_ERR_ARG,
               "bad dimensions");
    KF_REQUIRE(Q1 && N1 && (nm2 == 0 || (X2 && ad && aE && Q2 && N2)), KF_ERR_ARG,
               "null pointer");
    KF_HIP_TRY(hipGetDevice(&P->device));
    P->sigma = sigma;
    std::vector<int> q1, n1, q2, n2, flag;
    int rc;
    if ((rc = mv_read(Q1, N1, nm1, ma1, X2, ad, Q2, N2, nm2, ma2, rep, q1, n1, q2, n2, flag,
                      stream)))
        return rc;
    MvLayout &L = P->layout;
    mv_layout(q1, n1, nm1, ma1, q2, n2, nm2, ma2, rep, flag.data(), true, L);
    if ((rc = plan_alloc((void **)&P->meta, L.meta_bytes()))) return rc;
    if ((rc = plan_alloc((void **)&P->train, sizeof(double) * L.train_doubles()))) return rc;
    if ((rc = plan_alloc((void **)&P->query, sizeof(double) * L.query_doubles()))) return rc;
    if ((rc = plan_alloc((void **)&P->acc, sizeof(double) * L.acc_doubles(true)))) return rc;
    std::vector<char> meta(L.meta_bytes());
    L.write_meta(meta.data());
    KF_HIP_TRY(hipMemcpyAsync(P->meta, meta.data(), meta.size(), hipMemcpyHostToDevice, stream));
    P->dev = mv_place(L, P->meta, P->train, P->query, P->acc);
    if ((rc = mv_pack_train(L, P->dev, X2, ad, aE, ma2, stream))) return rc;
    // (executions do not write these rows)
    if ((rc = mv_zero_unmatched(L, P->dev, true, stream))) return rc;
    // the host vector above is released on return: wait for the copy that reads it
    KF_HIP_TRY(hipStreamSynchronize(stream));
    return KF_OK;
}

int plan_execute(const kf_matvec_plan *P, const double *X1, const double *dX1, double *E,
                 double *F, hipStream_t stream) {
    KF_REQUIRE(P && X1 && dX1 && E && F, KF_ERR_ARG, "null pointer");
    int dev = -1;
    KF_HIP_TRY(hipGetDevice(&dev));
    KF_REQUIRE(dev == P->device, KF_ERR_ARG, "plan was created on device %d, current is %d",
               P->device, dev);
    const int rc = mv_run(P->layout, P->dev, X1, dX1, P->sigma, 1 | 2, stream);
    return rc ? rc : mv_reduce(P->layout, P->dev, E, F, 1 | 2, stream);
}

}  // namespace
}  // namespace kf

using namespace kf;

extern "C" int kf_matvec_plan_create(const int *Q1, const int *N1, int nm1, int max_atoms1,
                                     const double *X2, const double *alpha_desc,
                                     const double *alpha_E, const int *Q2, const int *N2,
                                     int nm2, int max_atoms2, int rep, double sigma,
                                     kf_matvec_plan **plan, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    KF_REQUIRE(plan, KF_ERR_ARG, "null plan out-pointer");
    *plan = nullptr;
    auto *P = new (std::nothrow) kf_matvec_plan();
    KF_REQUIRE(P, KF_ERR_NOMEM, "plan allocation failed");
    const int rc = plan_create(Q1, N1, nm1, max_atoms1, X2, alpha_desc, alpha_E, Q2, N2, nm2,
                               max_atoms2, rep, sigma, P, as_stream(stream));
    if (rc) {
        delete P;
        return rc;
    }
    *plan = P;
    return KF_OK;
}

extern "C" int kf_matvec_plan_execute(const kf_matvec_plan *plan, const double *X1,
                                      const double *dX1, double *E, double *F, void *stream) {
    return plan_execute(plan, X1, dX1, E, F, as_stream(stream));
}

extern "C" int kf_matvec_plan_destroy(kf_matvec_plan *plan) {
    if (plan) {
        (void)hipDeviceSynchronize();  // no execution may still read the plan's memory
        delete plan;
    }
    return KF_OK;
}

extern "C" int kf_local_alpha_desc(const double *dX, const int *Q, const int *N, int nm,
                                   int max_atoms, int rep, const double *alpha, double *out,
                                   void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    (void)Q;
    KF_REQUIRE(nm >= 0 && max_atoms >= 0 && rep >= 1, KF_ERR_ARG, "bad dimensions");
    if (nm == 0 || max_atoms == 0) return KF_OK;
    KF_REQUIRE(dX && N && alpha && out, KF_ERR_ARG, "null pointer");
    hipStream_t st = as_stream(stream);
    std::vector<int> hN(nm);
    int *stage = static_cast<int *>(host_staging(WS_AUX0, sizeof(int) * (nm + 1)));
    KF_REQUIRE(stage, KF_ERR_NOMEM, "staging allocation failed");
    KF_HIP_TRY(hipMemcpyAsync(stage, N, sizeof(int) * nm, hipMemcpyDeviceToHost, st));
    KF_HIP_TRY(hipStreamSynchronize(st));
    std::vector<int> offs(nm + 1, 0);
    for (int a = 0; a < nm; ++a) offs[a + 1] = offs[a] + 3 * clamp_atoms(stage[a], max_atoms);
    int *d_offs = static_cast<int *>(workspace(WS_PLAN, sizeof(int) * (nm + 1), st));
    int *st2 = static_cast<int *>(host_staging(WS_PLAN, sizeof(int) * (nm + 1)));
    KF_REQUIRE(d_offs && st2, KF_ERR_NOMEM, "workspace allocation failed");
    std::copy(offs.begin(), offs.end(), st2);
    KF_HIP_TRY(hipMemcpyAsync(d_offs, st2, sizeof(int) * (nm + 1), hipMemcpyHostToDevice, st));
    const long atoms = (long)nm * max_atoms;
    hipLaunchKernelGGL(alpha_desc_kernel, dim3((unsigned)((atoms + 3) / 4)), dim3(NT), 0, st, dX,
                       N, d_offs, nm, max_atoms, rep, alpha, out);
    KF_HIP_TRY(hipGetLastError());
    return KF_OK;
}

extern "C" int kf_local_full_matvec(const double *X1, const double *dX1, const double *X2,
                                    const double *alpha_desc, const double *alpha_E,
                                    const int *Q1, const int *Q2, const int *N1, const int *N2,
                                    int nm1, int nm2, int max_atoms1, int max_atoms2, int rep,
                                    double sigma, double *E, double *F, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return matvec_impl(X1, dX1, X2, alpha_desc, alpha_E, Q1, Q2, N1, N2, nm1, nm2, max_atoms1,
                       max_atoms2, rep, sigma, E, F, 1 | 2 | 4, as_stream(stream));
}

// 100 float32 molecules of 21 atoms against 1,000, descriptors and Jacobians included: 1.7 ms
// (2.60 ms with FP64 copies of the operands made first; the Jacobians of the 100 molecules
// are 0.38 GB, written and read once, where they were 0.76 GB, copied and read).
extern "C" int kf_local_full_matvec_f32(const float *X1, const float *dX1, const float *X2,
                                        const float *alpha_desc, const float *alpha_E,
                                        const int *Q1, const int *Q2, const int *N1,
                                        const int *N2, int nm1, int nm2, int max_atoms1,
                                        int max_atoms2, int rep, double sigma, double *E,
                                        double *F, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return matvec_impl(X1, dX1, X2, alpha_desc, alpha_E, Q1, Q2, N1, N2, nm1, nm2, max_atoms1,
                       max_atoms2, rep, sigma, E, F, 1 | 2 | 4, as_stream(stream));
}

extern "C" int kf_local_hessian_matvec(const double *X1, const double *dX1, const double *X2,
                                       const double *alpha_desc, const int *Q1, const int *Q2,
                                       const int *N1, const int *N2, int nm1, int nm2,
                                       int max_atoms1, int max_atoms2, int rep, double sigma,
                                       double *F, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return matvec_impl<double>(X1, dX1, X2, alpha_desc, nullptr, Q1, Q2, N1, N2, nm1, nm2,
                               max_atoms1, max_atoms2, rep, sigma, nullptr, F, 2,
                               as_stream(stream));
}

extern "C" int kf_local_jacobian_t_matvec(const double *X1, const double *X2,
                                          const double *alpha_desc, const int *Q1,
                                          const int *Q2, const int *N1, const int *N2, int nm1,
                                          int nm2, int max_atoms1, int max_atoms2, int rep,
                                          double sigma, double *E, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return matvec_impl<double>(X1, nullptr, X2, alpha_desc, nullptr, Q1, Q2, N1, N2, nm1, nm2,
                               max_atoms1, max_atoms2, rep, sigma, E, nullptr, 1,
                               as_stream(stream));
}
