// local_direct.hip -- the scalar local kernels (local_scalar.hip) for small calls.
//
// The blocked kernel of local_scalar.hip packs and orders the molecules by the descriptor
// windows they use and gives each work-group a block of molecule pairs, whose labels and
// tiles it walks one after another.  For a few hundred thousand molecule pairs that leaves
// most of the GPU waiting on the longest chain, and the packing and ordering cost as much
// as the products.  This form has no packing: rows are read where they are, tile by tile of
// one label's Gram matrix.  While there are few tiles they are 32 x 32, and a work-group's
// four waves share a tile's descriptor columns, straight from global memory into registers
// (two 16-byte loads of a row at a time, with the summation index of a step permuted the same
// way in both operands, as in local_matvec.hip); beyond, they are 64 x 64 and both operands
// go through LDS.  A tile's rows pass through the registers whole in either, so their squared
// norms come from the same loads.  The exponentials go to memory (8 bytes per matched atom
// pair), and a second kernel sums those of each molecule pair in a fixed order.
// Measured for whole calls on molecules of 5-23 atoms, 720 columns: 50 molecules 77 us, 400
// 323 (719 of the blocked form with its smallest blocks, 2,657 with 64 x 64), 800 867 (1,108,
// 3,244); one molecule against 5,000 446 us (1,244 with 64 x 64).
#include <algorithm>
#include <cmath>

#include "local_direct.hpp"
#include "reg_pipeline.hpp"

namespace kf {
namespace {

constexpr int NT = 256;
constexpr int TE = 32;  // tile edge (rows of one label)
// Row tiles of a band: while the column tiles pass, its rows are read again and again, so the
// columns are fetched once per band instead of once per row tile.  Of 720 columns it is 2.9 MB
// in 32-row tiles, which stay in an XCD's 4 MB of L2, and 5.9 MB in 64-row ones, which do in part.
constexpr int BT = 16;
constexpr int kLdsTiles = 384;  // 64 x 64 tiles from which on they are taken (local_direct)
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

// One label: its packed rows of both sets and where its exponentials go: R1 rows of R2, or,
// in the symmetric forms, row tile after row tile from the diagonal tile on.
struct DirectSeg {
    int r1, R1, r2, R2;
    int it, pad;  // first tile
    size_t eoff;
};

// Exponentials of the row tiles before row c0, a multiple of te, of a symmetric label with R
// rows: a tile has te rows from its first column on.
__host__ __device__ inline size_t upper_rows(int c0, int te, int R) {
    return (size_t)c0 * R - ((size_t)c0 * (c0 - te) >> 1);
}

// Row i of a label's exponentials, indexed by column (symmetric: from its tile's first row on;
// te a power of 2).
template <bool SYMM>
__device__ inline double *exp_row(const DirectSeg &S, int te, int i, double *Ex) {
    if (!SYMM) return Ex + S.eoff + (size_t)i * S.R2;
    const int c0 = i & -te;
    return Ex + S.eoff + upper_rows(c0, te, S.R2) + (size_t)(i - c0) * (S.R2 - c0) - c0;
}

// Consecutive tiles (which share operands) on one XCD: work-groups are dealt round-robin
// over eight of them.
__device__ inline int xcd_tile() {
    const int g = blockIdx.x, G = gridDim.x;
    return (G % 8 == 0) ? (g % 8) * (G / 8) + g / 8 : g;
}

// Label of a tile: the last one whose first tile is not beyond it.
__device__ inline int seg_of(const DirectSeg *segs, int nseg, int tile) {
    int s = 0;
    for (int n = nseg; n > 1;) {
        const int h = n / 2;
        if (segs[s + h].it <= tile) s += h, n -= h;
        else n = h;
    }
    return s;
}

// Columns k + 2 g, + 1, + 8 and + 9 of a row for lane group g: two loads that together take
// 128 contiguous bytes of 16 rows, 64 at a time, or four where rows are not 16-byte aligned
// (VEC = false).
template <bool VEC>
__device__ inline void load4(const double *p, double (&v)[4]) {
    if (VEC) {
        const v2d a = *reinterpret_cast<const v2d *>(p), b = *reinterpret_cast<const v2d *>(p + 8);
        v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = p[u < 2 ? u : u + 6];
    }
}

// Row and column tile of tile `loc` of a label: bands of BT row tiles, each walked column
// tile by column tile.  False below the diagonal (first columns of a symmetric band).
template <bool SYMM>
__device__ inline bool tile_at(const DirectSeg &S, int te, int loc, int &rt, int &ct) {
    const int nrt = (S.R1 + te - 1) / te, nct = (S.R2 + te - 1) / te;
    int r0 = 0;
    for (;; r0 += BT) {
        const int n = min(BT, nrt - r0) * (SYMM ? nct - r0 : nct);
        if (loc < n) break;
        loc -= n;
    }
    const int h = min(BT, nrt - r0);
    rt = r0 + loc % h;
    ct = (SYMM ? r0 : 0) + loc / h;
    return !SYMM || ct >= rt;
}

// Exponentials of a 16 x 16 fragment: s its Gram entries, rows from row0 with squared norms
// in `nr` (lane r holds row r's), this lane's column with squared norm nc.
template <bool SYMM, int T>
__device__ inline void put_exps(const DirectSeg &S, const double (&s)[4], int row0, int col,
                                double nr, double nc, double cy, const double *etab, int lane,
                                double *Ex) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int rr = mfma16_row_f64(lane, v);
        const double e = exp_scaled(fma(s[v], -2.0 * cy, cy * __shfl(nr, rr, 64) + cy * nc), etab);
        if (row0 + rr < S.R1 && col < S.R2) exp_row<SYMM>(S, T, row0 + rr, Ex)[col] = e;
    }
}

// 32 x 32 tiles, one per work-group, its waves each taking every fourth 16 columns of the
// descriptors straight into registers: no barrier until the end, the shortest chain.
template <bool SYMM, bool VEC>
__global__ __launch_bounds__(NT, 3) void exp_tiles_kernel(const DirectSeg *__restrict__ segs,
                                                          int nseg, const double *__restrict__ X1,
                                                          const int *__restrict__ src1,
                                                          const double *__restrict__ X2,
                                                          const int *__restrict__ src2, int rep,
                                                          double cy, double *__restrict__ Ex) {
    constexpr int F = TE / 16, KW = 4;
    __shared__ double red[KW][F * F * 4][64];
    __shared__ double nrm[KW][2 * F * 16];
    __shared__ double etab[64];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    if (tid < 64) etab[tid] = kExp2Tab64[tid];
    const int tile = xcd_tile();
    const DirectSeg S = segs[seg_of(segs, nseg, tile)];
    int rt, ct;
    if (!tile_at<SYMM>(S, TE, tile - S.it, rt, ct)) return;
    const double *pa[F], *pb[F];
#pragma unroll
    for (int m = 0; m < F; ++m) {  // rows past the label's end repeat its last one
        pa[m] = X1 + (size_t)src1[S.r1 + min(rt * TE + 16 * m + r, S.R1 - 1)] * rep + 2 * g;
        pb[m] = X2 + (size_t)src2[S.r2 + min(ct * TE + 16 * m + r, S.R2 - 1)] * rep + 2 * g;
    }
    v4d c[F][F];
    double na[F], nb[F];
#pragma unroll
    for (int m = 0; m < F; ++m) {
        na[m] = nb[m] = 0.0;
#pragma unroll
        for (int n = 0; n < F; ++n) c[m][n] = (v4d){0.0, 0.0, 0.0, 0.0};
    }
    double a[2][F][4], b[2][F][4];
    auto load = [&](int buf, int k) {
#pragma unroll
        for (int m = 0; m < F; ++m) {
            load4<VEC>(pa[m] + k, a[buf][m]);
            load4<VEC>(pb[m] + k, b[buf][m]);
        }
    };
    auto mul = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int m = 0; m < F; ++m)
#pragma unroll
                for (int n = 0; n < F; ++n)
                    c[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[buf][m][u], b[buf][n][u],
                                                                   c[m][n], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < F; ++m) {
                na[m] = fma(a[buf][m][u], a[buf][m][u], na[m]);
                nb[m] = fma(b[buf][m][u], b[buf][m][u], nb[m]);
            }
        }
    };
    const int whole = rep & ~15, kb = 16 * wv;
    reg_pipeline((whole - kb + 16 * KW - 1) / (16 * KW),
                 [&](int buf, int i) { load(buf, kb + i * 16 * KW); }, mul);
    if (whole < rep && wv == KW - 1) {  // the last, partial 16 columns
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = whole + (u < 2 ? u : u + 6);
            const bool in = k + 2 * g < rep;
            const int at = in ? k : rep - 1 - 2 * g;
#pragma unroll
            for (int m = 0; m < F; ++m) {
                const double x = pa[m][at], y = pb[m][at];
                a[0][m][u] = in ? x : 0.0;
                b[0][m][u] = in ? y : 0.0;
            }
        }
        mul(0);
    }
#pragma unroll
    for (int m = 0; m < F; ++m) {
        na[m] += __shfl_xor(na[m], 16, 64);
        na[m] += __shfl_xor(na[m], 32, 64);
        nb[m] += __shfl_xor(nb[m], 16, 64);
        nb[m] += __shfl_xor(nb[m], 32, 64);
        if (g == 0) {
            nrm[wv][16 * m + r] = na[m];
            nrm[wv][16 * (F + m) + r] = nb[m];
        }
#pragma unroll
        for (int n = 0; n < F; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[wv][(m * F + n) * 4 + v][lane] = c[m][n][v];
    }
    __syncthreads();
    const int m = wv / F, n = wv % F;  // a fragment per wave
    double nr = 0.0, nc = 0.0, s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int w = 0; w < KW; ++w) {
        nr += nrm[w][16 * m + r];
        nc += nrm[w][16 * (F + n) + r];
#pragma unroll
        for (int v = 0; v < 4; ++v) s[v] += red[w][(m * F + n) * 4 + v][lane];
    }
    put_exps<SYMM, TE>(S, s, rt * TE + 16 * m, ct * TE + 16 * n + r, nr, nc, cy, etab, lane, Ex);
}

// 64 x 64 tiles, 16 columns of both operands at a time through LDS (double-buffered, one
// barrier a step), each wave a 32 x 32 quarter.  A row's 16 columns are four threads' loads
// of 64 contiguous bytes: with a lane per row instead (operands straight into registers)
// every lane is a cache access of its own, and the accesses, one a cycle, bound the kernel
// (92% of its cycles; 920 us at 800 molecules against 675 here).  LDS holds fragments in lane
// order, 16-byte units with the row XORed by 4 (column pair) so that neither the stores nor the
// reads conflict.
constexpr int TL = 64;
template <bool SYMM, bool VEC>
__global__ __launch_bounds__(NT, 4) void exp_tiles_lds_kernel(
    const DirectSeg *__restrict__ segs, int nseg, const double *__restrict__ X1,
    const int *__restrict__ src1, const double *__restrict__ X2, const int *__restrict__ src2,
    int rep, double cy, double *__restrict__ Ex) {
    // [buffer][operand][row group][8-column half][lane]
    __shared__ v2d sh[2][2][4][2][64];
    __shared__ double nrm[2][TL], etab[64];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    if (tid < 64) etab[tid] = kExp2Tab64[tid];
    const int tile = xcd_tile();
    const DirectSeg S = segs[seg_of(segs, nseg, tile)];
    int rt, ct;
    if (!tile_at<SYMM>(S, TL, tile - S.it, rt, ct)) return;
    const int row = tid >> 2, part = tid & 3;
    const double *pa = X1 + (size_t)src1[S.r1 + min(rt * TL + row, S.R1 - 1)] * rep + 2 * part;
    const double *pb = X2 + (size_t)src2[S.r2 + min(ct * TL + row, S.R2 - 1)] * rep + 2 * part;
    const int unit = 16 * part + ((row & 15) ^ (4 * part)), grp = row >> 4;
    const int rdu = 16 * g + (r ^ (4 * g)), wr = wv >> 1, wc = wv & 1;
    double a[4], b[4], na = 0.0, nb = 0.0;
    auto load = [&](int k) {
        load4<VEC>(pa + k, a);
        load4<VEC>(pb + k, b);
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            na = fma(a[u], a[u], na);
            nb = fma(b[u], b[u], nb);
        }
        sh[buf][0][grp][0][unit] = (v2d){a[0], a[1]};
        sh[buf][0][grp][1][unit] = (v2d){a[2], a[3]};
        sh[buf][1][grp][0][unit] = (v2d){b[0], b[1]};
        sh[buf][1][grp][1][unit] = (v2d){b[2], b[3]};
    };
    v4d c[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) c[m][n] = (v4d){0.0, 0.0, 0.0, 0.0};
    auto mul = [&](int buf) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v2d x[2], y[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                x[m] = sh[buf][0][2 * wr + m][h][rdu];
                y[m] = sh[buf][1][2 * wc + m][h][rdu];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int n = 0; n < 2; ++n)
                        c[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[m][u], y[n][u], c[m][n],
                                                                       0, 0, 0);
        }
    };
    const int whole = rep >> 4, steps = (rep + 15) >> 4;
    auto load_tail = [&]() {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = 16 * whole + (u < 2 ? u : u + 6);
            const bool in = k + 2 * part < rep;
            const int at = in ? k : rep - 1 - 2 * part;
            const double x = pa[at], y = pb[at];
            a[u] = in ? x : 0.0;
            b[u] = in ? y : 0.0;
        }
    };
    if (whole > 0) load(0);
    else load_tail();
    store(0);
    __syncthreads();
    for (int i = 0; i < steps; ++i) {
        const bool more = i + 1 < steps;  // uniform
        if (more) {
            if (i + 1 < whole) load(16 * (i + 1));
            else load_tail();
        }
        mul(i & 1);
        if (more) store((i + 1) & 1);
        __syncthreads();
    }
    na += __shfl_xor(na, 1, 64);
    na += __shfl_xor(na, 2, 64);
    nb += __shfl_xor(nb, 1, 64);
    nb += __shfl_xor(nb, 2, 64);
    if (part == 0) {
        nrm[0][row] = na;
        nrm[1][row] = nb;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int rl = 32 * wr + 16 * m, cl = 32 * wc + 16 * n;
            const double s[4] = {c[m][n][0], c[m][n][1], c[m][n][2], c[m][n][3]};
            put_exps<SYMM, TL>(S, s, rt * TL + rl, ct * TL + cl + r, nrm[0][rl + r],
                               nrm[1][cl + r], cy, etab, lane, Ex);
        }
}

// K[a, b] = sum over the labels and the label's rows of a and b of the exponentials (in
// tiles of te rows).  Eight lanes share a molecule pair, each taking every eighth row of a.
// The labels that a has are listed first: walking all of them for every pair, 500 labels on
// 2,000 molecules of 14 atoms took 5.7 ms, and 3,000 labels 40.
template <int MODE>
__global__ __launch_bounds__(NT) void pair_sums_kernel(const DirectSeg *__restrict__ segs,
                                                       double *__restrict__ Ex,
                                                       const int *__restrict__ mol1,
                                                       const int *__restrict__ mol2, int nseg,
                                                       int nm1, int nm2, int te, size_t first,
                                                       double *__restrict__ out) {
    constexpr bool SYMM = MODE != DIRECT_RECT;
    const int nbk = (nm2 + 31) / 32, sub = threadIdx.x & 7;
    const size_t blk = first + blockIdx.x;
    const int a = (int)(blk / nbk), b = (int)(blk % nbk) * 32 + (threadIdx.x >> 3);
    if (SYMM && (blk % nbk) * 32 + 31 < a) return;
    __shared__ int list[NT], rows[NT][2], have[NT / 64];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double s = 0.0;
    for (int l0 = 0; l0 < nseg; l0 += NT) {
        const int lt = l0 + threadIdx.x;
        int r0 = 0, r1 = 0;
        if (lt < nseg) {
            const int *ma = mol1 + (size_t)lt * (nm1 + 1) + a;
            r0 = ma[0] - segs[lt].r1, r1 = ma[1] - segs[lt].r1;
        }
        const unsigned long long hit = __ballot(r1 > r0);
        if (l0 > 0) __syncthreads();  // the last list is done with
        if (lane == 0) have[wv] = __popcll(hit);
        __syncthreads();
        int at = __popcll(hit & ((1ull << lane) - 1)), n = 0;
        for (int w = 0; w < NT / 64; ++w) {
            if (w < wv) at += have[w];
            n += have[w];
        }
        if (r1 > r0) list[at] = lt, rows[at][0] = r0, rows[at][1] = r1;
        __syncthreads();
        if (b >= nm2 || (SYMM && b < a)) continue;
        for (int u = 0; u < n; ++u) {
            const DirectSeg &S = segs[list[u]];
            const int *mb = mol2 + (size_t)list[u] * (nm2 + 1) + b;
            const int i0 = rows[u][0], i1 = rows[u][1], j0 = mb[0] - S.r2, j1 = mb[1] - S.r2;
            for (int i = i0 + sub; i < i1; i += 8) {
                if (SYMM && a == b) {  // only tiles of the upper triangle were formed
                    for (int j = j0; j < j1; ++j)
                        s += exp_row<SYMM>(S, te, min(i, j), Ex)[max(i, j)];
                } else {
                    const double *p = exp_row<SYMM>(S, te, i, Ex);
                    int j = j0;
                    for (; j + 4 <= j1; j += 4) s += (p[j] + p[j + 1]) + (p[j + 2] + p[j + 3]);
                    for (; j < j1; ++j) s += p[j];
                }
            }
        }
    }
    if (b >= nm2 || (SYMM && b < a)) return;
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 4, 64);
    if (sub) return;
    if (MODE == DIRECT_SYMM_RFP) {
        out[rfp_upper((size_t)nm1, a, b)] = s;
    } else {
        out[(size_t)a * nm2 + b] = s;
        if (SYMM) out[(size_t)b * nm2 + a] = s;
    }
}

}  // namespace

int local_direct(int mode, const LocalPlan &p1, const double *X1, const LocalPlan &p2,
                 const double *X2, int rep, double cy, double *out, int timer_id,
                 hipStream_t stream) {
    const bool symm = mode != DIRECT_RECT;
    const int L = p1.nlabels, nm1 = p1.nm, nm2 = p2.nm;
    std::vector<DirectSeg> segs(L);
    // 64 x 64 tiles once there are enough to fill the GPU and they are not mostly padding: one
    // costs about 2.8 of the 32 x 32 ones (800 molecules 675 us against 950; one molecule
    // against 10,000, whose 14 atoms fill neither, 257 against 185)
    auto count = [&](int te) {
        int n = 0;
        for (int l = 0; l < L; ++l) {
            const int *a = &p1.mol_row[(size_t)l * (nm1 + 1)], *b = &p2.mol_row[(size_t)l * (nm2 + 1)];
            const int t1 = ceil_div(a[nm1] - a[0], te), t2 = ceil_div(b[nm2] - b[0], te);
            segs[l].it = n;
            if (t1 > 0 && t2 > 0)
                for (int r0 = 0; r0 < t1; r0 += BT) n += std::min(BT, t1 - r0) * (symm ? t2 - r0 : t2);
        }
        return n;
    };
    int tiles = count(TL);
    const int small = count(TE);
    const bool lds = tiles >= kLdsTiles && 2.8 * tiles < small;
    tiles = lds ? count(TL) : small;
    const int te = lds ? TL : TE;
    size_t elen = 0;
    for (int l = 0; l < L; ++l) {
        const int *a = &p1.mol_row[(size_t)l * (nm1 + 1)], *b = &p2.mol_row[(size_t)l * (nm2 + 1)];
        const int R1 = a[nm1] - a[0], R2 = b[nm2] - b[0];
        segs[l] = {a[0], R1, b[0], R2, segs[l].it, 0, elen};
        elen += symm ? upper_rows(ceil_div(R1, te) * te, te, R1) : (size_t)R1 * R2;
    }
    // one upload: segments, then the rows' sources and the molecules' row ranges
    const size_t n1 = p1.src.size(), m1 = p1.mol_row.size();
    const size_t n2 = symm ? 0 : p2.src.size(), m2 = symm ? 0 : p2.mol_row.size();
    const size_t bytes = sizeof(DirectSeg) * L + sizeof(int) * (n1 + m1 + n2 + m2);
    double *Ex = static_cast<double *>(workspace(WS_PACK, sizeof(double) * elen, stream));
    char *dev = static_cast<char *>(workspace(WS_PLAN, bytes, stream));
    char *stage = static_cast<char *>(host_staging(WS_PLAN, bytes));
    KF_REQUIRE(dev && stage && Ex, KF_ERR_NOMEM, "workspace allocation failed (%zu B)",
               sizeof(double) * elen);
    std::copy(segs.begin(), segs.end(), reinterpret_cast<DirectSeg *>(stage));
    int *h = reinterpret_cast<int *>(stage + sizeof(DirectSeg) * L);
    h = std::copy(p1.src.begin(), p1.src.end(), h);
    h = std::copy(p1.mol_row.begin(), p1.mol_row.end(), h);
    if (!symm) {
        h = std::copy(p2.src.begin(), p2.src.end(), h);
        std::copy(p2.mol_row.begin(), p2.mol_row.end(), h);
    }
    KF_HIP_TRY(hipMemcpyAsync(dev, stage, bytes, hipMemcpyHostToDevice, stream));
    const DirectSeg *dseg = reinterpret_cast<const DirectSeg *>(dev);
    const int *src1 = reinterpret_cast<const int *>(dev + sizeof(DirectSeg) * L);
    const int *mol1 = src1 + n1, *src2 = symm ? src1 : mol1 + m1, *mol2 = symm ? mol1 : src2 + n2;
    ScopedTimer timer(timer_id, stream);
    const bool vec = rep % 2 == 0 && ((reinterpret_cast<size_t>(X1) | reinterpret_cast<size_t>(X2)) & 15) == 0;
    if (tiles > 0) {
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(tiles), dim3(NT), 0, stream, dseg, L, X1, src1, X2, src2,
                               rep, cy, Ex);
        };
        if (symm) {
            if (lds) vec ? launch(exp_tiles_lds_kernel<true, true>) : launch(exp_tiles_lds_kernel<true, false>);
            else vec ? launch(exp_tiles_kernel<true, true>) : launch(exp_tiles_kernel<true, false>);
        } else {
            if (lds) vec ? launch(exp_tiles_lds_kernel<false, true>) : launch(exp_tiles_lds_kernel<false, false>);
            else vec ? launch(exp_tiles_kernel<false, true>) : launch(exp_tiles_kernel<false, false>);
        }
        KF_HIP_TRY(hipGetLastError());
    }
    auto sums = [&](auto kern) {
        return for_groups((size_t)nm1 * ceil_div(nm2, 32), [&](size_t first, unsigned n) {
            hipLaunchKernelGGL(kern, dim3(n), dim3(NT), 0, stream, dseg, Ex, mol1, mol2, L, nm1,
                               nm2, te, first, out);
        });
    };
    if (mode == DIRECT_SYMM_RFP) return sums(pair_sums_kernel<DIRECT_SYMM_RFP>);
    if (mode == DIRECT_SYMM_DENSE) return sums(pair_sums_kernel<DIRECT_SYMM_DENSE>);
    return sums(pair_sums_kernel<DIRECT_RECT>);
}

}  // namespace kf
