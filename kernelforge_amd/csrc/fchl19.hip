// fchl19.hip -- FCHL19 atom-centred representation and its coordinate Jacobian
// on gfx950, FP64.
//
// Maths: reference src/fchl19_repr.cpp:89-299 (values) and :308-778 (values +
// Jacobian).  The Jacobian here is derived from the closed form (product rule
// over angular x radial x cutoff x Axilrod-Teller-Muto factors) rather than
// transcribed; it agrees with the reference to FP64 rounding.
//
// Work decomposition
//  * representation: a work-group per molecule, a batch of centres at a time.
//    Neighbour pairs are numbered by element-pair channel; threads evaluate one
//    (centre, pair) each into LDS, then own (channel, centre, radial term) and
//    sum the pairs in registers, so each rep entry has exactly one writer and a
//    fixed summation order.
//  * Jacobian: one or more workgroups per (molecule, centre).  Six scalars per
//    ordered neighbour pair in LDS; threads own (neighbour, radial term) and sum
//    over the partners in registers; an element-pair channel's rows are put
//    together in an LDS tile and leave as one contiguous run (dX rows are
//    contiguous per (centre, feature)).
#include <algorithm>
#include <cmath>

#include "kf_common.hpp"

namespace kf {
namespace {

constexpr int kMaxElem = 16;
constexpr int kMaxRs = 64;
constexpr int kMaxHarm = 8;
constexpr int kMaxAtoms = 128;
constexpr double kEps = 1e-12;
constexpr double kSqrt2Pi = 2.5066282746310005;

struct FchlParams {
    int nelem, nb2, nb3, na, nharm, nchan, rs, three_off, max_atoms;
    int elements[kMaxElem];
    double Rs2[kMaxRs], logRs2[kMaxRs], Rs3[kMaxRs];
    double angw[kMaxHarm];
    double eta2, eta3, rcut, acut, d2, d3, w3;
};

__device__ inline int elem_index(const FchlParams &P, int z) {
    for (int e = 0; e < P.nelem; ++e)
        if (P.elements[e] == z) return e;
    return -1;
}

__device__ inline int pair_channel(int nelem, int p, int q) {
    if (p > q) { int t = p; p = q; q = t; }
    return p * nelem - p * (p - 1) / 2 + (q - p);
}

// The x-th pair j < k of n, counted j by j.
__device__ inline void triangle_at(int n, int x, int &j, int &k) {
    j = (int)((2 * n - 1 - sqrtf((float)((2 * n - 1) * (2 * n - 1) - 8 * x))) * 0.5f);
    while (j > 0 && x < j * (2 * n - j - 1) / 2) --j;
    while (x >= (j + 1) * (2 * n - j - 2) / 2) ++j;
    k = j + 1 + x - j * (2 * n - j - 1) / 2;
}

__device__ inline double cut_fn(double r, double cut) {
    const double inv = cut > 0.0 ? 1.0 / cut : 0.0;
    return 0.5 * (cospi(r * inv) + 1.0);
}
__device__ inline double cut_dfn(double r, double cut) {
    const double inv = cut > 0.0 ? 1.0 / cut : 0.0;
    return -0.5 * M_PI * inv * sinpi(r * inv);
}

__device__ inline double dist(const double *R, int i, int j) {
    const double dx = R[3 * j] - R[3 * i], dy = R[3 * j + 1] - R[3 * i + 1],
                 dz = R[3 * j + 2] - R[3 * i + 2];
    return sqrt(dx * dx + dy * dy + dz * dz);
}

// Two-body pair quantities.  value_k = f * pref0 * exp(-L^2 / 2 s2) / Rs2_k with
// L = ln Rs2_k - mu; d value_k / dr = pref0 exp(..)/Rs2_k * (f * dlog0_k + df),
// dlog0_k = -d2/r - s'/s + L mu'/s2 + L^2 s'/s^3.  Returns false when the
// log-normal width vanishes.
struct TwoBody {
    double s2, s, mu, pref0, f, df, ds, dmu;
};
__device__ inline bool two_body(const FchlParams &P, double r, TwoBody &t, bool want_grad) {
    const double r2 = r * r;
    t.s2 = log1p(P.eta2 / (r2 > kEps ? r2 : kEps));
    t.s = sqrt(t.s2 > 0.0 ? t.s2 : 0.0);
    if (t.s < kEps) return false;
    t.mu = log(r) - 0.5 * t.s2;
    t.f = cut_fn(r, P.rcut);
    t.pref0 = 1.0 / (t.s * kSqrt2Pi * pow(r, P.d2));
    if (want_grad) {
        const double ds2 = -2.0 * P.eta2 / (r * (r2 + P.eta2));
        t.ds = ds2 / (2.0 * t.s);
        t.dmu = 1.0 / r - 0.5 * ds2;
        t.df = cut_dfn(r, P.rcut);
    }
    return true;
}

// ---------------------------------------------------------------------------
// Representation kernel: one work-group per molecule (several when the batch is small, each
// with a run of its rows), a batch of centres at a time.
//
// Atoms are sorted by element once.  Leaving out the centre then leaves every element's
// neighbours an index range, and the neighbour pairs of an element-pair channel too (a
// np x nq grid, or a triangle); which ranges depends only on the centre's element.  Per
// batch -- as many centres as have `pairs` neighbour pairs between them (13 of a 14-atom
// molecule) -- the threads evaluate one (centre, neighbour) each (unit vector, cutoff,
// two-body scalars), then one (centre, pair) each (rbar and the amplitude of every angular
// term), and then own one channel, centre and two radial terms each and sum its pairs in
// registers.  The lanes of a wave are of one channel and consecutive centres, whose pair
// counts differ by little, so they run the same number of steps.  Every output has one
// writing lane and a fixed summation order.  Bound by the FP64 VALU: the exponentials (one
// per pair and radial term) and the pair geometry.  20,000 molecules of 5-23 atoms take
// 2.30 ms (5.40 with a read-modify-write of an LDS accumulator per record and slot, 3.33 with
// a wave per centre, 2.65 with one radial term per thread); without the exponential sums 1.5,
// without the pair geometry 1.7, without both 1.0, of which the stores 0.4.
//
// LONG: molecules whose batches are of so few items (10 for one element and a centre at a time)
// that most of a work-group would be idle, or whose centres have more pairs than fit at once.
// Several lanes share an item and add up what they have at its end, and a chunk's pairs are
// found from their places instead of going through all pairs again.  1,000 molecules of one
// element: 60 atoms 4.8 ms (24.5 without, 12.0 with an accumulator in LDS), 128 atoms 51 (380,
// 104); of five elements 5.0 and 69 ms.
// ---------------------------------------------------------------------------
constexpr int kRepThreads = 256;
constexpr int kLB = 2;  // radial terms per thread
constexpr int kNbrFields = 8;  // unit vector, distance, cutoff, three two-body scalars

// LDS, in doubles: exp table | coordinates | neighbours (kNbrFields x nbrs) | pairs
// ((1 + na) x pairs) | ints: element, atoms by element, place of an atom in that order,
// first atom of an element, elements of a channel, first pair of a channel by the centre's
// element
struct RepLds {
    int R, nbr, pair, ints, nbrs, pairs, total_ints;
};
__host__ __device__ inline RepLds rep_lds(int ma, int nelem, int nchan, int na) {
    RepLds g;
    g.nbrs = ma > 192 ? ma : 192;
    g.pairs = 3072 / (1 + na) < 64 ? 64 : 3072 / (1 + na);
    g.R = 64;
    g.nbr = g.R + 3 * ma + (ma & 1);
    g.pair = g.nbr + kNbrFields * g.nbrs;
    g.ints = g.pair + (1 + na) * g.pairs;
    g.total_ints = 3 * ma + nelem + 1 + nchan + nelem * (nchan + 1);
    return g;
}
__host__ inline size_t rep_lds_bytes(int ma, int nelem, int nchan, int na) {
    const RepLds g = rep_lds(ma, nelem, nchan, na);
    return sizeof(double) * (size_t)g.ints + sizeof(int) * (size_t)g.total_ints;
}

// Centres of an n-atom molecule taken at a time.
__host__ __device__ inline int rep_batch(const RepLds &g, int n) {
    const int npair = (n - 1) * (n - 2) / 2;
    const int by_nbr = g.nbrs / n, by_pair = npair > 0 ? g.pairs / npair : n;
    const int b = by_nbr < by_pair ? by_nbr : by_pair;
    return b > 1 ? b : 1;
}
// Lanes that share one of a batch's (channel, centre, radial terms) items, as a power of 2: at
// most 64, up to four lanes of work per thread, and 32 and more of the centre's pairs each.
__host__ __device__ inline int rep_share_log(int items, int npair) {
    int lg = 0;
    while (lg < 6 && (2 << lg) * items <= 4 * kRepThreads && 64 << lg <= npair) ++lg;
    return lg;
}

template <typename O, bool LONG>
__global__ __launch_bounds__(kRepThreads, 4) void fchl19_rep_kernel(
    const double *__restrict__ coords, const int *__restrict__ Q, const int *__restrict__ N,
    FchlParams P, O *__restrict__ X, int *__restrict__ err) {
    extern __shared__ __align__(16) double smem[];
    __shared__ int next;
    const int m = blockIdx.x, tid = threadIdx.x;
    const int ma = P.max_atoms, nelem = P.nelem, nchan = P.nchan;
    int n = N[m];
    n = n < 0 ? 0 : (n > ma ? ma : n);
    const RepLds g = rep_lds(ma, nelem, nchan, P.na);
    double *tab = smem, *R = smem + g.R, *nbr = smem + g.nbr, *rbar = smem + g.pair,
           *amp = rbar + g.pairs;
    const double *ex = nbr, *ey = ex + g.nbrs, *ez = ey + g.nbrs, *rr = ez + g.nbrs,
                 *fc = rr + g.nbrs, *t_mu = fc + g.nbrs, *t_sc = t_mu + g.nbrs,
                 *t_f = t_sc + g.nbrs;
    int *el = reinterpret_cast<int *>(smem + g.ints), *ord = el + ma, *place = ord + ma,
        *est = place + ma, *chan = est + nelem + 1, *cst = chan + nchan;

    const double *Cm = coords + (size_t)m * ma * 3;
    bool bad = false;
    for (int t = tid; t < 3 * n; t += kRepThreads) R[t] = Cm[t];
    for (int t = tid; t < n; t += kRepThreads) {
        el[t] = elem_index(P, Q[(size_t)m * ma + t]);
        bad |= el[t] < 0;
    }
    if (tid < 64) tab[tid] = kExp2Tab64[tid];
    for (int c = tid; c < nchan; c += kRepThreads) {
        int p = 0, q = c;
        while (q >= nelem - p) q -= nelem - p, ++p;
        chan[c] = p << 16 | (p + q);
    }
    O *Xm = X + (size_t)m * ma * P.rs;
    // a molecule with an unknown element is reported through *err; its rows are zeroed
    if (__syncthreads_or(bad)) {
        if (tid == 0) *err = 1;
        n = 0;
    }
    const int per = (ma + gridDim.y - 1) / gridDim.y, row0 = blockIdx.y * per,
              row1 = min(row0 + per, ma), cen1 = min(row1, n);
    const int pad0 = max(row0, n);  // padding rows
    if (pad0 < row1) {
        O *d = Xm + (size_t)pad0 * P.rs;
        const int cnt = (row1 - pad0) * P.rs;
        for (int t = tid; t < cnt; t += kRepThreads) d[t] = O(0);
    }
    if (row0 >= cen1) return;
    for (int t = tid; t < n; t += kRepThreads) {
        int rank = 0;
        for (int s = 0; s < n; ++s) rank += (int)((el[s] < el[t]) | ((el[s] == el[t]) & (s < t)));
        ord[rank] = t;
        place[t] = rank;
    }
    for (int e = tid; e <= nelem; e += kRepThreads) {
        int c = 0;
        for (int s = 0; s < n; ++s) c += (int)(el[s] < e);
        est[e] = c;
    }
    __syncthreads();
    for (int t = tid; t < nelem * (nchan + 1); t += kRepThreads) {
        const int e = t / (nchan + 1), c1 = t - e * (nchan + 1);
        int off = 0;
        for (int c = 0; c < c1; ++c) {
            const int p = chan[c] >> 16, q = chan[c] & 0xffff;
            const int np = est[p + 1] - est[p] - (p == e), nq = est[q + 1] - est[q] - (q == e);
            off += p == q ? np * (np - 1) / 2 : np * nq;
        }
        cst[t] = off;
    }
    __syncthreads();

    const int npair = (n - 1) * (n - 2) / 2;
    const int batch = rep_batch(g, n);
    const int nlb = (P.nb3 + kLB - 1) / kLB;
    const int lg = LONG ? rep_share_log(nchan * nlb * batch, npair) : 0, share = 1 << lg;
    const double ysc = -P.eta3 * kExpScale;
    for (int i0 = row0; i0 < cen1; i0 += batch) {
        const int B = min(batch, cen1 - i0);
        __syncthreads();  // the previous batch's reads are done
        // ---- (centre, neighbour) ----
        for (int t = tid; t < B * n; t += kRepThreads) {
            const int b = t / n, j = t - b * n, i = i0 + b;
            double *f = nbr + t;
            const double r = dist(R, i, j), ir = 1.0 / (r > kEps ? r : kEps);
            for (int c = 0; c < 3; ++c) f[c * g.nbrs] = (R[3 * j + c] - R[3 * i + c]) * ir;
            f[3 * g.nbrs] = r;
            f[4 * g.nbrs] = cut_fn(r, P.acut);
            TwoBody tb;
            double mu = 0.0, sc = 0.0, fac = 0.0;
            if (j != i && !(r > P.rcut) && two_body(P, r, tb, false)) {
                mu = tb.mu;
                sc = -0.5 * kExpScale / tb.s2;
                fac = tb.f * tb.pref0;
            }
            f[5 * g.nbrs] = mu;
            f[6 * g.nbrs] = sc;
            f[7 * g.nbrs] = fac;
        }
        __syncthreads();
        // ---- two-body: (element, centre, k) ----
        for (int t = tid; t < nelem * B * P.nb2; t += kRepThreads) {
            const int eb = t / P.nb2, k = t - eb * P.nb2, e = eb / B, b = eb - e * B, i = i0 + b;
            double v = 0.0;
            for (int s = est[e]; s < est[e + 1]; ++s) {
                const int x = b * n + ord[s];
                if (t_f[x] != 0.0) {
                    const double L = P.logRs2[k] - t_mu[x];
                    v += t_f[x] * exp_scaled(L * L * t_sc[x], tab);
                }
            }
            Xm[(size_t)i * P.rs + e * P.nb2 + k] = O(v / P.Rs2[k]);
        }
        // ---- three-body, in one chunk unless a single centre has more than g.pairs ----
        for (int q0 = 0; q0 == 0 || q0 < npair; q0 += g.pairs) {
            const int qn = B > 1 ? npair : min(g.pairs, npair - q0);  // pairs of a centre here
            if (q0 > 0) __syncthreads();
            if (tid == 0) next = 0;
            // the neighbours' pairs (ja < ka in the order by element) as a triangle; a pair's
            // place is its channel's first one plus its index in the channel
            const float inv_np = 1.0f / (float)max(npair, 1);
            const int n1 = n - 1;
            const bool chunked = LONG && npair > g.pairs;
            for (int t = tid; t < (chunked ? qn : B * npair); t += kRepThreads) {
                const int b = chunked ? 0 : (int)(((float)t + 0.5f) * inv_np), i = i0 + b;
                const int pi = place[i], ei = el[i];
                int at, ja, ka;
                if (chunked) {  // the other way: from the place, channel by channel
                    const int *cs = cst + ei * (nchan + 1), x = q0 + t;
                    int c = 0;
                    for (int h = nchan; h - c > 1;) {
                        const int mid = (c + h) >> 1;
                        if (cs[mid] <= x) c = mid;
                        else h = mid;
                    }
                    const int p = chan[c] >> 16, q = chan[c] & 0xffff, y = x - cs[c];
                    const int np = est[p + 1] - est[p] - (p == ei), nq = est[q + 1] - est[q] - (q == ei);
                    int jl, kl;
                    if (p == q) triangle_at(np, y, jl, kl);
                    else jl = y / nq, kl = y - jl * nq;
                    at = t;
                    ja = est[p] + jl - (p > ei);
                    ka = est[q] + kl - (q > ei);
                } else {
                    triangle_at(n1, t - b * npair, ja, ka);
                }
                const int j = ord[ja + (ja >= pi)], k = ord[ka + (ka >= pi)];
                if (!chunked) {
                    const int p = el[j], q = el[k];
                    const int jl = ja - est[p] + (p > ei), kl = ka - est[q] + (q > ei);
                    const int np = est[p + 1] - est[p] - (p == ei), nq = est[q + 1] - est[q] - (q == ei);
                    at = cst[ei * (nchan + 1) + pair_channel(nelem, p, q)] +
                         (p == q ? jl * (2 * np - jl - 1) / 2 + kl - jl - 1 : jl * nq + kl);
                }
                const int xj = b * n + j, xk = b * n + k;
                const double rij = rr[xj], rik = rr[xk];
                double fa = 0.0, ci = 0.0, rb = 0.0;
                if (!(rij > P.acut) && !(rik > P.acut)) {
                    const double rjk = dist(R, j, k), ijk = 1.0 / (rjk > kEps ? rjk : kEps);
                    const double wx = (R[3 * k] - R[3 * j]) * ijk,
                                 wy = (R[3 * k + 1] - R[3 * j + 1]) * ijk,
                                 wz = (R[3 * k + 2] - R[3 * j + 2]) * ijk;
                    ci = ex[xj] * ex[xk] + ey[xj] * ey[xk] + ez[xj] * ez[xk];
                    ci = ci > 1.0 ? 1.0 : (ci < -1.0 ? -1.0 : ci);
                    const double cj = -(ex[xj] * wx + ey[xj] * wy + ez[xj] * wz);
                    const double ck = ex[xk] * wx + ey[xk] * wy + ez[xk] * wz;
                    const double prod = rik * rij * rjk;
                    fa = fc[xj] * fc[xk] * (1.0 + 3.0 * ci * cj * ck) * P.w3 /
                         pow(prod > kEps ? prod : kEps, P.d3);
                    rb = 0.5 * (rij + rik);
                }
                const int rec = b * qn + at;
                rbar[rec] = rb;
                const double si = sqrt(fmax(0.0, 1.0 - ci * ci));
                double cp = 1.0, sp = 0.0, cc = ci, sc = si;
                int o = 1;
                for (int h = 0; 2 * h < P.na; ++h) {
                    while (h < P.nharm && o < 2 * h + 1) {
                        const double cn = 2.0 * ci * cc - cp, sn = 2.0 * ci * sc - sp;
                        cp = cc; sp = sc; cc = cn; sc = sn; ++o;
                    }
                    const double w = h < P.nharm ? P.angw[h] * fa : 0.0;
                    amp[(2 * h) * g.pairs + rec] = w * cc;
                    amp[(2 * h + 1) * g.pairs + rec] = w * sc;
                }
            }
            __syncthreads();
            // (channel, centre, kLB radial terms), `share` lanes each
            for (;;) {
                // the waves draw 64 items at a time: channels differ in length
                int t0 = 0;
                if ((tid & 63) == 0) t0 = atomicAdd(&next, 64);
                const int t = __shfl(t0, 0, 64) + (tid & 63);
                if (t - (tid & 63) >= nchan * B * nlb << lg) break;
                if (t >= nchan * B * nlb << lg) continue;
                const int it = t >> lg, part = t & (share - 1);
                const int cb = it / nlb, l0 = (it - cb * nlb) * kLB, c = cb / B, b = cb - c * B,
                          i = i0 + b;
                const int *cs = cst + el[i] * (nchan + 1);
                const int lo = max(cs[c], q0) - q0, hi = min(cs[c + 1], q0 + qn) - q0;
                const bool first = q0 == 0 || q0 <= cs[c];  // nothing of it before this chunk
                if (hi <= lo && q0 > 0) continue;
                O *dst = Xm + (size_t)i * P.rs + P.three_off + (c * P.nb3 + l0) * P.na;
                const int ln = min(kLB, P.nb3 - l0);
                double rs3[kLB];
#pragma unroll
                for (int u = 0; u < kLB; ++u) rs3[u] = P.Rs3[min(l0 + u, P.nb3 - 1)];
                for (int ta = 0; ta < P.na; ta += 2) {
                    double v0[kLB], v1[kLB];
#pragma unroll
                    for (int u = 0; u < kLB; ++u) v0[u] = v1[u] = 0.0;
                    const double *a0 = amp + ta * g.pairs, *a1 = a0 + g.pairs;
                    for (int x = b * qn + lo + part; x < b * qn + hi; x += share) {
                        const double rb = rbar[x], c0 = a0[x], c1 = a1[x];
#pragma unroll
                        for (int u = 0; u < kLB; ++u) {
                            const double dr = rb - rs3[u];
                            const double e = exp_scaled(ysc * (dr * dr), tab);
                            v0[u] = fma(e, c0, v0[u]);
                            v1[u] = fma(e, c1, v1[u]);
                        }
                    }
                    for (int o = 1; o < share; o <<= 1) {
#pragma unroll
                        for (int u = 0; u < kLB; ++u) {
                            v0[u] += __shfl_xor(v0[u], o, 64);
                            v1[u] += __shfl_xor(v1[u], o, 64);
                        }
                    }
                    if (part) continue;
#pragma unroll
                    for (int u = 0; u < kLB; ++u) {
                        if (u >= ln) break;
                        O *d = dst + u * P.na + ta;
                        d[0] = O(first ? v0[u] : d[0] + v0[u]);
                        d[1] = O(first ? v1[u] : d[1] + v1[u]);
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Representation + Jacobian kernel: work-groups (centre, split) x molecule.
//
// The output is the work: 363 KB of Jacobian rows per centre of a 21-atom molecule, so the
// kernel is built to keep the stores going.  Everything a triplet contributes to the column
// of neighbour j is  rad_l * (alpha u_j + beta u_k) + rad_l dr_l c u_j  with u = R - R_i and
// six scalars per ordered pair (j, k) (alpha, beta and the value factor c of the cosine and
// the sine term), which fit in LDS for the whole molecule (48 n^2 bytes).  A thread owns
// (neighbour j, radial l) of one element-pair channel and sums over the partners k in
// registers, both angular terms and all three coordinates from one exponential; the
// centre's own column is minus the sum of the others (the descriptor does not change when
// the molecule moves).  The channel's rows are put together in an LDS tile and leave as one
// contiguous run; channels of elements the molecule does not hold are zero runs without
// any of that.  Two-body features use the same tile.  `splits` work-groups share a centre
// (each takes every splits-th feature block) when the batch has too few centres to fill the
// GPU.  Bound by the HBM stores: 500 molecules of 21
// atoms (3.8 GB) take 0.92 ms = 4.2 TB/s, against 0.57 ms for filling as much memory and
// 7.35 ms for the form with one triplet list per channel and read-modify-writes of the tile.
// (Non-temporal stores are no faster here and cost a following reader the cached rows: the
// back-projection of one molecule's matvec 1.8 ms instead of 1.1.)
// ---------------------------------------------------------------------------
constexpr int kGradThreads = 256;  // NTG: 64 for small molecules (fchl19_impl)
constexpr int kTwoW = 8;  // two-body scalars per neighbour

// LDS of one work-group, in doubles from the start (ints at the end).
struct GradLds {
    int tab, R, u4, f, df, two, rec, tile, vals, ints;
    int tile_rows, total_ints;
};
__host__ __device__ inline GradLds grad_lds(int ma, int nb2, int nb3, int na) {
    GradLds g;
    // rows of the tile: whole groups of angular terms, at least one group, at most what the
    // feature blocks need
    const int step = na > 0 ? na : 1;
    const int cap = step * (40 / step > 0 ? 40 / step : 1);
    const int need = nb2 > nb3 * na ? nb2 : nb3 * na;
    g.tile_rows = need < cap ? (need > step ? need : step) : cap;
    g.tab = 0;
    g.R = g.tab + 64;
    g.u4 = g.R + 4 * ((3 * ma + 3) / 4);
    g.f = g.u4 + 4 * ma;
    g.df = g.f + ma;
    g.two = g.df + ma;
    g.rec = g.two + kTwoW * ma;
    g.tile = g.rec + 6 * ma * ma;
    g.vals = g.tile + g.tile_rows * 3 * ma + (g.tile_rows * 3 * ma & 1);
    g.ints = g.vals + g.tile_rows * ma;
    g.total_ints = 2 * ma + kMaxElem + 2;
    return g;
}
__host__ inline size_t grad_lds_bytes(int ma, int nb2, int nb3, int na) {
    const GradLds g = grad_lds(ma, nb2, nb3, na);
    return sizeof(double) * (size_t)g.ints + sizeof(int) * (size_t)g.total_ints;
}

// n doubles of `src` (LDS; zeros when null) to dst, 16 bytes a lane where dst allows it.
template <int NTG, typename O>
__device__ inline void stream_out(O *dst, const double *src, int n) {
    constexpr int V = 16 / sizeof(O);
    typedef O vec __attribute__((ext_vector_type(V)));
    if (((reinterpret_cast<size_t>(dst) & 15) | (n % V)) == 0) {
        for (int t = threadIdx.x; t < n / V; t += NTG) {
            vec v;
#pragma unroll
            for (int u = 0; u < V; ++u) v[u] = src ? O(src[t * V + u]) : O(0);
            reinterpret_cast<vec *>(dst)[t] = v;
        }
    } else {
        for (int t = threadIdx.x; t < n; t += NTG) dst[t] = src ? O(src[t]) : O(0);
    }
}

template <typename O, int NTG>
__global__ __launch_bounds__(NTG) void fchl19_grad_kernel(
    const double *__restrict__ coords, const int *__restrict__ Q, const int *__restrict__ N,
    FchlParams P, int splits, O *__restrict__ X, O *__restrict__ dX,
    int *__restrict__ err) {
    extern __shared__ __align__(16) double smem[];
    const int m = blockIdx.y, i = blockIdx.x / splits, split = blockIdx.x % splits;
    const int tid = threadIdx.x;
    const int ma = P.max_atoms;
    const int ld = 3 * ma;
    int n = N[m];
    n = n < 0 ? 0 : (n > ma ? ma : n);
    O *Xi = X + ((size_t)m * ma + i) * P.rs;
    O *dXi = dX + ((size_t)m * ma + i) * P.rs * ld;
    const GradLds g = grad_lds(ma, P.nb2, P.nb3, P.na);
    double *tab = smem + g.tab, *R = smem + g.R, *u4 = smem + g.u4, *fc = smem + g.f,
           *dfc = smem + g.df, *two = smem + g.two, *rec = smem + g.rec, *tile = smem + g.tile,
           *vals = smem + g.vals;
    int *el = reinterpret_cast<int *>(smem + g.ints);  // element of an atom
    int *ord = el + ma;                                // neighbours sorted by element
    int *est = ord + ma;                               // first neighbour of an element

    // feature blocks (units): two-body elements in runs of tile_rows, then the radial terms
    // of each channel in runs of tile_rows / na
    const int nu2 = (P.nb2 + g.tile_rows - 1) / g.tile_rows;
    const int lrun = P.na > 0 ? g.tile_rows / P.na : 1;
    const int nu3 = P.na > 0 ? (P.nb3 + lrun - 1) / lrun : 0;
    const int nunits = P.nelem * nu2 + P.nchan * nu3;
    auto unit_rows = [&](int unit, int &f0, int &nr) {
        if (unit < P.nelem * nu2) {
            const int e = unit / nu2, k0 = (unit % nu2) * g.tile_rows;
            f0 = e * P.nb2 + k0;
            nr = min(g.tile_rows, P.nb2 - k0);
        } else {
            const int c = (unit - P.nelem * nu2) / nu3, l0 = ((unit - P.nelem * nu2) % nu3) * lrun;
            f0 = P.three_off + (c * P.nb3 + l0) * P.na;
            nr = min(lrun, P.nb3 - l0) * P.na;
        }
    };
    auto zero_rows = [&](int f0, int nr) {
        for (int t = tid; t < nr; t += NTG) Xi[f0 + t] = O(0);
        stream_out<NTG, O>(dXi + (size_t)f0 * ld, nullptr, nr * ld);
    };

    bool bad = false;
    if (i < n) {
        const double *Cm = coords + (size_t)m * ma * 3;
        for (int t = tid; t < 3 * n; t += NTG) R[t] = Cm[t];
        for (int t = tid; t < n; t += NTG) {
            const int e = elem_index(P, Q[(size_t)m * ma + t]);
            el[t] = e;
            bad |= e < 0;
        }
        for (int t = tid; t < 64; t += NTG) tab[t] = kExp2Tab64[t];
        for (int t = tid; t < g.tile_rows * ld; t += NTG) tile[t] = 0.0;
    }
    // a molecule with an unknown element is reported through *err; its rows are zeroed
    if (__syncthreads_or(bad)) {
        if (tid == 0) *err = 1;
        bad = true;
    }
    if (i >= n || bad || n == 1) {  // padding centre or nothing near it: zero rows
        const int f0 = (int)((long)P.rs * split / splits), f1 = (int)((long)P.rs * (split + 1) / splits);
        zero_rows(f0, f1 - f0);
        return;
    }

    // ---------------- per neighbour ----------------
    for (int j = tid; j < n; j += NTG) {
        const double r = dist(R, i, j);
        // (an atom at infinity adds nothing: its vector must not make NaN of a zero factor)
        const bool far = r > 1e150;
        for (int c = 0; c < 3; ++c) u4[4 * j + c] = far ? 0.0 : R[3 * j + c] - R[3 * i + c];
        u4[4 * j + 3] = far ? 1e150 : r;
        if (j != i) {
            fc[j] = cut_fn(r, P.acut);
            dfc[j] = cut_dfn(r, P.acut);
            TwoBody tb;
            double *w = two + kTwoW * j;
            w[7] = 0.0;  // pref0: no contribution
            if (!(r > P.rcut) && two_body(P, r, tb, true)) {
                w[0] = tb.mu;
                w[1] = 1.0 / tb.s2;
                w[2] = -P.d2 / r - tb.ds / tb.s;
                w[3] = tb.dmu / tb.s2;
                w[4] = tb.ds / (tb.s2 * tb.s);
                w[5] = tb.f;
                w[6] = tb.df;
                w[7] = tb.pref0;
            } else {
                for (int c = 0; c < 7; ++c) w[c] = 0.0;
            }
            int rank = 0;
            for (int t = 0; t < n; ++t)
                rank += (int)(t != i) & ((el[t] < el[j]) | ((el[t] == el[j]) & (t < j)));
            ord[rank] = j;
        }
    }
    for (int e = tid; e <= P.nelem; e += NTG) {
        int c = 0;
        for (int t = 0; t < n; ++t) c += (int)(t != i) & (el[t] < e);
        est[e] = c;
    }
    for (int t = tid; t < n * n; t += NTG) {  // no triplet (j, j)
        if (t / n == t % n)
            for (int c = 0; c < 6; ++c) rec[(size_t)(t / n * ma + t % n) * 6 + c] = 0.0;
    }
    __syncthreads();

    // ---------------- pair records: (j, k) and (k, j) of every neighbour pair ----------------
    const int n1 = n - 1, ntri = n1 * (n1 - 1) / 2;
    for (int t = tid; t < ntri; t += NTG) {
        int ja, ka;
        triangle_at(n1, t, ja, ka);
        const int j = ja + (ja >= i), k = ka + (ka >= i);  // neighbour index -> atom (not i)
        double *rj = rec + (size_t)(j * ma + k) * 6, *rk = rec + (size_t)(k * ma + j) * 6;
        const double rij = u4[4 * j + 3], rik = u4[4 * k + 3];
        if (rij > P.acut || rik > P.acut) {
            for (int c = 0; c < 6; ++c) rj[c] = rk[c] = 0.0;
            continue;
        }
        const double rjk = dist(R, j, k);
        double u[3], v[3], w[3];
        for (int c = 0; c < 3; ++c) {
            u[c] = u4[4 * j + c];
            v[c] = u4[4 * k + c];
            w[c] = R[3 * k + c] - R[3 * j + c];
        }
        const double uv = u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
        const double uw = u[0] * w[0] + u[1] * w[1] + u[2] * w[2];
        const double vw = v[0] * w[0] + v[1] * w[1] + v[2] * w[2];
        const double iij = 1.0 / rij, iik = 1.0 / rik, ijk = 1.0 / rjk;
        const double qjk = iij * iik, qij = iij * ijk, qik = iik * ijk, s_jk = ijk * ijk;
        double ci = uv * qjk;
        ci = ci > 1.0 ? 1.0 : (ci < -1.0 ? -1.0 : ci);
        const double cj = -uw * qij, ck = vw * qik;
        const double prod = rij * rik * rjk;
        const double wP = P.w3 * pow(prod > kEps ? prod : kEps, -P.d3);
        const double tn = 1.0 + 3.0 * ci * cj * ck, T = tn * wP;
        const double fij = fc[j], fik = fc[k], F = fij * fik, W = F * T;
        const double sden = sqrt(fmax(1e-10, rij * rij * rik * rik - uv * uv)) * qjk;
        const double aw = P.angw[0], si = sqrt(fmax(0.0, 1.0 - ci * ci)), cot = ci / sden;
        // own-vector (u) and partner-vector (v) coefficients of the gradient at one neighbour
        auto side = [&](double io, double c_own, double c_oth, double q_own, double q_oth,
                        double dF, double *out) {
            const double io2 = io * io;
            const double ac = -ci * io2, bc = qjk;                        // cos at the centre
            const double aj = 2.0 * q_own - c_own * (io2 + s_jk), bj = c_own * s_jk - q_own;
            const double ak = -c_oth * s_jk, bk = c_oth * s_jk - q_oth;
            const double aT = wP * (3.0 * (ac * cj * ck + ci * (aj * c_oth + ak * c_own)) -
                                    tn * P.d3 * (io2 + s_jk));
            const double bT = wP * (3.0 * (bc * cj * ck + ci * (bj * c_oth + bk * c_own)) +
                                    tn * P.d3 * s_jk);
            const double aW = dF * io * T + F * aT, bW = F * bT;
            out[0] = aw * (ac * W + ci * aW);
            out[1] = aw * (bc * W + ci * bW);
            out[2] = aw * (si * aW - cot * ac * W);
            out[3] = aw * (si * bW - cot * bc * W);
            out[4] = aw * ci * W;
            out[5] = aw * si * W;
        };
        side(iij, cj, ck, qij, qik, dfc[j] * fik, rj);
        side(iik, ck, cj, qik, qij, dfc[k] * fij, rk);
    }
    __syncthreads();

    // ---------------- feature blocks ----------------
    const double ysc = -P.eta3 * kExpScale;
    // species p (and q) of a block: neighbours ord[pb..pe) and ord[qb..qe); false where there
    // are none
    auto species = [&](int unit, int &p, int &q) {
        const bool two_body = unit < P.nelem * nu2;
        p = 0;
        if (two_body) {
            p = q = unit / nu2;
        } else {
            int c = (unit - P.nelem * nu2) / nu3;
            while (c >= P.nelem - p) c -= P.nelem - p, ++p;
            q = p + c;
        }
        const int np = est[p + 1] - est[p], nq = est[q + 1] - est[q];
        return np > 0 && nq > 0 && (two_body || p != q || np > 1);
    };
    for (int unit = split; unit < nunits; unit += splits) {
        int f0, nr, p, q;
        unit_rows(unit, f0, nr);
        const bool is2 = unit < P.nelem * nu2;
        if (!species(unit, p, q)) {
            if constexpr (NTG < kGradThreads)  // with the empty blocks that follow as one run
                for (int e0, en; splits == 1 && unit + 1 < nunits && !species(unit + 1, p, q);
                     ++unit) {
                    unit_rows(unit + 1, e0, en);
                    nr = e0 + en - f0;
                }
            zero_rows(f0, nr);
            continue;
        }
        const int pb = est[p], np = est[p + 1] - pb, qb = est[q], nq = est[q + 1] - qb;
        const int nact = p == q ? np : np + nq;
        const int nl = is2 ? nr : nr / P.na;
        // neighbour of item a: the block's first, then the others (their columns are zero)
        auto atom_of = [&](int a) {
            if (a < np) return ord[pb + a];
            if (a < nact) return ord[qb + a - np];
            a -= nact;
            if (a >= pb) a += np;
            if (p != q && a >= qb) a += nq;  // p < q, so its range lies behind p's
            return ord[a];
        };
        for (int item = tid; item < n1 * nl; item += NTG) {
            const int a = item / nl, l = item - a * nl, j = atom_of(a);
            if (a >= nact) {
                for (int row = is2 ? l : l * P.na, e = is2 ? row + 1 : row + P.na; row < e; ++row)
                    for (int d = 0; d < 3; ++d) tile[row * ld + 3 * j + d] = 0.0;
                continue;
            }
            if (is2) {
                double val = 0.0, dv = 0.0;
                const double *w = two + kTwoW * j;
                if (w[7] != 0.0) {
                    const int k = f0 - p * P.nb2 + l;
                    const double L = P.logRs2[k] - w[0];
                    const double E =
                        exp_scaled(-0.5 * kExpScale * (L * L * w[1]), tab) * w[7] / P.Rs2[k];
                    val = w[5] * E;
                    dv = E * (w[5] * (w[2] + L * (w[3] + L * w[4])) + w[6]) / u4[4 * j + 3];
                }
                vals[l * ma + a] = val;
                for (int d = 0; d < 3; ++d) tile[l * ld + 3 * j + d] = dv * u4[4 * j + d];
                continue;
            }
            double v0 = 0.0, v1 = 0.0, s0 = 0.0, s1 = 0.0, t0 = 0.0, t1 = 0.0;
            double g0[3] = {0.0, 0.0, 0.0}, g1[3] = {0.0, 0.0, 0.0};
            const int tr = l * P.na;
            const bool inp = a < np;
            const int kb = inp ? qb : pb, ke = kb + (inp ? nq : np);
            const double rs3 = P.Rs3[((f0 - P.three_off) / P.na) % P.nb3 + l];
            const double off = 0.5 * u4[4 * j + 3] - rs3;
            for (int t = kb; t < ke; ++t) {
                const int k = ord[t];
                const double *rr = rec + (size_t)(j * ma + k) * 6;
                const double dr = fma(0.5, u4[4 * k + 3], off);
                const double rad = exp_scaled(ysc * (dr * dr), tab);
                const double rd = rad * dr;
                const double b0 = rad * rr[1], b1 = rad * rr[3];
                s0 = fma(rad, rr[0], s0);
                s1 = fma(rad, rr[2], s1);
                v0 = fma(rad, rr[4], v0);
                v1 = fma(rad, rr[5], v1);
                t0 = fma(rd, rr[4], t0);
                t1 = fma(rd, rr[5], t1);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    g0[d] = fma(b0, u4[4 * k + d], g0[d]);
                    g1[d] = fma(b1, u4[4 * k + d], g1[d]);
                }
            }
            const double h = -P.eta3 / u4[4 * j + 3];
            s0 = fma(h, t0, s0);
            s1 = fma(h, t1, s1);
            for (int ta = 0; ta < P.na; ++ta)
                vals[(tr + ta) * ma + a] = ta == 0 ? v0 : (ta == 1 ? v1 : 0.0);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                double *col = tile + (size_t)tr * ld + 3 * j + d;
                col[0] = fma(s0, u4[4 * j + d], g0[d]);
                col[ld] = fma(s1, u4[4 * j + d], g1[d]);
                for (int ta = 2; ta < P.na; ++ta) col[ta * ld] = 0.0;
            }
        }
        __syncthreads();
        // centre column and value of each row; in a channel of two elements every pair is
        // seen from both, so the values are summed over the first element's atoms only
        for (int t = tid; t < 4 * nr; t += NTG) {
            const int row = t >> 2, d = t & 3;
            double s = 0.0;
            if (d < 3) {
                for (int a = 0; a < nact; ++a) s -= tile[row * ld + 3 * atom_of(a) + d];
                tile[row * ld + 3 * i + d] = s;
            } else {
                for (int a = 0; a < np; ++a) s += vals[row * ma + a];
                Xi[f0 + row] = O((!is2 && p == q) ? 0.5 * s : s);
            }
        }
        __syncthreads();
        stream_out<NTG, O>(dXi + (size_t)f0 * ld, tile, nr * ld);
        __syncthreads();
    }
}

int build_params(FchlParams &P, int max_atoms, const int *elements, int nelem, const double *Rs2,
                 int nRs2, const double *Rs3, int nRs3, int nabasis, double eta2, double eta3,
                 double zeta, double rcut, double acut, double d2, double d3, double w3,
                 bool grad) {
    KF_REQUIRE(nelem >= 1 && nelem <= kMaxElem, KF_ERR_BASIS, "nelem must be in [1, %d]",
               kMaxElem);
    KF_REQUIRE(nRs2 >= 1 && nRs2 <= kMaxRs && nRs3 >= 1 && nRs3 <= kMaxRs, KF_ERR_BASIS,
               "nRs2/nRs3 must be in [1, %d]", kMaxRs);
    KF_REQUIRE(nabasis >= 0 && nabasis % 2 == 0 && nabasis <= 2 * kMaxHarm, KF_ERR_BASIS,
               "Ts.size() (nabasis) must be even and <= %d", 2 * kMaxHarm);
    KF_REQUIRE(max_atoms >= 1, KF_ERR_ARG, "max_atoms must be >= 1");
    for (int k = 0; k < nRs2; ++k)
        KF_REQUIRE(Rs2[k] > 0.0, KF_ERR_BASIS, "All Rs2 must be > 0");
    P.nelem = nelem;
    P.nb2 = nRs2;
    P.nb3 = nRs3;
    P.na = nabasis;
    P.nharm = grad ? (nabasis >= 2 ? 1 : 0) : nabasis / 2;
    P.nchan = nelem * (nelem + 1) / 2;
    P.three_off = nelem * nRs2;
    P.rs = P.three_off + P.nchan * nRs3 * nabasis;
    P.max_atoms = max_atoms;
    for (int e = 0; e < kMaxElem; ++e) P.elements[e] = e < nelem ? elements[e] : 0;
    for (int k = 0; k < kMaxRs; ++k) {
        P.Rs2[k] = k < nRs2 ? Rs2[k] : 1.0;
        P.logRs2[k] = log(P.Rs2[k]);
        P.Rs3[k] = k < nRs3 ? Rs3[k] : 0.0;
    }
    for (int h = 0; h < kMaxHarm; ++h) {
        const double t = zeta * (2 * h + 1);
        P.angw[h] = 2.0 * exp(-0.5 * t * t);
    }
    P.eta2 = eta2;
    P.eta3 = eta3;
    P.rcut = rcut;
    P.acut = acut;
    P.d2 = d2;
    P.d3 = d3;
    P.w3 = w3;
    return KF_OK;
}

// Whether the kernels above take this batch (else kf_fchl19_f64 takes the FCHL19v2 kernel), and
// whether they write each value once: a representation whose centres have more pairs than one
// chunk holds is added up in X itself.
bool fchl19_fits(int ma, int nelem, int nchan, int nb2, int nb3, int na, bool grad) {
    return ma <= kMaxAtoms && (grad ? grad_lds_bytes(ma, nb2, nb3, na)
                                    : rep_lds_bytes(ma, nelem, nchan, na)) <= 160 * 1024;
}
bool fchl19_long(int ma, int nelem, int nchan, int nb3, int na) {
    const RepLds g = rep_lds(ma, nelem, nchan, na);
    const int npair = (ma - 1) * (ma - 2) / 2;  // (ma <= kMaxAtoms)
    return npair > g.pairs ||
           rep_share_log(nchan * ((nb3 + kLB - 1) / kLB) * rep_batch(g, ma), npair) > 0;
}
bool fchl19_one_chunk(int ma, int nelem, int nchan, int na) {
    return (long)(ma - 1) * (ma - 2) / 2 <= rep_lds(ma, nelem, nchan, na).pairs;
}

template <typename O>
int fchl19_impl(const double *coords, const int *Q, const int *N, int nm, int max_atoms,
                const int *elements, int nelem, const double *Rs2, int nRs2, const double *Rs3,
                int nRs3, int nabasis, double eta2, double eta3, double zeta, double rcut,
                double acut, double two_body_decay, double three_body_decay, double w3, O *X,
                O *dX, void *stream_) {
    hipStream_t stream = as_stream(stream_);
    KF_REQUIRE(nm >= 0, KF_ERR_ARG, "nm must be >= 0");
    if (nm == 0) return KF_OK;
    KF_REQUIRE(coords && Q && N && X && elements && Rs2 && Rs3, KF_ERR_ARG, "null pointer");
    FchlParams P;
    int rc = build_params(P, max_atoms, elements, nelem, Rs2, nRs2, Rs3, nRs3, nabasis, eta2,
                          eta3, zeta, rcut, acut, two_body_decay, three_body_decay, w3,
                          dX != nullptr);
    if (rc) return rc;
    // LDS of the kernels below (whole molecules staged per workgroup)
    const int ma = max_atoms;
    const size_t lds_rep = rep_lds_bytes(ma, P.nelem, P.nchan, P.na);
    const size_t lds_grad = grad_lds_bytes(ma, P.nb2, P.nb3, P.na);
    const size_t lds = dX ? lds_grad : lds_rep;
    const bool fits = fchl19_fits(ma, P.nelem, P.nchan, P.nb2, P.nb3, P.na, dX != nullptr);
    if constexpr (sizeof(O) == sizeof(float)) {
        KF_REQUIRE(fits && (dX || fchl19_one_chunk(ma, P.nelem, P.nchan, P.na)), KF_ERR_ARG,
                   "max_atoms %d is too large for float32 results (kf_fchl19_f32_fits)", ma);
    } else if (!fits) {
        // Large molecules: the FCHL19v2 kernel with the log-normal two-body and odd-Fourier
        // r_bar three-body bases is this representation (same values and Jacobian, the
        // gradient path's first-harmonic convention included) and stages no molecule in LDS.
        return kf_fchl19v2_f64(coords, Q, N, nm, max_atoms, elements, nelem, Rs2, nRs2, Rs3,
                               nRs3, nullptr, 0, nabasis, 0, 0, eta2, eta3, eta3, zeta, rcut,
                               acut, two_body_decay, three_body_decay, w3, X, dX, stream_);
    }
    // the kernels raise the flag in pinned host memory (one word per device), so a call needs
    // no launch to clear it and no copy to read it
    int dev = 0;
    KF_HIP_TRY(hipGetDevice(&dev));
    int *err = static_cast<int *>(host_staging(WS_ERR, sizeof(int) * kErrWords));
    KF_REQUIRE(err && dev >= 0 && dev < kErrWords / 2, KF_ERR_NOMEM, "pinned staging allocation failed");
    err += dev;
    *err = 0;
    ScopedTimer timer(TM_FCHL19, stream);
    if (!dX) {
        // up to a work-group per two rows while there are fewer molecules than the GPU takes
        // work-groups
        const int splits = std::max(1, std::min((ma + 1) / 2, 1024 / nm));
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(nm, splits), dim3(kRepThreads), lds, stream, coords, Q,
                               N, P, X, err);
        };
        if (fchl19_long(ma, P.nelem, P.nchan, P.nb3, P.na)) launch(fchl19_rep_kernel<O, true>);
        else launch(fchl19_rep_kernel<O, false>);
    } else {
        KF_REQUIRE(P.nelem * P.nb2 > 0, KF_ERR_BASIS, "empty two-body basis");
        // Several work-groups per centre while the batch has fewer centres than the GPU takes
        // work-groups (256 CUs, three each): one molecule of 21 atoms takes 20 us with 8 per centre (181 us before, one per centre)
        const long centres = (long)nm * ma;
        const int splits = centres >= 768 ? 1 : (int)std::min<long>(8, 768 / centres);
        auto launch = [&](auto kern, int threads) {
            hipLaunchKernelGGL(kern, dim3(ma * splits, nm), dim3(threads), lds, stream, coords, Q,
                               N, P, splits, X, dX, err);
        };
        // A small molecule's centre is a chain of short steps: one wave each keeps four times as
        // many in flight.  20,000 molecules of 2 atoms of one element 0.17 ms (0.45 with four
        // waves), 5,000 of 5 atoms of five elements 0.49 (1.14), 500 of 10 atoms 0.31 (0.41);
        // 500 of 14 atoms 0.80 (0.71), and 50 of 8 atoms, which do not fill the GPU, 103 us (87).
        if (ma <= 10 && centres >= 1024) launch(fchl19_grad_kernel<O, 64>, 64);
        else launch(fchl19_grad_kernel<O, kGradThreads>, kGradThreads);
    }
    KF_HIP_TRY(hipGetLastError());
    KF_HIP_TRY(hipStreamSynchronize(stream));
    KF_REQUIRE(*static_cast<volatile int *>(err) == 0, KF_ERR_ELEMENT, "nuclear_z contains an element not present in elements");
    return KF_OK;
}

}  // namespace
}  // namespace kf

extern "C" int kf_fchl19_f64(const double *coords, const int *Q, const int *N, int nm,
                             int max_atoms, const int *elements, int nelem, const double *Rs2,
                             int nRs2, const double *Rs3, int nRs3, int nabasis, double eta2,
                             double eta3, double zeta, double rcut, double acut,
                             double two_body_decay, double three_body_decay, double w3,
                             double *X, double *dX, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return kf::fchl19_impl<double>(coords, Q, N, nm, max_atoms, elements, nelem, Rs2, nRs2, Rs3,
                                   nRs3, nabasis, eta2, eta3, zeta, rcut, acut, two_body_decay,
                                   three_body_decay, w3, X, dX, stream);
}

extern "C" int kf_fchl19_f32_fits(int max_atoms, int nelem, int nRs2, int nRs3, int nabasis,
                                  int grad) {
    using namespace kf;
    if (max_atoms < 1 || nelem < 1 || nRs2 < 1 || nRs3 < 1 || nabasis < 1) return 0;
    const int nchan = nelem * (nelem + 1) / 2;
    return fchl19_fits(max_atoms, nelem, nchan, nRs2, nRs3, nabasis, grad != 0) &&
           (grad || fchl19_one_chunk(max_atoms, nelem, nchan, nabasis));
}

extern "C" int kf_fchl19_f32(const double *coords, const int *Q, const int *N, int nm,
                             int max_atoms, const int *elements, int nelem, const double *Rs2,
                             int nRs2, const double *Rs3, int nRs3, int nabasis, double eta2,
                             double eta3, double zeta, double rcut, double acut,
                             double two_body_decay, double three_body_decay, double w3, float *X,
                             float *dX, void *stream) {
    kf::EntryGuard kf_entry_guard_(kf::as_stream(stream));
    return kf::fchl19_impl<float>(coords, Q, N, nm, max_atoms, elements, nelem, Rs2, nRs2, Rs3,
                                  nRs3, nabasis, eta2, eta3, zeta, rcut, acut, two_body_decay,
                                  three_body_decay, w3, X, dX, stream);
}
