// feature_compact.hip -- gather descriptor sets onto their non-zero columns.
//
// A descriptor column that is zero for every atom of the sets a call works on, in X and in
// the Jacobian, adds nothing to any kernel entry or matvec product built from them (the
// FCHL19 channels of neighbour elements a data set does not contain: N and S for C9H8O4
// conformers use 312 of the 720 columns).  The derivative kernels and the matrix-free
// solver gather their sets once onto the used columns and run on those; the results
// differ only in the order of the FP64 additions.
#include <algorithm>
#include <vector>

#include "feature_compact.hpp"

namespace kf {
namespace {

__device__ inline int clamp_n(int v, int hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

__global__ __launch_bounds__(256) void fill_int_kernel(int *p, int n, int v) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

// flag[f] = 1 when column f is non-zero in X or dX for some atom of the set.  A work-group
// takes the columns of one atom (row step * (first + blockIdx.x) of the set) that no earlier one
// has flagged: it reads the flags once, lists the others in LDS and streams their runs of
// the Jacobian.  Launched first on a few atoms spread over the set, which find nearly every
// used column, then on all: the second launch then reads little but the unused columns.
// (Every flag is only ever raised, so one that is not yet seen costs a read, no more.)
// Bound by that read: 200 conformers of 21 atoms (1.5 GB, 408 of 720 columns unused)
// 0.22 ms (1.95 with one work-group per molecule reading everything a run a wave), 37 mixed
// molecules, whose columns are nearly all used, 0.04 (2.19).
__global__ __launch_bounds__(256) void active_cols_kernel(const double *__restrict__ X,
                                                          const double *__restrict__ dX,
                                                          const int *__restrict__ N, int ma,
                                                          int rep, int step, size_t first,
                                                          int *__restrict__ flag) {
    extern __shared__ int lds[];  // unseen columns, then a flag for each
    __shared__ int count;
    const int tid = threadIdx.x;
    const size_t row = (first + blockIdx.x) * step;
    const int a = (int)(row / ma), i = (int)(row - (size_t)a * ma);
    if (i >= clamp_n(N[a], ma)) return;
    int *list = lds, *seen = lds + rep;
    if (tid == 0) count = 0;
    __syncthreads();
    const double *x = X + row * rep;
    for (int f = tid; f < rep; f += 256) {
        if (flag[f]) continue;
        if (x[f] != 0.0) {
            flag[f] = 1;
        } else if (dX) {
            const int at = atomicAdd(&count, 1);
            list[at] = f;
            seen[at] = 0;
        }
    }
    __syncthreads();
    const int n = count;
    if (n == 0) return;
    // the threads take nrow runs of L coordinates at a time (one for 85 atoms and more)
    const int L = 3 * ma;
    const double *J = dX + row * rep * L;
    for (int c0 = 0; c0 < L; c0 += 256) {
        const int cn = min(L - c0, 256), nrow = 256 / cn, rr = tid / cn, c = c0 + tid - rr * cn;
        if (rr >= nrow) continue;
        for (int u = rr; u < n; u += 4 * nrow) {
            double v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = J[(size_t)list[min(u + k * nrow, n - 1)] * L + c];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (v[k] != 0.0) seen[min(u + k * nrow, n - 1)] = 1;
        }
    }
    __syncthreads();
    for (int u = tid; u < n; u += 256)
        if (seen[u]) flag[list[u]] = 1;
}

int flag_columns(const double *X, const double *dX, const int *N, int nm, int ma, int rep,
                 int *flag, hipStream_t stream) {
    const long rows = (long)nm * ma;
    if (rows == 0) return KF_OK;
    const size_t lds = 2 * sizeof(int) * rep;
    const int probe = (int)(rows / 64);  // an atom in so many, in the first launch
    auto scan = [&](int step) {
        return for_groups((rows + step - 1) / step, [&](size_t first, unsigned n) {
            hipLaunchKernelGGL(active_cols_kernel, dim3(n), dim3(256), lds, stream, X, dX, N, ma,
                               rep, step, first, flag);
        });
    };
    int rc = KF_OK;
    if (dX && probe > 1) rc = scan(probe);
    return rc ? rc : scan(1);
}

// Y[r][g][c] = X[r][cols[g]][c]: row r of rep runs of L doubles -> nf runs.  One
// work-group per row.
__global__ __launch_bounds__(256) void gather_cols_kernel(const double *__restrict__ X, int rep,
                                                          int L, const int *__restrict__ cols,
                                                          int nf, double *__restrict__ Y) {
    const size_t r = blockIdx.x;
    const double *src = X + r * rep * L;
    double *dst = Y + r * nf * L;
    const int n = nf * L;
    for (int e = threadIdx.x; e < n; e += 256) {
        const int g = e / L, c = e - g * L;
        dst[e] = src[(size_t)cols[g] * L + c];
    }
}

// Gather X (and dX, if given) of one set onto the columns cols (device) into ws.
int gather_set(const double *X, const double *dX, int nm, int ma, int rep, const int *cols,
               int nf, int ws, hipStream_t stream, const double **Xc, const double **dXc) {
    const size_t rows = (size_t)nm * ma, L = 3 * (size_t)ma;
    const size_t nx = rows * nf, nj = dX ? rows * nf * L : 0;
    double *buf = static_cast<double *>(workspace(ws, sizeof(double) * (nx + nj + 1), stream));
    KF_REQUIRE(buf, KF_ERR_NOMEM, "workspace allocation failed (%zu B)", sizeof(double) * (nx + nj));
    *Xc = buf;
    *dXc = dX ? buf + nx : nullptr;
    if (rows == 0) return KF_OK;
    auto gather = [&](const double *from, size_t run, double *to) {
        return for_groups(rows, [&](size_t first, unsigned n) {
            hipLaunchKernelGGL(gather_cols_kernel, dim3(n), dim3(256), 0, stream,
                               from + first * rep * run, rep, (int)run, cols, nf,
                               to + first * nf * run);
        });
    };
    const int rc = gather(X, 1, buf);
    return rc || !dX ? rc : gather(dX, L, buf + nx);
}

}  // namespace

int compact_columns(CompactSets &c, int rep, int ws1, int ws2, hipStream_t stream, int *nf_out) {
    *nf_out = rep;
    if (rep < 1 || (c.nm1 == 0 && c.nm2 == 0)) return KF_OK;
    if (rep > 16384) return KF_OK;  // (128 KB of LDS) wider than one work-group's flags: run on every column
    const bool same = c.x1 == c.x2 && c.dx1 == c.dx2 && c.n1 == c.n2 && c.nm1 == c.nm2 &&
                      c.ma1 == c.ma2;
    int *flag = static_cast<int *>(workspace(WS_AUX1, sizeof(int) * (2 * (size_t)rep + 1), stream));
    int *hflag = static_cast<int *>(host_staging(WS_AUX1, sizeof(int) * rep));
    KF_REQUIRE(flag && hflag, KF_ERR_NOMEM, "workspace allocation failed");
    hipLaunchKernelGGL(fill_int_kernel, dim3((rep + 255) / 256), dim3(256), 0, stream, flag, rep, 0);
    KF_HIP_TRY(hipGetLastError());
    int rc;
    if ((rc = flag_columns(c.x1, c.dx1, c.n1, c.nm1, c.ma1, rep, flag, stream))) return rc;
    if (!same && (rc = flag_columns(c.x2, c.dx2, c.n2, c.nm2, c.ma2, rep, flag, stream))) return rc;
    KF_HIP_TRY(hipMemcpyAsync(hflag, flag, sizeof(int) * rep, hipMemcpyDeviceToHost, stream));
    KF_HIP_TRY(hipStreamSynchronize(stream));
    std::vector<int> cols;
    for (int f = 0; f < rep; ++f)
        if (hflag[f]) cols.push_back(f);
    if ((int)cols.size() == rep) return KF_OK;
    if (cols.empty()) cols.push_back(0);  // all-zero sets: one (zero) column keeps rep >= 1
    const int nf = (int)cols.size();
    std::copy(cols.begin(), cols.end(), hflag);
    int *dcols = flag + rep;
    KF_HIP_TRY(hipMemcpyAsync(dcols, hflag, sizeof(int) * nf, hipMemcpyHostToDevice, stream));
    const double *x1 = nullptr, *dx1 = nullptr, *x2 = nullptr, *dx2 = nullptr;
    if ((rc = gather_set(c.x1, c.dx1, c.nm1, c.ma1, rep, dcols, nf, ws1, stream, &x1, &dx1)))
        return rc;
    if (same) {
        x2 = x1;
        dx2 = dx1;
    } else if ((rc = gather_set(c.x2, c.dx2, c.nm2, c.ma2, rep, dcols, nf, ws2, stream, &x2,
                                &dx2))) {
        return rc;
    }
    c.x1 = x1; c.dx1 = dx1; c.x2 = x2; c.dx2 = dx2;
    *nf_out = nf;
    // the staging copy above must land before hflag is reused by a later call
    KF_HIP_TRY(hipStreamSynchronize(stream));
    return KF_OK;
}

}  // namespace kf
