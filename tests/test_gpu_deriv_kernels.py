"""GPU parity: energy+force forms of the local kernel (jacobian, jacobian_t, hessian,
full, and the symmetric dense / RFP forms) vs the FP64 oracle.

Bar: every entry within 1e-10 relative to the largest |entry| of the oracle's block
(FP64 throughout; the GPU sums in a different order, so bit equality is not expected).
Random inputs use random (not physical) Jacobians, which exercises the algebra of every
block independently; the conformer case uses real FCHL19 descriptors and Jacobians."""

import numpy as np
import pytest

import oracle
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.fixture(scope="module")
def lk():
    from kernelforge_amd import local_kernels

    return local_kernels


def rand_set(nm, ma, rep, nlab, seed, nmin=0):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((nm, ma, rep)) * 0.3
    dX = rng.standard_normal((nm, ma, rep, 3 * ma)) * 0.2
    Q = rng.integers(1, nlab + 1, (nm, ma)).astype(np.int32)
    N = rng.integers(nmin, ma + 1, nm).astype(np.int32)
    return X, dX, Q, N


# (nm1, ma1, nm2, ma2, rep, nlab): single-atom molecules (one 16-column block), 2 and 4
# force-column blocks, more than 64 columns (a second round of column blocks), the
# 32-atom maximum, and more partners per molecule than one projection group holds (8).
CASES = [(3, 1, 4, 2, 9, 1), (5, 3, 6, 4, 33, 2), (4, 7, 5, 9, 40, 3), (3, 21, 4, 21, 72, 3),
         (2, 23, 3, 25, 50, 2), (2, 32, 2, 32, 24, 2), (3, 5, 20, 7, 16, 2)]


@pytest.mark.parametrize("case", CASES)
def test_rect_forms(lk, case):
    nm1, ma1, nm2, ma2, rep, nlab = case
    X1, dX1, Q1, N1 = rand_set(nm1, ma1, rep, nlab, 1 + ma1)
    X2, dX2, Q2, N2 = rand_set(nm2, ma2, rep, nlab, 100 + ma2)
    s = 1.7
    got = lk.kernel_gaussian_jacobian(X1, X2, dX2, Q1, Q2, N1, N2, s)
    assert got.shape == (nm1, 3 * int(np.clip(N2, 0, ma2).sum()))
    assert rel_err(got, oracle.jacobian(X1, X2, dX2, Q1, Q2, N1, N2, s)) < TOL
    got = lk.kernel_gaussian_jacobian_t(X1, dX1, X2, Q1, Q2, N1, N2, s)
    assert rel_err(got, oracle.jacobian_t(X1, dX1, X2, Q1, Q2, N1, N2, s)) < TOL
    got = lk.kernel_gaussian_hessian(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)
    assert rel_err(got, oracle.hessian(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)) < TOL
    got = lk.kernel_gaussian_full(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)
    ref = oracle.full(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)
    assert got.shape == ref.shape
    assert rel_err(got, ref) < TOL


@pytest.mark.parametrize("case", [(4, 2, 10, 2), (7, 6, 33, 3), (5, 21, 64, 3), (3, 24, 20, 2),
                                  (2, 32, 12, 1), (19, 6, 20, 3)])
def test_symm_forms(lk, case):
    nm, ma, rep, nlab = case
    X, dX, Q, N = rand_set(nm, ma, rep, nlab, 7 * ma + nm)
    s = 1.3
    for name, fn in (("kernel_gaussian_hessian_symm", oracle.hessian_symm),
                     ("kernel_gaussian_hessian_symm_rfp", oracle.hessian_symm_rfp),
                     ("kernel_gaussian_full_symm", oracle.full_symm),
                     ("kernel_gaussian_full_symm_rfp", oracle.full_symm_rfp)):
        got = getattr(lk, name)(X, dX, Q, N, s)
        ref = fn(X, dX, Q, N, s)
        assert got.shape == ref.shape, name
        assert rel_err(got, ref) < TOL, name


def test_zero_columns(lk):
    """Columns that are zero in X and in the Jacobian for every atom of both sets are
    dropped before the kernels run; columns zero in X but not in the Jacobian stay (their
    Jacobian rows still enter the force-force blocks)."""
    X1, dX1, Q1, N1 = rand_set(4, 6, 50, 2, 31)
    X2, dX2, Q2, N2 = rand_set(5, 5, 50, 2, 32)
    x_only = [3, 4, 17, 30, 31, 32]     # zero in X, Jacobian kept
    both = [0, 1, 2, 10, 11, 40, 49]    # zero in X and in the Jacobian
    for X, dX in ((X1, dX1), (X2, dX2)):
        X[..., x_only + both] = 0.0
        dX[..., both, :] = 0.0
    dX2[..., 5, :] = 0.0                # zero in one set's Jacobian only: kept
    s = 1.3
    assert rel_err(lk.kernel_gaussian_full(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s),
                   oracle.full(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)) < TOL
    assert rel_err(lk.kernel_gaussian_jacobian(X1, X2, dX2, Q1, Q2, N1, N2, s),
                   oracle.jacobian(X1, X2, dX2, Q1, Q2, N1, N2, s)) < TOL
    got = lk.kernel_gaussian_full_symm_rfp(X1, dX1, Q1, N1, s)
    assert rel_err(got, oracle.full_symm_rfp(X1, dX1, Q1, N1, s)) < TOL
    got = lk.kernel_gaussian_hessian_symm(X2, dX2, Q2, N2, s)
    assert rel_err(got, oracle.hessian_symm(X2, dX2, Q2, N2, s)) < TOL
    # every column zero: the kernel of the constant descriptor
    Z, dZ = np.zeros_like(X1), np.zeros_like(dX1)
    assert rel_err(lk.kernel_gaussian_full_symm(Z, dZ, Q1, N1, s),
                   oracle.full_symm(Z, dZ, Q1, N1, s)) < TOL


def test_full_symm_conformers(lk):
    """Real FCHL19 descriptors + Jacobians of 10 C9H8O4 conformers: the RFP E+F
    kernel, its dense form, and the block identities of the full kernel."""
    from kernelforge_amd import synthetic

    base, z = synthetic.aspirin_base()
    C, Z, _, _ = synthetic.conformers(base, z, 10, 5)
    Q = np.tile(Z, (10, 1)).astype(np.int32)
    N = np.full(10, 21, np.int32)
    X, dX = oracle.fchl19_batch(C, Q, N, grad=True)
    arf = lk.kernel_gaussian_full_symm_rfp(X, dX, Q, N, 2.0)
    assert rel_err(arf, oracle.full_symm_rfp(X, dX, Q, N, 2.0)) < TOL
    K = lk.kernel_gaussian_full_symm(X, dX, Q, N, 2.0)
    nm = 10
    # blocks of the symmetric full kernel against the standalone forms
    assert rel_err(K[:nm, :nm], lk.kernel_gaussian_symm(X, Q, N, 2.0)) < TOL
    jt = lk.kernel_gaussian_jacobian_t(X, dX, X, Q, Q, N, N, 2.0)
    assert rel_err(K[nm:, :nm], -jt) < TOL            # FE = dK/dR1 = -jacobian_t
    assert rel_err(K[:nm, nm:], -jt.T) < TOL          # EF = dK/dR2
    assert rel_err(K[nm:, nm:], lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 2.0)) < TOL
    assert rel_err(K, K.T) < 1e-13


def test_zero_atoms_and_no_shared_labels(lk):
    X, dX, Q, N = rand_set(4, 3, 8, 2, 3, nmin=0)
    N[:] = [0, 2, 0, 3]
    got = lk.kernel_gaussian_full_symm_rfp(X, dX, Q, N, 1.1)
    assert rel_err(got, oracle.full_symm_rfp(X, dX, Q, N, 1.1)) < TOL
    K = lk.kernel_gaussian_full(X, dX, X, dX, Q, Q + 10, N, N, 1.1)
    assert np.all(K == 0.0)
    N0 = np.zeros(4, np.int32)
    assert lk.kernel_gaussian_hessian(X, dX, X, dX, Q, Q, N0, N, 1.0).shape == (0, 15)
    assert lk.kernel_gaussian_jacobian_t(X, dX, X, Q, Q, N0, N, 1.0).shape == (0, 4)


@pytest.mark.parametrize("ma1,ma2", [(5, 9), (30, 6), (9, 30)])
def test_any_label_value(lk, ma1, ma2):
    # labels are compared and nothing else: negative ones are labels too, also where molecules
    # have places past their atoms and a group of partners is not full; the two sets' molecules
    # may differ in size by any amount
    X1, dX1, Q1, N1 = rand_set(3, ma1, 20, 3, 5, 1)
    X2, dX2, Q2, N2 = rand_set(5, ma2, 20, 3, 6, 1)
    N1[0], N2[-1] = ma1, 2
    s = 1.6
    for lab in (np.array([0, -2, -1, 7]), np.array([0, 0, -(2**31), 2**31 - 1])):
        q1, q2 = lab[Q1].astype(np.int32), lab[Q2].astype(np.int32)
        got = lk.kernel_gaussian_full(X1, dX1, X2, dX2, q1, q2, N1, N2, s)
        assert rel_err(got, oracle.full(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)) < TOL
        got = lk.kernel_gaussian_hessian(X1, dX1, X2, dX2, q1, q2, N1, N2, s)
        assert rel_err(got, oracle.hessian(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)) < TOL
        got = lk.kernel_gaussian_hessian_symm(X2, dX2, q2, N2, s)
        assert rel_err(got, oracle.hessian_symm(X2, dX2, Q2, N2, s)) < TOL


def test_errors(lk):
    X, dX, Q, N = rand_set(3, 2, 6, 2, 4)
    with pytest.raises(ValueError):
        lk.kernel_gaussian_full_symm(X, dX, Q, N, 0.0)
    with pytest.raises(ValueError):
        lk.kernel_gaussian_full_symm(X, dX[..., :5], Q, N, 1.0)
    with pytest.raises(ValueError):
        lk.kernel_gaussian_hessian(X, dX, X[..., :4], dX, Q, Q, N, N, 1.0)
    # more than 32 atoms per molecule is no error: the size-general kernel takes it
    Xb, dXb, Qb, Nb = rand_set(2, 33, 4, 1, 5)
    assert rel_err(lk.kernel_gaussian_hessian_symm(Xb, dXb, Qb, Nb, 1.0),
                   oracle.hessian_symm(Xb, dXb, Qb, Nb, 1.0)) < 1e-12


def test_keywords(lk):
    X, dX, Q, N = rand_set(3, 2, 6, 2, 6)
    a = lk.kernel_gaussian_full(X1=X, dX1=dX, X2=X, dX2=dX, Q1=Q, Q2=Q, N1=N, N2=N, sigma=1.2)
    np.testing.assert_array_equal(a, lk.kernel_gaussian_full(X, dX, X, dX, Q, Q, N, N, 1.2))
    b = lk.kernel_gaussian_jacobian(X1=X, X2=X, dX2=dX, Q1=Q, Q2=Q, N1=N, N2=N, sigma=1.2)
    np.testing.assert_array_equal(b, lk.kernel_gaussian_jacobian(X, X, dX, Q, Q, N, N, 1.2))


# ---------------------------------------------------------------------------
# alpha_desc and the matrix-free matvecs (the PCG operator) vs the oracle and
# vs the explicit full kernel: K_full @ [aE; aF] == full_matvec(aE, alpha_desc(aF)).
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("case", [(4, 3, 5, 4, 17, 2), (6, 9, 7, 8, 40, 3), (3, 21, 4, 21, 72, 3),
                                  (2, 30, 3, 26, 20, 2)])
def test_alpha_desc_and_matvecs(lk, case):
    nm1, ma1, nm2, ma2, rep, nlab = case
    X1, dX1, Q1, N1 = rand_set(nm1, ma1, rep, nlab, 11 + ma1)
    X2, dX2, Q2, N2 = rand_set(nm2, ma2, rep, nlab, 111 + ma2)
    rng = np.random.default_rng(5)
    naq2 = 3 * int(np.clip(N2, 0, ma2).sum())
    aF, aE = rng.standard_normal(naq2), rng.standard_normal(nm2)
    ad = lk.kernel_gaussian_local_compute_alpha_desc(dX2, Q2, N2, aF)
    ad_o = oracle.alpha_desc(dX2, Q2, N2, aF)
    assert ad.shape == ad_o.shape and rel_err(ad, ad_o) < 1e-13
    s = 1.6
    E, F = lk.kernel_gaussian_local_full_matvec(X1, dX1, X2, ad_o, aE, Q1, Q2, N1, N2, s)
    Eo, Fo = oracle.full_matvec(X1, dX1, X2, ad_o, aE, Q1, Q2, N1, N2, s)
    assert rel_err(E, Eo) < TOL and rel_err(F, Fo) < TOL
    Fh = lk.kernel_gaussian_local_hessian_matvec(X1, dX1, X2, ad_o, Q1, Q2, N1, N2, s)
    assert rel_err(Fh, oracle.hessian_matvec(X1, dX1, X2, ad_o, Q1, Q2, N1, N2, s)) < TOL
    Ej = lk.kernel_gaussian_local_jacobian_t_matvec(X1, X2, ad_o, Q1, Q2, N1, N2, s)
    assert rel_err(Ej, oracle.jacobian_t_matvec(X1, X2, ad_o, Q1, Q2, N1, N2, s)) < TOL
    # the matvec is the explicit full kernel applied to [aE; aF]
    K = lk.kernel_gaussian_full(X1, dX1, X2, dX2, Q1, Q2, N1, N2, s)
    y = K @ np.concatenate([aE, aF])
    assert rel_err(np.concatenate([E, F]), y) < 1e-9


# (nm1, ma1, nm2, ma2, rep, labels, zero columns of the training side): 16-row tiles with the
# summation shared by four waves, 32-row tiles with and without that, a training side
# without a query label, atoms without a match, columns that only the query has, more
# rows than one pass holds (two rounds of the 1 GiB coefficient block), and more columns
# than threads in the back-projection's work-group
@pytest.mark.parametrize("case", [
    (1, 16, 9, 5, 37, 1, 20), (1, 17, 5, 16, 16, 1, 0), (1, 90, 2, 3, 6, 2, 1),
    (7, 12, 11, 9, 33, 4, 33), (60, 25, 62, 25, 17, 1, 1), (830, 10, 830, 10, 3, 1, 1)])
def test_matvec_variants(lk, case):
    nm1, ma1, nm2, ma2, rep, nlab, nzero = case
    full = nm1 > 100  # every atom present, so that the coefficient block is over its limit
    X1, dX1, Q1, N1 = rand_set(nm1, ma1, rep, nlab, 31 + ma1, ma1 if full or nm1 == 1 else 0)
    X2, _, Q2, N2 = rand_set(nm2, ma2, rep, max(1, nlab - 1), 131 + ma2, ma2 if full else 0)
    rng = np.random.default_rng(6)
    ad = rng.standard_normal((nm2, ma2, rep))
    live = np.arange(ma2)[None] < N2[:, None]
    ad[~live] = 0.0
    X2[..., rep - nzero:] = 0.0
    ad[..., rep - nzero:] = 0.0
    aE = rng.standard_normal(nm2)
    s = 1.6
    E, F = lk.kernel_gaussian_local_full_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s)
    Eo, Fo = oracle.full_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s)
    assert rel_err(E, Eo) < TOL and rel_err(F, Fo) < TOL
    Fh = lk.kernel_gaussian_local_hessian_matvec(X1, dX1, X2, ad, Q1, Q2, N1, N2, s)
    assert rel_err(Fh, oracle.hessian_matvec(X1, dX1, X2, ad, Q1, Q2, N1, N2, s)) < TOL
    Ej = lk.kernel_gaussian_local_jacobian_t_matvec(X1, X2, ad, Q1, Q2, N1, N2, s)
    assert rel_err(Ej, oracle.jacobian_t_matvec(X1, X2, ad, Q1, Q2, N1, N2, s)) < TOL


def plan_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s):
    """(E, F) of a matvec plan on host arrays."""
    import ctypes

    from kernelforge_amd import capi

    L, DA = capi.lib(), capi.DeviceArray
    dq1, dn1, dq2, dn2 = (DA.from_numpy(a) for a in (Q1, N1, Q2, N2))
    dx1, ddx1, dx2, dad, dae = (DA.from_numpy(a) for a in (X1, dX1, X2, ad, aE))
    E, F = DA(len(X1)), DA(3 * int(np.clip(N1, 0, Q1.shape[1]).sum()))
    h = ctypes.c_void_p()
    capi.check(L.kf_matvec_plan_create(dq1.ptr, dn1.ptr, *Q1.shape, dx2.ptr, dad.ptr, dae.ptr,
                                       dq2.ptr, dn2.ptr, *Q2.shape, X1.shape[2], s,
                                       ctypes.byref(h), None), "plan")
    try:
        for _ in range(2):
            capi.check(L.kf_matvec_plan_execute(h, dx1.ptr, ddx1.ptr, E.ptr, F.ptr, None), "plan")
        capi.synchronize()
        return E.numpy(), F.numpy()
    finally:
        L.kf_matvec_plan_destroy(h)


def test_matvec_ignores_unmatched_atoms(lk):
    """Query atoms whose label the training side lacks contribute nothing, whatever their
    descriptors and Jacobians hold: all results are bit for bit those of finite ones."""
    X1, dX1, Q1, N1 = rand_set(4, 5, 24, 2, 41, 5)
    X2, _, Q2, N2 = rand_set(6, 4, 24, 2, 42, 1)
    Q1[0, 2] = Q1[2, :] = 9
    rng = np.random.default_rng(3)
    ad, aE, s = rng.standard_normal(X2.shape), rng.standard_normal(6), 1.4
    ad[np.arange(4)[None] >= N2[:, None]] = 0.0
    Xb, dXb = X1.copy(), dX1.copy()
    Xb[0, 2], Xb[2, 1, 3] = np.nan, np.inf
    dXb[0, 2, 5], dXb[2] = np.inf, np.nan

    def results(X, dX):
        E, F = lk.kernel_gaussian_local_full_matvec(X, dX, X2, ad, aE, Q1, Q2, N1, N2, s)
        return [E, F, lk.kernel_gaussian_local_hessian_matvec(X, dX, X2, ad, Q1, Q2, N1, N2, s),
                lk.kernel_gaussian_local_jacobian_t_matvec(X, X2, ad, Q1, Q2, N1, N2, s),
                *plan_matvec(X, dX, X2, ad, aE, Q1, Q2, N1, N2, s)]

    want = results(X1, dX1)
    Eo, Fo = oracle.full_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s)
    assert rel_err(want[0], Eo) < TOL and rel_err(want[1], Fo) < TOL
    assert want[0][2] == 0.0 and not want[1][30:45].any()
    for got, w in zip(results(Xb, dXb), want):
        np.testing.assert_array_equal(got, w)
    # no atom of the query set has a partner
    Q1[:] = 9
    for got in results(Xb, dXb):
        assert not got.any()


def test_matvec_far_and_non_finite_query_rows(lk):
    """A query row so far away that its squared norm overflows has no neighbours: exactly as
    if its label were absent.  An infinity in a column that the training side does not use
    still shows as NaN."""
    X1, dX1, Q1, N1 = rand_set(3, 4, 20, 2, 51, 4)
    X2, _, Q2, N2 = rand_set(5, 4, 20, 2, 52, 4)
    rng = np.random.default_rng(4)
    ad, aE, s = rng.standard_normal(X2.shape), rng.standard_normal(5), 1.4
    X2[..., 15:] = ad[..., 15:] = 0.0
    Qa = Q1.copy()
    Qa[1, 0] = Qa[2, 3] = 9
    want = lk.kernel_gaussian_local_full_matvec(X1, dX1, X2, ad, aE, Qa, Q2, N1, N2, s)
    X1[1, 0, 2], X1[2, 3, 17] = 1e160, -1e160
    got = lk.kernel_gaussian_local_full_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s)
    for g, w in zip(got, want):
        assert rel_err(g, w) < TOL
    X1[1, 0, 2], X1[2, 3, 17] = 0.1, np.inf
    E, F = lk.kernel_gaussian_local_full_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s)
    assert np.isnan(E[2]) and np.isnan(F[24:]).all()
    assert np.isfinite(E[:2]).all() and np.isfinite(F[:24]).all()


def test_matvec_float32_operands(lk):
    """float32 operands give what the same numbers held in FP64 give."""
    from kernelforge_amd import capi

    X1, dX1, Q1, N1 = rand_set(6, 11, 41, 3, 5)
    X2, _, Q2, N2 = rand_set(9, 8, 41, 3, 6)
    rng = np.random.default_rng(8)
    ad, aE = rng.standard_normal((9, 8, 41)), rng.standard_normal(9)
    X2[..., 30:] = 0.0
    ad[..., 30:] = 0.0
    naq = 3 * int(N1.sum())
    ints = [capi.DeviceArray.from_numpy(a.astype(np.int32)) for a in (Q1, Q2, N1, N2)]
    out = []
    for dtype, fn in ((np.float32, "kf_local_full_matvec_f32"), (np.float64, "kf_local_full_matvec")):
        ops = [capi.DeviceArray.from_numpy(a.astype(np.float32).astype(dtype)) for a in (X1, dX1, X2, ad, aE)]
        E, F = capi.DeviceArray(6), capi.DeviceArray(naq)
        capi.check(getattr(capi.lib(), fn)(*(o.ptr for o in ops), *(i.ptr for i in ints), 6, 9, 11,
                                           8, 41, 1.6, E.ptr, F.ptr, None), fn)
        capi.synchronize()
        out.append((E.numpy(), F.numpy()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


def test_matvec_wide_descriptors(lk):
    """More features than LDS holds for one query row, and query rows enough for one run."""
    nm, rep = 1040, 21000
    rng = np.random.default_rng(4)
    X1 = np.tile(rng.standard_normal((nm, 1, 300)) * 0.02, 70)
    dX1 = np.tile(rng.standard_normal((nm, 1, 300, 3)) * 0.2, (70, 1))
    X2, ad = rng.standard_normal((2, 1, rep)) * 0.02, rng.standard_normal((2, 1, rep)) * 0.02
    one, two = np.ones(nm, np.int32), np.ones(2, np.int32)
    args = (X1, dX1, X2, ad, np.ones(2), one[:, None], two[:, None], one, two, 2.0)
    E, F = lk.kernel_gaussian_local_full_matvec(*args)
    Eo, Fo = oracle.full_matvec(*args)
    assert rel_err(E, Eo) < TOL and rel_err(F, Fo) < TOL


def test_matvec_conformers_symmetric(lk):
    """Training-set operator on C9H8O4 conformers equals the RFP E+F kernel times alpha."""
    from kernelforge_amd import synthetic

    base, z = synthetic.aspirin_base()
    C, Z, _, _ = synthetic.conformers(base, z, 8, 9)
    Q = np.tile(Z, (8, 1)).astype(np.int32)
    N = np.full(8, 21, np.int32)
    X, dX = oracle.fchl19_batch(C, Q, N, grad=True)
    rng = np.random.default_rng(2)
    a = rng.standard_normal(8 + 8 * 63)
    ad = lk.kernel_gaussian_local_compute_alpha_desc(dX, Q, N, a[8:])
    E, F = lk.kernel_gaussian_local_full_matvec(X, dX, X, ad, a[:8], Q, Q, N, N, 2.0)
    K = oracle.full_symm(X, dX, Q, N, 2.0)
    assert rel_err(np.concatenate([E, F]), K @ a) < 1e-9


# pairs whose features are dealt over several work-groups: 22 runs, runs of unequal length
# (the last shorter, or left out: 61 of 33 features hold 2,003), two runs, one run from 2,048
# pairs on; groups of one molecule shared by eight work-groups and by one
@pytest.mark.parametrize("nm,ma,rep", [(2, 23, 720), (5, 7, 101), (44, 4, 67), (65, 3, 64),
                                       (2, 3, 2003)])
def test_feature_runs(lk, nm, ma, rep):
    X, dX, Q, N = rand_set(nm, ma, rep, 2, nm + rep)
    got = lk.kernel_gaussian_full_symm(X, dX, Q, N, 2.1)
    assert rel_err(got, oracle.full_symm(X, dX, Q, N, 2.1)) < TOL
    got = lk.kernel_gaussian_full_symm_rfp(X, dX, Q, N, 2.1)
    assert rel_err(got, oracle.full_symm_rfp(X, dX, Q, N, 2.1)) < TOL
    m = max(1, nm // 3)
    got = lk.kernel_gaussian_hessian(X[:m], dX[:m], X, dX, Q[:m], Q, N[:m], N, 2.1)
    assert rel_err(got, oracle.hessian(X[:m], dX[:m], X, dX, Q[:m], Q, N[:m], N, 2.1)) < TOL


# Jacobians that are zero in whole blocks, as a descriptor's are for atoms a feature does not
# depend on: molecules of one to 32 atoms in every bucket, labels that start at multiples of 4
# rows and ones that cannot (too many of them), last force columns alone in their block, small
# values that decide whether a block counts, and a feature with a value that is not finite
@pytest.mark.parametrize("ma,nlab", [(1, 1), (5, 2), (10, 3), (16, 3), (21, 3), (22, 5), (24, 9),
                                     (32, 4)])
def test_zero_blocks(lk, ma, nlab):
    nm, rep = 6, 70
    X, dX, Q, N = rand_set(nm, ma, rep, nlab, 50 + ma, max(1, ma - 3))
    rng = np.random.default_rng(ma)
    lab = rng.integers(0, nlab + 1, (rep, 2))  # a feature's labels (0: none)
    for m in range(nm):
        on = (lab[:, :1] == Q[m]) | (lab[:, 1:] == Q[m])  # (rep, atom)
        keep = on[None] | np.eye(ma, dtype=bool)[:, None]  # and the centre itself
        dX[m] *= np.repeat(keep, 3, axis=2) * np.where(rng.random((ma, rep, 1)) < 0.3, 1e-9, 1.0)
        dX[m, N[m]:] = 0.0
        dX[m, :, :, 3 * N[m]:] = 0.0
    a = lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.7)
    assert rel_err(a, oracle.hessian_symm(X, dX, Q, N, 1.7)) < TOL
    for _ in range(10):
        np.testing.assert_array_equal(lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.7), a)
    got = lk.kernel_gaussian_full(X[:2], dX[:2], X[1:], dX[1:], Q[:2], Q[1:], N[:2], N[1:], 1.7)
    assert rel_err(got, oracle.full(X[:2], dX[:2], X[1:], dX[1:], Q[:2], Q[1:], N[:2], N[1:],
                                    1.7)) < TOL
    dX[2, 0, 7, 3 * N[2] - 1] = np.inf
    got = lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.7)
    col = int(3 * N[:3].sum()) - 1
    assert not np.isfinite(got[col, col])
    far = np.ones(len(got), bool)
    far[3 * N[:2].sum(): 3 * N[:3].sum()] = False
    np.testing.assert_array_equal(got[np.ix_(far, far)], a[np.ix_(far, far)])


@pytest.mark.parametrize("nm,ma,rep", [(1, 2, 5), (70, 2, 300), (3, 30, 97), (40, 5, 17)])
def test_unused_columns_found_anywhere(lk, nm, ma, rep):
    """A column used by a single entry -- of the last live atom, in the Jacobian only, or of a
    padded atom, which does not count -- in sets of fewer and of more atoms than the first
    look samples."""
    X, dX, Q, N = rand_set(nm, ma, rep, 2, 17 * nm + rep, 1)
    live = np.arange(ma)[None] < N[:, None]
    X[live] *= rng_mask(X[live].shape, 3)
    dX[:, :, rep // 2:] = 0.0
    X[:, :, rep // 2:] = 0.0
    a, i = nm - 1, N[-1] - 1
    dX[a, i, rep - 1, 3 * N[-1] - 1] = 0.7
    X[a, i, rep - 2] = -0.4
    dX[~live] = 0.0
    X[~live, rep - 3] = 9.0
    X[~live, : rep // 2] = 0.0
    got = lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.3)
    assert rel_err(got, oracle.hessian_symm(X, dX, Q, N, 1.3)) < TOL


def rng_mask(shape, seed):
    return (np.random.default_rng(seed).random(shape) < 0.5).astype(np.float64)


def test_refused_scratch(lk):
    """Each device workspace request of a Hessian kernel refused in turn: an error, or the
    result without what the scratch was for (features in several runs)."""
    from kernelforge_amd import capi

    X, dX, Q, N = rand_set(5, 12, 130, 3, 77, 5)
    want = lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.7)
    assert rel_err(want, oracle.hessian_symm(X, dX, Q, N, 1.7)) < TOL
    done = []
    for nth in range(1, 9):
        capi.lib().kf_workspace_refuse(nth)
        try:
            got = lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.7)
        except (MemoryError, RuntimeError):
            got = None
        left = capi.lib().kf_workspace_refuse(0)
        if got is not None:
            assert rel_err(got, want) < TOL
            done.append(left)
    assert done[:1] == [0]  # the last request is one that it can do without
    assert rel_err(lk.kernel_gaussian_hessian_symm(X, dX, Q, N, 1.7), want) < TOL


@pytest.mark.parametrize("nlab2", [3, 2, 1])
def test_matvec_refused_scratch(lk, nlab2):
    """Each workspace request of the matvecs refused in turn: the product goes label by label,
    labels without a partner among them, or the call says that memory is out."""
    from kernelforge_amd import capi

    X1, dX1, Q1, N1 = rand_set(9, 6, 70, 3, 91, 2)
    X2, _, Q2, N2 = rand_set(12, 5, 70, nlab2, 92, 1)
    rng = np.random.default_rng(9)
    ad, aE, s = rng.standard_normal(X2.shape), rng.standard_normal(12), 1.5
    ad[np.arange(5)[None] >= N2[:, None]] = 0.0
    calls = {
        "full": lambda: lk.kernel_gaussian_local_full_matvec(X1, dX1, X2, ad, aE, Q1, Q2, N1, N2, s),
        "forces": lambda: (lk.kernel_gaussian_local_hessian_matvec(X1, dX1, X2, ad, Q1, Q2, N1,
                                                                   N2, s),),
        "energies": lambda: (lk.kernel_gaussian_local_jacobian_t_matvec(X1, X2, ad, Q1, Q2, N1,
                                                                        N2, s),)}
    for name, call in calls.items():
        want, went_on = call(), 0
        for nth in range(1, 6):
            capi.lib().kf_workspace_refuse(nth)
            try:
                got = call()
            except (MemoryError, RuntimeError):
                got = None
            left = capi.lib().kf_workspace_refuse(0)
            if got is not None:
                assert all(rel_err(g, w) < TOL for g, w in zip(got, want)), (name, nth)
                went_on += left == 0
        assert went_on == 3, name  # the plan, the operands and the per-atom sums
