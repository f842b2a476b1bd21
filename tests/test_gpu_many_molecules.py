"""Calls on more molecules or atoms than a grid has threads for one work-group each (2^32
threads; 2^24 work-groups of 256): small descriptors, checked in closed form or against the
oracle on both ends of the set."""

import numpy as np
import pytest

import oracle
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

MANY = (1 << 24) + 4321


@pytest.mark.parametrize("nm2", [2, 3])
def test_rect_kernel_many_molecules(nm2):
    """One-atom molecules, below (2) and above (3) the matched pairs of the packing-free
    form, with one value each in the first or in the second 16 columns: every entry is
    exp(-(x - y)^2 / 2) or, in different columns, exp(-(x^2 + y^2) / 2)."""
    from kernelforge_amd import capi

    rng = np.random.default_rng(nm2)
    rep = 17
    x, y = rng.standard_normal(MANY), rng.standard_normal(nm2)
    cx, cy = np.arange(MANY) % 3 == 1, np.arange(nm2) % 2 == 1  # in column 16
    X, Y = np.zeros((MANY, rep)), np.zeros((nm2, rep))
    X[~cx, 0], X[cx, 16], Y[~cy, 0], Y[cy, 16] = x[~cx], x[cx], y[~cy], y[cy]
    DA = capi.DeviceArray
    one = lambda n: DA.from_numpy(np.ones(n, np.int32))
    dx, dy, K = DA.from_numpy(X), DA.from_numpy(Y), DA((MANY, nm2))
    q1, n1, q2, n2 = one(MANY), one(MANY), one(nm2), one(nm2)
    capi.check(capi.lib().kf_local_kernel(capi.KF_PREC_F64, dx.ptr, dy.ptr, q1.ptr, q2.ptr,
                                          n1.ptr, n2.ptr, MANY, nm2, 1, 1, rep, 1.0, K.ptr,
                                          None),
               "kf_local_kernel")
    capi.synchronize()
    cross = np.where(cx[:, None] == cy[None], 2.0 * x[:, None] * y[None], 0.0)
    want = np.exp(-0.5 * (x[:, None] ** 2 + y[None] ** 2 - cross))
    # x^2 + y^2 - 2 x y in the exponent, |x|, |y| < 6
    assert np.abs(K.numpy() - want).max() < 1e-13


def test_matvec_many_molecules():
    """E and F of one-atom query molecules with one descriptor value and unit Jacobians:
    E = sum_j e_j (aE_j + d_j ad_j), F = dE/dx.  Every third has no partner."""
    from kernelforge_amd import capi

    rng = np.random.default_rng(5)
    x, y, ad, aE = rng.standard_normal(MANY), *rng.standard_normal((3, 2))
    q = np.where(np.arange(MANY) % 3 == 2, 7, 1).astype(np.int32)
    DA = capi.DeviceArray
    dX = np.zeros((MANY, 3))
    dX[:, 1] = 1.0
    dq1, dn1 = DA.from_numpy(q), DA.from_numpy(np.ones(MANY, np.int32))
    dq2, dn2 = DA.from_numpy(np.ones(2, np.int32)), DA.from_numpy(np.ones(2, np.int32))
    dx, ddx, dy, dad, dae = (DA.from_numpy(a) for a in (x, dX, y, ad, aE))
    E, F = DA(MANY), DA((MANY, 3))
    capi.check(capi.lib().kf_local_full_matvec(dx.ptr, ddx.ptr, dy.ptr, dad.ptr, dae.ptr, dq1.ptr,
                                               dq2.ptr, dn1.ptr, dn2.ptr, MANY, 2, 1, 1, 1, 1.0,
                                               E.ptr, F.ptr, None), "kf_local_full_matvec")
    capi.synchronize()
    d = x[:, None] - y[None]
    e = np.exp(-0.5 * d * d) * (q == 1)[:, None]
    assert rel_err(E.numpy(), (e * (aE + d * ad)).sum(1)) < 1e-12
    # the force rows: c ad - (e inner) d - c aE d with sigma = 1
    G = (e * (ad - d * ad * d - aE * d)).sum(1)
    got = F.numpy()
    assert rel_err(got[:, 1], G) < 1e-12
    assert not got[:, 0].any() and not got[:, 2].any()


def test_derivative_kernel_many_atoms():
    """A Jacobian kernel whose first set has more atom rows than work-groups fit: the column
    scan of a padded set."""
    from kernelforge_amd import capi

    nm, ma, rep = MANY // 23 + 50, 23, 3
    rng = np.random.default_rng(8)
    X1 = rng.standard_normal((nm, ma, rep)) * 0.3
    X1[..., 1] = 0.0
    X1[-1, 1, 1] = 0.4  # a column used by one of the last atoms only
    Q1 = rng.integers(1, 3, (nm, ma)).astype(np.int32)
    N1 = np.full(nm, 2, np.int32)
    X2, dX2 = rng.standard_normal((2, 2, rep)) * 0.3, rng.standard_normal((2, 2, rep, 6)) * 0.2
    dX2[:, :, 1] = 0.0
    X2[..., 1] = 0.0
    Q2, N2 = rng.integers(1, 3, (2, 2)).astype(np.int32), np.full(2, 2, np.int32)
    DA = capi.DeviceArray
    dev = [DA.from_numpy(a) for a in (X1, X2, dX2, Q1, Q2, N1, N2)]
    K = DA((nm, 12))
    capi.check(capi.lib().kf_local_kernel_jacobian(*(d.ptr for d in dev), nm, 2, ma, 2, rep, 1.2,
                                                   K.ptr, None), "kf_local_kernel_jacobian")
    capi.synchronize()
    got = K.numpy()
    for s in (slice(0, 40), slice(nm - 40, nm)):
        want = oracle.jacobian(X1[s], X2, dX2, Q1[s], Q2, N1[s], N2, 1.2)
        assert rel_err(got[s], want) < 1e-10
