"""GPU parity: FCHL19 descriptors and Jacobians (kf_fchl19_f64) vs the oracle and the
reference golden vectors.  Bar: per-atom relative error <= 1e-12 (tests/helpers.py)."""

import numpy as np
import pytest

import oracle
from tests.helpers import row_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fr():
    from kernelforge_amd import fchl19_repr

    return fchl19_repr


def test_golden_rep_and_grad(fr, golden_fchl19):
    g = golden_fchl19
    for t in range(10):
        rep = fr.generate_fchl_acsf(g[f"coords_{t}"], g[f"z_{t}"])
        assert rep.shape == g[f"rep_{t}"].shape
        assert row_rel_err(rep, g[f"rep_{t}"]) < 1e-12
    for t in range(3):
        rep, grad = fr.generate_fchl_acsf_and_gradients(g[f"gcoords_{t}"], g[f"gz_{t}"])
        assert row_rel_err(rep, g[f"grep_{t}"]) < 1e-12
        assert grad.shape == g[f"ggrad_{t}"].shape
        assert row_rel_err(grad, g[f"ggrad_{t}"]) < 1e-12


def test_golden_nondefault(fr, golden_fchl19):
    from tests.golden.make_golden import NONDEFAULT

    g = golden_fchl19
    assert row_rel_err(fr.generate_fchl_acsf(g["nd_coords"], g["nd_z"], **NONDEFAULT),
                       g["nd_rep"]) < 1e-12
    rep, grad = fr.generate_fchl_acsf_and_gradients(g["nd_coords"], g["nd_z"], **NONDEFAULT)
    assert row_rel_err(rep, g["nd_grep"]) < 1e-12
    assert row_rel_err(grad, g["nd_ggrad"]) < 1e-12


def test_batch_config0_vs_oracle(fr, config0):
    _, _, _, C, Q, N = config0
    X = fr.generate_fchl_acsf_batch(C, Q, N)
    Xo = oracle.fchl19_batch(C, Q, N)
    assert X.shape == Xo.shape == (1000, 23, 720)
    assert row_rel_err(X, Xo, lead=2) < 1e-12


def test_batch_gradients_vs_oracle(fr, config0):
    _, _, _, C, Q, N = config0
    sl = slice(0, 40)
    X, dX = fr.generate_fchl_acsf_batch(C[sl], Q[sl], N[sl], with_gradients=True)
    Xo, dXo = oracle.fchl19_batch(C[sl], Q[sl], N[sl], grad=True)
    assert dX.shape == dXo.shape
    assert row_rel_err(X, Xo, lead=2) < 1e-12
    assert row_rel_err(dX, dXo, lead=2) < 1e-12


@pytest.mark.parametrize("kw", [dict(nFourier=2), dict(nRs2=10, nRs3=7, rcut=3.0, acut=2.6),
                                dict(three_body_weight=0.0), dict(elements=[1, 6, 7, 8, 16, 9])])
def test_parameter_variants(fr, config0, kw):
    coords, zs, *_ = config0
    for m in range(4):
        assert row_rel_err(fr.generate_fchl_acsf(coords[m], zs[m], **kw),
                           oracle.fchl19(coords[m], zs[m], **kw)) < 1e-12
        r, g = fr.generate_fchl_acsf_and_gradients(coords[m], zs[m], **kw)
        ro, go = oracle.fchl19(coords[m], zs[m], grad=True, **kw)
        assert row_rel_err(r, ro) < 1e-12
        assert row_rel_err(g, go) < 1e-12


def test_flat_coords_and_errors(fr, config0):
    coords, zs, *_ = config0
    a = fr.generate_fchl_acsf(coords[0], zs[0])
    b = fr.generate_fchl_acsf(coords[0].reshape(-1), zs[0])
    np.testing.assert_array_equal(a, b)
    with pytest.raises(RuntimeError):
        fr.generate_fchl_acsf(coords[0], np.full(len(zs[0]), 9, np.int32))
    with pytest.raises(ValueError):
        fr.generate_fchl_acsf(np.zeros((0, 3)), np.zeros(0, np.int32))
    with pytest.raises(ValueError):
        fr.generate_fchl_acsf(np.zeros((4, 2)), np.ones(4, np.int32))
    assert fr.compute_rep_size(5, 24, 20, 2) == 720


def test_c_abi_device_resident(config0):
    from kernelforge_amd import capi

    _, _, _, C, Q, N = config0
    ma = Q.shape[1]
    dC = capi.DeviceArray.from_numpy(C[:64])
    dQ = capi.DeviceArray.from_numpy(Q[:64])
    dN = capi.DeviceArray.from_numpy(N[:64])
    X = capi.DeviceArray((64, ma, 720))
    dX = capi.DeviceArray((64, ma, 720, 3 * ma))
    capi.fchl19(dC.ptr, dQ.ptr, dN.ptr, 64, ma, X.ptr, dX.ptr)
    capi.synchronize()
    Xo, dXo = oracle.fchl19_batch(C[:64], Q[:64], N[:64], grad=True)
    assert row_rel_err(X.numpy(), Xo, lead=2) < 1e-12
    assert row_rel_err(dX.numpy(), dXo, lead=2) < 1e-12


# (atoms of the largest molecule, molecules, parameters): one atom to the most whose pair
# records fit in LDS, batches that share a centre among 8, 2 and 1 work-groups, feature
# blocks that do not fill a tile and ones that take several
@pytest.mark.parametrize("ma,nm,kw", [
    (1, 3, {}), (2, 1, {}), (3, 5, dict(nFourier=3)), (9, 40, dict(nRs2=41, nRs3=37)),
    (13, 70, dict(nRs2=3, nRs3=1, nFourier=8)), (32, 2, dict(elements=[8])), (44, 1, {})])
def test_jacobian_kernel_edges(fr, ma, nm, kw):
    from kernelforge_amd import synthetic

    rng = np.random.default_rng(100 * ma + nm)
    el = np.array(kw.get("elements", [1, 6, 7, 8, 16]))
    Ns = np.concatenate([[ma], rng.integers(1, ma + 1, nm - 1)]).astype(int)
    C, Q, N = synthetic.pad_batch([synthetic._place_atoms(rng, n) for n in Ns],
                                  [rng.choice(el, n).astype(np.int32) for n in Ns])
    X, dX = fr.generate_fchl_acsf_batch(C, Q, N, with_gradients=True, **kw)
    Xo, dXo = oracle.fchl19_batch(C, Q, N, grad=True, **kw)
    assert row_rel_err(X, Xo, lead=2) < 1e-12
    assert row_rel_err(dX, dXo, lead=2) < 1e-12


# float32 results are the FP64 ones rounded: rows whose blocks are and are not whole 16-byte
# words, and sizes that the float32 entry point leaves to the FP64 one
@pytest.mark.parametrize("ma,nm,grad,kw", [
    (1, 2, True, {}), (9, 30, True, dict(nRs2=41, nRs3=37)), (12, 3, True, dict(nRs3=3)),
    (45, 1, True, {}), (3, 700, False, dict(nRs3=1)), (23, 20, False, {}), (47, 3, False, {})])
def test_float32_results(fr, ma, nm, grad, kw):
    from kernelforge_amd import capi, synthetic

    rng = np.random.default_rng(7 * ma + nm)
    Ns = np.concatenate([[ma], rng.integers(1, ma + 1, nm - 1)]).astype(int)
    C, Q, N = synthetic.pad_batch([synthetic._place_atoms(rng, n) for n in Ns],
                                  [rng.choice([1, 6, 7, 8, 16], n).astype(np.int32) for n in Ns])
    p = dict(nRs2=24, nRs3=20) | kw
    rep = capi.rep_size(5, p["nRs2"], p["nRs3"], 2)
    Cd, Qd, Nd = (capi.DeviceArray.from_numpy(a) for a in (C, Q.astype(np.int32), N.astype(np.int32)))
    out = []
    for f32 in (False, True):
        X = capi.DeviceArray((nm, ma, rep), np.float32 if f32 else np.float64)
        J = capi.DeviceArray((nm, ma, rep, 3 * ma), X.dtype) if grad else None
        if f32 and not capi.lib().kf_fchl19_f32_fits(ma, 5, p["nRs2"], p["nRs3"], 2, int(grad)):
            with pytest.raises(ValueError):
                capi.fchl19(Cd.ptr, Qd.ptr, Nd.ptr, nm, ma, X.ptr, J.ptr if grad else 0, f32=True, **p)
            return
        capi.fchl19(Cd.ptr, Qd.ptr, Nd.ptr, nm, ma, X.ptr, J.ptr if grad else 0, f32=f32, **p)
        capi.synchronize()
        out.append([X.numpy()] + ([J.numpy()] if grad else []))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a.astype(np.float32), b)


# one atom to more than the pair storage holds in one go (47 atoms: 1,035 pairs a centre),
# batches of a few centres, one radial term left over per thread, many angular terms (a
# smaller pair storage: several chunks from 21 atoms on), one element, work-groups sharing
# a molecule
@pytest.mark.parametrize("ma,nm,kw", [
    (1, 2, {}), (2, 1, {}), (3, 1500, dict(nRs3=1)), (8, 130, dict(nRs2=41, nRs3=37)),
    (23, 1, dict(nFourier=8, nRs3=7)), (47, 3, {}), (60, 2, dict(elements=[8], nRs3=3))])
def test_representation_kernel_edges(fr, ma, nm, kw):
    from kernelforge_amd import synthetic

    rng = np.random.default_rng(10 * ma + nm)
    el = np.array(kw.get("elements", [1, 6, 7, 8, 16]))
    Ns = np.concatenate([[ma], rng.integers(1, ma + 1, nm - 1)]).astype(int)
    C, Q, N = synthetic.pad_batch([synthetic._place_atoms(rng, n) for n in Ns],
                                  [rng.choice(el, n).astype(np.int32) for n in Ns])
    X = fr.generate_fchl_acsf_batch(C, Q, N, **kw)
    assert row_rel_err(X, oracle.fchl19_batch(C, Q, N, **kw), lead=2) < 1e-12


# molecules whose items are shared by 2 to 64 lanes: of few elements and radial terms, at the
# sizes where the number of lanes changes, and centres whose pairs take several chunks, with
# channels that end inside one and absent elements; a chunk's pairs with no sharing (16 elements)
@pytest.mark.parametrize("ma,nm,kw", [
    (13, 3, dict(elements=[8], nRs3=3)), (22, 600, dict(elements=[8])),
    (31, 40, dict(elements=[1, 8])), (47, 3, dict(elements=[6], nRs3=1)),
    (66, 2, dict(elements=[1, 6, 7], nFourier=3)), (101, 1, dict(elements=[1, 6])),
    (128, 2, {}), (128, 1, dict(elements=[1], nRs3=7)), (50, 1, dict(elements=list(range(1, 17))))])
def test_representation_long_molecules(fr, ma, nm, kw):
    test_representation_kernel_edges(fr, ma, nm, kw)
    if len(kw.get("elements", [])) > 1:  # one of the elements absent
        from kernelforge_amd import synthetic

        rng = np.random.default_rng(ma)
        z = rng.choice(kw["elements"][1:], ma).astype(np.int32)
        C, Q, N = synthetic.pad_batch([synthetic._place_atoms(rng, ma)], [z])
        assert row_rel_err(fr.generate_fchl_acsf_batch(C, Q, N, **kw),
                           oracle.fchl19_batch(C, Q, N, **kw), lead=2) < 1e-12


# small molecules in batches that fill the GPU, a wave per centre: none, one and some
# neighbours, blocks of absent elements on end, alone and at the end of a row
@pytest.mark.parametrize("ma,nm,kw", [
    (1, 1100, {}), (2, 700, dict(elements=[1, 8])), (2, 600, {}), (3, 400, dict(nRs2=3, nRs3=1)),
    (4, 300, dict(nRs2=41, nRs3=37)), (7, 160, dict(nFourier=3)), (10, 110, {})])
def test_jacobian_small_molecules(fr, ma, nm, kw):
    test_jacobian_kernel_edges(fr, ma, nm, kw)
    test_float32_results(fr, ma, nm, True, {k: v for k, v in kw.items() if k.startswith("nRs")})
