"""The work that programs on this framework spend their GPU time on, as cases to time.

`listed()` has one case for each kind of call at a size it is used at, `draw()` gives more of
the same kinds over their whole ranges.  `prepare()` makes what a program has in hand before
the call (descriptors, kernels, a model or a matvec plan), `run()` is the call itself through
the public entry points (the torch modules, the C ABI through `capi`, and the model layer),
`exact()` is the same result from plain torch in float64.

Molecules follow `kernelforge_amd.synthetic`: 5-23 atoms of H, C, N, O, S for the ragged
sets, conformers of one molecule (Gaussian displacements of 0.05 Angstrom) for energy and
force models; they are drawn here by a vectorised form of the same rule, since thousands are
needed per case.
"""

import ctypes
import math

import numpy as np
import torch  # before any module that loads the library

from kernelforge_amd import capi, cuda_fchl19_repr, cuda_local_kernels

ELEMENTS = (1, 6, 7, 8, 16)
ELEMENT_P = (0.5, 0.3, 0.1, 0.08, 0.02)
SIGMA = 2.0
REP = 720
# mean atoms of a ragged molecule (uniform 5..23) and of each label in it
MEAN_ATOMS = 14.0
# descriptor columns that are not zero: 16-wide windows that two rows of one label share in
# the ragged sets, and columns of a C/H/O molecule
RAGGED_FILL, CONFORMER_FILL = 0.465, 312.0 / 720.0


def listed():
    return [
        # one molecular-dynamics step: descriptors and Jacobian of the new geometry, then
        # energy and forces from a trained model; bound by launches and latency
        {"name": "md_step_21x200", "kind": "md_step", "atoms": 21, "train": 200, "dtype": "f64"},
        # descriptors of a whole training set (the energy fit's first stage)
        {"name": "descriptors_20000", "kind": "descriptors", "mols": 20000, "dtype": "f64"},
        # descriptors and Jacobians of a conformer set (the energy+force fit's first stage)
        {"name": "jacobians_500x21", "kind": "jacobians", "mols": 500, "atoms": 21,
         "dtype": "f64"},
        # the training kernel of a small energy model, and of the benchmark's large one
        {"name": "symm_800", "kind": "symm", "mols": 800, "dtype": "f64"},
        {"name": "symm_20000", "kind": "symm", "mols": 20000, "dtype": "f64"},
        # energies of new molecules from a large energy model
        {"name": "rect_333x10000", "kind": "rect", "query": 333, "train": 10000, "dtype": "f64"},
        # the training kernel of an energy+force model of one molecule
        {"name": "ef_kernel_200x21", "kind": "ef_kernel", "mols": 200, "atoms": 21,
         "form": "full", "dtype": "f64"},
        # the force-only training kernel of a small mixed set (ragged atom counts)
        {"name": "force_kernel_ragged_37", "kind": "ef_kernel", "mols": 37, "atoms": 0,
         "form": "hessian", "dtype": "f64"},
        # the regularised solve of a small model (several property columns) and of the large one
        {"name": "solve_1501x3", "kind": "solve", "order": 1501, "nrhs": 3},
        {"name": "solve_20000", "kind": "solve", "order": 20000, "nrhs": 1},
        # energies and forces of a batch of conformers from an energy+force model, in the
        # single precision that callers of the torch modules keep their tensors in
        {"name": "predict_ef_100x1000", "kind": "predict_ef", "query": 100, "train": 1000,
         "atoms": 21, "dtype": "f32"},
        # the model layer's prediction, host arrays in and out
        {"name": "model_predict_8x150", "kind": "model_predict", "query": 8, "train": 150},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["md_step", "descriptors", "jacobians", "symm", "symm", "rect", "ef_kernel",
                       "ef_kernel", "solve", "solve", "predict_ef", "model_predict"])
    dtype = rng.choice(["f64", "f64", "f32"])
    if kind == "md_step":
        return {"kind": kind, "atoms": rng.randint(5, 30), "train": _log(rng, 20, 1000),
                "dtype": dtype}
    if kind == "descriptors":
        return {"kind": kind, "mols": _log(rng, 1, 20000), "dtype": dtype}
    if kind == "jacobians":
        return {"kind": kind, "mols": _log(rng, 1, 500), "atoms": rng.choice([0, rng.randint(5, 23)]),
                "dtype": dtype}
    if kind == "symm":
        return {"kind": kind, "mols": _log(rng, 50, 12000), "dtype": dtype}
    if kind == "rect":
        return {"kind": kind, "query": _log(rng, 1, 2000), "train": _log(rng, 100, 12000),
                "dtype": "f64"}
    if kind == "ef_kernel":
        return {"kind": kind, "mols": _log(rng, 4, 200), "atoms": rng.choice([0, rng.randint(5, 23)]),
                "form": rng.choice(["full", "full", "hessian"]), "dtype": "f64"}
    if kind == "solve":
        return {"kind": kind, "order": _log(rng, 100, 20000), "nrhs": rng.choice([1, 1, 2, 5])}
    if kind == "predict_ef":
        return {"kind": kind, "query": _log(rng, 1, 200), "train": _log(rng, 20, 1000),
                "atoms": rng.randint(5, 23), "dtype": dtype}
    return {"kind": kind, "query": _log(rng, 1, 10), "train": _log(rng, 20, 150)}


# ---------------------------------------------------------------- inputs


def _molecules(n_mols, rng, counts=None):
    """Padded coordinates (nm, max, 3), charges and atom counts: atoms placed one at a time in
    a box of 1.6 n^(1/3) Angstrom, redrawn while closer than 0.9 Angstrom to a placed one.
    The counts of a set are the same for every seed, in another order, so that the outputs
    of a case have one size."""
    if counts is None:
        n = rng.permutation(np.random.default_rng(n_mols).integers(5, 24, n_mols))
    else:
        n = np.full(n_mols, counts)
    ma = int(n.max())
    side = 1.6 * n ** (1.0 / 3.0)
    C = np.zeros((n_mols, ma, 3))
    for k in range(ma):
        todo = np.nonzero(n > k)[0]
        while todo.size:
            p = rng.uniform(size=(todo.size, 3)) * side[todo, None]
            d2 = ((C[todo, :k] - p[:, None]) ** 2).sum(-1)
            ok = (d2 >= 0.81).all(1)
            C[todo[ok], k] = p[ok]
            todo = todo[~ok]
    live = np.arange(ma)[None] < n[:, None]
    Z = np.where(live, rng.choice(np.array(ELEMENTS), (n_mols, ma), p=ELEMENT_P), 0)
    return C, Z.astype(np.int32), n.astype(np.int32)


def _conformers(n_conf, atoms, rng):
    """Conformers of one H/C/O molecule."""
    C, _, _ = _molecules(1, rng, atoms)
    z = np.sort(rng.choice(np.array([1, 6, 8]), atoms, p=[0.4, 0.4, 0.2])).astype(np.int32)
    C = C + rng.normal(0.0, 0.05, (n_conf, atoms, 3))
    return C, np.tile(z, (n_conf, 1)), np.full(n_conf, atoms, np.int32)


def _sets(case, seed):
    """(coordinates, charges, counts) of the case's training (or only) set and of its query
    set, as NumPy arrays."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    nt = case.get("mols", case.get("train", 0))
    nq = 1 if kind == "md_step" else case.get("query", 0)
    if case.get("atoms", 0):
        C, Z, N = _conformers(nt + nq, case["atoms"], rng)
    else:
        C, Z, N = _molecules(nt, rng)
        if nq:
            return rng, (C, Z, N), _molecules(nq, rng)
    return rng, (C[:nt], Z[:nt], N[:nt]), (C[nt:], Z[nt:], N[nt:])


def _gpu(a, dtype=None):
    return torch.as_tensor(a, device="cuda", dtype=dtype)


def _index(Z):
    """Element indices, as the torch descriptor module takes them."""
    lut = np.zeros(32, np.int32)
    lut[list(ELEMENTS)] = np.arange(len(ELEMENTS))
    return lut[Z]


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.float64


def _describe(S, dtype, grad):
    """Labels, counts, descriptors (and Jacobians) of a set on the GPU."""
    C, Z, N = S
    Q, N = _gpu(_index(Z)), _gpu(N)
    C = _gpu(C, dtype)
    if not grad:
        return Q, N, cuda_fchl19_repr.generate_fchl_acsf(C, Q, N, len(ELEMENTS)), None
    X, dX = cuda_fchl19_repr.generate_fchl_acsf_and_gradients(C, Q, N, len(ELEMENTS))
    return Q, N, X, dX


def _alphas(rng, nt, naq):
    """Weights of a trained energy+force model."""
    return rng.normal(0.0, 0.1, nt), rng.normal(0.0, 0.01, naq)


def _rfp_system(order, seed):
    """A kernel matrix of `order` points in RFP (TRANSR='N', UPLO='U') as the solver takes it,
    dense and packed: the Gaussian kernel of random points, well above the rounding noise."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    P = torch.rand((order, 12), generator=g, device="cuda", dtype=torch.float64)
    sq = (P * P).sum(1)
    D = (sq[:, None] + sq[None] - 2.0 * (P @ P.T)).clamp_(min=0.0)
    K = torch.exp_(D.mul_(-2.0))
    K.diagonal().fill_(1.0)
    return K


def _to_rfp_u(A):
    """Lower triangle of A as an RFP array, TRANSR='N', UPLO='U' (its transpose's upper)."""
    n = A.shape[0]
    k, s = n // 2, n + (n % 2 == 0)
    M = torch.zeros((n - k, s), dtype=A.dtype, device=A.device)
    M[:, :n] = torch.tril(A[k:], k)
    if k:
        M[:k, k + 1:k + 1 + k] += torch.triu(A[:k, :k].T)
    return M.reshape(-1)


def _to_rfp_l(A):
    """Lower triangle of A as an RFP array, TRANSR='N', UPLO='L'."""
    n = A.shape[0]
    k = n // 2
    n1, off = n - k, int(n % 2 == 0)
    s = n + off
    M = torch.zeros((n1, s), dtype=A.dtype, device=A.device)
    M[:, off:] = torch.tril(A).T[:n1]
    if k:
        c0 = 1 - off  # the trailing triangle, transposed, fills the columns from c0 on
        M[c0:c0 + k, :k] += torch.tril(A[n1:, n1:])
    return M.reshape(-1)


class _Plan:
    """A matvec plan of the C ABI with its output buffers."""

    def __init__(self, Q, N, Xt, ad, aE, Qt, Nt):
        nt, ma, rep = Xt.shape
        h = ctypes.c_void_p()
        capi.check(capi.lib().kf_matvec_plan_create(
            Q.data_ptr(), N.data_ptr(), 1, ma, Xt.data_ptr(), ad.data_ptr(), aE.data_ptr(),
            Qt.data_ptr(), Nt.data_ptr(), nt, ma, rep, SIGMA, ctypes.byref(h),
            torch.cuda.current_stream().cuda_stream), "kf_matvec_plan_create")
        self.handle = h.value

    def __del__(self):
        torch.cuda.synchronize()
        capi.lib().kf_matvec_plan_destroy(self.handle)


def prepare(case, seed):
    kind, dt = case["kind"], _dtype(case)
    if kind == "solve":
        K = _rfp_system(case["order"], seed)
        rng = np.random.default_rng(seed)
        y = _gpu(rng.normal(size=(case["nrhs"], case["order"])))
        arf = _to_rfp_u(K)
        return {"case": case, "arf": arf, "y": y, "work": torch.empty_like(arf),
                "alpha": torch.empty_like(y)}
    rng, T, S = _sets(case, seed)
    if kind in ("descriptors", "jacobians"):
        C, Z, N = T
        return {"case": case, "C": _gpu(C, dt), "Q": _gpu(_index(Z)), "N": _gpu(N)}
    if kind == "model_predict":
        from kernelforge_amd import synthetic
        from kernelforge_amd.krr import LocalKRRModel

        def lists(S):
            return [c[:n] for c, n in zip(S[0], S[2])], [z[:n] for z, n in zip(S[1], S[2])]

        coords, zs = lists(T)
        E = np.array([synthetic.molecule_energy(c, z) for c, z in zip(coords, zs)])
        model = LocalKRRModel(sigma=SIGMA, l2=1e-6).fit(coords, zs, energies=E)
        q = lists(S)
        return {"case": case, "model": model, "coords": q[0], "zs": q[1]}
    grad = kind in ("ef_kernel", "md_step", "predict_ef")
    Qt, Nt, Xt, dXt = _describe(T, dt, grad)
    st = {"case": case, "Qt": Qt, "Nt": Nt, "Xt": Xt}
    if kind == "rect":
        st["Q"], st["N"], st["X"], _ = _describe(S, dt, False)
    if kind == "ef_kernel":
        st["dXt"] = dXt.reshape(*dXt.shape[:3], -1)
        st["naq"] = 3 * int(T[2].sum())
    if kind in ("md_step", "predict_ef"):
        aE, aF = _alphas(rng, case["train"], 3 * int(T[2].sum()))
        st["aE"] = _gpu(aE, dt)
        st["ad"] = cuda_local_kernels.compute_alpha_desc(dXt, Nt, _gpu(aF, dt))
        st["C"], st["Q"], st["N"] = _gpu(S[0], dt), _gpu(_index(S[1])), _gpu(S[2])
    if kind == "md_step":
        f64 = [t.to(torch.float64) for t in (Xt, st["ad"], st["aE"])]
        st["plan"] = _Plan(st["Q"], st["N"], *f64, Qt, Nt)
        st["E"] = torch.empty(1, dtype=torch.float64, device="cuda")
        st["F"] = torch.empty(3 * case["atoms"], dtype=torch.float64, device="cuda")
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    ne = len(ELEMENTS)
    if kind == "descriptors":
        return cuda_fchl19_repr.generate_fchl_acsf(st["C"], st["Q"], st["N"], ne)
    if kind == "jacobians":
        return cuda_fchl19_repr.generate_fchl_acsf_and_gradients(st["C"], st["Q"], st["N"], ne)
    if kind == "symm":
        return cuda_local_kernels.kernel_gaussian_symm_rfp(st["Xt"], st["Qt"], st["Nt"], SIGMA)
    if kind == "rect":
        return cuda_local_kernels.kernel_gaussian_rect(st["X"], st["Q"], st["N"], st["Xt"],
                                                       st["Qt"], st["Nt"], SIGMA)
    if kind == "ef_kernel" and case["form"] == "full":
        return cuda_local_kernels.kernel_gaussian_full_symm_rfp(st["Xt"], st["dXt"], st["Qt"],
                                                                st["Nt"], SIGMA)
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "ef_kernel":
        X, naq = st["Xt"], st["naq"]
        nm, ma, rep = X.shape
        K = torch.empty(naq * (naq + 1) // 2, dtype=torch.float64, device="cuda")
        capi.check(capi.lib().kf_local_kernel_hessian_symm_rfp(
            X.data_ptr(), st["dXt"].data_ptr(), st["Qt"].data_ptr(), st["Nt"].data_ptr(), nm, ma,
            rep, SIGMA, K.data_ptr(), stream), "kf_local_kernel_hessian_symm_rfp")
        return K
    if kind == "solve":
        n, nrhs = case["order"], case["nrhs"]
        st["work"].copy_(st["arf"])
        st["alpha"].copy_(st["y"])
        capi.rfp_potrf(capi.KF_PREC_F64, st["work"].data_ptr(), n, 1e-8, stream)
        capi.rfp_potrs(capi.KF_PREC_F64, st["work"].data_ptr(), n, st["alpha"].data_ptr(), nrhs,
                       stream)
        return st["alpha"], st["work"]
    if kind == "predict_ef":
        X, dX = cuda_fchl19_repr.generate_fchl_acsf_and_gradients(st["C"], st["Q"], st["N"], ne)
        return cuda_local_kernels.kernel_gaussian_full_matvec(
            X, dX, st["Q"], st["N"], st["Xt"], st["Qt"], st["Nt"], st["aE"], st["ad"], SIGMA)
    if kind == "md_step":
        X, dX = cuda_fchl19_repr.generate_fchl_acsf_and_gradients_md_single(
            st["C"], st["Q"], st["N"], ne)
        X, dX = X.to(torch.float64), dX.to(torch.float64)
        capi.check(capi.lib().kf_matvec_plan_execute(
            st["plan"].handle, X.data_ptr(), dX.data_ptr(), st["E"].data_ptr(),
            st["F"].data_ptr(), stream), "kf_matvec_plan_execute")
        return st["E"], st["F"]
    return st["model"].predict(st["coords"], st["zs"])


# ---------------------------------------------------------------- work


def work(case):
    """Bytes and flops that a pass cannot do without: operands read and results written once,
    products over the descriptor columns that are not zero."""
    kind = case["kind"]
    b = 4 if case.get("dtype") == "f32" else 8
    atoms = case.get("atoms", 0) or MEAN_ATOMS
    fill = CONFORMER_FILL if case.get("atoms", 0) else RAGGED_FILL
    p2 = sum(p * p for p in ELEMENT_P) if not case.get("atoms", 0) else 0.36
    trip = atoms * (atoms - 1) * (atoms - 2) / 2
    xrow, pad = REP * b, atoms if case.get("atoms", 0) else 23
    # a triplet costs about 20 exponentials of some 15 operations and 40 products
    desc = trip * 20 * 20
    jac = trip * 40 * 9 * 2
    if kind == "descriptors":
        return {"bytes": case["mols"] * 23 * xrow, "flops": case["mols"] * desc}
    if kind == "jacobians":
        return {"bytes": case["mols"] * pad * xrow * (1 + 3 * pad),
                "flops": case["mols"] * (desc + jac)}
    if kind == "symm":
        n = case["mols"]
        return {"bytes": n * MEAN_ATOMS * xrow + n * (n + 1) / 2 * b,
                "flops": REP * fill * p2 * (n * MEAN_ATOMS) ** 2}
    if kind == "rect":
        n1, n2 = case["query"], case["train"]
        return {"bytes": (n1 + n2) * MEAN_ATOMS * xrow + n1 * n2 * b,
                "flops": 2 * REP * fill * p2 * n1 * n2 * MEAN_ATOMS ** 2}
    if kind == "ef_kernel":
        n, nc, f = case["mols"], 3 * atoms, REP * fill
        matched = p2 * atoms * atoms
        pair = matched * (6 * f * nc + 2 * nc * nc) + atoms * 2 * nc * nc * f
        order = n * (nc + (case["form"] == "full"))
        return {"bytes": n * atoms * f * b * (1 + nc) + order * (order + 1) / 2 * b,
                "flops": pair * n * (n + 1) / 2}
    if kind == "solve":
        n, r = case["order"], case["nrhs"]
        return {"bytes": n * (n + 1) * 8.0 + 2 * n * r * 8, "flops": n ** 3 / 3 + 2.0 * n * n * r}
    nq, nt = case.get("query", 1), case["train"]
    product = 2 * REP * fill * p2 * atoms * atoms * nq * nt
    if kind == "model_predict":
        return {"bytes": (nq + nt) * atoms * REP * 8, "flops": 2 * product + nq * (desc + jac)}
    # E and F: the products with the training rows and their weights, and back to rows
    return {"bytes": nq * atoms * 3 * 8 * 2 + 2 * nt * atoms * REP * fill * b,
            "flops": 4 * product + nq * (desc + jac + atoms * 2 * REP * fill * 3 * atoms)}


# ---------------------------------------------------------------- exact values


def _rep_exact(R, E, L):
    """FCHL19 (default parameters) of coordinates R (B, n, 3), element one-hots E (B, n, 5) and
    live atoms L (B, n): (B, n, 720), by plain torch operations."""
    B, n, _ = R.shape
    dev = R.device
    eye = torch.eye(n, dtype=torch.float64, device=dev)
    u = R[:, None, :, :] - R[:, :, None, :]  # u[i, j] = R_j - R_i
    D = torch.sqrt((u * u).sum(-1) + eye)
    pair = L[:, :, None] & L[:, None, :] & (eye == 0) & (D <= 8.0)
    D = torch.where(pair, D, torch.ones_like(D))
    f = torch.where(pair, 0.5 * (torch.cos(math.pi * D / 8.0) + 1.0), torch.zeros_like(D))
    Rs2 = torch.arange(1, 25, dtype=torch.float64, device=dev) * (8.0 / 24)
    Rs3 = torch.arange(1, 21, dtype=torch.float64, device=dev) * (8.0 / 20)
    s2 = torch.log1p(0.32 / (D * D))
    l = torch.log(Rs2) - (torch.log(D) - 0.5 * s2)[..., None]
    g = (f / (torch.sqrt(s2) * math.sqrt(2 * math.pi) * D ** 1.8))[..., None] \
        * torch.exp(-0.5 * l * l / s2[..., None]) / Rs2
    two = torch.einsum("bijk,bje->biek", g, E).reshape(B, n, 120)
    # triplets: centre i, neighbours j < k
    up = torch.triu(torch.ones((n, n), dtype=torch.bool, device=dev), 1)
    live3 = pair[:, :, :, None] & pair[:, :, None, :] & up
    Dij, Dik, Djk = D[:, :, :, None], D[:, :, None, :], D[:, None, :, :]
    # Djk may exceed the cutoff: it needs its own value
    Djk = torch.sqrt((u * u).sum(-1) + eye)[:, None]
    uv = torch.einsum("bijt,bikt->bijk", u, u)
    uw = uv - (u * u).sum(-1)[:, :, :, None]  # (R_j - R_i).(R_k - R_j)
    vw = (u * u).sum(-1)[:, :, None, :] - uv  # (R_k - R_i).(R_k - R_j)
    one = torch.ones_like(uv)
    ci = torch.where(live3, uv / (Dij * Dik), 0.5 * one)
    cj, ck = -uw / (Dij * Djk), vw / (Dik * Djk)
    w3 = math.sqrt(2.7 / math.pi) * 13.4
    amp = (1.0 + 3.0 * ci * cj * ck) * w3 * (Dij * Dik * Djk) ** -0.57 * f[:, :, :, None] * f[:, :, None, :]
    amp = torch.where(live3, amp, torch.zeros_like(amp))
    w = 2.0 * math.exp(-0.5 * math.pi ** 2)
    ang = torch.stack([w * ci, w * torch.sqrt(1.0 - ci * ci)], -1)
    rad = torch.exp(-2.7 * (0.5 * (Dij + Dik)[..., None] - Rs3) ** 2) * amp[..., None]
    chan = torch.zeros((5, 5, 15), dtype=torch.float64, device=dev)
    c = 0
    for p in range(5):
        for q in range(p, 5):
            chan[p, q, c] = chan[q, p, c] = 1.0
            c += 1
    P = torch.einsum("bjp,bkq,pqc->bjkc", E, E, chan).reshape(B, n * n, 15)
    feat = (rad[..., :, None] * ang[..., None, :]).reshape(B, n, n * n, 40)
    three = torch.matmul(P.transpose(1, 2).contiguous()[:, None], feat).reshape(B, n, 600)
    return torch.cat([two, three], -1) * L[..., None]


def _describe_exact(S, dtype, grad):
    """(label index, live, X, dX or None) of a set; inputs rounded to the case's dtype."""
    C, Z, N = S
    R = _gpu(C, dtype).to(torch.float64)
    Q, L = _gpu(_index(Z)).long(), _gpu(np.arange(Z.shape[1])[None] < N[:, None])
    E = torch.nn.functional.one_hot(Q, 5).to(torch.float64) * L[..., None]
    nm, ma = Q.shape
    X = torch.empty((nm, ma, REP), dtype=torch.float64, device="cuda")
    dX = torch.empty((nm, ma, REP, 3 * ma), dtype=torch.float64, device="cuda") if grad else None
    for b in range(0, nm, 64):
        s = slice(b, b + 64)
        if not grad:
            X[s] = _rep_exact(R[s], E[s], L[s])
            continue
        for t in range(3 * ma):
            d = torch.zeros_like(R[s]).reshape(-1, 3 * ma)
            d[:, t] = 1.0
            X[s], dX[s, :, :, t] = torch.func.jvp(lambda r: _rep_exact(r, E[s], L[s]), (R[s],),
                                                  (d.reshape(R[s].shape),))
    if grad:
        dX *= L.repeat_interleave(3, 1)[:, None, None, :]
    return Q, L, X, dX


def _rows(Q, L, X, e):
    """Rows of label e, in molecule order, and their molecules."""
    m = (Q == e) & L
    return X[m], m.nonzero()[:, 0]


def _kernel_exact(A, B):
    """(nm_a, nm_b) scalar kernel of two sets (label index, live, X)."""
    na, nb = A[0].shape[0], B[0].shape[0]
    K = torch.zeros((na, nb), dtype=torch.float64, device="cuda")
    for e in range(5):
        xa, ma = _rows(*A[:3], e)
        xb, mb = _rows(*B[:3], e)
        if not len(xa) or not len(xb):
            continue
        sb = (xb * xb).sum(1)
        for r in range(0, len(xa), 2048):
            x = xa[r:r + 2048]
            G = torch.exp(-((x * x).sum(1)[:, None] + sb - 2.0 * (x @ xb.T)).clamp(min=0.0)
                          / (2 * SIGMA ** 2))
            cols = torch.zeros((nb, len(x)), dtype=torch.float64, device="cuda")
            cols.index_add_(0, mb, G.T.contiguous())
            K.index_add_(0, ma[r:r + 2048], cols.T.contiguous())
    return K


def _ef_exact(Q, L, X, dX, nf):
    """Dense energy+force kernel over the live coordinates (nm + naq square)."""
    nm, ma = Q.shape
    keep = L.repeat_interleave(3, 1).reshape(-1).nonzero()[:, 0]
    s2 = SIGMA ** 2
    act = ((X != 0).reshape(-1, REP).any(0) | (dX != 0).any(-1).reshape(-1, REP).any(0)).nonzero()[:, 0]
    X, dX = X[:, :, act].contiguous(), dX[:, :, act].contiguous()
    f, nc = len(act), 3 * ma
    order = nm + nm * nc
    K = torch.zeros((order, order), dtype=torch.float64, device="cuda")
    FF = K[nm:, nm:].view(nm, nc, nm, nc)
    step = max(1, int(2e9 / (ma * ma * f * 8)))
    for a in range(nm):
        Ja = dX[a]  # (ma, f, nc)
        for b in range(0, nm, step):
            t = slice(b, min(b + step, nm))
            m = t.stop - b
            same = (Q[a][:, None, None] == Q[t][None]) & L[a][:, None, None] & L[t][None]
            d = X[a][:, None, None, :] - X[t][None]  # (ma, m, ma, f)
            k = torch.exp(-(d * d).sum(-1) / (2 * s2)) * same
            v = torch.matmul(d.reshape(ma, m * ma, f), Ja).reshape(ma, m, ma, nc)
            dt = d.permute(1, 2, 0, 3).reshape(m * ma, ma, f)
            u = torch.matmul(dt, dX[t].reshape(m * ma, f, nc)).reshape(m, ma, ma, nc)
            u = u.permute(2, 0, 1, 3)  # (i, m, j, nc)
            K[a, t] = k.sum((0, 2))
            K[a, nm + b * nc: nm + t.stop * nc] = ((k / s2)[..., None] * u).sum((0, 2)).reshape(-1)
            K[nm + a * nc: nm + (a + 1) * nc, t] = -((k / s2)[..., None] * v).sum((0, 2)).T
            for x in range(b, t.stop):
                c = k[:, x - b] / s2  # (ma, ma)
                T = (c @ dX[x].reshape(ma, f * nc)).reshape(ma * f, nc)
                FF[a, :, x] = Ja.reshape(ma * f, nc).T @ T
                w = (k[:, x - b] / (s2 * s2)).reshape(-1, 1)
                FF[a, :, x] -= (v[:, x - b].reshape(-1, nc) * w).T @ u[:, x - b].reshape(-1, nc)
    idx = nm + keep if nf else torch.cat([torch.arange(nm, device="cuda"), nm + keep])
    return K[idx][:, idx]


def _predict_exact(S, T, ad, aE):
    """Energies and energy gradients of set S = (Q, L, X, dX) from training set T and its
    weights in descriptor space."""
    Q, L, X, dX = S
    nq, s2 = Q.shape[0], SIGMA ** 2
    E = torch.zeros(nq, dtype=torch.float64, device="cuda")
    G = torch.zeros_like(X)
    for e in range(5):
        xa, ma = _rows(Q, L, X, e)
        xb, mb = _rows(*T[:3], e)
        if not len(xa) or not len(xb):
            continue
        al, w = ad[(T[0] == e) & T[1]], aE[mb]
        d2 = ((xa * xa).sum(1)[:, None] + (xb * xb).sum(1) - 2.0 * (xa @ xb.T)).clamp(min=0.0)
        k = torch.exp(-d2 / (2 * s2))
        p = xa @ al.T - (xb * al).sum(1)  # d . alpha
        E.index_add_(0, ma, (k * (w + p / s2)).sum(1))
        c = k * (w / s2 + p / (s2 * s2))  # factor of -d
        G[(Q == e) & L] = (k / s2) @ al - c.sum(1, keepdim=True) * xa + c @ xb
    F = torch.einsum("bif,bifz->bz", G, dX)
    return E, F[L.repeat_interleave(3, 1)]


def exact(case, seed):
    kind, dt = case["kind"], _dtype(case)
    if kind == "solve":
        K = _rfp_system(case["order"], seed)
        y = _gpu(np.random.default_rng(seed).normal(size=(case["nrhs"], case["order"])))
        K.diagonal().add_(1e-8)
        U = torch.linalg.cholesky(K)
        return torch.cholesky_solve(y.T.contiguous(), U).T.contiguous(), _to_rfp_u(U)
    rng, T, S = _sets(case, seed)
    if kind == "descriptors":
        return _describe_exact(T, dt, False)[2]
    if kind == "jacobians":
        Q, L, X, dX = _describe_exact(T, dt, True)
        return X, dX.reshape(*dX.shape[:3], -1, 3)
    if kind == "model_predict":
        from kernelforge_amd import synthetic

        E = np.array([synthetic.molecule_energy(c[:n], z[:n]) for c, z, n in zip(*T)])
        el = [e for e in ELEMENTS if (T[1] == e).any()]
        count = lambda Z: np.stack([(Z == e).sum(1) for e in el], 1).astype(float)  # noqa: E731
        base, *_ = np.linalg.lstsq(count(T[1]), E, rcond=None)
        A = _describe_exact(T, dt, False)
        K = _kernel_exact(A, A)
        K.diagonal().add_(1e-6)
        alpha = torch.linalg.solve(K, _gpu(E - count(T[1]) @ base))
        e, g = _predict_exact(_describe_exact(S, dt, True), A, torch.zeros_like(A[2]), alpha)
        return e.cpu().numpy() + count(S[1]) @ base, -g.cpu().numpy()
    if kind == "symm":
        A = _describe_exact(T, dt, False)
        A = (A[0], A[1], A[2].to(dt).to(torch.float64))
        return _to_rfp_l(_kernel_exact(A, A))
    if kind == "rect":
        return _kernel_exact(_describe_exact(S, dt, False), _describe_exact(T, dt, False))
    if kind == "ef_kernel":
        if case["mols"] * (case["atoms"] or 16) ** 2 > 100000:
            return None
        full = case["form"] == "full"
        K = _ef_exact(*_describe_exact(T, dt, True), not full)
        return _to_rfp_l(K) if full else _to_rfp_u(K)
    aE, aF = _alphas(rng, case["train"], 3 * int(T[2].sum()))
    aF = _gpu(aF, dt).to(torch.float64).reshape(case["train"], -1)
    Q, L, X, dX = _describe_exact(T, dt, True)
    X, dX = X.to(dt).to(torch.float64), dX.to(dt).to(torch.float64)
    ad = torch.einsum("bifz,bz->bif", dX, aF).to(dt).to(torch.float64)
    q = _describe_exact(S, dt, True)
    q = (q[0], q[1], q[2].to(dt).to(torch.float64), q[3].to(dt).to(torch.float64))
    return _predict_exact(q, (Q, L, X), ad, _gpu(aE, dt).to(torch.float64))
