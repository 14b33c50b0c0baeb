"""Timed cases: what a program using this package has it compute.

Every case goes through the package's public entry points, on inputs made
from a seed, and returns quantities that do not depend on the gauge of a
tensor train (states as vectors, kept two-site tensors, energies, overlaps):

* ``overlap``    ``scprod`` of two MPS, the building block of norms and fidelities;
* ``batch``      ``BatchedOverlap``: the overlaps of many uneven MPS in one graph;
* ``matvec``     ``QuadraticForm.two_site_matvec``, the product DMRG and TDVP repeat;
* ``split``      the truncated SVD of a two-site tensor (both sweep directions);
* ``apply``      ``MPO.apply`` followed by the variational simplify;
* ``sum``        ``simplify`` of a weighted sum of two uneven MPS (one in complex64);
* ``tebd``       one second-order Trotter step (gates and splits, forth and back);
* ``dmrg``       two-site DMRG from a random guess (growing bonds);
* ``learned``    two-site DMRG with the learned-rank splits from a nearly converged state.
"""

import math

import numpy as np
import torch

import seemps2_amd as S
from seemps2_amd import core, learned
from seemps2_amd.batch import BatchedOverlap
from seemps2_amd.evolution.trotter import Trotter2ndOrder

EPS = float(np.finfo(np.float64).eps)


def listed():
    return [
        # one bond update of a small sweep: the 64 x 64 split a sweep at chi = 32 makes
        {"name": "split-chi32", "kind": "split", "left": 32, "d1": 2, "d2": 2, "right": 32,
         "cap": 32, "direction": 1, "decades": 8.0},
        # a bond between different local dimensions with odd bonds, sweeping left
        {"name": "split-odd", "kind": "split", "left": 87, "d1": 2, "d2": 3, "right": 61,
         "cap": 75, "direction": -1, "decades": 0.0},
        # the capped bond of a chi = 256 sweep: a 512 x 512 split
        {"name": "split-chi256", "kind": "split", "left": 256, "d1": 2, "d2": 2, "right": 256,
         "cap": 256, "direction": 1, "decades": 10.0},
        # the effective Hamiltonian of a Heisenberg-like chain (MPO bond 5) at chi = 256
        {"name": "matvec-chi256", "kind": "matvec", "left": 256, "d": 2, "w": 5, "right": 256},
        # fidelity of two long states of a large sweep
        {"name": "overlap-n64-chi256", "kind": "overlap", "n": 64, "bra": 256, "ket": 200},
        # overlaps of many uneven states (N ~ U[10, 40], chi ~ U[8, 128])
        {"name": "batch-64-pairs", "kind": "batch", "pairs": 64, "longest": 40, "chi": 128},
        # a small operator application without truncation: launches and latency
        {"name": "apply-n10-chi8", "kind": "apply", "n": 10, "chi": 8, "cap": 0},
        # MPO.apply + simplify of a random 20-site state, chi = 32 to 64
        {"name": "apply-n20-chi32", "kind": "apply", "n": 20, "chi": 32, "cap": 64},
        # one sum of the many-state workload: uneven bonds, tolerance 1e-8
        {"name": "sum-n16-uneven", "kind": "sum", "n": 16, "chi": 37, "chi2": 101},
        # a Trotter step of the Heisenberg chain at a bond cap
        {"name": "tebd-n16-chi64", "kind": "tebd", "n": 16, "chi": 64},
        # DMRG from a random state: bonds grow to their cap in two sweeps
        {"name": "dmrg-n20-chi96", "kind": "dmrg", "n": 20, "chi": 48, "cap": 96, "sweeps": 2},
        # DMRG sweeps of a nearly converged state with the learned-rank splits
        {"name": "learned-n20-chi64", "kind": "learned", "n": 20, "cap": 64, "sweeps": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["overlap", "batch", "matvec", "split", "split", "apply", "sum", "tebd",
                       "dmrg", "learned"])
    if kind == "overlap":
        return {"kind": kind, "n": _log(rng, 10, 64), "bra": _log(rng, 8, 256),
                "ket": _log(rng, 8, 256)}
    if kind == "batch":
        return {"kind": kind, "pairs": _log(rng, 8, 64), "longest": rng.randint(12, 40),
                "chi": _log(rng, 16, 128)}
    if kind == "matvec":
        d = rng.choice([2, 2, 3])
        top = 256 if d == 2 else 170
        return {"kind": kind, "left": _log(rng, 16, top), "d": d, "w": rng.randint(3, 6),
                "right": _log(rng, 16, top)}
    if kind == "split":
        d1, d2 = rng.choice([2, 2, 3, 4]), rng.choice([2, 2, 3, 4])
        left, right = _log(rng, 12, 512 // d1), _log(rng, 12, 512 // d2)
        small = min(left * d1, right * d2)
        return {"kind": kind, "left": left, "d1": d1, "d2": d2, "right": right,
                "cap": max(4, int(small * rng.uniform(0.35, 0.8))),
                "direction": rng.choice([1, -1]), "decades": rng.choice([0.0, 4.0, 8.0, 10.0])}
    if kind == "apply":
        n = rng.randint(10, 20)
        chi = _log(rng, 4, 32)
        return {"kind": kind, "n": n, "chi": chi, "cap": rng.choice([2 * chi, chi + 5])}
    if kind == "sum":
        return {"kind": kind, "n": rng.randint(10, 16), "chi": _log(rng, 8, 110),
                "chi2": _log(rng, 8, 110)}
    if kind == "tebd":
        return {"kind": kind, "n": rng.randint(8, 16), "chi": _log(rng, 8, 64)}
    if kind == "dmrg":
        chi = _log(rng, 8, 48)
        # even chains: an odd one has a degenerate ground state
        return {"kind": kind, "n": 2 * rng.randint(5, 10), "chi": chi, "cap": 2 * chi,
                "sweeps": 2}
    return {"kind": kind, "n": 2 * rng.randint(7, 10), "cap": _log(rng, 33, 64), "sweeps": 2}


# --- inputs -------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, dtype=torch.complex128, device="cuda", generator=g)


def _chain(g, n, chi, d=2):
    """Random MPS tensors with the largest bonds up to chi, norm of order one."""
    bonds = [min(chi, d ** min(i, n - i, 40)) for i in range(n + 1)]
    return [_randn(g, bonds[i], d, bonds[i + 1]) / math.sqrt(d * bonds[i]) for i in range(n)]


def _theta(case, g):
    """A two-site tensor; `decades` > 0: singular values falling by about that
    many decades (a converged sweep's), 0: the flat spectrum of a random state."""
    m, n = case["left"] * case["d1"], case["d2"] * case["right"]
    r = min(m, n)
    if case["decades"] > 0:
        w = torch.pow(10.0, -case["decades"] * torch.arange(r, dtype=torch.float64,
                                                            device="cuda") / r)
        t = (_randn(g, m, r) * w) @ _randn(g, r, n)
    else:
        t = _randn(g, m, n)
    return (t / torch.linalg.vector_norm(t)).reshape(case["left"], case["d1"], case["d2"],
                                                     case["right"]).contiguous()


def _batch_states(case, g, seed):
    rng = np.random.default_rng(seed)
    states = []
    for _ in range(case["pairs"]):
        n = int(rng.integers(10, case["longest"] + 1))
        states.append((_chain(g, n, int(rng.integers(8, case["chi"] + 1))),
                       _chain(g, n, int(rng.integers(8, case["chi"] + 1)))))
    return states


def _matvec_parts(case, g):
    """Four sites around the bond: the environments come from the outer two."""
    left, right, d, w = case["left"], case["right"], case["d"], case["w"]
    mps = [_randn(g, 1, d, left), _randn(g, left, d, 40) / math.sqrt(left),
           _randn(g, 40, d, right) / math.sqrt(40), _randn(g, right, d, 1) / math.sqrt(right)]
    mpo = [_randn(g, 1, d, d, w), _randn(g, w, d, d, w), _randn(g, w, d, d, w),
           _randn(g, w, d, d, 1)]
    v = _randn(g, left, d, d, right)
    return mps, mpo, v / torch.linalg.vector_norm(v)


def _delta(seed):
    return 0.3 + 0.6 * float(np.random.default_rng(int(seed)).random())


def _strategy(case):
    kind = case["kind"]
    if kind == "split":
        return S.DEFAULT_STRATEGY.replace(max_bond_dimension=case["cap"])
    if kind == "apply":
        kw = {"max_bond_dimension": case["cap"]} if case["cap"] else {}
        return S.Strategy(tolerance=1e-10, simplification_tolerance=1e-10, max_sweeps=2, **kw)
    if kind == "sum":
        return S.Strategy(tolerance=1e-8, simplification_tolerance=1e-8, max_sweeps=2)
    if kind == "tebd":
        return S.Strategy(tolerance=1e-10, max_bond_dimension=case["chi"])
    return S.DEFAULT_STRATEGY.replace(max_bond_dimension=case["cap"])


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    state = {"case": case}
    if kind == "overlap":
        state["bra"] = S.MPS(_chain(g, case["n"], case["bra"]))
        state["ket"] = S.MPS(_chain(g, case["n"], case["ket"]))
    elif kind == "batch":
        pairs = _batch_states(case, g, seed)
        a, b = [S.MPS(p[0]) for p in pairs], [S.MPS(p[1]) for p in pairs]
        # the three overlaps that simplify(a + b) starts from
        state["plan"] = BatchedOverlap(a + b + a, a + b + b)
    elif kind == "matvec":
        mps, mpo, v = _matvec_parts(case, g)
        psi = S.CanonicalMPS(mps, center=1, is_canonical=True, normalize=False)
        state["form"] = S.QuadraticForm(S.MPO(mpo), psi, start=1)
        state["form"].two_site_block(1)
        state["v"] = v
    elif kind == "split":
        state["theta"], state["strategy"] = _theta(case, g), _strategy(case)
    elif kind == "apply":
        state["op"] = S.HeisenbergHamiltonian(case["n"]).to_mpo()
        state["psi"], state["strategy"] = S.MPS(_chain(g, case["n"], case["chi"])), _strategy(case)
    elif kind == "sum":
        state["sum"] = S.MPSSum([1.0, 0.7], _sum_states(case, g))
        state["strategy"] = _strategy(case)
    elif kind == "tebd":
        state["step"] = Trotter2ndOrder(S.HeisenbergHamiltonian(case["n"]), 0.05, _strategy(case))
        state["psi"] = S.CanonicalMPS(_chain(g, case["n"], case["chi"]), center=0,
                                      strategy=S.NO_TRUNCATION, normalize=False)
    elif kind == "dmrg":
        state["H"] = S.XXZHamiltonian(case["n"], 1.0, _delta(seed)).to_mpo()
        state["psi"], state["strategy"] = S.MPS(_chain(g, case["n"], case["chi"])), _strategy(case)
    else:
        H = S.XXZHamiltonian(case["n"], 1.0, _delta(seed)).to_mpo()
        st = _strategy(case)
        near = S.dmrg(H, S.MPS(_chain(g, case["n"], 24)), maxiter=3, tol=0.0, tol_up=1.0,
                      tol_eigs=1e-10, strategy=st)
        state.update(H=H, psi=near.state, strategy=st, net=learned.RankPredictor(seed=int(seed)))
    return state


def _sum_states(case, g):
    return [S.MPS(_chain(g, case["n"], case["chi"])),
            S.MPS([A.to(torch.complex64) for A in _chain(g, case["n"], case["chi2"])])]


# --- one pass -----------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "overlap":
        return np.complex128(S.scprod(state["bra"], state["ket"]))
    if kind == "batch":
        return state["plan"].run_async()
    if kind == "matvec":
        return state["form"].two_site_matvec(1, state["v"])
    if kind == "split":
        cut = core._left_orth_2site if case["direction"] > 0 else core._right_orth_2site
        A, B, error = cut(state["theta"], state["strategy"])
        return {"kept": core._contract_last_and_first(A, B), "error": float(error),
                "bond": int(A.shape[2])}
    if kind == "apply":
        out = state["op"].apply(state["psi"], strategy=state["strategy"], simplify=True)
        return out.to_vector()
    if kind == "sum":
        return S.simplify(state["sum"], strategy=state["strategy"]).to_vector()
    if kind == "tebd":
        return state["step"].apply(state["psi"]).to_vector()
    if kind == "dmrg":
        res = S.dmrg(state["H"], state["psi"], maxiter=case["sweeps"], tol=0.0, tol_up=1.0,
                     tol_eigs=1e-10, strategy=state["strategy"])
    else:
        with learned.learned_truncation(learned.LearnedTruncation(state["net"])):
            res = S.dmrg(state["H"], state["psi"].copy(), maxiter=case["sweeps"], tol=0.0,
                         tol_up=1.0, tol_eigs=1e-10, strategy=state["strategy"])
    return {"energies": np.array(res.trajectory), "state": res.state.to_vector()}


# --- what a pass cannot do without ------------------------------------------------


def _bonds(n, chi, d=2):
    return [min(chi, d ** min(i, n - i, 40)) for i in range(n + 1)]


def _overlap_work(n, chi1, chi2, d=2):
    a, b = _bonds(n, chi1, d), _bonds(n, chi2, d)
    flops = sum(8.0 * d * (a[i] * b[i] * b[i + 1] + a[i] * a[i + 1] * b[i + 1])
                for i in range(n))
    size = sum(16.0 * d * (a[i] * a[i + 1] + b[i] * b[i + 1]) for i in range(n))
    return size, flops


def _svd_flops(m, n):
    m, n = max(m, n), min(m, n)
    return 4.0 * (6.0 * m * n * n + 16.0 * n * n * n)


def _sweep_flops(n, inner, cap, terms, d=2):
    """Two-site sweep over bonds min(cap, ..) of a target with bonds `inner`."""
    c = _bonds(n, cap, d)
    flops = 0.0
    for i in range(n - 1):
        flops += _svd_flops(c[i] * d, d * c[i + 2])
        for b in inner:
            flops += 8.0 * d * (2 * c[i] * b[i] * b[i + 1] + c[i + 2] * b[i + 1] * b[i + 2]
                                + d * c[i] * b[i + 1] * c[i + 2] + c[i] * c[i + 1] * b[i + 1])
    return flops * max(terms, 1)


def work(case):
    kind = case["kind"]
    if kind == "overlap":
        size, flops = _overlap_work(case["n"], case["bra"], case["ket"])
        return {"bytes": size, "flops": flops}
    if kind == "batch":
        # mean sizes of the uneven states
        n, chi = (10 + case["longest"]) // 2, (8 + case["chi"]) // 2
        size, flops = _overlap_work(n, chi, chi)
        return {"bytes": case["pairs"] * size, "flops": 3 * case["pairs"] * flops}
    if kind == "matvec":
        a, f, d, w = case["left"], case["right"], case["d"], case["w"]
        return {"bytes": 16.0 * (a * a * w + f * f * w + 2 * a * d * d * f),
                "flops": 8.0 * (w * a * a * d * d * f + w * a * d * d * f * f)}
    if kind == "split":
        m, n = case["left"] * case["d1"], case["right"] * case["d2"]
        k = min(case["cap"], m, n)
        return {"bytes": 16.0 * (2 * m * n), "flops": _svd_flops(m, n) + 8.0 * m * n * k}
    n = case["n"]
    if kind == "apply":
        wide = _bonds(n, 5 * case["chi"])
        cap = case["cap"] or 5 * case["chi"]
        size = 16.0 * 2 * sum(a * b for a, b in zip(_bonds(n, case["chi"]),
                                                    _bonds(n, case["chi"])[1:])) + 16.0 * 2 ** n
        return {"bytes": size, "flops": 2 * _sweep_flops(n, [wide], cap, 1)}
    if kind == "sum":
        a, b = _bonds(n, case["chi"]), _bonds(n, case["chi2"])
        size = 16.0 * 2 * sum(x[i] * x[i + 1] for x in (a, b) for i in range(n)) + 16.0 * 2 ** n
        return {"bytes": size,
                "flops": 3 * _sweep_flops(n, [a, b], case["chi"] + case["chi2"], 1)}
    cap = case["chi"] if kind == "tebd" else case["cap"]
    c = _bonds(n, cap)
    size = 16.0 * (2 * 2 * sum(c[i] * c[i + 1] for i in range(n)) + 2 ** n)
    cuts = sum(_svd_flops(2 * c[i], 2 * c[i + 2]) for i in range(n - 1))
    if kind == "tebd":
        join = sum(8.0 * 4 * (c[i] * c[i + 1] * c[i + 2] + 4 * c[i] * c[i + 2])
                   for i in range(n - 1))
        return {"bytes": size, "flops": 2 * (cuts + join)}
    # five products with the effective Hamiltonian per bond, one environment update
    products = sum(8.0 * 5 * 4 * (c[i] * c[i] * c[i + 2] + c[i] * c[i + 2] * c[i + 2])
                   for i in range(n - 1))
    return {"bytes": size, "flops": case["sweeps"] * (cuts + 6 * products)}


# --- the same results in 64 bits without this package -------------------------------


def _host(x):
    return x.detach().cpu().to(torch.complex128).numpy()


def _rank(s, tol, cap):
    """Kept size: discarded squares at most tol of the total, at most `cap`."""
    tail = np.cumsum((s * s)[::-1])
    drop = int(np.sum(tail <= tol * tail[-1]))
    return max(1, min(len(s) - drop, cap))


def _np_overlap(bra, ket):
    rho = np.ones((1, 1), dtype=np.complex128)
    for A, B in zip(bra, ket):
        rho = np.tensordot(A.conj(), np.tensordot(rho, B, 1), ((0, 1), (0, 1)))
    return rho[0, 0]


def _np_vector(tensors):
    out = np.ones((1, 1), dtype=np.complex128)
    for A in tensors:
        out = np.tensordot(out, A, 1).reshape(-1, A.shape[2])
    return out[:, 0]


def _np_simplify(weights, terms, tol, cap, sweeps):
    """Variational two-site simplify of sum_k weights[k] terms[k] from its
    truncated canonical form, `sweeps` sweeps unless the first one is exact."""
    n = len(terms[0])
    data = []
    for i in range(n):
        parts = [t[i] * (weights[k] if i == 0 else 1.0) for k, t in enumerate(terms)]
        rows = 1 if i == 0 else sum(p.shape[0] for p in parts)
        cols = 1 if i == n - 1 else sum(p.shape[2] for p in parts)
        W = np.zeros((rows, parts[0].shape[1], cols), dtype=np.complex128)
        l = r = 0
        for p in parts:
            W[l:l + p.shape[0], :, r:r + p.shape[2]] += p
            l += 0 if i == 0 else p.shape[0]
            r += 0 if i == n - 1 else p.shape[2]
        data.append(W)
    for i in range(n - 1, 0, -1):
        a, d, b = data[i].shape
        U, s, V = np.linalg.svd(data[i].reshape(a, d * b), full_matrices=False)
        k = _rank(s, tol, cap)
        data[i] = V[:k].reshape(k, d, b)
        data[i - 1] = np.tensordot(data[i - 1], U[:, :k] * s[:k], 1)
    one = np.ones((1, 1), dtype=np.complex128)
    L, R = [[one] * n for _ in terms], [[one] * n for _ in terms]

    def grow_left(i):
        for k, t in enumerate(terms):
            x = np.tensordot(L[k][i], t[i], 1)
            L[k][i + 1] = np.tensordot(data[i].conj(), x, ((0, 1), (0, 1)))

    def grow_right(i):
        for k, t in enumerate(terms):
            x = np.tensordot(t[i], R[k][i], 1)
            R[k][i - 1] = np.tensordot(x, data[i].conj(), ((1, 2), (1, 2)))

    for i in range(n - 1, 0, -1):
        grow_right(i)
    total = sum((np.conj(u) * v * _np_overlap(x, y)).real for u, x in zip(weights, terms)
                for v, y in zip(weights, terms))
    for sweep in range(sweeps):
        right = sweep % 2 == 0
        for i in (range(n - 1) if right else range(n - 2, -1, -1)):
            theta = 0.0
            for k, t in enumerate(terms):
                x = np.tensordot(np.tensordot(L[k][i], t[i], 1), t[i + 1], 1)
                theta = theta + weights[k] * np.tensordot(x, R[k][i + 1], 1)
            a, d, e, b = theta.shape
            U, s, V = np.linalg.svd(theta.reshape(a * d, e * b), full_matrices=False)
            k = _rank(s, tol, cap)
            U, V = (U[:, :k], s[:k, None] * V[:k]) if right else (U[:, :k] * s[:k], V[:k])
            data[i], data[i + 1] = U.reshape(a, d, k), V.reshape(k, e, b)
            if right and i < n - 2:
                grow_left(i)
            if not right and i > 0:
                grow_right(i + 1)
        norm = sum(np.vdot(A, A).real for A in [data[n - 1 if right else 0]])
        cross = sum(w * _np_overlap(data, t) for w, t in zip(weights, terms)).real
        if 2 * abs(1 - cross / math.sqrt(norm * total)) < tol:
            break
        if right:
            grow_left(n - 2)
        else:
            grow_right(1)
    return _np_vector(data)


def _heisenberg():
    x = np.array([[0, 1], [1, 0]], dtype=complex)
    y = np.array([[0, -1j], [1j, 0]])
    z = np.diag([1.0 + 0j, -1.0])
    return 0.25 * sum(np.kron(p, p) for p in (x, y, z))


def _np_mpo(n):
    """The Heisenberg chain as MPO tensors W[a, out, in, b] with bond 5."""
    x = np.array([[0, 1], [1, 0]], dtype=complex) / 2
    y = np.array([[0, -1j], [1j, 0]]) / 2
    z = np.diag([0.5 + 0j, -0.5])
    W = np.zeros((5, 2, 2, 5), dtype=complex)
    W[0, :, :, 0] = W[4, :, :, 4] = np.eye(2)
    for k, p in enumerate((x, y, z)):
        W[0, :, :, 1 + k] = p
        W[1 + k, :, :, 4] = p
    return [W[:1] if i == 0 else W[..., 4:] if i == n - 1 else W for i in range(n)]


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "overlap":
        bra, ket = _chain(g, case["n"], case["bra"]), _chain(g, case["n"], case["ket"])
        return np.complex128(_np_overlap([_host(A) for A in bra], [_host(A) for A in ket]))
    if kind == "batch":
        pairs = [([_host(A) for A in p], [_host(A) for A in q])
                 for p, q in _batch_states(case, g, seed)]
        return np.array([_np_overlap(p, p) for p, _ in pairs]
                        + [_np_overlap(q, q) for _, q in pairs]
                        + [_np_overlap(p, q) for p, q in pairs])
    if kind == "matvec":
        mps, mpo, v = _matvec_parts(case, g)
        mps, mpo, v = [_host(A) for A in mps], [_host(W) for W in mpo], _host(v)
        # L[bra, w, ket] of site 0 and R[bra, w, ket] of site 3
        left = np.einsum("ix,ijw,jy->xwy", mps[0][0].conj(), mpo[0][0], mps[0][0])
        right = np.einsum("xi,wij,yj->xwy", mps[3][..., 0].conj(), mpo[3][..., 0],
                          mps[3][..., 0])
        x = np.tensordot(left, v, 1)                                      # a w k l f
        x = np.tensordot(x, mpo[1], ((1, 2), (0, 2)))                     # a l f K e
        x = np.tensordot(x, mpo[2], ((1, 4), (2, 0)))                     # a f K L e
        return np.tensordot(x, right, ((1, 4), (2, 1)))                   # a K L g
    if kind == "split":
        t = _host(_theta(case, g))
        U, s, V = np.linalg.svd(t.reshape(case["left"] * case["d1"], -1), full_matrices=False)
        k = _rank(s, EPS, case["cap"])
        return {"kept": ((U[:, :k] * s[:k]) @ V[:k]).reshape(t.shape),
                "error": float(math.sqrt(np.sum(s[k:] ** 2))), "bond": int(k)}
    if kind == "apply":
        psi = [_host(A) for A in _chain(g, case["n"], case["chi"])]
        out = []
        for W, A in zip(_np_mpo(case["n"]), psi):
            x = np.tensordot(A, W, ((1,), (2,))).transpose(0, 2, 3, 1, 4)
            a, w, d, b, v = x.shape
            out.append(x.reshape(a * w, d, b * v))
        if not case["cap"]:
            return _np_vector(out)
        return _np_simplify([1.0], [out], 1e-10, case["cap"], 2)
    if kind == "sum":
        a = [_host(A) for A in _chain(g, case["n"], case["chi"])]
        b = [_host(A.to(torch.complex64)) for A in _chain(g, case["n"], case["chi2"])]
        return _np_simplify([1.0, 0.7], [a, b], 1e-8, 1 << 30, 2)
    if kind == "tebd":
        n = case["n"]
        e, U = np.linalg.eigh(_heisenberg())
        gate = (U * np.exp(-0.025j * e)) @ U.conj().T
        v = _np_vector([_host(A) for A in _chain(g, n, case["chi"])])

        def cut(v, bond):
            u, s, w = np.linalg.svd(v.reshape(2 ** bond, -1), full_matrices=False)
            k = _rank(s, 1e-10, case["chi"])
            return (u[:, :k] * s[:k]) @ w[:k]

        for j in list(range(n - 1)) + list(range(n - 2, -1, -1)):
            v = cut(np.einsum("ab,xbz->xaz", gate, v.reshape(2 ** j, 4, -1)), j + 1)
        return v.reshape(-1)
    return None  # a fixed number of DMRG sweeps has no closed form
