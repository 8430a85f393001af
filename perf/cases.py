"""Performance cases of the sweep engine: the steps of a region (effective-Hamiltonian
apply, Krylov solvers, environment update, truncated factorisation) on dense, block-sparse
and complex tensors, and two whole calls (a DMRG run, a tree TDVP step).

``prepare`` makes seeded inputs on the device and the operators a sweep holds at that
point; ``run`` is one pass through the public entry points; ``exact`` restates the result
in FP64 numpy.  Results stay in HBM, as a sweep leaves them, and are copied to the host
when they are read (``Results``).
"""
import functools
import math

import numpy as np

import networksolvers_amd as ns
from networksolvers_amd import qn


@functools.lru_cache(maxsize=None)
def _ctx():
    """The one device context that a program works with."""
    return ns.Context(0)


class Results(list):
    """Outputs of one pass: device tensors, copied to the host when the list is read."""

    def __iter__(self):
        return (x.numpy() if isinstance(x, ns.DeviceTensor) else x for x in list.__iter__(self))


def _num(x):
    """A scalar result as an FP64 array."""
    return np.array([x], dtype=np.float64)


# --------------------------------------------------------------------- cases
def listed():
    return [
        # The effective-Hamiltonian apply at the benchmark chain's bond-dimension cap
        # (XXZ, maxdim 1024): every Krylov step of a large solve is one of these.
        dict(name="heff_fp64_chi1024", kind="heff", l=1024, r=1024, d=2, sites=2, precision="fp64"),
        # The same apply in the split-BF16 form on ragged links, an ordinary mid-size region.
        dict(name="heff_bf16x3_ragged", kind="heff", l=613, r=487, d=2, sites=2, precision="bf16x3"),
        # The updater of a dense region at the benchmark chain's converged links, in its
        # timed FP32 form: operator set-up and the 3-vector Lanczos solve.
        dict(name="eigsolve_fp32_chi200", kind="eigsolve", l=197, r=211, d=2, precision="fp32"),
        # Real-time evolution of a complex two-site region (TDVP, Krylov exponential).
        dict(name="expm_c128_chi60", kind="expm", l=61, r=64, d=2),
        # One environment update of a spin-1 chain, odd sizes.
        dict(name="env_spin1_ragged", kind="env", l=389, r=421, d=3, side=0),
        # The truncated split at the benchmark chain's converged links (cutoff 1e-12: SVD).
        dict(name="svd_chi200", kind="factorize", m=394, n=422, decay=11.7, cutoff=1e-12, maxdim=1024, trailing=False),
        # The truncated split where maxdim 1024 binds: the largest step of a sweep.
        dict(name="svd_chi1024", kind="factorize", m=2048, n=2048, decay=8, cutoff=0.0, maxdim=1024, trailing=True),
        # The split of a small solve as the request loop runs it (cutoff 1e-10: eigen route).
        dict(name="eigen_chi80", kind="factorize", m=154, n=166, decay=5, cutoff=1e-10, maxdim=77, trailing=True),
        # Block-sparse spin-1 chain with conserved Sz: the sector split and the updater.
        dict(name="qn_factorize_spin1", kind="qn_factorize", l=270, r=259, d=3, maxdim=270, trailing=False),
        dict(name="qn_eigsolve_spin1", kind="qn_eigsolve", l=270, r=259, d=3, precision="fp64"),
        # Whole calls: a small spin-1 DMRG solve from a random state, and one fourth-order
        # two-site TDVP step of a transverse-field Ising quench on a binary tree.
        dict(name="dmrg_spin1_n20", kind="dmrg", N=20, maxdim=40, nsweeps=2),
        dict(name="tree_tdvp_n15", kind="tree_tdvp", n=15, dt=0.05),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["heff", "heff", "eigsolve", "expm", "env", "factorize", "factorize", "factorize",
                       "qn_factorize", "qn_eigsolve", "dmrg", "tree_tdvp"])
    if kind == "heff":
        return dict(kind=kind, l=_log(rng, 8, 1000), r=_log(rng, 8, 1000), d=rng.choice([2, 2, 3]) if rng.random() < .5
                    else 2, sites=rng.choice([1, 2, 2]), precision=rng.choice(["fp64", "fp32", "bf16x3"]))
    if kind == "eigsolve":
        return dict(kind=kind, l=_log(rng, 8, 512), r=_log(rng, 8, 512), d=rng.choice([2, 3]),
                    precision=rng.choice(["fp64", "fp32"]))
    if kind == "expm":
        return dict(kind=kind, l=_log(rng, 4, 128), r=_log(rng, 4, 128), d=2)
    if kind == "env":
        return dict(kind=kind, l=_log(rng, 8, 1000), r=_log(rng, 8, 1000), d=rng.choice([2, 3]), side=rng.choice([0, 1]))
    if kind == "factorize":
        m, n = _log(rng, 8, 1700), _log(rng, 8, 1700)
        if rng.random() < 0.6:
            n = max(8, min(1700, int(m * rng.uniform(0.5, 2.0))))
        if rng.random() < 0.6:   # the SVD route: truncated by the cutoff, as the benchmark chain
            return dict(kind=kind, m=m, n=n, decay=11.7, cutoff=1e-12, maxdim=1024, trailing=rng.random() < 0.5)
        m, n = min(m, 1024), min(n, 1024)
        return dict(kind=kind, m=m, n=n, decay=5, cutoff=1e-10, maxdim=max(2, min(m, n) // 2),
                    trailing=rng.random() < 0.5)
    if kind == "qn_factorize":
        l = _log(rng, 20, 300)
        return dict(kind=kind, l=l, r=max(20, int(l * rng.uniform(0.7, 1.3))), d=rng.choice([2, 3]), maxdim=l,
                    trailing=rng.random() < 0.5)
    if kind == "qn_eigsolve":
        l = _log(rng, 20, 300)
        return dict(kind=kind, l=l, r=max(20, int(l * rng.uniform(0.7, 1.3))), d=rng.choice([2, 3]),
                    precision=rng.choice(["fp64", "fp32"]))
    if kind == "dmrg":
        return dict(kind=kind, N=rng.randint(8, 24), maxdim=rng.randint(16, 48), nsweeps=rng.choice([1, 2]))
    return dict(kind=kind, n=rng.randint(6, 15), dt=round(rng.uniform(0.02, 0.06), 4))


# -------------------------------------------------------------------- inputs
def _spin(d):
    S = (d - 1) / 2
    m = S - np.arange(d)
    Sp = np.zeros((d, d))
    for k in range(1, d):
        Sp[k - 1, k] = math.sqrt(S * (S + 1) - m[k] * (m[k] + 1))
    return np.diag(m), Sp


def _mpo_site(d, Jz=1.0):
    """Bulk XXZ tensor W[wl, wr, s', s], D = 5."""
    Sz, Sp = _spin(d)
    W = np.zeros((5, 5, d, d))
    W[0, 0] = W[4, 4] = np.eye(d)
    W[1, 0], W[2, 0], W[3, 0] = Sp, Sp.T, Sz
    W[4, 1], W[4, 2], W[4, 3] = 0.5 * Sp.T, 0.5 * Sp, Jz * Sz
    return W


def _env_pair(rng, l, r, cplx=False, mask=None):
    """Left and right environments [bra, mpo, ket] of a Hermitian effective
    Hamiltonian: the identity channel, the accumulated block Hamiltonian (spectrum of
    order 1) and the boundary spin operators (S+ and S- adjoint to each other)."""
    def rand(n):
        g = rng.standard_normal((n, n)) / math.sqrt(n)
        return g + 1j * rng.standard_normal((n, n)) / math.sqrt(n) if cplx else g

    def herm(n, scale):
        g = rand(n)
        return scale * (g + g.conj().T) / 2

    def env(n, identity, block, lower):
        E = np.zeros((n, 5, n), dtype=np.complex128 if cplx else np.float64)
        E[:, identity, :] = np.eye(n)
        E[:, block, :] = herm(n, 2.0)
        s = 0.5 * rand(n)
        E[:, 1, :], E[:, 2, :] = (s.conj().T, s) if lower else (s, s.conj().T)
        E[:, 3, :] = herm(n, 0.5)
        return E
    L, R = env(l, 4, 0, False), env(r, 0, 4, True)
    if mask is not None:
        L, R = np.where(mask[0], L, 0.0), np.where(mask[1], R, 0.0)
        for E in (L, R):   # masked S+ and S- stay adjoint: their masks are transposes
            E[:, 2, :] = E[:, 1, :].T
    return L, R


def _unit(rng, shape, cplx=False):
    x = rng.standard_normal(shape)
    if cplx:
        x = x + 1j * rng.standard_normal(shape)
    return x / np.linalg.norm(x)


def _decaying(rng, m, n, decay, exact_spectrum=True):
    """m x n matrix whose singular values fall ``decay`` decades over min(m, n), as a
    two-site tensor's Schmidt spectrum does; with ``exact_spectrum`` they are the same
    for every seed, so a cutoff keeps the same number of them."""
    p = min(m, n)
    s = 10.0 ** (-decay * np.arange(p) / p)
    X, Y = rng.standard_normal((m, p)) / math.sqrt(m), rng.standard_normal((n, p)) / math.sqrt(n)
    if exact_spectrum:
        X, Y = np.linalg.qr(X)[0], np.linalg.qr(Y)[0]
    M = (X * s) @ Y.T
    return M / np.linalg.norm(M)


def _sectors(total, step=2):
    """Link sectors (charge, dim) of about ``total`` states, a Gaussian profile over the
    charges of a spin chain's bond."""
    half = 4 if total > 60 else 2
    w = np.exp(-(np.arange(-half, half + 1) / (0.45 * half)) ** 2)
    dims = np.maximum(1, np.round(total * w / w.sum())).astype(int)
    return [(step * k, int(n)) for k, n in zip(range(-half, half + 1), dims)]


def _charges(sectors):
    return np.concatenate([np.full(n, q) for q, n in sectors])


# charges of the XXZ MPO link channels (H, S+, S-, Sz, I): what each has still to give back
_C_MPO = np.array([0, -2, 2, 0, 0])


def _qn_setup(case, rng):
    sl, sr = _sectors(case["l"]), _sectors(case["r"])
    ql, qr = _charges(sl), _charges(sr)
    qs = np.array([case["d"] - 1 - 2 * i for i in range(case["d"])])
    return sl, sr, ql, qr, qs


def _theta_mask(ql, qs, qr):
    return (ql[:, None, None, None] + qs[None, :, None, None] + qs[None, None, :, None]) == qr[None, None, None, :]


def _qn_theta(case, rng):
    """Block-sparse two-site tensor (dense storage) whose charge sectors have decaying
    spectra, and its sectors as (charge, row ids, column ids)."""
    sl, sr, ql, qr, qs = _qn_setup(case, rng)
    d = case["d"]
    rows = (ql[:, None] + qs[None, :]).reshape(-1)
    cols = (qr[None, :] - qs[:, None]).reshape(-1)
    M = np.zeros((len(ql) * d, d * len(qr)))
    parts = []
    for q in sorted(set(rows) & set(cols)):
        i, j = np.nonzero(rows == q)[0], np.nonzero(cols == q)[0]
        M[np.ix_(i, j)] = _decaying(rng, len(i), len(j), 5) * math.exp(0.03 * q - (q / 5.0) ** 2)
        parts.append((int(q), i, j))
    M /= np.linalg.norm(M)
    return M.reshape(len(ql), d, d, len(qr)), parts


def _qn_operator(case, rng):
    sl, sr, ql, qr, qs = _qn_setup(case, rng)
    ml = (ql[:, None, None] - ql[None, None, :]) == _C_MPO[None, :, None]
    mr = (qr[:, None, None] - qr[None, None, :]) == _C_MPO[None, :, None]
    L, R = _env_pair(rng, len(ql), len(qr), mask=(ml, mr))
    x = np.where(_theta_mask(ql, qs, qr), rng.standard_normal((len(ql), case["d"], case["d"], len(qr))), 0.0)
    return L, R, x / np.linalg.norm(x)


def _inputs(case, seed):
    rng = np.random.default_rng([int(seed), 17])
    k = case["kind"]
    if k in ("heff", "eigsolve", "expm"):
        cplx = k == "expm"
        L, R = _env_pair(rng, case["l"], case["r"], cplx)
        shape = (case["l"],) + (case["d"],) * case.get("sites", 2) + (case["r"],)
        return L, R, _mpo_site(case["d"]), _unit(rng, shape, cplx)
    if k == "env":
        n_in, n_out = (case["l"], case["r"]) if case["side"] == 0 else (case["r"], case["l"])
        E, _ = _env_pair(rng, n_in, 2)
        A = rng.standard_normal((case["l"], case["d"], case["r"])) / math.sqrt(case["d"] * n_in)
        return E, A, _mpo_site(case["d"])
    if k == "factorize":
        return (_decaying(rng, case["m"], case["n"], case["decay"], case["cutoff"] == 1e-12),)
    raise ValueError(k)


# --------------------------------------------------------------------- passes
def prepare(case, seed):
    ctx = _ctx()
    k = case["kind"]
    up = ctx.upload
    if k in ("heff", "eigsolve", "expm", "env", "factorize"):
        arrays = _inputs(case, seed)
        if k == "factorize":
            M = arrays[0]   # as a two-site tensor [l, s1, s2, r] wherever the sizes are even
            m, n = M.shape
            return dict(case=case, x=up(M.reshape((m // 2, 2, n) if m % 2 == 0 else (m, 1, n))))
        t = [up(a) for a in arrays[:2]]
        W = up(arrays[2])
        if k == "env":
            return dict(case=case, E=t[0], A=t[1], W=W)
        s = dict(case=case, L=t[0], R=t[1], W=W, x=up(arrays[3]))
        if k == "heff":
            s["op"] = ns.HeffMap(s["L"], W, W if case["sites"] == 2 else None, s["R"], case["precision"])
            s["y"] = ctx.empty(s["x"].shape)
        return s
    rng = np.random.default_rng([int(seed), 23])
    if k in ("qn_factorize", "qn_eigsolve"):
        site = qn.spin_site_index(case["d"])
        l, r = (qn.QNIndex(_sectors(case[e])) for e in "lr")
        if k == "qn_factorize":
            theta, _ = _qn_theta(case, rng)
            return dict(case=case, x=qn.QNTensor.from_dense(ctx, theta, [l, site, site, r], [1, 1, 1, -1]))
        L, R, x = _qn_operator(case, rng)
        H = qn.QNMPO(ctx, ns.xxz_mpo(4, d=case["d"]), site)
        return dict(case=case, H=H, x=qn.QNTensor.from_dense(ctx, x, [l, site, site, r], [1, 1, 1, -1]),
                    L=qn.QNTensor.from_dense(ctx, L, [l, H.links[1], l], [1, -1, -1]),
                    R=qn.QNTensor.from_dense(ctx, R, [r, H.links[3], r], [1, -1, -1]))
    if k == "dmrg":
        H = ns.TTNO(ctx, ns.xxz_mpo(case["N"], d=3, Jz=float(rng.uniform(0.5, 2.0))))
        return dict(case=case, H=H, psi=ns.TTN.from_arrays(ctx, ns.random_mps(case["N"], 3, 8, seed=int(seed))))
    G = ns.Graph(list(range(case["n"])), [((i - 1) // 2, i) for i in range(1, case["n"])])
    W = ns.tree_mpo(G, 2, onsite=-float(rng.uniform(0.8, 1.2)) * np.array([[0.0, 1.0], [1.0, 0.0]]),
                    bond_terms=[(-1.0, np.diag([1.0, -1.0]), np.diag([1.0, -1.0]))])
    psi = ns.product_ttn(ctx, G, {v: 0 for v in range(case["n"])}, 2)
    return dict(case=case, H=ns.TreeTTNO(ctx, G, W), psi=psi)


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "heff":
        return Results([state["op"].apply(state["x"], state["y"])])
    if k == "eigsolve":
        H = ns.HeffMap(state["L"], state["W"], state["W"], state["R"], case["precision"])
        e, x = ns.eigsolve_solver(H, state["x"])
        H.close()
        return Results([_num(e), x])
    if k == "expm":
        H = ns.HeffMap(state["L"], state["W"], state["W"], state["R"], "fp64")
        x, _ = ns.exponentiate_solver(H, -0.05j, state["x"])
        H.close()
        return Results([x])
    if k == "env":
        return Results([ns.env_update(state["E"], state["A"], state["W"], case["side"])])
    if k == "factorize":
        U, C, info = ns.factorize(state["x"], 2, case["trailing"], cutoff=case["cutoff"], maxdim=case["maxdim"])
        return Results([U, C, _num(info.truncerr), _num(info.total), info.kept])
    if k == "qn_factorize":
        left, right, mid, info = qn.factorize(state["x"], case["trailing"], cutoff=1e-10, maxdim=case["maxdim"])
        return Results([left.data, right.data, _num(info.truncerr), _num(info.total), np.array(mid.n), np.array(mid.q)])
    if k == "qn_eigsolve":
        H, x = state["H"], state["x"]
        op = qn.heff2(state["L"], H.W[1], H.W[2], state["R"], x, H.c[1], H.c[3], x.ctx, case["precision"])
        e, y = ns.eigsolve_solver(op, x)
        op.close()
        return Results([_num(e), y.data])
    if k == "dmrg":
        E, psi = ns.dmrg(state["H"], state["psi"], nsweeps=case["nsweeps"], nsites=2,
                         inserter_kwargs=dict(trunc=dict(cutoff=1e-10, maxdim=case["maxdim"])))
        z2 = ns.expect_local(psi, np.diag([1.0, 0.0, 1.0]))
        return Results([_num(E), np.array([z2[v] for v in psi.vertices()])])
    psi = ns.tdvp(state["H"], state["psi"], [0.0, case["dt"]], nsites=2, tdvp_order=4,
                  updater_kwargs=dict(solver=ns.exponentiate_solver),
                  inserter_kwargs=dict(trunc=dict(cutoff=1e-10, maxdim=256)))
    z = ns.expect_local(psi, np.diag([1.0, -1.0]))
    return Results([np.array([z[v] for v in psi.vertices()])])


# ------------------------------------------------------------------ work, tolerance
def work(case):
    k = case["kind"]
    D = 5
    if k in ("heff", "eigsolve", "expm"):
        l, r, d = case["l"], case["r"], case["d"]
        n = d ** case.get("sites", 2)
        applies = {"heff": 1, "eigsolve": 3, "expm": 8}[k]
        c = 2 if k == "expm" else 1
        return dict(bytes=8.0 * c * (D * (l * l + r * r) + 2 * n * l * r),
                    flops=applies * (4 if c == 2 else 1) * 2.0 * D * n * l * r * (l + r))
    if k == "env":
        l, r, d = case["l"], case["r"], case["d"]
        return dict(bytes=8.0 * (D * (l * l + r * r) + d * l * r), flops=2.0 * D * d * l * r * (l + r))
    if k == "factorize":
        m, n = case["m"], case["n"]
        s, t = min(m, n), max(m, n)
        kept = min(case["maxdim"], s // 2 if case["cutoff"] > 0 else s)
        return dict(bytes=8.0 * (m * n + kept * (m + n)), flops=4.0 * s * s * (t - s / 3.0) + 4.0 * kept * m * n)
    if k in ("qn_factorize", "qn_eigsolve"):
        l, r, d = case["l"], case["r"], case["d"]
        nq = 2.5   # about this many sectors hold most of the states
        s = d * min(l, r) / nq
        if k == "qn_factorize":
            return dict(bytes=8.0 * (d * d * l * r / nq + 2 * d * l * r / nq), flops=nq * 6.0 * s ** 3)
        return dict(bytes=8.0 * (D * (l * l + r * r) + 2 * d * d * l * r) / nq,
                    flops=3 * 2.0 * D * d * d * l * r * (l + r) / nq ** 2)
    if k == "dmrg":
        c, N = case["maxdim"], case["N"]
        return dict(bytes=16.0 * N * 3 * c * c, flops=case["nsweeps"] * 2.0 * N * (3 * 180.0 * c ** 3 + 150.0 * c ** 3))
    return dict(bytes=16.0 * case["n"] * 64, flops=case["n"] * 12.0 * 4e4)


def tolerance(case):
    k = case["kind"]
    p = case.get("precision", "fp64")
    if k in ("heff", "eigsolve", "qn_eigsolve"):
        return {"fp64": {"rel": 1e-12}, "fp32": {"rel": 1e-5}, "bf16x3": {"rel": 1e-4}}[p]
    if k == "env":
        return {"rel": 1e-12}
    if k == "expm":
        return {"rel": 1e-10}
    if k in ("factorize", "qn_factorize"):
        # a singular vector is fixed to eps * sigma_max / gap: up to ~1e-8 at the cut
        return {"rel": 1e-7, "max": 1e-5}
    # whole runs: a perturbation of 1e-14 of one start tensor moves the profile by 5e-12
    # (DMRG; every split adds its own rounding) and 2e-16 (the quench)
    return {"rel": 1e-8, "max": 1e-7} if k == "dmrg" else {"rel": 1e-10, "max": 1e-9}


# ----------------------------------------------------------------------- exact
def _apply(L, Ws, R, x):
    """y = H x by contracting one tensor after the other."""
    t = np.tensordot(L, x, axes=(2, 0))                               # a' w s.. b
    for W in Ws:                                                      # w s -> s' w'
        t = np.tensordot(t, W, axes=([1, 2], [0, 3]))                 # a' s.. b .. w' s'
        t = np.moveaxis(t, [-2, -1], [1, -1])
    return np.tensordot(t, R, axes=([1, 2], [1, 2]))                  # a' s1'.. b'


def _lanczos(A, x, K):
    V = [x / np.linalg.norm(x)]
    HV = []
    for j in range(K):
        w = A(V[j])
        HV.append(w)
        if j + 1 < K:
            for _ in range(2):
                for v in V:
                    w = w - np.vdot(v, w) * v
            V.append(w / np.linalg.norm(w))
    T = np.array([[np.vdot(V[i], HV[j]) for j in range(K)] for i in range(K)])
    return V, (T + T.conj().T) / 2


def _ritz(A, x):
    V, T = _lanczos(A, x, 3)
    w, S = np.linalg.eigh(T)
    y = S[:, 0] * (1.0 if S[0, 0] >= 0 else -1.0)
    return float(w[0]), sum(c * v for c, v in zip(y, V))


def _gauge(U):
    """Columns with their largest-magnitude entry positive."""
    j = np.argmax(np.abs(U), axis=0)
    return U * np.where(U[j, np.arange(U.shape[1])] < 0, -1.0, 1.0)


def _truncate(P, maxdim, cutoff):
    """(kept, discarded weight, total) of a decreasing spectrum."""
    n, err, total = len(P), 0.0, P.sum()
    while n > maxdim:
        n -= 1
        err += P[n]
    while n > 1 and err + P[n - 1] <= cutoff * total:
        n -= 1
        err += P[n]
    return n, err / total, total


def _isometry(M, trailing):
    """(isometry columns in the gauge, singular values)."""
    U, s, Vt = np.linalg.svd(M, full_matrices=False)
    return (Vt.T if trailing else U), s


def exact(case, seed):
    k = case["kind"]
    if k in ("heff", "eigsolve", "expm"):
        L, R, W, x = _inputs(case, seed)
        Ws = [W] * case.get("sites", 2)

        def A(v):
            return _apply(L, Ws, R, v)
        if k == "heff":
            return [A(x)]
        if k == "eigsolve":
            e, y = _ritz(A, x)
            return [_num(e), y]
        V, T = _lanczos(A, x, 24)
        w, S = np.linalg.eigh(T)
        c = S @ (np.exp(-0.05j * w) * S[0].conj()) * np.linalg.norm(x)
        return [sum(a * v for a, v in zip(c, V))]
    if k == "env":
        E, A, W = _inputs(case, seed)
        if case["side"] == 0:
            t = np.tensordot(E, A, axes=(2, 0))                        # a' w s b
            t = np.tensordot(t, W, axes=([1, 2], [0, 3]))              # a' b w' s'
            return [np.tensordot(A, t, axes=([0, 1], [0, 3])).transpose(0, 2, 1)]
        t = np.tensordot(E, A, axes=(2, 2))                            # b' v a s
        t = np.tensordot(t, W, axes=([1, 3], [1, 3]))                  # b' a w s'
        return [np.tensordot(A, t, axes=([1, 2], [3, 0])).transpose(0, 2, 1)]
    if k == "factorize":
        M, = _inputs(case, seed)
        Q, s = _isometry(M, case["trailing"])
        kept, err, total = _truncate(s * s, case["maxdim"], case["cutoff"])
        Q = _gauge(Q[:, :kept])
        m, n = M.shape
        split = (m // 2, 2) if m % 2 == 0 else (m, 1)
        if case["trailing"]:
            return [np.ascontiguousarray(Q.T), (M @ Q).reshape(split + (kept,)), _num(err), _num(total), kept]
        return [Q.reshape(split + (kept,)), Q.T @ M, _num(err), _num(total), kept]
    if k == "qn_factorize":
        rng = np.random.default_rng([int(seed), 23])
        theta, parts = _qn_theta(case, rng)
        return _qn_exact_split(case, theta, parts)
    if k == "qn_eigsolve":
        rng = np.random.default_rng([int(seed), 23])
        L, R, x = _qn_operator(case, rng)
        W = _mpo_site(case["d"])
        e, y = _ritz(lambda v: _apply(L, [W, W], R, v), x)
        _, _, ql, qr, qs = _qn_setup(case, None)
        return [_num(e), _pack(y, [ql, qs, qs, qr], [1, 1, 1, -1])]
    return None   # whole runs: a truncated trajectory has no 64-bit value of its own


def _qn_exact_split(case, theta, parts):
    trailing, d = case["trailing"], case["d"]
    _, _, ql, qr, qs = _qn_setup(case, None)
    M = theta.reshape(len(ql) * d, d * len(qr))
    split = [_isometry(M[np.ix_(i, j)], trailing) for _, i, j in parts]
    P = np.sort(np.concatenate([s * s for _, s in split]))[::-1]
    n, err, total = _truncate(P, case["maxdim"], 1e-10)
    cut = -1.0
    if n < len(P):
        cut = (P[n - 1] + P[n]) / 2
        if abs(P[n - 1] - P[n]) < 1e-3 * P[n - 1]:
            cut += 1e-3 * P[n - 1]
    left, right, qm = [], [], []
    for (q, i, j), (Q, s) in zip(parts, split):
        kq = int(np.sum(s * s > cut))
        if kq == 0:
            continue
        Q = _gauge(Q[:, :kq])
        B = M[np.ix_(i, j)]
        lf, rt = np.zeros((len(ql) * d, kq)), np.zeros((kq, d * len(qr)))
        lf[i], rt[:, j] = (B @ Q, Q.T) if trailing else (Q, Q.T @ B)
        left.append(lf)
        right.append(rt)
        qm.append((q, kq))
    q_mid = _charges(qm)
    return [_pack(np.hstack(left).reshape(len(ql), d, -1), [ql, qs, q_mid], [1, 1, -1]),
            _pack(np.vstack(right).reshape(-1, d, len(qr)), [q_mid, qs, qr], [1, 1, -1]), _num(err), _num(total),
            np.array([n for _, n in qm]), np.array([q for q, _ in qm])]


def _pack(a, charges, dirs):
    """The charge-allowed blocks of a dense array, flattened in the order of their sectors
    (a sector: a run of equal charges; site states are sectors of their own)."""
    runs = []
    for q in charges:
        edges = np.concatenate([[0], np.nonzero(np.diff(q))[0] + 1, [len(q)]])
        runs.append([(int(q[a0]), slice(a0, a1)) for a0, a1 in zip(edges[:-1], edges[1:])])
    out = []

    def walk(axis, total, where):
        if axis == len(runs):
            if total == 0:
                out.append(a[tuple(where)].reshape(-1))
            return
        for q, sl in runs[axis]:
            walk(axis + 1, total + dirs[axis] * q, where + [sl])
    walk(0, 0, [])
    return np.concatenate(out)
