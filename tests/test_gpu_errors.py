"""Non-finite input on the device paths, through the C ABI: NaN or Inf in theta,
in a Krylov start vector or in H_eff comes back as NSMI_ERR_NOT_FINITE (no
library eigensolver or SVD is handed such values), and the context keeps working
afterwards.  The reference has no such check (a NaN would surface inside LAPACK);
the status is this library's own, declared in include/nsmi.h."""
import numpy as np
import pytest

from oracle import chain, linalg, models

pytestmark = pytest.mark.gpu

NOT_FINITE = -5


@pytest.fixture(scope="module")
def ctx():
    import networksolvers_amd as ns
    c = ns.Context(0)
    yield c
    c.close()


def _graded(m, n, seed):
    rng = np.random.default_rng(seed)
    r = min(m, n)
    U0, _ = np.linalg.qr(rng.standard_normal((m, r)))
    V0, _ = np.linalg.qr(rng.standard_normal((n, r)))
    return (U0 * np.exp(-np.arange(r) / 25.0)) @ V0.T


def _factorize_still_works(ctx, m, n, route):
    import networksolvers_amd as ns
    M = _graded(m, n, 7)
    U, C, info = ns.factorize(ctx.upload(M.reshape(m, 1, 1, n)), 2, False, cutoff=1e-9, which_decomp=route)
    Uo, Co, io = linalg.factorize(M, cutoff=1e-9, which_decomp=route)
    assert info.kept == io.kept
    np.testing.assert_allclose(U.numpy().reshape(m, -1) @ C.numpy().reshape(-1, n), Uo @ Co, atol=1e-12)


# one case per eigensolver path: batched Jacobi (Gram size <= 40), the tridiagonal
# reductions on one XCD (two plans) and over all of them, dsyevd above 1024, and a small
# matrix on the "svd" route
@pytest.mark.parametrize("m,n,route", [(20, 24, "eigen"), (100, 110, "eigen"), (300, 320, "eigen"),
                                       (700, 700, "eigen"), (1100, 1000, "eigen"), (12, 20, "svd")])
@pytest.mark.parametrize("bad,where", [(np.nan, "middle"), (np.inf, "middle"), (np.nan, "corner"),
                                       (-np.inf, "first")])
def test_factorize_rejects_non_finite_theta(ctx, m, n, route, bad, where):
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    M = _graded(m, n, m + n)
    i, j = {"middle": (m // 3, n // 2), "corner": (m - 1, n - 1), "first": (0, 0)}[where]
    M[i, j] = bad
    print(f"factorize non-finite m={m} n={n} route={route} bad={bad} at {where}", flush=True)
    with pytest.raises(NsmiError, match="non-finite") as err:
        ns.factorize(ctx.upload(M.reshape(m, 1, 1, n)), 2, False, cutoff=1e-9, which_decomp=route)
    assert err.value.code == NOT_FINITE
    _factorize_still_works(ctx, min(m, 64), min(n, 70), route)


def test_complex_factorize_rejects_non_finite_theta(ctx):
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    rng = np.random.default_rng(3)
    th = rng.standard_normal((30, 2, 2, 40)) + 1j * rng.standard_normal((30, 2, 2, 40))
    th[4, 1, 0, 17] = complex(0.0, np.nan)
    with pytest.raises(NsmiError, match="non-finite") as err:
        ns.factorize(ctx.upload(th), 2, False, cutoff=1e-10, maxdim=32)
    assert err.value.code == NOT_FINITE
    th[4, 1, 0, 17] = 1.0 + 0.5j
    U, C, info = ns.factorize(ctx.upload(th), 2, False, cutoff=1e-10, maxdim=32)
    assert np.isfinite(info.truncerr) and info.kept == 32


def _tiny_heff(ctx, poison=None, dtype=np.float64):
    """H_eff of the 2-site XXZ chain (dimension 4), optionally with a NaN or Inf
    in L; complex environments (the MPO stays real) when dtype is complex128."""
    import networksolvers_amd as ns
    W = models.xxz_mpo(2)
    L = np.full((1, 1, 1), 1.0 if poison is None else poison, dtype)
    R = np.ones((1, 1, 1), dtype)
    return ns.HeffMap(ctx.upload(L), ctx.upload(W[0]), ctx.upload(W[1]), ctx.upload(R)), W, L, R


def _lanczos_still_works(ctx):
    import networksolvers_amd as ns
    H, W, L, R = _tiny_heff(ctx)
    w = np.linalg.eigvalsh(chain.heff2_dense_matrix(L, W[0], W[1], R))
    x = ctx.upload(np.random.default_rng(5).standard_normal((1, 2, 2, 1)))
    res = ns.lanczos_eig(H, x, krylovdim=4, tol=1e-14)
    assert abs(res.eigval - w[0]) < 1e-12


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_lanczos_rejects_non_finite_start_vector(ctx, bad):
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    H, *_ = _tiny_heff(ctx)
    x0 = np.random.default_rng(1).standard_normal((1, 2, 2, 1))
    x0[0, 1, 0, 0] = bad
    with pytest.raises(NsmiError, match="non-finite") as err:
        ns.lanczos_eig(H, ctx.upload(x0), krylovdim=3)
    assert err.value.code == NOT_FINITE
    _lanczos_still_works(ctx)


def test_lanczos_rejects_non_finite_operator(ctx):
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    H, *_ = _tiny_heff(ctx, poison=np.nan)
    x0 = np.random.default_rng(2).standard_normal((1, 2, 2, 1))
    with pytest.raises(NsmiError, match="non-finite recurrence coefficient") as err:
        ns.lanczos_eig(H, ctx.upload(x0), krylovdim=3)
    assert err.value.code == NOT_FINITE
    _lanczos_still_works(ctx)


@pytest.mark.parametrize("tau", [-0.1, -0.1j])
def test_expm_rejects_non_finite_input(ctx, tau):
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    dt = np.complex128 if isinstance(tau, complex) else np.float64
    x0 = np.random.default_rng(4).standard_normal((1, 2, 2, 1)).astype(dt)
    bad = x0.copy()
    bad[0, 0, 1, 0] = np.nan
    H, *_ = _tiny_heff(ctx, dtype=dt)
    with pytest.raises(NsmiError, match="non-finite") as err:
        ns.krylov_expm(H, ctx.upload(bad), tau, krylovdim=4)
    assert err.value.code == NOT_FINITE
    Hp, *_ = _tiny_heff(ctx, poison=np.inf, dtype=dt)
    with pytest.raises(NsmiError, match="non-finite") as err:
        ns.krylov_expm(Hp, ctx.upload(x0), tau, krylovdim=4)
    assert err.value.code == NOT_FINITE
    _lanczos_still_works(ctx)


def _sector_case(shapes, seed):
    mats = [_graded(m, n, seed + i) for i, (m, n) in enumerate(shapes)]
    offs, flat = [], []
    for M in mats:
        offs.append(sum(x.size for x in flat))
        flat.append(M.reshape(-1))
    return mats, offs, np.concatenate(flat)


def _check_sectors(ctx, mats, offs, buf, shapes):
    from networksolvers_amd import qn
    from oracle import qn as oqn
    rows, cols = [m for m, _ in shapes], [n for _, n in shapes]
    U, C, kept, info = qn._factorize_sectors(ctx, ctx.upload(buf), offs, rows, cols, False, 1e-10, None, 1, "eigen")
    res, okept, oinfo = oqn.factorize_sectors(mats, False, cutoff=1e-10, which_decomp="eigen")
    assert kept == okept
    Uh, Ch = U.numpy(), C.numpy()
    uo = co = 0
    for q, (M, k, (m, n)) in enumerate(zip(mats, kept, shapes)):
        Uq = Uh[uo:uo + m * k].reshape(m, k)
        Cq = Ch[co:co + k * n].reshape(k, n)
        np.testing.assert_allclose(Uq.T @ Uq, np.eye(k), atol=1e-12)
        # the truncated product (cutoff 1e-10 cuts into the graded spectra)
        Uo, Co = res[q] if k else (np.zeros((m, 0)), np.zeros((0, n)))
        np.testing.assert_allclose(Uq @ Cq, Uo @ Co, atol=1e-9)
        uo += m * k
        co += k * n


# sectors on every one-XCD reduction plan (three each on the 65..128 and 129..256 plans, one
# above, one on the 41..64 plan), one Jacobi (30)
_MANY_SHAPES = [(80, 90), (100, 110), (120, 100), (150, 160), (200, 180), (256, 256), (300, 320), (60, 70),
                (30, 35)]


def test_sector_factorize_many_sectors(ctx):
    """Nine sectors spread over the auxiliary streams: every sector's factors equal
    the oracle's (kept counts, U^T U = I, the truncated product U C), a NaN in one
    sector is reported as NSMI_ERR_NOT_FINITE, a give-up forced from the host
    (the timeout flag of the first multi-workgroup reduction raised before its launch)
    as NSMI_ERR_SOLVER, and after each the same context factorises exactly."""
    from networksolvers_amd import qn
    from networksolvers_amd._lib import NsmiError
    mats, offs, buf = _sector_case(_MANY_SHAPES, 40)
    rows, cols = [m for m, _ in _MANY_SHAPES], [n for _, n in _MANY_SHAPES]
    print("many sectors: exact case", flush=True)
    _check_sectors(ctx, mats, offs, buf, _MANY_SHAPES)
    bad = buf.copy()
    bad[offs[4] + 11] = np.nan
    print("many sectors: NaN in sector 4", flush=True)
    with pytest.raises(NsmiError, match="non-finite") as err:
        qn._factorize_sectors(ctx, ctx.upload(bad), offs, rows, cols, False, 1e-10, None, 1, "eigen")
    assert err.value.code == NOT_FINITE
    _check_sectors(ctx, mats, offs, buf, _MANY_SHAPES)
    print("many sectors: injected barrier time-out", flush=True)
    ctx.check(ctx.lib.nsmi_inject_barrier_timeout(ctx.h, 1))
    with pytest.raises(NsmiError, match="timed out at a grid barrier") as err:
        qn._factorize_sectors(ctx, ctx.upload(buf), offs, rows, cols, False, 1e-10, None, 1, "eigen")
    assert err.value.code == -4
    assert "columns, in those from 0 on)" in str(err.value)
    _check_sectors(ctx, mats, offs, buf, _MANY_SHAPES)


@pytest.mark.parametrize("bad_sector", [0, 1, 2])
def test_sector_factorize_rejects_non_finite(ctx, bad_sector):
    """The sector factorisation (independent sectors on several streams: two on the
    reduction path, one on the batched Jacobi path) reports a NaN in any sector as
    NSMI_ERR_NOT_FINITE, and the next call on the same context is exact."""
    from networksolvers_amd import qn
    from networksolvers_amd._lib import NsmiError
    from oracle import qn as oqn
    shapes = [(80, 90), (60, 70), (30, 35)]
    rng = np.random.default_rng(9)
    mats = [_graded(m, n, 20 + i) for i, (m, n) in enumerate(shapes)]
    offs, flat = [], []
    for M in mats:
        offs.append(sum(x.size for x in flat))
        flat.append(M.reshape(-1))
    buf = np.concatenate(flat)
    bad = buf.copy()
    bad[offs[bad_sector] + 7] = np.nan
    rows, cols = [m for m, _ in shapes], [n for _, n in shapes]
    with pytest.raises(NsmiError, match="non-finite") as err:
        qn._factorize_sectors(ctx, ctx.upload(bad), offs, rows, cols, False, 1e-10, None, 1, "eigen")
    assert err.value.code == NOT_FINITE
    U, C, kept, info = qn._factorize_sectors(ctx, ctx.upload(buf), offs, rows, cols, False, 1e-10, None, 1, "eigen")
    res, okept, _ = oqn.factorize_sectors(mats, False, cutoff=1e-10, which_decomp="eigen")
    assert kept == okept
    Uh, Ch = U.numpy(), C.numpy()
    uo = co = 0
    for M, k, (m, n) in zip(mats, kept, shapes):
        Uq = Uh[uo:uo + m * k].reshape(m, k)
        Cq = Ch[co:co + k * n].reshape(k, n)
        np.testing.assert_allclose(Uq.T @ Uq, np.eye(k), atol=1e-12)
        np.testing.assert_allclose(Uq @ Cq, M, atol=1e-9)
        uo += m * k
        co += k * n


def test_frees_from_other_threads_while_the_owner_computes():
    """Tensors whose last reference is dropped on other threads (as a finalizer
    on another serving worker would) while the owner thread keeps allocating and
    applying H_eff on the same context: the pool stays consistent (everything
    released once all handles are gone) and the owner's results stay exact."""
    import queue
    import threading

    import networksolvers_amd as ns
    from networksolvers_amd.kernels import HeffMap

    rng = np.random.default_rng(5)
    cl, cr, D, d = 24, 20, 5, 2
    L = rng.standard_normal((cl, D, cl))
    R = rng.standard_normal((cr, D, cr))
    W = models.heisenberg_mpo(4)[1]
    x = rng.standard_normal((cl, d, d, cr))
    ref = chain.heff2_apply(L, W, W, R, x)
    c = ns.Context(0)
    try:
        base = c.pool_stats()["in_use"]
        inbox = queue.Queue()
        stop = threading.Event()

        def dropper():
            while not stop.is_set() or not inbox.empty():
                try:
                    t = inbox.get(timeout=0.01)
                except queue.Empty:
                    continue
                del t  # the last reference: the free runs on this thread

        workers = [threading.Thread(target=dropper) for _ in range(4)]
        for w in workers:
            w.start()
        H = HeffMap(c.upload(L), c.upload(W), c.upload(W), c.upload(R))
        xd = c.upload(x)
        print("cross-thread frees: 300 H_eff applies, 4 dropper threads", flush=True)
        for it in range(300):
            for k in range(4):
                inbox.put(c.upload(rng.standard_normal(64 + 37 * k)))
            y = H(xd)
            if it % 50 == 0:
                np.testing.assert_allclose(y.numpy(), ref, rtol=1e-12, atol=1e-12 * np.abs(ref).max())
            inbox.put(y)
        stop.set()
        for w in workers:
            w.join()
        del y, xd, H
        import gc
        gc.collect()
        assert c.pool_stats()["in_use"] == base
    finally:
        c.close()


@pytest.mark.parametrize("m,n,route", [(100, 110, "eigen"), (300, 320, "eigen"), (200, 220, "svd"),
                                       (700, 700, "svd"), (1500, 1500, "svd"), (2048, 1024, "svd"),
                                       (128, 100, "svd"), (512, 512, "svd"), (512, 520, "eigen"), (600, 610, "eigen")])
def test_reduction_barrier_give_up_is_reported_and_recovered(ctx, m, n, route):
    """In every column of the one-launch reductions each workgroup waits for all the
    others, with a bounded number of polls; when a wait gives up, every workgroup
    leaves and the call reports NSMI_ERR_SOLVER.  The host forces that path: the
    timeout flag is raised before the launch, the first workgroup then leaves before
    its first column, and the others, waiting for it, in theirs (the error names the
    last block of columns that any of them got to: the first one).  Then the same
    context factorises the same matrix correctly."""
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    M = _graded(m, n, 3)
    print(f"injected barrier time-out m={m} n={n} route={route}", flush=True)
    ctx.check(ctx.lib.nsmi_inject_barrier_timeout(ctx.h, 1))
    with pytest.raises(NsmiError, match="timed out at a grid barrier") as err:
        ns.factorize(ctx.upload(M.reshape(m, 1, 1, n)), 2, False, cutoff=1e-9, which_decomp=route)
    assert err.value.code == -4
    assert f"(of {min(m, n)} columns, in those from 0 on)" in str(err.value)
    _factorize_still_works(ctx, m, n, route)
