"""The one-launch reductions behind the truncated factorisation at the edges of their plans.

Tolerances: an SVD's backward error is c n eps ||M|| with a small c; n <= 4096 gives
1e-12, and the measured values are 5e-15.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import networksolvers_amd as ns
    c = ns.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("m,n", [(32, 31), (33, 32), (65, 64), (129, 63), (257, 64), (2049, 5), (129, 128), (257, 65),
                                 (1025, 128), (2049, 127), (257, 256), (513, 129), (1025, 256), (513, 512),
                                 (600, 512), (2049, 513), (1025, 1025)])
def test_bidiagonalisation_plan_edges(ctx, m, n):
    """First shapes past each plan's limits (rows and columns; one workgroup, one XCD with
    and without sliced columns, all XCDs): M = U C, orthonormal U, the row norms of C the
    singular values, on both sides."""
    import networksolvers_amd as ns
    M = np.random.default_rng(m * 5000 + n).standard_normal((m, n))
    s = np.linalg.svd(M, compute_uv=False)
    print(f"bidiagonalisation m={m} n={n}", flush=True)
    x = ctx.upload(M)
    for trailing in (False, True):
        U, C, info = ns.factorize(x, 1, trailing, cutoff=0.0, which_decomp="svd")
        assert info.route == "svd" and info.kept == n
        u, c = (U.numpy().T, C.numpy().T) if trailing else (U.numpy(), C.numpy())
        A = M.T if trailing else M
        assert np.linalg.norm(u @ c - A) < 1e-12 * np.linalg.norm(M)
        assert np.abs(u.T @ u - np.eye(n)).max() < 1e-12
        assert np.abs(np.linalg.norm(c, axis=1) - s).max() < 1e-12 * s[0]


@pytest.mark.parametrize("n", [41, 64, 65, 100, 128, 129, 192, 256, 257, 385, 512, 513, 1000, 1024])
def test_tridiagonalisation_plan_edges(ctx, n):
    """The eigen route at the edges of the tridiagonalisation's plans, on a matrix with
    well-separated squares: the kept eigenvalues, orthonormal U, C = U^T M, and each
    column an eigenvector of the Gram matrix to n eps of its norm."""
    import networksolvers_amd as ns
    M = np.random.default_rng(n).standard_normal((n, n + 3))
    k = n // 2
    print(f"tridiagonalisation n={n}", flush=True)
    U, C, info = ns.factorize(ctx.upload(M), 1, False, cutoff=0.0, maxdim=k, which_decomp="eigen")
    u, c = U.numpy(), C.numpy()
    s = np.linalg.svd(M, compute_uv=False)
    assert info.route == "eigen" and info.kept == k
    assert np.abs(u.T @ u - np.eye(k)).max() < 1e-12
    assert np.linalg.norm(u.T @ M - c) < 1e-12 * np.linalg.norm(M)
    assert np.abs(np.linalg.norm(c, axis=1) - s[:k]).max() < 1e-12 * s[0]
    assert np.abs(M @ (M.T @ u) - u * s[:k] ** 2).max() < 1e-12 * s[0] ** 2


def test_bidiagonalisation_of_special_matrices(ctx):
    """Zero and rank-one matrices, and entries whose squares are near the ends of the range:
    finite results, orthonormal U, the rank-one matrix reproduced."""
    import networksolvers_amd as ns
    rng = np.random.default_rng(11)
    for m, n in ((40, 40), (150, 130), (300, 280)):
        one = np.outer(rng.standard_normal(m), rng.standard_normal(n))
        for name, M in (("zero", np.zeros((m, n))), ("rank one", one), ("small", 1e-146 * rng.standard_normal((m, n))),
                        ("large", 1e145 * rng.standard_normal((m, n)))):
            print(f"special {name} m={m} n={n}", flush=True)
            U, C, info = ns.factorize(ctx.upload(M), 1, False, cutoff=0.0, maxdim=7, which_decomp="svd")
            u, c = U.numpy(), C.numpy()
            assert np.isfinite(u).all() and np.isfinite(c).all()
            assert np.abs(u.T @ u - np.eye(info.kept)).max() < 1e-11
            if name == "rank one":
                assert np.linalg.norm(u @ c - M) < 1e-12 * np.linalg.norm(M)


def test_reductions_on_more_streams_than_places(ctx):
    """18 contexts (streams) share the 16 places of the one-XCD groups: results equal to
    the first context's, bit for bit, with all launches in flight from several threads."""
    import threading

    import networksolvers_amd as ns
    M = np.random.default_rng(3).standard_normal((150, 140))
    ctxs = [ns.Context(0) for _ in range(18)]
    want = ns.factorize(ctx.upload(M), 1, False, cutoff=0.0, maxdim=20, which_decomp="svd")[1].numpy()
    got, errors = {}, []

    def work(ids):
        try:
            for _ in range(3):
                for i in ids:
                    got[i] = ns.factorize(ctxs[i].upload(M), 1, False, cutoff=0.0, maxdim=20,
                                          which_decomp="svd")[1].numpy()
        except Exception as ex:   # noqa: BLE001
            errors.append(ex)
    ts = [threading.Thread(target=work, args=(range(t, 18, 6),)) for t in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for c in ctxs:
        c.close()
    assert not errors
    for i in range(18):
        np.testing.assert_array_equal(got[i], want)


def _reduce_launches(ctx, fn):
    """fn() with the reductions' launches counted."""
    ctx.profile(True)
    ctx.profile_reset()
    out = fn()
    n = ctx.profile_stats()["fact_reduce"]["launches"]
    ctx.profile(False)
    return out, n


@pytest.mark.parametrize("m,n,route", [(60, 64, "svd"), (128, 100, "svd"), (300, 70, "svd"), (300, 280, "svd"),
                                       (512, 500, "svd"), (700, 520, "svd"), (64, 90, "eigen"), (130, 140, "eigen"),
                                       (300, 310, "eigen"), (512, 520, "eigen")])
def test_misplaced_groups_give_the_same_result(ctx, m, n, route):
    """A group that does not get the XCD it asks for leaves without having started and is
    launched again over the whole device (up to 512 columns and rows), once more when that
    placement times out; one over all XCDs (700 x 520) is formed in the grid's order.  Every
    sum has a fixed order, so the factors are the same bit for bit."""
    import networksolvers_amd as ns
    x = ctx.upload(np.random.default_rng(m + n).standard_normal((m, n)))
    print(f"misplaced m={m} n={n} route={route}", flush=True)

    def run():
        U, C, info = ns.factorize(x, 1, False, cutoff=1e-10, maxdim=20, which_decomp=route)
        return U.numpy(), C.numpy(), info.route
    (u, c, r), once = _reduce_launches(ctx, run)
    assert once == 1
    for count in (1,) if m == 700 else (1, 2):
        ctx.check(ctx.lib.nsmi_inject_misplacement(ctx.h, count))
        (u1, c1, r1), launches = _reduce_launches(ctx, run)
        assert launches == (1 if m == 700 else 1 + count) and r == r1
        np.testing.assert_array_equal(u, u1)
        np.testing.assert_array_equal(c, c1)


def test_misplaced_sector_groups_give_the_same_result(ctx):
    """Three of six sectors' groups, on four streams, are launched again; the sectors' factors
    are the same bit for bit."""
    from networksolvers_amd import qn
    shapes = [(80, 90), (60, 70), (300, 200), (30, 35), (150, 149), (45, 200)]
    rng = np.random.default_rng(5)
    offs = np.concatenate([[0], np.cumsum([m * n for m, n in shapes])])[:-1].tolist()
    buf = ctx.upload(rng.standard_normal(sum(m * n for m, n in shapes)))
    rows, cols = [m for m, _ in shapes], [n for _, n in shapes]

    def run():
        U, C, kept, _ = qn._factorize_sectors(ctx, buf, offs, rows, cols, False, 1e-10, 100, 1, "eigen")
        return U.numpy(), C.numpy(), kept
    (u, c, k), once = _reduce_launches(ctx, run)
    print("misplaced sectors", flush=True)
    ctx.check(ctx.lib.nsmi_inject_misplacement(ctx.h, 3))
    (u1, c1, k1), more = _reduce_launches(ctx, run)
    assert (once, more) == (5, 8) and k == k1
    np.testing.assert_array_equal(u, u1)
    np.testing.assert_array_equal(c, c1)


@pytest.mark.parametrize("m,n,route,limit", [(250, 250, "svd", 4506624), (422, 394, "svd", 15894016),
                                             (600, 600, "svd", 32049664), (1000, 800, "svd", 61934080),
                                             (2048, 2048, "svd", 312611328), (700, 710, "eigen", 27339264)])
def test_factorisation_fits_the_pool_it_fitted(m, n, route, limit):
    """Pool limits that held a factorisation with k = n / 2 when the reductions' exchange was
    smaller (two buffers, 8 to 256 workgroups) still hold it: the exchange is given back before
    the vectors' solves, where the peak is."""
    import networksolvers_amd as ns
    c = ns.Context(0)
    x = c.upload(np.random.default_rng(1).standard_normal((m, n)))
    ns.factorize(x, 1, False, cutoff=0.0, maxdim=min(m, n) // 2, which_decomp=route)
    assert c.pool_stats()["peak"] <= limit
    del x
    c.close()


def _same_from_threads(ctx, ctxs, work, rounds):
    """Every context factorises the matrices of `work` in turn, five threads sharing the
    contexts; C is compared with that of `ctx` alone."""
    import threading

    import networksolvers_amd as ns

    def run(c, M, route):
        return ns.factorize(c.upload(M), 1, False, cutoff=0.0, maxdim=20, which_decomp=route)[1].numpy()
    want = [run(ctx, M, route) for M, route in work]
    errors = []

    def worker(t):
        try:
            for it in range(rounds):
                for i in range(t, len(ctxs), 5):
                    j = (t + it + i) % len(work)
                    np.testing.assert_array_equal(run(ctxs[i], *work[j]), want[j])
        except BaseException as ex:   # noqa: BLE001
            errors.append(ex)
    ts = [threading.Thread(target=worker, args=(t,)) for t in range(5)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors


def test_full_groups_of_many_streams_at_once(ctx):
    """Groups of up to 32 workgroups that fill half of an XCD each (four waves of 256 registers,
    n = 500 on the eigen route; eight of 128, 500 x 490 on the svd route), from ten contexts on
    five threads, several of them in flight at any time on places of the same XCD: every
    result equals the first context's, bit for bit."""
    import networksolvers_amd as ns
    rng = np.random.default_rng(4)
    work = [(rng.standard_normal((500, 510)), "eigen"), (rng.standard_normal((500, 490)), "svd"),
            (rng.standard_normal((1000, 120)), "svd")]
    ctxs = [ns.Context(0) for _ in range(10)]
    print("full groups of ten streams", flush=True)
    _same_from_threads(ctx, ctxs, work, 4)
    for c in ctxs:
        c.close()


def test_groups_over_the_device_beside_groups_of_one_xcd(ctx):
    """Contexts on five threads mix groups over all XCDs (1100 x 520 and 700 x 700 on the svd
    route, n = 600 on the eigen route) with groups that fill half of an XCD: every result
    equals the first context's, bit for bit."""
    import networksolvers_amd as ns
    rng = np.random.default_rng(6)
    work = [(rng.standard_normal((1100, 520)), "svd"), (rng.standard_normal((500, 490)), "svd"),
            (rng.standard_normal((700, 700)), "svd"), (rng.standard_normal((500, 510)), "eigen"),
            (rng.standard_normal((600, 610)), "eigen")]
    ctxs = [ns.Context(0) for _ in range(10)]
    print("groups over the device beside groups of one XCD", flush=True)
    _same_from_threads(ctx, ctxs, work, 5)
    for c in ctxs:
        c.close()


_PROCESS = """
import sys
import numpy as np
import networksolvers_amd as ns
seed = int(sys.argv[1])
ctx = ns.Context(0)
rng = np.random.default_rng(seed)
work = [(rng.standard_normal((500, 490)), "svd"), (rng.standard_normal((500, 510)), "eigen"),
        (rng.standard_normal((150, 140)), "svd"), (rng.standard_normal((700, 600)), "svd")]
print("ready", flush=True)
sys.stdin.readline()
for it in range(8):
    for M, route in work:
        C = ns.factorize(ctx.upload(M), 1, False, cutoff=0.0, maxdim=20, which_decomp=route)[1].numpy()
        s = np.linalg.svd(M, compute_uv=False) if it == 0 else None
        if it == 0:
            assert np.abs(np.linalg.norm(C, axis=1) - s[:20]).max() < 1e-12 * s[0]
            first = globals().setdefault("first", {})
            first[M.shape] = C
        assert np.array_equal(C, first[M.shape])
ctx.close()
"""


def test_groups_of_several_processes(ctx):
    """Three processes, started together, factorise at the same time, with groups that fill half
    of an XCD and groups over all of them; none knows of the others' launches."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, OMP_NUM_THREADS="4")
    procs = [subprocess.Popen([sys.executable, "-c", _PROCESS, str(seed)], cwd=root, env=env, text=True,
                              stdin=subprocess.PIPE, stdout=subprocess.PIPE, stderr=subprocess.PIPE)
             for seed in range(3)]
    try:
        for p in procs:
            assert p.stdout.readline().strip() == "ready"
        print("three processes", flush=True)
        for p in procs:
            p.stdin.write("go\n")
            p.stdin.flush()
        for p in procs:
            _, err = p.communicate(timeout=60)
            assert p.returncode == 0, err[-2000:]
    finally:
        for p in procs:
            if p.poll() is None:
                p.kill()
