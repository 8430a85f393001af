"""The MFMA products at the edges of their tiles and K slabs, through the H_eff apply and the
environment update, against NumPy in FP64.

The sizes: one element; below, at and past a 16 x 16 block, a 32 x 32 tile and a K slab
of 16 or 32 (K = chi for the first product, 5 chi for the second); odd leading dimensions
(odd chi); the 64 x 64 tile of FP32 (1505 x 1268); the 128 x 128 tile, ragged on both
sides and in K (2105 x 1796 x 421).  Complex: K below, at and past the 8 of a slab and the 16
of a wave's chunk, fewer and more chunks than the 8 waves, and both sides of the rule between
the forms (252 and 286 tiles of 32 x 32).

Bar: a sum of K rounded products in random signs is off by about sqrt(K) u, three
contractions follow each other and the inputs are rounded once, so 8 sqrt(K) u with K the
longest inner dimension (u = 2^-53, 2^-24 in FP32); the largest seen is about a quarter of that.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DW, D = 5, 2


@pytest.fixture(scope="module")
def ctx():
    import networksolvers_amd as ns
    c = ns.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision,u", [("fp64", 2.0**-53), ("fp32", 2.0**-24)])
@pytest.mark.parametrize("cl,cr", [(1, 1), (3, 2), (15, 17), (16, 16), (17, 31), (32, 33), (63, 65), (129, 95),
                                   (301, 317), (421, 449)])
def test_products_at_tile_edges(ctx, cl, cr, precision, u):
    import networksolvers_amd as ns
    rng = np.random.default_rng(cl * 1000 + cr)
    L, R = rng.standard_normal((cl, DW, cl)), rng.standard_normal((cr, DW, cr))
    W = rng.standard_normal((DW, DW, D, D))
    x = rng.standard_normal((cl, D, D, cr))
    from oracle import chain
    want = chain.heff2_apply(L, W, W, R, x)
    H = ns.HeffMap(ctx.upload(L), ctx.upload(W), ctx.upload(W), ctx.upload(R), precision)
    got = H(ctx.upload(x)).numpy()
    K = DW * max(cl, cr)
    assert np.linalg.norm(got - want) <= 8 * np.sqrt(K) * u * np.linalg.norm(want)


@pytest.mark.parametrize("precision,bar", [("bf16x3", 2.0**-15), ("bf16", 2.0**-7)])
@pytest.mark.parametrize("cl,cr", [(1, 1), (7, 9), (15, 17), (33, 31), (63, 65), (129, 95), (251, 259), (421, 449)])
def test_bf16_products_at_tile_edges(ctx, cl, cr, precision, bar):
    """Tiles of 32, 64 (1255 x 1036, 340 of them) and 128 (2105 x 1796).  Two products follow
    each other, each with two operands rounded to 2^-9 (split in two: 2^-17, and 2^-18 for the
    product of the low parts that is left out): at most 4 x 2^-9 and 5 x 2^-17 of the norm."""
    import networksolvers_amd as ns
    from oracle import chain
    rng = np.random.default_rng(cl * 1000 + cr)
    L, R = rng.standard_normal((cl, DW, cl)), rng.standard_normal((cr, DW, cr))
    W = rng.standard_normal((DW, DW, D, D))
    x = rng.standard_normal((cl, D, D, cr))
    want = chain.heff2_apply(L, W, W, R, x)
    got = ns.HeffMap(ctx.upload(L), ctx.upload(W), ctx.upload(W), ctx.upload(R), precision)(ctx.upload(x)).numpy()
    assert np.linalg.norm(got - want) <= bar * np.linalg.norm(want)


@pytest.mark.parametrize("Dw,d,sites", [(1, 2, 1), (6, 2, 1), (7, 2, 1), (5, 2, 2), (3, 3, 2), (5, 3, 2), (7, 3, 2)])
@pytest.mark.parametrize("cl,cr", [(2, 255), (300, 257)])
def test_bf16_mixing_widths(ctx, Dw, d, sites, cl, cr):
    """Widths (Dw d^sites = 2 to 63) on both sides of the padded ones (12, 20, 32, 48, 64), with an
    output count that is no multiple of four, columns at the edge of a workgroup, few and many rows."""
    import networksolvers_amd as ns
    from oracle import chain
    rng = np.random.default_rng(Dw * 100 + d)
    L, R, W = rng.standard_normal((cl, Dw, cl)), rng.standard_normal((cr, Dw, cr)), rng.standard_normal((Dw, Dw, d, d))
    x = rng.standard_normal((cl,) + (d,) * sites + (cr,))
    want = chain.heff2_apply(L, W, W, R, x) if sites == 2 else chain.heff1_apply(L, W, R, x)
    H = ns.HeffMap(ctx.upload(L), ctx.upload(W), ctx.upload(W) if sites == 2 else None, ctx.upload(R), "bf16x3")
    assert np.linalg.norm(H(ctx.upload(x)).numpy() - want) <= 2.0**-15 * np.linalg.norm(want)


def _crand(rng, shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("precision,u", [("fp64", 2.0**-53), ("fp32", 2.0**-24)])
@pytest.mark.parametrize("cl,cr", [(1, 1), (8, 9), (9, 2), (15, 17), (16, 16), (17, 31), (33, 32), (129, 95), (135, 97)])
def test_complex_products_at_tile_edges(ctx, cl, cr, precision, u):
    import networksolvers_amd as ns
    from oracle import chain
    rng = np.random.default_rng(cl * 1000 + cr)
    L, R, W = _crand(rng, (cl, DW, cl)), _crand(rng, (cr, DW, cr)), rng.standard_normal((DW, DW, D, D))
    x = _crand(rng, (cl, D, D, cr))
    want = chain.heff2_apply(L, W, W, R, x)
    H = ns.HeffMap(ctx.upload(L), ctx.upload(W), ctx.upload(W), ctx.upload(R), precision)
    got = H(ctx.upload(x)).numpy()
    K = DW * max(cl, cr)
    assert np.linalg.norm(got - want) <= 8 * np.sqrt(2 * K) * u * np.linalg.norm(want)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("ca,cb", [(1, 9), (8, 16), (17, 15), (31, 65), (129, 95)])
def test_complex_environment_products_at_tile_edges(ctx, ca, cb, side):
    import networksolvers_amd as ns
    from oracle import chain
    rng = np.random.default_rng(ca * 1000 + cb)
    A, W = _crand(rng, (ca, D, cb)), rng.standard_normal((DW, DW, D, D))
    E = _crand(rng, (ca, DW, ca) if side == 0 else (cb, DW, cb))
    want = chain.env_left(E, A, W) if side == 0 else chain.env_right(E, A, W)
    got = ns.env_update(ctx.upload(E), ctx.upload(A), ctx.upload(W), side).numpy()
    K = DW * max(ca, cb)
    assert np.linalg.norm(got - want) <= 8 * np.sqrt(2 * K) * 2.0**-53 * np.linalg.norm(want)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("ca,cb", [(1, 3), (15, 17), (31, 65), (95, 129), (451, 449)])
def test_environment_products_at_tile_edges(ctx, ca, cb, side):
    import networksolvers_amd as ns
    from oracle import chain
    rng = np.random.default_rng(ca * 1000 + cb)
    A, W = rng.standard_normal((ca, D, cb)), rng.standard_normal((DW, DW, D, D))
    E = rng.standard_normal((ca, DW, ca) if side == 0 else (cb, DW, cb))
    want = chain.env_left(E, A, W) if side == 0 else chain.env_right(E, A, W)
    got = ns.env_update(ctx.upload(E), ctx.upload(A), ctx.upload(W), side).numpy()
    K = DW * max(ca, cb)
    assert np.linalg.norm(got - want) <= 8 * np.sqrt(K) * 2.0**-53 * np.linalg.norm(want)


def test_fp32_partial_sums_are_added_in_fp64(ctx):
    """The FP32 form writes y in FP64: where a product splits its K = 512 over waves or
    workgroups, the partial sums are added in FP64 and not rounded on the way.  Two terms,
    2^24 at k = 0 and 1 at k = 144, lie in different parts of every split (parts of 16 dealt to
    8 waves; parts of 128): their sum needs 25 bits and comes out exactly."""
    import networksolvers_amd as ns
    n = 512
    L, W, R = np.ones((1, 1, 1)), np.eye(D).reshape(1, 1, D, D), np.zeros((n, 1, n))
    R[0, 0, :] = 1.0
    x = np.zeros((1, D, D, n))
    x[0, 0, 0, 0], x[0, 0, 0, 144] = 2.0**24, 1.0
    H = ns.HeffMap(ctx.upload(L), ctx.upload(W), ctx.upload(W), ctx.upload(R), "fp32")
    got = H(ctx.upload(x)).numpy()
    assert got[0, 0, 0, 0] == 2.0**24 + 1.0
    assert np.count_nonzero(got) == 1
