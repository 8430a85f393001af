"""nsmi_heff_apply_noalloc against nsmi_heff_apply, through the C ABI.

The no-allocation entry point takes the GEMMs' split-K partial sums from a
per-device array instead of the pool; it runs the same kernels with the same
split, so its result must equal the allocating apply bit for bit.  Two calls in a
row on the shared array, the second with a smaller operator (the array keeps the
first call's contents), in the FP64 and FP32 forms, at shapes whose GEMM2 is split
over K (chi = 150: 600 x 150 output on 95 tiles of 32 x 32, K = 750 in 5 splits;
chi 130 x 120: 520 x 120 on 68 tiles, K = 600 in 4), then one whose products need no
partial sums in memory (chi 90 x 70: 36 tiles, K = 350, the one-block form); an operator
form it does not serve is rejected.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import chain, models

pytestmark = pytest.mark.gpu


def _case(ctx, cl, cr, precision, seed):
    import networksolvers_amd as ns
    rng = np.random.default_rng(seed)
    W = models.xxz_mpo(6, Jz=1.0)[2]
    L = rng.standard_normal((cl, 5, cl))
    R = rng.standard_normal((cr, 5, cr))
    th = rng.standard_normal((cl, 2, 2, cr))
    H = ns.HeffMap(ctx.upload(L), ctx.upload(W), ctx.upload(W), ctx.upload(R), precision)
    return H, ctx.upload(th), chain.heff2_apply(L, W, W, R, th)


@pytest.mark.parametrize("precision,bar", [("fp64", 1e-12), ("fp32", 2e-5)])
def test_noalloc_apply_equals_apply(precision, bar):
    import networksolvers_amd as ns
    ctx = ns.Context(0)
    try:
        assert ctx.lib.nsmi_noalloc_scratch_bytes() == 32 << 20
        for cl, cr, seed in [(150, 150, 1), (130, 120, 3), (90, 70, 2)]:
            print(f"noalloc apply {precision} chi_l={cl} chi_r={cr}", flush=True)
            H, x, want = _case(ctx, cl, cr, precision, seed)
            y_ref = H(x).numpy()
            y = ctx.empty(x.shape)
            ctx.check(ctx.lib.nsmi_heff_apply_noalloc(ctx.h, H.h, x.h, y.h))
            got = y.numpy()
            assert np.array_equal(got, y_ref)
            assert np.linalg.norm(got - want) <= bar * np.linalg.norm(want)
    finally:
        ctx.close()


def test_noalloc_rejects_unserved_operators():
    import networksolvers_amd as ns
    from networksolvers_amd._lib import NsmiError
    ctx = ns.Context(0)
    try:
        H, x, _ = _case(ctx, 20, 24, "bf16x3", 3)
        y = ctx.empty(x.shape)
        with pytest.raises(NsmiError, match="FP64 and FP32 forms"):
            ctx.check(ctx.lib.nsmi_heff_apply_noalloc(ctx.h, H.h, x.h, y.h))
        # the context keeps working
        H2, x2, want = _case(ctx, 20, 24, "fp64", 4)
        ctx.check(ctx.lib.nsmi_heff_apply_noalloc(ctx.h, H2.h, x2.h, y.h))
        assert np.linalg.norm(y.numpy() - want) <= 1e-12 * np.linalg.norm(want)
    finally:
        ctx.close()
