"""The launch shape of a problem nobody tuned, at the edges of its rule
(minor extents around one wavefront, the unchunked limits and the largest;
partly filled workgroups; red-black halves): the same bits as the plainest
shape, one site per 64-thread workgroup without a gather pipeline, for Dhop
and the fused x - b Dhop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MINOR = [(1, 1), (3, 1), (5, 2), (17, 1), (13, 5), (8, 8), (11, 8), (89, 1), (16, 8), (43, 3), (16, 16), (257, 1),
         (64, 64)]


@pytest.mark.parametrize("Ls,nrhs", MINOR)
@pytest.mark.parametrize("prec", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("half", [False, True])
def test_default_shape_matches_the_plain_one(gpu, gbx, Ls, nrhs, prec, half):
    dims = (4, 2, 2, 6) if half else (3, 2, 5, 2)
    dbl = gbx.gen_doubled_gauge(dims, 61)
    if half:
        gout, gin = gbx.Geometry.rb_pair(dims)
    else:
        gout = gin = gbx.Geometry(dims)
    U = gbx.GaugeField(gout, prec).upload(dbl)
    src = gbx.SpinorField(gin, Ls, nrhs, prec).fill_gaussian(62)
    x = gbx.SpinorField(gout, Ls, nrhs, prec).fill_gaussian(63)
    a, b = (gbx.SpinorField(gout, Ls, nrhs, prec) for _ in range(2))
    plain = gbx.kcfg(1, 64)
    for dag in (False, True):
        gbx.dhop(U, a, src, dag=dag)
        gbx.dhop(U, b, src, dag=dag, cfg=plain)
        assert np.array_equal(a.download(), b.download())
        gbx.dhop_xpay(U, a, x, src, 1.0, -0.12, dag=dag)
        gbx.dhop_xpay(U, b, x, src, 1.0, -0.12, dag=dag, cfg=plain)
        assert np.array_equal(a.download(), b.download())
