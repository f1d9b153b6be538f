"""Links staged into LDS in 16-byte pieces: workgroups of one site to many more
pieces than one round of loads holds, a partly filled last workgroup, 18- and
12-real links (16-bit pieces then straddle links).  The same bits as one site
per 64-thread workgroup, which other tests pin to the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spw,threads", [(2, 64), (5, 64), (11, 64), (23, 64), (48, 64), (64, 256), (3, 256)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("c12", [False, True])
def test_any_number_of_sites_a_workgroup(gpu, gbx, spw, threads, prec, c12):
    dims, Ls = (5, 3, 7, 4), 3
    g = gbx.Geometry(dims)
    U = gbx.GaugeField(g, prec, c12).upload(gbx.gen_doubled_gauge(dims, 64))
    src = gbx.SpinorField(g, Ls, 1, prec).fill_gaussian(65)
    a, b = (gbx.SpinorField(g, Ls, 1, prec) for _ in range(2))
    gbx.dhop(U, a, src, cfg=gbx.kcfg(spw, threads))
    gbx.dhop(U, b, src, cfg=gbx.kcfg(1, 64))
    assert np.array_equal(a.download(), b.download())
