"""Batch work items at the edges of their size rule (minor extents below, at
and above a workgroup's points, a lattice smaller than an item): the same bits
as one application per lattice, from the graph and the no-allocation entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32", "f16", "bf16"])
def test_items_cover_every_point(gpu, gbx, prec):
    shapes = [((2, 3, 2, 2), 1, 1), ((3, 2, 4, 5), 24, 1), ((2, 2, 2, 3), 17, 15), ((2, 2, 3, 2), 16, 16),
              ((2, 2, 2, 2), 257, 1), ((4, 4, 2, 2), 3, 1)]
    U, src, dst, want = [], [], [], []
    for i, (dims, Ls, nrhs) in enumerate(shapes):
        g = gbx.Geometry(dims)
        U.append(gbx.GaugeField(g, prec).upload(gbx.gen_doubled_gauge(dims, 41 + i)))
        src.append(gbx.SpinorField(g, Ls, nrhs, prec).fill_gaussian(51 + i))
        dst.append(gbx.SpinorField(g, Ls, nrhs, prec).zero())
        want.append(gbx.dhop(U[-1], gbx.SpinorField(g, Ls, nrhs, prec), src[-1]).download())
    b = gbx.Batch(U, dst, src)
    for _ in range(2):
        b.run()
        for d, w in zip(dst, want):
            assert np.array_equal(d.download(), w)
            d.zero()
    gbx.batch_run_noalloc(U, dst, src)
    for d, w in zip(dst, want):
        assert np.array_equal(d.download(), w)
