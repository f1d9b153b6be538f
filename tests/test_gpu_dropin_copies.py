"""Drop-in calls whose host arrays go through the pinned staging ring: pieces
that do not divide the arrays, more pieces than buffers, arrays on both sides
of the size that takes the ring, on both device paths and on a context used
for several shapes in turn.  Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("canonical", [True, False])
def test_staged_arrays_arrive_whole(gpu, gbx, orc, dtype, canonical):
    with gbx.DslashContext() as ctx:
        for dims, Ls in (((4, 4, 4, 4), 3), ((8, 8, 8, 12), 9), ((12, 12, 8, 16), 7), ((4, 6, 4, 4), 5)):
            V = int(np.prod(dims))
            nbr, prm = orc.tables(dims, 1, Ls)
            if not canonical:
                nbr = nbr.copy()
                nbr[5 * 8 + 2], nbr[-3] = V * Ls - 1, 0  # still valid, no periodic lattice's
            U = orc.aligned_copy(orc.pack_gauge(dims, 1, gbx.gen_doubled_gauge(dims, 31)).astype(dtype))
            src = orc.aligned_copy(orc.pack_spinor(dims, 1, Ls, gbx.gen_spinor(dims, Ls, 1, 32)[0]).astype(dtype))
            want = orc.hand(U, src, nbr, prm, V, Ls, 1, nthreads=8)
            for _ in range(2):
                out = np.full_like(src, np.nan)
                ctx.kernel(1, U, out, src, nbr, V, Ls, prm, 1)
                assert ctx.last_path() == (1 if canonical else 2)
                assert np.array_equal(out, want)
