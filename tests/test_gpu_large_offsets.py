"""Fused hopping kernels on fields next to 4 GiB: below it gathers go by 32-bit
byte offsets (here up to 4.2e9, beyond the signed range), above it by 64-bit
addresses.  A right-hand side in the last place of a large field gives the bits
it gives in a field of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrhs", [42, 44])  # 4.228e9 and 4.429e9 bytes; 2^32 = 4.295e9
@pytest.mark.parametrize("dag", [False, True])
def test_last_right_hand_side_of_a_large_field(gpu, gbx, nrhs, dag):
    dims, Ls = (16, 16, 16, 16), 16
    g = gbx.Geometry(dims)
    U = gbx.GaugeField(g, "f32").upload(gbx.gen_doubled_gauge(dims, 61))
    psi = gbx.gen_spinor(dims, Ls, 1, 62)
    out = []
    for n in (1, nrhs):
        x = gbx.SpinorField(g, Ls, n, "f32").zero()
        x.upload_rhs(n - 1, psi[0])
        y = gbx.SpinorField(g, Ls, n, "f32").zero()
        gbx.dwf_apply(U, y, x, dag=dag)
        out.append(y.download_rhs(n - 1))
    assert np.array_equal(out[0], out[1])
