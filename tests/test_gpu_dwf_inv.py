"""The closed-form Mooee^-1 kernel where its LDS columns change shape: the
smallest and largest Ls, workgroups with idle threads (Ls not dividing 256),
several right-hand sides, every storage type (a 16-bit chunk holds both
chiralities), both adjoints, and an infinite input.  Reference: the Ls x Ls
matrices of test_gpu_dwf.py, on the values as stored."""
import numpy as np
import pytest

from conftest import rel_l2, round_storage, storage_tol
from test_gpu_dwf import MASS, M5, mooee_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ls,nrhs", [(2, 3), (3, 1), (17, 2), (64, 1), (129, 1), (256, 1)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("dag", [False, True])
def test_inverse_at_the_edges_of_its_columns(gpu, gbx, Ls, nrhs, prec, dag):
    dims = (2, 3, 1, 2)
    psi = gbx.gen_spinor(dims, Ls, nrhs, 77)
    g = gbx.Geometry(dims)
    x = gbx.SpinorField(g, Ls, nrhs, prec).upload(psi)
    y = gbx.SpinorField(g, Ls, nrhs, prec)
    gbx.dwf_mooee(y, x, M5, MASS, inv=True, dag=dag)
    want = mooee_np(round_storage(psi, prec), M5, MASS, inv=True, dag=dag)
    assert rel_l2(y.download(), want) <= storage_tol(prec, psi)


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_infinite_input_stays_in_its_column(gpu, gbx, prec):
    dims, Ls, s0 = (2, 2, 2, 2), 6, 2
    psi = gbx.gen_spinor(dims, Ls, 1, 78)
    psi[0, 3, s0, 1, 2, 0] = np.inf  # P+: reaches s >= s0 directly, s < s0 around the wall with factor -mass
    g = gbx.Geometry(dims)
    x = gbx.SpinorField(g, Ls, 1, prec).upload(psi)
    y = gbx.SpinorField(g, Ls, 1, prec)
    gbx.dwf_mooee(y, x, M5, MASS, inv=True)
    got = y.download()
    col = got[0, 3, :, 1, 2, 0].copy()
    assert np.array_equal(col, np.where(np.arange(Ls) >= s0, np.inf, -np.inf))
    got[0, 3, :, 1, 2, 0] = 0.0
    assert np.isfinite(got).all()
