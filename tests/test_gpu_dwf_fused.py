"""The domain-wall operator in one pass (the hopping kernel adds the
fifth-dimension term to what it writes) at the edges of its launch shapes:
workgroups with idle threads, several right-hand sides and minor chunks, the
smallest Ls, 16-bit chunks that hold both chiralities, compressed links.
Reference: the Mooee matrices plus the library's Dhop of the same field in
FP64 (itself pinned to the oracle)."""
import numpy as np
import pytest

from conftest import rel_l2, round_storage, storage_tol
from test_gpu_dwf import MASS, M5, mooee_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ls,nrhs", [(2, 1), (3, 2), (16, 1), (17, 1), (11, 9), (24, 6), (256, 1)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("dag", [False, True])
def test_operator_matches_its_terms(gpu, gbx, Ls, nrhs, prec, dag):
    dims = (4, 3, 2, 4)
    dbl = round_storage(gbx.gen_doubled_gauge(dims, 91), prec)
    psi = round_storage(gbx.gen_spinor(dims, Ls, nrhs, 92), prec)
    g = gbx.Geometry(dims)
    U64 = gbx.GaugeField(g, "f64").upload(dbl)
    x64 = gbx.SpinorField(g, Ls, nrhs, "f64").upload(psi)
    h64 = gbx.dhop(U64, gbx.SpinorField(g, Ls, nrhs, "f64"), x64, dag=dag).download()
    want = mooee_np(psi, M5, MASS, dag=dag) - 0.5 * h64
    U = gbx.GaugeField(g, prec).upload(dbl)
    x = gbx.SpinorField(g, Ls, nrhs, prec).upload(psi)
    y = gbx.SpinorField(g, Ls, nrhs, prec)
    gbx.dwf_apply(U, y, x, dag=dag)
    assert rel_l2(y.download(), want) <= storage_tol(prec, gbx.gen_spinor(dims, Ls, nrhs, 92))


def test_operator_with_compressed_links(gpu, gbx):
    dims, Ls = (4, 4, 2, 4), 8
    dbl, psi = gbx.gen_doubled_gauge(dims, 93), gbx.gen_spinor(dims, Ls, 1, 94)
    g = gbx.Geometry(dims)
    x = gbx.SpinorField(g, Ls, 1, "f64").upload(psi)
    out = []
    for c12 in (False, True):
        U = gbx.GaugeField(g, "f64", c12).upload(dbl)
        y = gbx.SpinorField(g, Ls, 1, "f64")
        gbx.dwf_apply(U, y, x)
        out.append(y.download())
    assert rel_l2(out[1], out[0]) <= 1e-14


@pytest.mark.parametrize("Ls", [2, 5, 17, 64, 96])  # 96: sliced in minor chunks, Mooee^-1 in a kernel of its own
@pytest.mark.parametrize("lo", [None, "f32", "f16"])
def test_even_odd_solve_at_the_edges_of_its_shapes(gpu, gbx, Ls, lo):
    dims = (4, 2, 4, 2)
    dbl, psi = gbx.gen_doubled_gauge(dims, 95), gbx.gen_spinor(dims, Ls, 1, 96)
    pair = gbx.Geometry.rb_pair(dims)
    U = [gbx.GaugeField(g, "f64").upload(dbl) for g in pair]
    low = None if lo is None else [gbx.GaugeField(g, lo).upload(dbl) for g in pair]
    b = [gbx.SpinorField(g, Ls, 1, "f64").upload(h) for g, h in zip(pair, gbx.rb_split(dims, psi))]
    x = [gbx.SpinorField(g, Ls, 1, "f64").zero() for g in pair]
    st = gbx.dwf_solve_eo(U, low, x, b, tol=1e-10, max_outer=60)
    assert st["true_resid"] <= 1e-10
    g = gbx.Geometry(dims)
    xl = gbx.SpinorField(g, Ls, 1, "f64").upload(gbx.rb_merge(dims, x[0].download(), x[1].download()))
    y = gbx.dhop(gbx.GaugeField(g, "f64").upload(dbl), gbx.SpinorField(g, Ls, 1, "f64"), xl)
    Dx = mooee_np(xl.download(), M5, MASS) - 0.5 * y.download()
    assert rel_l2(Dx, psi) <= 2e-10
