"""The device-resident inner CG at the edges of its control flow: the smallest
lattices (one partly filled workgroup), an iteration limit below and above
what the tolerance needs, an inner tolerance no precision can reach, and many
partial sums.  Every solution is checked against b with the library's FP64
kernels (pinned to the oracle), and two solves give the same bits."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

KAPPA = 0.11


def system(gbx, dims, Ls, lo, seed=71):
    dbl = gbx.gen_doubled_gauge(dims, seed)
    g = gbx.Geometry(dims)
    U = gbx.GaugeField(g, "f64").upload(dbl)
    Ulo = None if lo is None else gbx.GaugeField(g, lo).upload(dbl)
    b = gbx.SpinorField(g, Ls, 1, "f64").upload(gbx.gen_spinor(dims, Ls, 1, seed + 1))
    return g, U, Ulo, b, gbx.SpinorField(g, Ls, 1, "f64").zero()


def residual(gbx, g, U, x, b):
    t, y = (gbx.SpinorField(g, x.Ls, 1, "f64") for _ in range(2))
    gbx.dhop_axpby(U, t, x, 1.0, -KAPPA)
    gbx.dhop_axpby(U, y, t, 1.0, -KAPPA, dag=True)
    return rel_l2(y.download(), b.download())


@pytest.mark.parametrize("dims,Ls", [((2, 2, 2, 2), 1), ((3, 1, 2, 5), 3), ((4, 4, 4, 4), 16), ((6, 10, 8, 12), 37)])
@pytest.mark.parametrize("lo", [None, "f32", "f16", "bf16"])
def test_solution_at_small_and_ragged_sizes(gpu, gbx, dims, Ls, lo):
    g, U, Ulo, b, x = system(gbx, dims, Ls, lo)
    st = gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-10, max_outer=60)
    assert st["true_resid"] <= 1e-10
    assert residual(gbx, g, U, x, b) <= 2e-10
    assert st["inner_iters"] == st["lo_applies"]
    first = x.download()
    x.zero()
    st2 = gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-10, max_outer=60)
    assert st2["inner_iters"] == st["inner_iters"]
    assert np.array_equal(first, x.download())


@pytest.mark.parametrize("max_inner", [1, 2, 3, 4, 5])
def test_iteration_limit(gpu, gbx, max_inner):
    g, U, Ulo, b, x = system(gbx, (4, 4, 4, 4), 4, "f32")
    st = gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-8, max_outer=400, max_inner=max_inner)
    assert st["true_resid"] <= 1e-8
    assert st["inner_iters"] == max_inner * st["outer_iters"]  # inner_tol is out of reach in 5 steps
    assert residual(gbx, g, U, x, b) <= 2e-8


@pytest.mark.parametrize("lo", ["f32", "f16"])
def test_unreachable_inner_tolerance_stops_at_the_limit(gpu, gbx, lo):
    g, U, Ulo, b, x = system(gbx, (4, 2, 4, 4), 4, lo)
    st = gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-10, inner_tol=1e-60, max_outer=60, max_inner=100)
    assert st["true_resid"] <= 1e-10
    assert st["inner_iters"] <= 100 * st["outer_iters"]
    assert residual(gbx, g, U, x, b) <= 2e-10


def test_no_convergence_is_reported(gpu, gbx):
    g, U, Ulo, b, x = system(gbx, (4, 4, 4, 4), 4, "f32")
    with pytest.raises(gbx.GbxError) as e:
        gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-10, max_outer=1, max_inner=2)
    assert e.value.status == 10
    gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-10)  # and the next solve is not disturbed
    assert residual(gbx, g, U, x, b) <= 2e-10


# the solution is brought up to date every other iteration and when the solve
# ends: an iteration limit at either parity must leave nothing out
@pytest.mark.parametrize("max_inner", [1, 2, 3, 8, 9])
@pytest.mark.parametrize("lo", [None, "f32", "bf16"])
def test_limit_at_either_parity_follows_the_textbook_iteration(gpu, gbx, max_inner, lo):
    dims, Ls = (4, 4, 2, 6), 3
    g, U, Ulo, b, x = system(gbx, dims, Ls, lo)
    with pytest.raises(gbx.GbxError):
        gbx.cg_solve(U, Ulo, x, b, KAPPA, tol=1e-14, inner_tol=1e-13, max_outer=1, max_inner=max_inner)

    t, y = (gbx.SpinorField(g, Ls, 1, "f64") for _ in range(2))
    f = gbx.SpinorField(g, Ls, 1, "f64")

    def A(v):
        f.upload(v)
        gbx.dhop_axpby(U, t, f, 1.0, -KAPPA)
        gbx.dhop_axpby(U, y, t, 1.0, -KAPPA, dag=True)
        return y.download()

    r = b.download()
    e, p, rr = np.zeros_like(r), r.copy(), np.sum(r * r)
    for _ in range(max_inner):
        q = A(p)
        a = rr / np.sum(p * q)
        e += a * p
        r -= a * q
        new = np.sum(r * r)
        p = r + (new / rr) * p
        rr = new
    # p and t are rounded once an iteration to the inner precision (unit 2^-24,
    # 2^-9), which moves a step by at most its condition (1 + 8 KAPPA)^2 /
    # (1 - 8 KAPPA)^2 times that; the steps here shrink, so a few units in all
    unit = {None: 2.0 ** -53, "f32": 2.0 ** -24, "bf16": 2.0 ** -9}[lo]
    assert rel_l2(x.download(), e) <= max(8 * max_inner * unit, 1e-13)
