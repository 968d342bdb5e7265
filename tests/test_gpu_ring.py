"""The solvers' ring of search directions (PRing, wl_internal.h: x += alpha_i p_i of several
iterations in one pass) on the GPU: solves that stop or take a reliable update at every place in
the ring.  The one-launch CG updates x in every iteration, with the same sums, so the ring gives
its bits; a solve with a reliable update must reach its true residual, and the FP64 solution to
that residual over the smallest eigenvalue of M^dag M (above 1e-3 for these links)."""
import numpy as np
import pytest

from hila_amd import wilson as W

pytestmark = pytest.mark.gpu
KAPPA = 0.124


@pytest.fixture(scope="module", params=[(8, 8, 8, 8), (12, 6, 10, 14), (16, 16, 16, 32)])
def lattice(request):
    dims = request.param
    lat = W.Lattice(dims)
    lat.upload_gauge(W.gen_gauge(dims, "smooth", 0.3, 11))
    return dims, lat


def _solve(lat, b, n, tol, maxiters, **how):
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    x = W.Field(lat, nrhs=n)
    x.upload(W.gen_spinor(lat.dims, 5) * 0.1, 0)  # a guess: x is read before it is written
    st = W.CG(D, tol, maxiters, **how).apply(b, x)
    return [x.download(j) for j in range(n)], st


@pytest.mark.parametrize("maxiters", [0, 1, 2, 3, 7, 8, 9, 10, 10000])
@pytest.mark.parametrize("mode", [0, -1])
def test_fp64_solve_has_the_bits_of_the_one_launch_solve(lattice, maxiters, mode):
    dims, lat = lattice
    lat.set_option(W.OPT_SMALL_HOP, -1)  # one lane per site, as the one-launch solve
    b = W.Field(lat).upload(W.gen_spinor(dims, 6))
    lat.set_option(W.OPT_CG_PERSISTENT, mode)
    (x,), (st,) = _solve(lat, b, 1, 1e-10, maxiters)
    lat.set_option(W.OPT_CG_PERSISTENT, 1)
    (y,), (su,) = _solve(lat, b, 1, 1e-10, maxiters)
    lat.set_option(W.OPT_CG_PERSISTENT, 0)
    lat.set_option(W.OPT_SMALL_HOP, 0)
    assert np.array_equal(x, y)
    assert (st["iterations"], st["true_resid"]) == (su["iterations"], su["true_resid"])


@pytest.mark.parametrize("update_every", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("precision,n", [("f32", 1), ("f64-mixed", 1), ("f32", 3), ("f16", 1), ("f16", 6)])
def test_reliable_update_at_every_place_in_the_ring(lattice, precision, n, update_every):
    dims, lat = lattice
    lat.set_option(W.OPT_SMALL_HOP, -1)
    b = W.Field(lat, nrhs=n)
    for j in range(n):
        b.upload(W.gen_spinor(dims, 6 + j), j)
    tol = 1e-9
    xs, sts = _solve(lat, b, n, tol, 20000, precision=precision, delta=1e-4, update_every=update_every)
    refs, _ = _solve(lat, b, n, 1e-12, 20000)
    lat.set_option(W.OPT_SMALL_HOP, 0)
    for j in range(n):
        assert sts[j]["converged"] == 1 and sts[j]["true_resid"] <= tol
        assert np.linalg.norm(xs[j] - refs[j]) <= 1e3 * tol * np.linalg.norm(b.download(j))


@pytest.mark.parametrize("maxiters", [1, 2, 3, 4, 5, 11])
@pytest.mark.parametrize("precision", ["f64", "f32", "f16"])
def test_batched_solve_that_stops_at_maxiters(lattice, precision, maxiters):
    # the true residual that the solve reports is that of the x it returns: recomputed from x by a
    # solve of no iterations
    dims, lat = lattice
    n = 2
    b = W.Field(lat, nrhs=n)
    for j in range(n):
        b.upload(W.gen_spinor(dims, 6 + j), j)
    xs, sts = _solve(lat, b, n, 1e-13, maxiters, precision=precision, delta=1e-4, update_every=100)
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    for j in range(n):
        assert sts[j]["iterations"] == maxiters and sts[j]["converged"] == 0
        one, x = W.Field(lat).upload(b.download(j)), W.Field(lat).upload(xs[j])
        (again,) = W.CG(D, 1e-13, 0).apply(one, x)
        assert abs(again["true_resid"] - sts[j]["true_resid"]) <= 1e-10 * sts[j]["true_resid"]
        assert sts[j]["true_resid"] < 1.0
