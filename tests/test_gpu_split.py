"""The direction-split FP64 multi-rhs hopping kernel (wl_split.h) on the GPU, against the lane-per-site
kernel (wl_rb.h), which a caller's WL_OPT_RHS_BLOCK selects, and against the FP64 oracle.

Both kernels form the same products and add the eight hops in another order.  A component of
a hop's sum goes through at most 16 roundings (projection 1, link product 6, the eight hops
and the four directions 9), so the two differ by at most 2 x 16 eps times the sum of the absolute
terms; the terms of one hop have a norm of at most 2 |in| (|1 +- gamma_mu| = 2, links unitary),
and there are eight: |a - b| <= 512 eps |in|.  M = 1 - kappa^2 H H: twice that times kappa^2 |H|
(8 on unit links: at most 16) x 512 eps, and the roundings of its own sum, 4 eps."""
import numpy as np
import pytest

from hila_amd import wilson as W
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
KAPPA = 0.12
EPS = 2.0 ** -53
HOP = 512
M = 2 * KAPPA ** 2 * 16 * HOP + 4

# lattices that take the split kernel: whole tiles of 128 sites, tiles with idle lanes, partial tiles
# in y or z, rows that are no power of two, short and long ones
LATTICES = [(16, 16, 16, 32), (20, 20, 20, 20), (14, 18, 14, 64), (28, 14, 18, 38), (10, 26, 24, 32), (40, 20, 16, 20)]


def _fields(lat, dims, n, parity=W.EVEN):
    f = W.Field(lat, parity, W.F64, n)
    for j in range(n):
        f.upload(W.gen_spinor(dims, 100 + j, 1 if parity == W.EVEN else 2), j)
    return f


@pytest.mark.parametrize("dims", LATTICES)
@pytest.mark.parametrize("rows,n", [(3, 12), (2, 13)])
def test_agrees_with_the_lane_per_site_kernel(dims, rows, n):
    lat = W.Lattice(dims, antiperiodic_t=n != 13)
    lat.set_option(W.OPT_LINK_ROWS, rows)
    # two-row storage takes links that are special unitary to 1e-13 only: the smooth ones are
    lat.upload_gauge(W.gen_gauge(dims, "haar" if rows == 3 else "smooth", 0 if rows == 3 else 0.3, 5))
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    H = W.Hasenbusch_operator(D, 0.1)
    got = []
    for nr in (0, 1):
        lat.set_option(W.OPT_RHS_BLOCK, nr)
        outs = []
        for parity in (W.EVEN, W.ODD):
            fin = _fields(lat, dims, n, parity)
            norm = [np.linalg.norm(fin.download(j)) for j in range(n)]
            hop, m = W.Field(lat, 3 - parity, W.F64, n), W.Field(lat, W.EVEN, W.F64, n)
            for sign in (1, -1):
                D.hop_set(fin, hop, sign)
                outs += [(hop.download(j), norm[j], HOP) for j in range(n)]
            if parity == W.EVEN:
                H.apply(fin, m)
                outs += [(m.download(j), norm[j], M) for j in range(n)]
                D.dagger(fin, m)
                outs += [(m.download(j), norm[j], M) for j in range(n)]
        got.append(outs)
    for (a, norm, bar), (b, _, _) in zip(*got):
        assert np.linalg.norm(a - b) <= bar * EPS * norm


def test_against_the_oracle():
    dims, n = (20, 20, 20, 20), 9
    U = W.gen_gauge(dims, "haar", 0, 6)
    lat = W.Lattice(dims)
    lat.upload_gauge(U)
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    fin, out = _fields(lat, dims, n), W.Field(lat, W.EVEN, W.F64, n)
    orc = Oracle(dims)
    D.apply(fin, out)
    for j in (0, n - 1):
        src = W.gen_spinor(dims, 100 + j)
        ref = orc.meo(U, KAPPA, src, 1)
        assert np.linalg.norm(out.to_full(j) - ref) <= M * EPS * np.linalg.norm(src)


@pytest.mark.parametrize("dims", [(16, 16, 16, 16), (10, 26, 24, 32)])  # in one group, in four
def test_most_right_hand_sides(dims):
    n = 64
    lat = W.Lattice(dims)
    lat.upload_gauge(W.gen_gauge(dims, "haar", 0, 7))
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    fin, out = W.Field(lat, W.EVEN, W.F64, n), W.Field(lat, W.ODD, W.F64, n)
    src = [W.gen_spinor(dims, 100 + j) for j in range(4)]
    for j in range(n):
        fin.upload(src[j % 4], j)
    D.hop_set(fin, out)
    first = [out.download(j) for j in range(4)]
    for j in range(4, n):
        assert np.array_equal(out.download(j), first[j % 4])


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_solve_with_right_hand_sides_that_finish_apart(precision):
    dims, n, tol = (16, 16, 16, 32), 7, 1e-9
    lat = W.Lattice(dims)
    lat.upload_gauge(W.gen_gauge(dims, "smooth", 0.3, 8))
    D = W.Dirac_Wilson_evenodd(0.124, lat)
    b, x, ref = (W.Field(lat, W.EVEN, W.F64, n) for _ in range(3))
    for j in range(n):
        if j == 3:
            b.upload(np.zeros((lat.V, 24)), j)
        elif j % 2:
            b.upload(W.gen_point(dims, 40 + j, j % 4, j % 3)[0] + W.gen_spinor(dims, 50 + j) * 1e-12, j)
        else:
            b.upload(W.gen_spinor(dims, 60 + j), j)
    x.zero(), ref.zero()
    st = W.CG(D, tol, 2000, precision=precision, delta=1e-2).apply(b, x, raise_on_noconv=True)
    lat.set_option(W.OPT_RHS_BLOCK, 1)
    W.CG(D, 1e-12, 2000).apply(b, ref, raise_on_noconv=True)
    for j in range(n):
        assert st[j]["converged"] == 1 and st[j]["true_resid"] <= tol
        r = ref.download(j)
        if j == 3:
            assert not x.download(j).any()
        else:
            # |x - ref| <= |(M^dag M)^-1| |residual|: M^dag M of these links has no eigenvalue below 1e-3
            assert np.linalg.norm(x.download(j) - r) <= 1e3 * tol * np.linalg.norm(b.download(j))
