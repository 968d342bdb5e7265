"""The LDS-tiled FP16 multi-rhs hopping kernel (wl_tile.h) on the GPU.  It forms every sum in the
order of the lane-per-site kernel (wl_rb.h), which a caller's WL_OPT_RHS_BLOCK selects, so the
two agree bit for bit; against the FP64 oracle the bar is FP16 storage's, 2e-3."""
import numpy as np
import pytest

from hila_amd import wilson as W
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
KAPPA = 0.12

# lattices that take the tiled kernel: whole tiles of four waves, tiles with idle lanes, partial
# tiles in y or z, rows that are no power of two, workgroups of two waves
LATTICES = [(16, 16, 16, 32), (20, 20, 20, 20), (14, 18, 14, 64), (14, 26, 6, 64), (28, 14, 18, 38), (8, 26, 10, 64)]


def _fields(lat, dims, n, parity=W.EVEN):
    f = W.Field(lat, parity, W.F16, n)
    for j in range(n):
        f.upload(W.gen_spinor(dims, 100 + j, 1 if parity == W.EVEN else 2), j)
    return f


@pytest.mark.parametrize("dims", LATTICES)
@pytest.mark.parametrize("n", [6, 7, 13])
def test_same_bits_as_the_lane_per_site_kernel(dims, n):
    lat = W.Lattice(dims, antiperiodic_t=n != 7)
    lat.upload_gauge(W.gen_gauge(dims, "haar", 0, 5))
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    H = W.Hasenbusch_operator(D, 0.1)
    got = []
    for nr in (0, 1):
        lat.set_option(W.OPT_RHS_BLOCK, nr)
        outs = []
        for parity in (W.EVEN, W.ODD):
            fin = _fields(lat, dims, n, parity)
            hop, m = W.Field(lat, 3 - parity, W.F16, n), W.Field(lat, W.EVEN, W.F16, n)
            for sign in (1, -1):
                D.hop_set(fin, hop, sign)
                outs += [hop.download(j) for j in range(n)]
            if parity == W.EVEN:
                H.apply(fin, m)
                outs += [m.download(j) for j in range(n)]
                D.dagger(fin, m)
                outs += [m.download(j) for j in range(n)]
        got.append(outs)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_against_the_oracle():
    dims, n = (20, 20, 20, 20), 6
    U = W.gen_gauge(dims, "haar", 0, 6)
    lat = W.Lattice(dims)
    lat.upload_gauge(U)
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    fin, out = _fields(lat, dims, n), W.Field(lat, W.EVEN, W.F16, n)
    orc = Oracle(dims)
    D.apply(fin, out)
    for j in (0, n - 1):
        ref = orc.meo(U, KAPPA, W.gen_spinor(dims, 100 + j), 1)
        assert np.linalg.norm(out.to_full(j) - ref) / np.linalg.norm(ref) <= 2e-3


def test_most_right_hand_sides():
    dims, n = (20, 20, 20, 20), 64
    lat = W.Lattice(dims)
    lat.upload_gauge(W.gen_gauge(dims, "haar", 0, 7))
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    fin, out = W.Field(lat, W.EVEN, W.F16, n), W.Field(lat, W.ODD, W.F16, n)
    src = [W.gen_spinor(dims, 100 + j) for j in range(4)]
    for j in range(n):
        fin.upload(src[j % 4], j)
    D.hop_set(fin, out)
    first = [out.download(j) for j in range(4)]
    for j in range(4, n):
        assert np.array_equal(out.download(j), first[j % 4])
    lat.set_option(W.OPT_RHS_BLOCK, 1)
    D.hop_set(fin, out)
    assert all(np.array_equal(out.download(j), first[j]) for j in range(4))


def test_solve_with_right_hand_sides_that_finish_apart():
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
    st = W.CG(D, tol, 2000, precision="f16", delta=1e-2).apply(b, x, raise_on_noconv=True)
    W.CG(D, 1e-12, 2000).apply(b, ref, raise_on_noconv=True)
    for j in range(n):
        assert st[j]["converged"] == 1 and st[j]["true_resid"] <= tol
        r = ref.download(j)
        if j == 3:
            assert not x.download(j).any()
        else:
            # |x - ref| <= |(M^dag M)^-1| |residual|: M^dag M of these links has no eigenvalue below 1e-3
            assert np.linalg.norm(x.download(j) - r) <= 1e3 * tol * np.linalg.norm(b.download(j))
