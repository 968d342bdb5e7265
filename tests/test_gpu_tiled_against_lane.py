"""The LDS-tiled multi-rhs kernels (wl_tile.h in FP16, wl_split.h in FP64) against the lane-per-site
kernel (wl_rb.h), WL_OPT_TILED_HOP = 1 against -1, on lattices with whole tiles, tiles with idle
lanes, partial tiles in y and z, and short and long rows.

Operators: FP16 ones form the same sums in the same order, so they agree bit for bit; the FP64 ones to
the rounding bound that test_gpu_split.py derives.

Solves add what operators do not show: ||.||^2 of partial and idle tiles, the residual update, and
rhs that are finished.  After one iteration from x = 0 the residual is r - alpha A r with alpha =
|r|^2 / |M r|^2, so |r_1|^2 / |b|^2 differs between the kernels by the rounding of both sums (of
at most 24 V terms, added in blocks: 30 eps) and of M (M eps, M about 250, as test_gpu_split.py), times
the condition of the update, |r_0|^2 / |r_1|^2 (under 100 here: one iteration takes no more than a
factor of ten from |r|).  A sum that misses one tile would change alpha by more than 1e-4.  With an
FP16 inner precision M agrees bit for bit and only the sums differ: the stored r_1 of a few
sites may round to its other neighbour, 2^-11 of them."""
import numpy as np
import pytest

from hila_amd import wilson as W
from test_gpu_split import EPS, HOP, KAPPA, M

pytestmark = pytest.mark.gpu
LATTICES = [(16, 16, 16, 16), (20, 20, 20, 20), (14, 18, 14, 16), (28, 14, 18, 6), (8, 26, 10, 16), (40, 20, 16, 4),
            (6, 10, 30, 8), (4, 6, 6, 10), (2, 2, 4, 6)]


def _lattice(dims, rows=3, antiperiodic=True):
    lat = W.Lattice(dims, antiperiodic_t=antiperiodic)
    lat.set_option(W.OPT_LINK_ROWS, rows)
    lat.upload_gauge(W.gen_gauge(dims, "smooth", 0.3, 5))
    return lat


def _kernels(lat, prec, n):
    """1, then -1, with the kernel that each takes."""
    for value, kernel in ((1, {W.F64: 2, W.F16: 1}[prec]), (-1, 0)):
        lat.set_option(W.OPT_TILED_HOP, value)
        assert lat.hop_kernel(prec, n) == kernel
        yield value


@pytest.mark.parametrize("dims", LATTICES)
@pytest.mark.parametrize("prec,rows,n", [(W.F64, 3, 5), (W.F64, 2, 2), (W.F16, 3, 1), (W.F16, 3, 7)])
def test_operators(dims, prec, rows, n):
    lat = _lattice(dims, rows, antiperiodic=n != 7)
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    H = W.Hasenbusch_operator(D, 0.1)
    fields = {p: W.Field(lat, p, prec, n) for p in (W.EVEN, W.ODD)}
    norm = {}
    for p, f in fields.items():
        for j in range(n):
            f.upload(W.gen_spinor(dims, 100 + j, 1 if p == W.EVEN else 2), j)
            norm[p, j] = np.linalg.norm(f.download(j))
    got = []
    for _ in _kernels(lat, prec, n):
        outs = []
        for p, f in fields.items():
            hop = W.Field(lat, 3 - p, prec, n)
            for sign in (1, -1):
                D.hop_set(f, hop, sign)
                outs += [(hop.download(j), norm[p, j], HOP) for j in range(n)]
        m = W.Field(lat, W.EVEN, prec, n)
        for op in (H.apply, D.dagger):
            op(fields[W.EVEN], m)
            outs += [(m.download(j), norm[W.EVEN, j], M) for j in range(n)]
        got.append(outs)
    for (a, size, bar), (b, _, _) in zip(*got):
        if prec == W.F16:
            assert np.array_equal(a, b)
        else:
            assert np.linalg.norm(a - b) <= bar * EPS * size
    lat.close()


@pytest.mark.parametrize("dims", LATTICES[:7])
@pytest.mark.parametrize("precision,rows", [("f64", 3), ("f64", 2), ("f16", 3)])
def test_first_iteration(dims, precision, rows):
    n, prec = 3, {"f64": W.F64, "f16": W.F16}[precision]
    lat = _lattice(dims, rows)
    b, x = W.Field(lat, nrhs=n), W.Field(lat, nrhs=n)
    b.upload(W.gen_spinor(dims, 60), 0)
    b.upload(np.zeros((lat.V, 24)), 1)
    b.upload(W.gen_spinor(dims, 61) * 1e-3, 2)
    got = []
    for _ in _kernels(lat, prec, n):
        x.zero()
        got.append(W.CG(W.Dirac_Wilson_evenodd(KAPPA, lat), 1e-12, 1, precision=precision, delta=1e-6).apply(b, x))
    bar = 100 * (30 + M) * EPS if precision == "f64" else 100 * 2.0 ** -22
    for s, t in zip(*got):
        assert s["iterations"] == t["iterations"]
        assert abs(s["rr_rel"] - t["rr_rel"]) <= bar * t["rr_rel"]
    assert got[0][0]["iterations"] == 1 and got[0][0]["rr_rel"] > 1e-2 and got[0][1]["iterations"] == 0
    lat.close()


@pytest.mark.parametrize("dims", [(16, 16, 16, 16), (20, 20, 20, 20), (10, 26, 24, 32), (14, 18, 14, 16)])
@pytest.mark.parametrize("precision", ["f64", "f32", "f16"])
def test_solve(dims, precision):
    # the iteration counts of the two kernels differ by what rounding moves the last one: one, and
    # with an FP16 inner precision, where rounding also moves the updates, one in ten
    n, tol = 5, 1e-9
    lat = _lattice(dims)
    b, x = W.Field(lat, nrhs=n), W.Field(lat, nrhs=n)
    for j in range(n):
        b.upload(W.gen_spinor(dims, 60 + j), j)
    counts = []
    for value in (1, -1):
        lat.set_option(W.OPT_TILED_HOP, value)
        x.zero()
        st = W.CG(W.Dirac_Wilson_evenodd(0.124, lat), tol, 2000, precision=precision, delta=1e-2).apply(b, x)
        assert all(s["converged"] == 1 and s["true_resid"] <= tol for s in st)
        counts.append([s["iterations"] for s in st])
    for s, t in zip(*counts):
        assert abs(s - t) <= (max(1, t // 10) if precision == "f16" else 1)
    lat.close()


@pytest.mark.parametrize("precision,n", [("f64", 4), ("f32", 4), ("f16", 8)])
def test_captured_chunks(precision, n):
    """Chunks with the tiled kernels (144 KB of dynamic LDS in FP64) captured into a HIP graph and
    replayed, with eager work between the solves, give the bits of the eager solve."""
    lat = _lattice((16, 16, 16, 32))
    prec = {"f64": W.F64, "f32": W.F32, "f16": W.F16}[precision]
    assert lat.hop_kernel(W.F64, n) == 2 and lat.hop_kernel(prec, n) == {W.F64: 2, W.F32: 0, W.F16: 1}[prec]
    D = W.Dirac_Wilson_evenodd(0.124, lat)
    cg = W.CG(D, 1e-9, 2000, precision=precision, delta=1e-1)
    b, x, tmp = W.Field(lat, nrhs=n), W.Field(lat, nrhs=n), W.Field(lat, nrhs=n)
    for j in range(n):
        b.upload(W.gen_spinor(lat.dims, 60 + j), j)
    x.zero()
    eager = cg.apply(b, x, raise_on_noconv=True)
    ref = [x.download(j) for j in range(n)]
    lat.set_option(W.OPT_GRAPHS, 1)
    for _ in range(3):
        D.apply(b, tmp)
        lat.sync()
        x.zero()
        st = cg.apply(b, x)
        assert [(s["iterations"], s["true_resid"]) for s in st] == [(s["iterations"], s["true_resid"]) for s in eager]
        assert all(np.array_equal(x.download(j), ref[j]) for j in range(n))
    lat.close()
