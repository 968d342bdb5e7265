"""Which kernel a multi-rhs hopping launch takes follows from the lattice, the precision and the
rhs count alone.  So where the LDS-tiled kernels (wl_tile.h, wl_split.h) are the default, whose
sums are taken in another order than the lane-per-site kernel's, the launch-shape options and the
autotuner leave every bit of an operator and of a solve as it was.  FP32 has no tiled kernel: the
options that choose no other instantiation of its lane-per-site kernel leave every bit too."""
import numpy as np
import pytest

from hila_amd import wilson as W

pytestmark = pytest.mark.gpu

# the same kernel code: workgroups, passes, cache policy
SAME = [(W.OPT_RHS_LAUNCH, 2), (W.OPT_BLOCK, 128), (W.OPT_LDS_RESERVE, -1), (W.OPT_LDS_RESERVE, 32768),
        (W.OPT_LINK_LOAD, 1)]
# other instantiations of the lane-per-site kernel, whose FMA contraction may differ
OTHER = [(W.OPT_RHS_BLOCK, 1), (W.OPT_RHS_BLOCK, 2), (W.OPT_LINK_LOAD, 3), (W.OPT_PIPELINE, 1)]


def _lattice(dims):
    lat = W.Lattice(dims)
    lat.upload_gauge(W.gen_gauge(dims, "smooth", 0.3, 8))
    return lat


def _results(lat, prec, n):
    """Bits of hop, M, M^dag and of a solve of n rhs with operator fields of this storage."""
    D = W.Dirac_Wilson_evenodd(0.124, lat)
    fin, hop, m = W.Field(lat, W.EVEN, prec, n), W.Field(lat, W.ODD, prec, n), W.Field(lat, W.EVEN, prec, n)
    b, x = W.Field(lat, W.EVEN, W.F64, n), W.Field(lat, W.EVEN, W.F64, n)
    for j in range(n):
        s = W.gen_spinor(lat.dims, 60 + j)
        fin.upload(s, j), b.upload(s, j)
    out = []
    D.hop_set(fin, hop)
    out += [hop.download(j) for j in range(n)]
    for op in (D.apply, D.dagger):
        op(fin, m)
        out += [m.download(j) for j in range(n)]
    x.zero()
    st = W.CG(D, 1e-8, 500, precision={W.F64: "f64", W.F32: "f32", W.F16: "f16"}[prec], delta=1e-2).apply(b, x)
    out += [x.download(j) for j in range(n)]
    out += [np.array([s["iterations"], s["rr_rel"], s["true_resid"]]) for s in st]
    return out


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("prec,n,options", [(W.F64, 4, SAME + OTHER), (W.F64, 8, SAME + OTHER),
                                            (W.F16, 8, SAME + OTHER), (W.F32, 4, SAME)],
                         ids=["f64-4", "f64-8", "f16-8", "f32-4"])
def test_launch_shape_options_leave_every_bit(prec, n, options):
    lat = _lattice((16, 16, 16, 32))
    kernel = lat.hop_kernel(prec, n)
    assert kernel == {W.F64: 2, W.F16: 1, W.F32: 0}[prec]
    ref = _results(lat, prec, n)
    for option, value in options:
        lat.set_option(option, value)
        assert lat.hop_kernel(prec, n) == kernel
        assert _same(_results(lat, prec, n), ref), (option, value)
        lat.set_option(option, 0)
    lat.close()


@pytest.mark.parametrize("tuned", [W.F64, W.F32, W.F16], ids=["f64", "f32", "f16"])
def test_autotuner_leaves_every_bit_of_the_tiled_kernels(tuned):
    # a solve's FP64 updates run on the context that was tuned for its inner precision
    n = 8
    lat = _lattice((16, 16, 16, 32))
    ref = [_results(lat, prec, n) for prec in (W.F64, W.F16)]
    t = lat.autotune(tuned, n)
    assert (t["candidates"] == 1) == (lat.hop_kernel(tuned, n, "hop") != 0)
    for prec, r in zip((W.F64, W.F16), ref):
        assert _same(_results(lat, prec, n), r), prec
    lat.close()


def test_tiled_hop_option():
    lat = _lattice((16, 16, 16, 32))
    assert lat.get_option(W.OPT_TILED_HOP) == 0
    lat.set_option(W.OPT_TILED_HOP, -1)
    assert [lat.hop_kernel(p, 8) for p in (W.F64, W.F32, W.F16)] == [0, 0, 0]
    for bad in (-2, 2):
        with pytest.raises(W.WilsonError):
            lat.set_option(W.OPT_TILED_HOP, bad)
    assert lat.get_option(W.OPT_TILED_HOP) == -1
    lat.set_option(W.OPT_TILED_HOP, 1)
    assert [lat.hop_kernel(p, 2) for p in (W.F64, W.F32, W.F16)] == [2, 0, 1]
    for prec, n in ((3, 8), (W.F64, 0), (W.F64, 65)):
        with pytest.raises(W.WilsonError):
            lat.hop_kernel(prec, n)
    lat.close()
