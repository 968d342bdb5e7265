"""The launch-folded CG whose first hop also ends the iteration before and forms p = beta p + r
(k_dslash_dir_xpay, wl_dslash.hip), against the unfolded CG, whose kernels the oracle tests pin:
the same bits and statistics, where a solve ends at any place among the iterations between two
looks of the host, from a guess, on lattices whose last workgroup has few sites and whose x
neighbours are the site itself (extent 2)."""
import numpy as np
import pytest

from hila_amd import wilson as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("antiperiodic", [False, True])
@pytest.mark.parametrize("rows", [2, 3])
@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (4, 4, 4, 4), (2, 6, 4, 6), (6, 2, 10, 4), (4, 6, 8, 10)])
def test_merged_first_hop_has_the_bits_of_the_unfolded_solve(dims, rows, antiperiodic):
    lat = W.Lattice(dims, antiperiodic_t=antiperiodic)
    lat.set_option(W.OPT_LINK_ROWS, rows)
    lat.upload_gauge(W.gen_gauge(dims, "smooth", 0.4, 21))
    D = W.Dirac_Wilson_evenodd(0.12, lat)
    b = W.Field(lat).upload(W.gen_spinor(dims, 22))
    for maxiters in [*range(0, 12), 1000]:
        got = []
        for mode in (-1, 0):
            lat.set_option(W.OPT_CG_PERSISTENT, mode)
            x = W.Field(lat).upload(W.gen_spinor(dims, 23) * 0.1)
            (st,) = W.CG(D, 1e-10, maxiters).apply(b, x)
            got.append((x.download(), st))
        (x, s), (y, t) = got
        assert np.array_equal(x, y), maxiters
        for key in ("iterations", "converged", "rr_rel", "true_resid"):
            assert s[key] == t[key], (maxiters, key)
    lat.close()
