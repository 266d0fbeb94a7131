"""The compressed mode's SU(3) check of uploaded links: one link among unit
links is stretched in its first row, which moves |U U^dag - 1| by d; links are
refused from 1e-6 on, wherever they lie, with their index, and a refused upload
leaves the field as it was.  d just below the bound is where the device hands
the decision to the host."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

N = (4, 6, 2, 10)
V = 480


def unit_links():
    U = np.zeros((4, V, 18))
    U[..., 0] = U[..., 8] = U[..., 16] = 1.0
    return U


@pytest.mark.parametrize("mu, site", [(0, 0), (3, V - 1), (1, 255), (2, 256)])
@pytest.mark.parametrize("d, refused", [(1e-9, False), (9.99e-7, False), (9.999995e-7, False), (1.0000005e-6, True),
                                        (3e-6, True)])
def test_bound(mu, site, d, refused):
    print(f"\n[gpu case] SU(3) check mu={mu} site={site} d={d}", flush=True)
    U = unit_links()
    U[mu, site, 0] = np.sqrt(1.0 + d)
    U[mu, site, 8] = 1.0 / U[mu, site, 0]
    with glacx.Lattice(N, glacx.FP32_COMPRESSED) as L:
        L.hot_start(4)
        before = L.download()
        if refused:
            with pytest.raises(glacx.GlacxError, match=f"link {site} deviates"):
                L.upload(U)
            assert np.array_equal(L.download(), before)
        else:
            L.upload(U)
            assert np.abs(L.download() - U).max() < 2e-6


def test_links_that_are_no_numbers_pass_as_the_host_loop_lets_them():
    U = unit_links()
    U[2, 17, 3] = np.nan
    with glacx.Lattice(N, glacx.FP32_COMPRESSED) as L:
        L.upload(U)
        assert np.isnan(L.download()[2, 17]).any()
