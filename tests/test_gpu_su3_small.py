"""The compressed mode's SU(3) check on both sides of the line up to which the host looks at all links (1024): the
last link, stretched in its first row by just less and just more than the bound of 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")


@pytest.mark.parametrize("n", [(2, 2, 2, 2), (4, 4, 4, 4), (4, 4, 6, 4)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("d, refused", [(9.99e-7, False), (1.001e-6, True)])
def test_bound(n, d, refused, tmp_path):
    print(f"\n[gpu case] SU(3) check of few links {n} d={d}", flush=True)
    V = int(np.prod(n))
    U = np.zeros((4, V, 18))
    U[..., 0] = U[..., 8] = U[..., 16] = 1.0
    U[3, V - 1, 0] = np.sqrt(1.0 + d)
    U[3, V - 1, 8] = 1.0 / U[3, V - 1, 0]
    U.transpose(1, 0, 2).tofile(tmp_path / "u.bin")
    with glacx.Lattice(n, glacx.FP32_COMPRESSED) as L:
        for put, link in ((lambda: L.upload(U), V - 1), (lambda: L.load_bin(tmp_path / "u.bin"), 4 * V - 1)):
            L.hot_start(4)
            before = L.download()
            if refused:
                with pytest.raises(glacx.GlacxError, match=f"link {link} deviates"):
                    put()
                assert np.array_equal(L.download(), before)
            else:
                put()
                assert np.abs(L.download() - U).max() < 2e-6
