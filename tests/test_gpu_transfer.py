"""Fields go to the device and come back to the last bit, below and above the
size from which they travel through pinned slices (16 MiB; slices of 4 MiB, the
last one partial), from several contexts at once, and through the file calls."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

SHAPES = [(8, 8, 8, 8), (16, 16, 14, 10), (16, 16, 16, 16), (18, 22, 20, 24)]


def links(n, seed):
    return np.random.default_rng(seed).normal(size=(4, int(np.prod(n)), 18))


@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_round_trip(n, tmp_path):
    print(f"\n[gpu case] transfer {n}", flush=True)
    U, W = links(n, 1), links(n, 2)
    with glacx.Lattice(n, glacx.FP64) as L:
        L.upload(U, glacx.MAIN)
        L.upload(W, glacx.FLOW)
        assert np.array_equal(L.download(glacx.MAIN), U) and np.array_equal(L.download(glacx.FLOW), W)
        L.save_bin(tmp_path / "u.bin", glacx.MAIN)
        site_major = np.fromfile(tmp_path / "u.bin").reshape(-1, 4, 18)
        assert np.array_equal(site_major, U.transpose(1, 0, 2))
        L.load_bin(tmp_path / "u.bin", glacx.FLOW)
        assert np.array_equal(L.download(glacx.FLOW), U)


def test_contexts_in_threads():
    n, fails = (16, 16, 14, 10), []

    def chain(seed):
        U = links(n, seed)
        with glacx.Lattice(n, glacx.FP64) as L:
            for _ in range(3):
                L.upload(U)
                if not np.array_equal(L.download(), U):
                    fails.append(seed)

    threads = [threading.Thread(target=chain, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not fails
