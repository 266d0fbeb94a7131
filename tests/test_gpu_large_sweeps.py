"""Sub-sweeps of more than 3072 blocks run with more wavefronts per SIMD than
smaller ones: the oracle's decisions hold there too, with a last block that is
not whole.

In FP32 exp(-dS) rounds at ~1e-7, so of 10^6 decisions a fraction of one flips
and takes some of the ~24 links whose staples hold its link along with it: at
most 200 links may differ for every 10^6 decisions."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

N, HITS = (34, 32, 30, 50), 2  # 816000 links of a direction and parity: 3187.5 blocks


@pytest.fixture(scope="module")
def swept():
    U = O.hot_start_haar(N, 5)
    accepted = O.cb_sweep(U, N, 6.0, 0.24, HITS, 9, 3, True)
    return U, accepted


@pytest.mark.parametrize("prec", [glacx.FP32_LINKS, glacx.FP32_COMPRESSED], ids=["fp32", "fp32c"])
def test_large_sweep_follows_oracle(swept, prec):
    print(f"\n[gpu case] large sweep {N} hits={HITS} prec={prec}", flush=True)
    U, accepted = swept
    with glacx.Lattice(N, prec) as L:
        L.hot_start(5)
        acc = L.metropolis(1, 6.0, 0.24, HITS, seed=9, sweep_offset=3)[0]
        chain = L.download()
    decisions = 4 * HITS * int(np.prod(N))
    off = np.abs(chain - U).max(-1) > 1e-4
    allowed = 200e-6 * decisions
    assert off.sum() <= allowed and abs(acc - accepted) * decisions <= allowed * HITS
