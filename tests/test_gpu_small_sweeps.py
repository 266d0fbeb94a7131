"""Sub-sweeps that do not fill the chip run with a block of several wavefronts
per 64 links (up to 256 groups of links, up to 768 in FP32 and 512 in FP64 with
fewer wavefronts each), with rounds of ten hits.  Same streams and decisions
as the oracle at the edges: a partial group, fewer hits than wavefronts that
propose them, hits on both sides of a round, and group counts on both sides of
the lines between the variants.

FP64 makes the oracle's decisions.  In FP32 exp(-dS) rounds at ~1e-7, so of
10^6 decisions a fraction of one flips, and takes some of the ~24 links whose
staples hold its link along with it: at most 200 links may differ."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

CASES = [((2, 2, 2, 2), 1), ((2, 2, 2, 2), 10), ((4, 6, 4, 6), 4), ((4, 6, 4, 6), 11), ((4, 6, 4, 6), 23),
         ((16, 16, 16, 8), 10),                                # 256 groups
         ((12, 14, 14, 14), 11),                               # 258
         ((16, 16, 16, 16), 3), ((16, 16, 14, 20), 3),         # 512 and 560
         ((16, 16, 16, 24), 3), ((16, 16, 18, 22), 3)]         # 768 and 792


@pytest.mark.parametrize("prec", [glacx.FP64, glacx.FP32_LINKS, glacx.FP32_COMPRESSED], ids=["fp64", "fp32", "fp32c"])
@pytest.mark.parametrize("n, hits", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_small_sweep_follows_oracle(n, hits, prec):
    print(f"\n[gpu case] small sweep {n} hits={hits} prec={prec}", flush=True)
    U = O.hot_start_haar(n, 5)
    accepted = O.cb_sweep(U, n, 6.0, 0.24, hits, 9, 3, True)
    with glacx.Lattice(n, prec) as L:
        L.hot_start(5)
        acc = L.metropolis(1, 6.0, 0.24, hits, seed=9, sweep_offset=3)[0]
        chain = L.download()
    decisions = 4 * hits * int(np.prod(n))
    off = np.abs(chain - U).max(-1) > (1e-10 if prec == glacx.FP64 else 1e-4)
    if prec == glacx.FP64:
        assert round(acc * decisions) == round(accepted * decisions) and not off.any()
    else:
        assert off.sum() <= 200 and abs(acc - accepted) * decisions <= 200 * hits
