"""Learned sub-sweeps of more than 1536 blocks run with more wavefronts per SIMD than
smaller ones: the oracle's decisions hold there too, with a last block that is not
whole.  The first layer's weights are zero, so that the network's output does not
depend on how FP32 and FP64 round a feature to bf16.

In FP32 exp(-dS) rounds at ~1e-7, so of 10^6 decisions a fraction of one flips
and takes some of the ~24 links whose staples hold its link along with it: at most
200 links may differ for every 10^6 decisions."""
import numpy as np
import pytest

import oracle as O
import oracle.training as T

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

N, HITS = (34, 30, 26, 30), 2  # 397800 links of a direction and parity: 1553.9 blocks


def test_large_learned_sweep_follows_oracle():
    print(f"\n[gpu case] large learned sweep {N} hits={HITS}", flush=True)
    rng = np.random.default_rng(11)
    p = T.init_params(rng, scale0=0.3)
    p[T.SLICES["W3"]] += rng.normal(size=36 * 32) * 0.02
    p[T.SLICES["W1"]] = 0.0
    p = (p.astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)  # exact in bf16
    U = O.hot_start_haar(N, 3)
    f = np.array([O.staple_features(O.staple(U, N, x, 1, 2, t, mu), 6.0)
                  for x in range(N[0]) for t in range(N[3]) for mu in range(4)])
    mean, std = f.mean(0).astype(np.float32), (f.std(0) + 1e-3).astype(np.float32)
    with glacx.Lattice(N, glacx.FP32_LINKS) as L:
        L.upload(U)
        L.proposal_set(p, mean, std)
        got_acc = L.metropolis_learned(1, 6.0, 0.24, HITS, reunit_every=1, seed=21)[0]
        got = L.download()
    acc = O.learned_cb_sweep(U, N, 6.0, HITS, 21, 0, p.astype(np.float64), mean.astype(np.float64),
                             std.astype(np.float64))
    decisions = 4 * HITS * int(np.prod(N))
    off = np.abs(got - U).max(-1) > 1e-4
    allowed = 200e-6 * decisions
    assert off.sum() <= allowed and abs(acc - got_acc) * decisions <= allowed * HITS
