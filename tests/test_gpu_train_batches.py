"""The training step at the edges of its 16-sample wavefronts, of the 256-sample
prefetch of its batch sums and of its split of the draws over four lanes,
against the FP64 numpy reference.

Tolerance: a sample's FP32 chain (features, three layers of sums over up to 32
terms, draws, and back) rounds at ~100 x 6e-8 of its terms; a pre-activation
within ~1e-6 of zero may take the other slope, which happens to a few units
among 33 000 samples and moves the gradient by at most a sample's share.  2e-4
of the largest entry covers both."""
import numpy as np
import pytest

import oracle as O
import oracle.training as T
from fieldtools import random_su3

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")


@pytest.mark.parametrize("n, draws", [(1, 1), (15, 4), (17, 5), (256, 2), (273, 7), (33000, 2)])
def test_train_gradient_at_block_edges(n, draws):
    print(f"\n[gpu case] train_grad n={n} draws={draws}", flush=True)
    rng = np.random.default_rng(n)
    A, U = random_su3(rng, (6, n)).sum(0), random_su3(rng, (n,))
    smp = np.concatenate([O.to_pairs(A), O.to_pairs(U)], axis=1).astype(np.float32)
    f = T.features(A, 6.0)
    mean = f.mean(0).astype(np.float32)
    std = (f.std(0) + 0.1 * (np.abs(f).mean(0) + 1)).astype(np.float32)
    p = T.init_params(rng, scale0=0.3)
    p[T.SLICES["W3"]] += rng.normal(size=36 * 32) * 0.05
    p[T.SLICES["b1"]] = rng.normal(size=32) * 0.1
    p = p.astype(np.float32)
    z = rng.normal(size=(n, draws, 8)).astype(np.float32)
    with glacx.Lattice((2, 2, 2, 2), glacx.FP32_LINKS) as L:
        L.proposal_set(p, mean, std)
        loss, g = L.train_grad(smp, z, 6.0)
    want_loss, want = T.loss_and_grad(p.astype(np.float64), mean.astype(np.float64), std.astype(np.float64),
                                      A.astype(np.complex64).astype(np.complex128),
                                      U.astype(np.complex64).astype(np.complex128), 6.0, z.astype(np.float64))
    assert abs(loss - want_loss) < 2e-5 * abs(want_loss)
    err = np.abs(g - want)
    assert err.max() < 2e-4 * np.abs(want).max(), (err.argmax(), err.max() / np.abs(want).max())
