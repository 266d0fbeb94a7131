"""FP64 plain flow stages take the x- and y-neighbours that a block holds itself
from LDS: rows that a block's run of 32 entries cuts, x-y planes that it
cuts, whole planes with both ends of a row inside, and lattices whose slabs are
not whole runs, where nothing is taken.  Against the oracle, links to 1e-12 as for
every FP64 flow."""
import numpy as np
import pytest

import oracle as O
from fieldtools import near_unit_field

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")


@pytest.mark.parametrize("n", [(2, 2, 2, 2), (6, 2, 2, 4), (4, 4, 4, 4), (2, 16, 4, 4), (64, 2, 2, 4), (16, 2, 8, 4),
                               (6, 4, 2, 8), (10, 6, 4, 4), (24, 24, 4, 4), (12, 10, 6, 6)],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("measured", [True, False], ids=["measured", "plain"])
def test_flow_follows_oracle(n, measured):
    print(f"\n[gpu case] flow with neighbours from LDS {n} measured={measured}", flush=True)
    U = near_unit_field(n, np.random.default_rng(sum(n)), 0.4)
    with glacx.Lattice(n, glacx.FP64) as L:
        L.upload(U, glacx.FLOW)
        (L.flow if measured else L.flow_super)(2, 0.02)
        links = L.download(glacx.FLOW)
    for _ in range(2):
        O.flow_step(U, n, 0.02)
    assert np.abs(links - U).max() < 1e-12
