"""Flow steps on both sides of the lines between the flow stages' variants: FP64 launches of up to 768 blocks of 64
sites gather their links in pairs, larger ones four at a time with in-block neighbours from LDS (rows and planes that
a block's run of 32 entries cuts, and slabs that are not whole runs, where nothing is taken); stores are streamed while
two fields take less than 16 (FP64) or 28 MiB (FP32).  Against the oracle, links to 1e-12 in FP64 and 2e-6 in FP32 as
for every flow."""
import numpy as np
import pytest

import oracle as O
from fieldtools import near_unit_field

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

FEW = [(10, 12, 12, 10), (12, 12, 12, 10), (16, 16, 16, 12)]  # 15.8 and 19.0 MiB; 768 blocks
MANY = [(6, 12, 32, 22),                                      # 792 blocks
        (2, 16, 40, 40), (64, 2, 20, 20), (6, 4, 46, 48), (24, 24, 8, 12), (12, 10, 22, 20), (10, 6, 30, 28)]
CASES = [(n, "FP64") for n in FEW + MANY]
CASES += [((16, 16, 14, 14), "FP32_LINKS"), ((16, 16, 14, 16), "FP32_LINKS")]                # 27.6 and 31.5 MiB
CASES += [((16, 16, 16, 18), "FP32_COMPRESSED"), ((16, 16, 18, 18), "FP32_COMPRESSED")]      # 27.0 and 30.4 MiB


@pytest.mark.parametrize("n, prec", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_flow_follows_oracle(n, prec):
    print(f"\n[gpu case] flow lines {n} {prec}", flush=True)
    start = near_unit_field(n, np.random.default_rng(sum(n)), 0.4)
    got = []
    with glacx.Lattice(n, getattr(glacx, prec)) as L:
        for measure in (True, False):
            L.upload(start, glacx.FLOW)
            L.flow(2, 0.02, measure=measure)
            got.append(L.download(glacx.FLOW))
    U = start.copy()
    for _ in range(2):
        O.flow_step(U, n, 0.02)
    for links in got:
        assert np.abs(links - U).max() < (1e-12 if prec == "FP64" else 2e-6)
