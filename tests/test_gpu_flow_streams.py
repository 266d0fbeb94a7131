"""Flow stages on both sides of the lines from which the accumulator (two fields and
it take 256 MiB) and the stored links (two fields exceed 256 MiB) are streamed past the
caches: one step against the oracle, links to 1e-12 in FP64 and 2e-6 in FP32 as for
every flow."""
import numpy as np
import pytest

import oracle as O
from fieldtools import near_unit_field

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")


@pytest.mark.parametrize("n, prec", [((24, 24, 24, 12), "FP64"),              # 223 MiB, fields 182
                                     ((24, 24, 24, 16), "FP64"),              # 297, 243
                                     ((24, 24, 24, 20), "FP64"),              # 371, 304
                                     ((32, 32, 32, 16), "FP32_COMPRESSED"),   # 256, 192
                                     ((32, 32, 32, 24), "FP32_LINKS")],       # 528, 432
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_flow_step_follows_oracle(n, prec):
    print(f"\n[gpu case] streamed flow step {n} {prec}", flush=True)
    U = near_unit_field(n, np.random.default_rng(sum(n)), 0.4)
    with glacx.Lattice(n, getattr(glacx, prec)) as L:
        L.upload(U, glacx.FLOW)
        L.flow(1, 0.02)
        links = L.download(glacx.FLOW)
    O.flow_step(U, n, 0.02)
    assert np.abs(links - U).max() < (1e-12 if prec == "FP64" else 2e-6)
