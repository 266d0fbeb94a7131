"""Measured flows whose blocks fill the chip: the four wavefronts of a block hand
over their parts of F once, after their last term.  Lattices just above the line to
the kernel for small ones, with x-y planes that blocks cut, against the oracle.
Tolerances as for every measured flow: FP64 1e-11 relative for E, 1e-12 for the
others (sums of up to 32768 sites); FP32 2e-6 and Q 1e-4."""
import numpy as np
import pytest

import oracle as O
from fieldtools import near_unit_field

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")


@pytest.mark.parametrize("prec", [glacx.FP64, glacx.FP32_LINKS, glacx.FP32_COMPRESSED], ids=["fp64", "fp32", "fp32c"])
@pytest.mark.parametrize("n", [(8, 16, 16, 10), (10, 16, 16, 8), (6, 8, 20, 24)], ids=lambda n: "x".join(map(str, n)))
def test_measured_flow(n, prec):
    print(f"\n[gpu case] measured flow, phases {n} prec={prec}", flush=True)
    U = near_unit_field(n, np.random.default_rng(sum(n)), 0.4)
    with glacx.Lattice(n, prec) as L:
        L.upload(U, glacx.FLOW)
        p, e, q, qt = L.flow(2, 0.02)
        links = L.download(glacx.FLOW)
    for i in range(3):
        wp, we, wq, wqt = O.measure(U, n)
        if prec == glacx.FP64:
            assert abs(p[i] - wp) < 1e-12 and abs(e[i] / we - 1) < 1e-11
            assert abs(q[i] - wq) < 1e-12 and np.abs(qt[i] - wqt).max() < 1e-12
        else:
            assert abs(p[i] - wp) < 2e-6 and abs(e[i] / we - 1) < 2e-6
            assert abs(q[i] - wq) < 1e-4 and np.abs(qt[i] - wqt).max() < 1e-4
        if i < 2:
            O.flow_step(U, n, 0.02)
    assert np.abs(links - U).max() < (1e-12 if prec == glacx.FP64 else 2e-6)
