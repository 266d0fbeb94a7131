"""A flow sums its measurements' partials to result rows in groups (all steps,
or as many as its buffer holds): the rows of a long flow, whose groups wrap,
are those of the same flow in two shorter calls, which stay within one group.
16^4 sums a row in one kernel and wraps after 1008 measurements, 24^3 x 48 in
two kernels after 101 (50 without allocation)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")


@pytest.mark.parametrize("n, first, second", [((16, 16, 16, 16), 600, 500), ((24, 24, 24, 48), 45, 100)],
                         ids=["16x16x16x16", "24x24x24x48"])
def test_rows_of_a_wrapping_flow(n, first, second):
    print(f"\n[gpu case] flow rows {n} {first} + {second}", flush=True)
    with glacx.Lattice(n, glacx.FP32_COMPRESSED) as L:
        L.hot_start(3, kind=glacx.HOT_RST)
        L.copy(glacx.FLOW, glacx.MAIN)
        a = L.flow(first, 0.001)
        b = L.flow(second, 0.001)
        for flow in (L.flow, L.flow_noalloc):
            L.copy(glacx.FLOW, glacx.MAIN)
            whole = flow(first + second, 0.001)
            for w, x, y in zip(whole, a, b):
                # row `first` is measured by the clover kernel at the end of the
                # first call, inside a flow stage in the other two
                assert np.array_equal(w[:first], x[:first]) and np.array_equal(w[first:], y)
