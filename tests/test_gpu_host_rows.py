"""Results that fit the context's pinned rows (8192 doubles) are stored there by the
kernels, longer ones are copied; a chain's plaquettes are summed together, in batches of
32 MiB of partials: a long call gives what two short ones give."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

N = (2, 2, 2, 4)


@pytest.mark.parametrize("sweeps", [4096, 4097, 5000])  # plaquettes and counts: 8192, 8194, 10000
def test_long_chain_equals_two_short_ones(sweeps):
    print(f"\n[gpu case] host rows, {sweeps} sweeps", flush=True)
    with glacx.Lattice(N, glacx.FP64) as L:
        L.hot_start(3)
        acc, plaq = L.metropolis(sweeps, 6.0, 0.24, 2, seed=5, plaquette=True)
        links = L.download()
        L.hot_start(3)
        half = [L.metropolis(n, 6.0, 0.24, 2, seed=5, sweep_offset=o, plaquette=True)
                for n, o in ((sweeps // 2, 0), (sweeps - sweeps // 2, sweeps // 2))]
        assert np.array_equal(links, L.download())
    assert np.array_equal(acc, np.concatenate([h[0] for h in half]))
    assert np.array_equal(plaq, np.concatenate([h[1] for h in half]))


def test_plaquettes_summed_in_two_batches():
    """1024 partials a sweep at 16^4: 4096 sweeps fill the batch."""
    print("\n[gpu case] host rows, plaquettes in two batches", flush=True)
    n = (16, 16, 16, 16)
    with glacx.Lattice(n, glacx.FP32_COMPRESSED) as L:
        L.hot_start(3)
        _, plaq = L.metropolis(4099, 6.0, 0.24, 1, seed=5, plaquette=True)
        L.hot_start(3)
        _, a = L.metropolis(4090, 6.0, 0.24, 1, seed=5, plaquette=True)
        _, b = L.metropolis(9, 6.0, 0.24, 1, seed=5, sweep_offset=4090, plaquette=True)
    assert np.array_equal(plaq, np.concatenate([a, b]))


@pytest.mark.parametrize("steps", [1169, 1170, 1500])  # rows of 7 doubles: 8190, 8197, 10507
def test_long_flow_equals_two_short_ones(steps):
    print(f"\n[gpu case] host rows, {steps} flow steps", flush=True)
    first = steps // 2
    with glacx.Lattice(N, glacx.FP64) as L:
        L.hot_start(3)
        L.copy(glacx.FLOW, glacx.MAIN)
        whole = L.flow(steps, 0.01)
        links = L.download(glacx.FLOW)
        L.copy(glacx.FLOW, glacx.MAIN)
        a = L.flow(first, 0.01)
        b = L.flow(steps - first, 0.01)
        assert np.array_equal(links, L.download(glacx.FLOW))
    for w, x, y in zip(whole, a, b):
        # the first call's last row is the second one's first
        assert np.array_equal(w[:first], x[:first]) and np.array_equal(w[first:], y)
