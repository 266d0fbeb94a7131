"""The accepted hits of a chain are counted in slots that hold 1024 sweeps at a time:
a call that goes round them counts what shorter calls count, and its memory grows by
its result rows alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

N = (2, 2, 4, 2)


def chain(L, proposal, sweeps, offset=0):
    update = L.metropolis if proposal == "rst" else L.metropolis_learned
    return update(sweeps, 6.0, 0.24, 1, seed=5, sweep_offset=offset)


@pytest.mark.parametrize("proposal", ["rst", "learned"])
@pytest.mark.parametrize("sweeps", [1024, 1025, 5000])  # 4097 and more: sums in device memory
def test_counts_of_a_call_that_goes_round(sweeps, proposal):
    print(f"\n[gpu case] count batches, {sweeps} {proposal} sweeps", flush=True)
    with glacx.Lattice(N, glacx.FP64) as L:
        rng = np.random.default_rng(3)
        L.proposal_set(rng.normal(size=glacx.PROPOSAL_NPARAM).astype(np.float32) * 0.1, np.zeros(6, np.float32),
                       np.full(6, 1e4, np.float32))
        L.hot_start(3)
        whole = chain(L, proposal, sweeps)
        links = L.download()
        L.hot_start(3)
        parts = [chain(L, proposal, min(700, sweeps - o), o) for o in range(0, sweeps, 700)]
        assert np.array_equal(links, L.download())
    assert np.array_equal(whole, np.concatenate(parts)) and whole.max() > 0


@pytest.mark.parametrize("proposal", ["rst", "learned"])
def test_memory_of_a_long_chain(proposal):
    print(f"\n[gpu case] memory of a long {proposal} chain", flush=True)
    sweeps = 20000
    with glacx.Lattice(N, glacx.FP64) as L:
        L.proposal_set(np.zeros(glacx.PROPOSAL_NPARAM, np.float32), np.zeros(6, np.float32), np.ones(6, np.float32))
        L.hot_start(3)
        before = L.device_bytes
        chain(L, proposal, sweeps)
        # slots of 1024 sweeps, 2 KiB each, and a count per sweep
        assert L.device_bytes - before <= (2 << 20) + 8 * sweeps
