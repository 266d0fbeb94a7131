"""FP32 sweeps against the oracle where their last group of 64 links or block of 256 is not whole, with bounds that
follow from the decisions made.

FP32 rounds dS at about 1e-6, so a decision whose exp(-dS) lies that close to its random number falls the other way:
of D decisions at most about 1e-6 D = m.  A flip takes some of the ~24 links whose staples hold its link along with
it, so 25 links for each of m + 4 sqrt(m) flips may differ, and none where m is below 0.01.  The links of the last
group or block are bounded on their own, below what one lost sub-sweep of them makes: a flip near them reaches a few
of them."""
import math

import numpy as np
import pytest

import oracle as O

glacx = pytest.importorskip("glac_amd")

# lattice, hits, links of a last group or block that is not whole
SMALL = [((2, 2, 2, 2), 1, 8), ((2, 2, 2, 2), 10, 8), ((4, 6, 4, 6), 4, 32), ((4, 6, 4, 6), 23, 32),
         ((12, 14, 14, 14), 11, 16), ((6, 10, 14, 90), 3, 40)]
LARGE = ((34, 32, 30, 50), 2, 128)


def tail_links(n, rest):
    """Which links of a parity's last `rest` storage entries: (V,) of one direction, both parities.  The last block
    of z and t holds the last entries, in (t, z, y, x / 2) order."""
    nx, ny, nz, nt = n
    bz, bt = (4 if nz % 4 == 0 else 2), (4 if nt % 4 == 0 else 2)
    t, z, y, x = np.meshgrid(np.arange(nt - bt, nt), np.arange(nz - bz, nz), np.arange(ny), np.arange(nx),
                             indexing="ij")
    site = (x + nx * (y + ny * (z + nz * t))).ravel()
    parity = ((x + y + z + t) & 1).ravel()
    mask = np.zeros(int(np.prod(n)), bool)
    for p in (0, 1):
        mask[site[parity == p][-rest:]] = True
    assert mask.sum() == 2 * rest
    return mask


def allowed(decisions):
    m = 1e-6 * decisions
    return 0 if m < 0.01 else 25 * math.ceil(m + 4 * math.sqrt(m))


def agrees(got, want, n, hits, rest):
    off = np.abs(got - want).max(-1) > 1e-4
    decisions = 4 * hits * int(np.prod(n))
    return off.sum() <= allowed(decisions) and off[:, tail_links(n, rest)].sum() <= min(rest // 4, allowed(decisions))


def oracle_sweep(n, hits):
    start = O.hot_start_haar(n, 5)
    U = start.copy()
    return start, U, O.cb_sweep(U, n, 6.0, 0.24, hits, 9, 3, True)


@pytest.mark.parametrize("n, hits, rest", SMALL, ids=str)
def test_bounds_see_a_lost_tail(n, hits, rest):
    """Planted in the oracle's result: the last group's links of one direction and parity left as they were."""
    start, U, _ = oracle_sweep(n, hits)
    assert (int(np.prod(n)) // 2) % 64 == rest
    tail = np.flatnonzero(tail_links(n, rest))
    c = np.stack([tail // int(np.prod(n[:k])) % n[k] for k in range(4)])
    lost = tail[c.sum(0) % 2 == 1]
    moved = np.abs(U - start)[2, lost].max(-1) > 1e-4
    bad = U.copy()
    bad[2, lost] = start[2, lost]
    assert agrees(U, U, n, hits, rest)
    if moved.sum() > rest // 4:  # one hit in ten is accepted: with a single one most links stay as they are
        assert not agrees(bad, U, n, hits, rest)
    else:
        assert hits < 4


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [glacx.FP32_LINKS, glacx.FP32_COMPRESSED], ids=["fp32", "fp32c"])
@pytest.mark.parametrize("n, hits, rest", SMALL + [LARGE], ids=str)
def test_last_links_follow_oracle(n, hits, rest, prec):
    print(f"\n[gpu case] sweep edges {n} hits={hits} prec={prec}", flush=True)
    _, U, accepted = oracle_sweep(n, hits)
    with glacx.Lattice(n, prec) as L:
        L.hot_start(5)
        acc = L.metropolis(1, 6.0, 0.24, hits, seed=9, sweep_offset=3)[0]
        chain = L.download()
    decisions = 4 * hits * int(np.prod(n))
    assert agrees(chain, U, n, hits, rest)
    assert abs(acc - accepted) * decisions <= allowed(decisions) * hits + 0.5
