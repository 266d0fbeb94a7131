"""A chain follows its seed to the last bit whichever kernel a lattice's size picks.  A link's streams and its hot start
depend on its GLAC site number, so lattices that differ in Nt alone have the same links and draws on their common time
slices; after one sweep (eight sub-sweeps, each reading links up to one slice away) all slices more than eight from the
shorter one's ends must be equal.  The pairs lie on the two sides of every line between the kernels:

FP32   256 | 257 groups of 64 links of a direction and parity (3 + 5 | 1 + 1 wavefronts per group), 768 | 769 groups
       (| one wavefront per group, three per SIMD), 2048 | 2049 blocks of four groups, with two stored rows 3072 | 3073
       (| more per SIMD)
FP64   512 | 513 groups
learned  1536 | 1537 blocks (FP32)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
glacx = pytest.importorskip("glac_amd")

PREC = {"fp64": glacx.FP64, "fp32": glacx.FP32_LINKS, "fp32c": glacx.FP32_COMPRESSED}


def swept(n, prec, hits, reunit, learned):
    with glacx.Lattice(n, PREC[prec]) as L:
        L.hot_start(5)
        args = dict(n_hit=hits, reunit_every=reunit, seed=9, sweep_offset=3)
        if learned:
            rng = np.random.default_rng(11)
            L.proposal_set(rng.normal(size=glacx.PROPOSAL_NPARAM).astype(np.float32) * 0.1,
                           np.array([0, 50, 2500, 0, 0, 6], np.float32),
                           np.array([10, 290, 2200, 21, 5.5, 1], np.float32))
            L.metropolis_learned(1, 6.0, 0.24, **args)
        else:
            L.metropolis(1, 6.0, 0.24, **args)
        return L.download().reshape((4, n[3], -1, 18))


def compare(space, short, long, prec, hits, reunit=1, learned=False):
    print(f"\n[gpu case] chain bits {space} x {short} | {long} {prec} hits={hits} reunit={reunit} learned={learned}",
          flush=True)
    a = swept(space + (short,), prec, hits, reunit, learned)
    b = swept(space + (long,), prec, hits, reunit, learned)
    common = slice(8, short - 8)
    assert a[:, common].shape[1] >= 8 and np.array_equal(a[:, common], b[:, common])


@pytest.mark.parametrize("hits, reunit", [(3, 0), (11, 1)])
@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp32c"])
@pytest.mark.parametrize("space, short, long", [((8, 8, 8), 24, 160),       # 96 | 640 groups
                                                ((8, 8, 8), 160, 256),     # 640 | 1024
                                                ((6, 10, 14), 26, 90),     # 170.6 | 590.6
                                                ((6, 10, 14), 90, 150)],   # 590.6 | 984.4
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_small_lattices(space, short, long, prec, hits, reunit):
    compare(space, short, long, prec, hits, reunit)


@pytest.mark.parametrize("prec", ["fp32", "fp32c"])
def test_across_2048_and_3072_blocks(prec):
    compare((16, 16, 16), 32, 392, prec, 4)  # 256 | 3136 blocks


@pytest.mark.parametrize("prec", ["fp32", "fp32c"])
def test_learned_across_1536_blocks(prec):
    compare((16, 16, 16), 32, 200, prec, 4, learned=True)  # 256 | 1600 blocks
