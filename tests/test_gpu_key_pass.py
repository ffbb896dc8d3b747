"""Keys and block insertions of particles in the order the host has them: around the key
pass's groups of 512 particles, blocks that come back all through the order or never (more
different ones than a group's set holds), and several scenes in one order.  The block set and
the canonical sort against the oracle, and the call without allocation to the same bits."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

from parity import compare_sort, oracle_pair
from test_zz_no_alloc import _Device, _compare, _step_noalloc

pytestmark = pytest.mark.gpu
H = 1 / 32


def _scene(n, per_block, seed):
    """n particles, per_block of them in each block of a cube of blocks, in random order."""
    rng = np.random.default_rng([n, per_block, seed])
    blocks = -(-n // per_block)
    side = int(np.ceil(blocks ** (1 / 3)))
    b = np.stack(np.unravel_index(np.arange(n) // per_block, (side,) * 3), -1) - side // 2
    x = ((b * 4 + rng.uniform(1.0, 4.9, (n, 3))) * H)[rng.permutation(n)]
    return scenes.make_scene(scenes.particles(x, H / 4, 1000.0, scenes.model_neo_hookean(1e4, 0.3),
                                              velocity=rng.normal(0, 0.3, (n, 3))), H, 5e-4)


@pytest.mark.parametrize("n,per_block", [(1, 1), (64, 1), (65, 2), (511, 1), (512, 1), (513, 3), (1025, 1), (4096, 1),
                                         (6001, 64), (8191, 40), (8192, 40), (16383, 40), (16384, 40)])
def test_key_pass(pipeline, n, per_block):
    sc = _scene(n, per_block, 0)
    cap = 32768
    st = mpm.MpmState.from_scene(pipeline, sc, cap)
    pipeline.step(st)
    x0 = sc.x.copy()
    o32, _ = oracle_pair(sc.copy(), 1)
    compare_sort(st.read_sort_canonical(), o32, x0, sc.cell_width)
    ref = st.read_particles()
    st.close()
    if n // per_block < 4096:   # (its scratch holds a grid of 4096 blocks)
        d = _Device(sc)
        _step_noalloc(pipeline, sc, d, 4096)
        _compare(d.read(), ref, sc)


def test_key_pass_scenes(pipeline):
    """Scenes of different sizes in one batch: the same bits as alone."""
    scs = [_scene(n, p, 1) for n, p in [(700, 1), (3, 1), (1500, 20), (513, 2)]]
    batch = mpm.Batch(pipeline)
    sts = [mpm.MpmState.from_scene(pipeline, sc, 8192) for sc in scs]
    for st in sts:
        batch.add(st)
    batch.step()
    got = [st.read_particles() for st in sts]
    for sc, p in zip(scs, got):
        alone = mpm.MpmState.from_scene(pipeline, sc, 8192)
        pipeline.step(alone)
        q = alone.read_particles()
        for f in ("x", "v", "C", "F", "enabled"):
            assert np.array_equal(p[f], q[f]), f
        alone.close()
