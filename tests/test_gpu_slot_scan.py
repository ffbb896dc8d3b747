"""The scans of the sort over the sizes of the hash: one tile, a slot over one and over two, the
two tile sizes' border, and many small scenes whose regions share a row of 64 slots."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

from parity import compare_sort, oracle_pair

pytestmark = pytest.mark.gpu
H = 1 / 32


def _scene(n, seed):
    rng = np.random.default_rng([n, seed])
    x = rng.uniform(-1, 1, (n, 3)) * H * 4 * max(1.0, n ** (1 / 3))
    return scenes.make_scene(scenes.particles(x, H / 4, 1000.0, scenes.model_neo_hookean(1e4, 0.3)), H, 5e-4)


@pytest.mark.parametrize("capacity,n", [(8, 1), (256, 20), (512, 60), (1024, 100), (1 << 18, 900), (1 << 19, 900),
                                        (1 << 19, 1)])
def test_slot_scan(pipeline, capacity, n):
    sc = _scene(n, 0)
    st = mpm.MpmState.from_scene(pipeline, sc, capacity)
    for k in range(2):     # keys by the key pass, then by the particle update
        x0 = st.read_particles()["x"].copy()
        pipeline.step(st)
        cur = _scene(n, 0)
        o32, _ = oracle_pair(cur, k + 1)
        can = st.read_sort_canonical()
        if k == 0:
            compare_sort(can, o32, x0, sc.cell_width)
        assert can["np"].sum() == n
    st.close()


def test_slot_scan_of_small_scenes(pipeline):
    """40 scenes of 17 and 33 slots in one world: the same bits as alone."""
    scs = [_scene(1 + k % 2, k) for k in range(40)]
    caps = [8 << (k % 2) for k in range(40)]
    batch = mpm.Batch(pipeline)
    sts = [mpm.MpmState.from_scene(pipeline, sc, cap) for sc, cap in zip(scs, caps)]
    for st in sts:
        batch.add(st)
    for _ in range(3):
        batch.step()
    for sc, cap, st in zip(scs, caps, sts):
        alone = mpm.MpmState.from_scene(pipeline, sc, cap)
        for _ in range(3):
            pipeline.step(alone)
        p, q = st.read_particles(), alone.read_particles()
        for f in ("x", "v", "C", "F", "enabled"):
            assert np.array_equal(p[f], q[f]), f
        alone.close()
