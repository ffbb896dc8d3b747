"""State readback (rows gathered by particle id on the device, copied through two pinned
chunks of 4 MiB): exact values in id order at sizes around a wave, a chunk (349,525
positions or 34,952 whole states are just under one) and two chunks, before and after the
sort has reordered the arena, and after a batch has put scenes behind one another."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

pytestmark = pytest.mark.gpu


def _scene(n, seed):
    rng = np.random.default_rng(seed)
    x = 0.3 + 0.4 * rng.random((n, 3))
    sc = scenes.make_scene(scenes.particles(x, 1 / 256, 1000.0, scenes.model_neo_hookean(1e3, 0.3)), 1 / 64, 1e-4,
                           gravity=(0.0, 0.0, 0.0))
    # constants that name their particle
    sc.mass = (1.0 + np.arange(n) / 2 ** 22).astype(np.float32)
    sc.vol0 = (1e-6 * (1.0 + np.arange(n) / 2 ** 22)).astype(np.float32)
    sc.fixed = (np.arange(n) % 3 == 0).astype(np.uint32)
    return sc


@pytest.mark.parametrize("n", [1, 63, 65, 34_952, 34_953, 349_525, 349_526, 700_001])
def test_state_comes_back_in_id_order(pipeline, n):
    sc = _scene(n, n)
    st = mpm.MpmState.from_scene(pipeline, sc)
    for k in range(3):
        pipeline.step(st)
        p = st.read_particles()
        assert np.array_equal(p["mass"], sc.mass) and np.array_equal(p["vol0"], sc.vol0)
        assert np.array_equal(p["fixed"], sc.fixed) and p["enabled"].all()
        assert np.array_equal(p["x"], st.read_positions())
        # fixed particles stay where they were put
        assert np.array_equal(p["x"][sc.fixed != 0], sc.x[sc.fixed != 0])
        assert np.array_equal(st.prep_readback()["position"], p["x"])
    can = st.read_sort_canonical()             # its inputs are not touched by the readbacks
    cell = np.floor(p["x"][sc.fixed != 0].astype(np.float64) * 64 + 0.5).astype(np.int64) - 1
    assert np.array_equal(can["vid"][can["particle_block"]][sc.fixed != 0], cell >> 2)
    st.close()


def test_batch_members_read_their_own_rows(pipeline):
    scs = [_scene(n, n) for n in (1000, 1, 40_001)]
    batch = mpm.Batch(pipeline)
    states = [mpm.MpmState.from_scene(pipeline, sc) for sc in scs]
    for st in states:
        batch.add(st)
    batch.run(2)
    for st, sc in zip(states, scs):
        p = st.read_particles()
        assert np.array_equal(p["mass"], sc.mass) and np.array_equal(p["x"], st.read_positions())
    batch.remove(states[0])                    # back to the host, then on alone
    pipeline.step(states[0])
    assert np.array_equal(states[0].read_particles()["mass"], scs[0].mass)
    batch.close()
    for st in states:
        st.close()
