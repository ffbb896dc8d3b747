"""P2G over the ways it takes a block: counts around the lanes-per-particle remainders (2, 7,
21), a wave (64), the single wave's limit (128), a team's round (256) and the ordering
window (512), with and without CPIC affinity in the block.  One substep against the oracle
to the parity bar (tests/parity.py), and the same bits for any order of the particles."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

from parity import assert_field_close, oracle_pair

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 3, 7, 8, 9, 21, 22, 63, 64, 65, 66, 71, 85, 127, 128, 129, 191, 255, 256, 257, 511, 512, 513, 1025]


def _scene(counts, cpic, seed=5, order=None):
    """counts[k] particles in block (3 k, 0, 0), all eight spill regions reached by the
    larger blocks; a floor under them."""
    h = 0.25
    rng = np.random.default_rng(seed)
    pos = np.concatenate([(np.array([12 * k, 0, 0]) + 0.5 + rng.random((n, 3)) * 3.98) * h for k, n in enumerate(counts)])
    pos += h                                    # base cells 0..3 of the block
    v = rng.normal(0, 0.5, pos.shape)
    sc = scenes.make_scene(scenes.particles(pos, h / 4, 1000.0, scenes.model_neo_hookean(1e5, 0.3), velocity=v), h, 1e-3,
                           colliders=scenes.cuboid((0.0, 0.02, 0.0), (200.0, 0.3, 200.0), bc=scenes.BC_SEPARATE, friction=0.4),
                           cpic=cpic)
    sc.C = rng.normal(0, 2.0, (sc.n, 9)).astype(np.float32)
    if order is not None:
        for f in ("x", "v", "F", "C", "mass", "vol0", "radius", "damping", "enabled", "fixed", "tag", "model"):
            setattr(sc, f, np.ascontiguousarray(getattr(sc, f)[order]))
    return sc


@pytest.mark.parametrize("cpic", [False, True])
@pytest.mark.parametrize("counts", [COUNTS, [513], [129, 1], [4097]], ids=["all", "one_crowded", "crowded_and_one", "very_crowded"])
def test_block_counts(pipeline, counts, cpic):
    sc = _scene(counts, cpic)
    st = mpm.MpmState.from_scene(pipeline, sc)
    pipeline.step(st)
    got = st.read_particles()
    o32, o64 = oracle_pair(_scene(counts, cpic), 1)
    for f in ("x", "v", "C", "F"):
        assert_field_close(f, got[f], getattr(o32.s, f), getattr(o64.s, f), o64.s)
    # another order of the particles, and three more substeps of each: the same bits
    order = np.random.default_rng(9).permutation(sc.n)
    other = mpm.MpmState.from_scene(pipeline, _scene(counts, cpic, order=order))
    for k in range(4):
        pipeline.step(other)
        if k:
            pipeline.step(st)
    a, b = st.read_particles(), other.read_particles()
    for f in ("x", "v", "C", "F", "enabled"):
        assert np.array_equal(a[f][order], b[f]), f
    st.close()
    other.close()


def test_values_that_are_not_finite_reach_only_their_nodes(pipeline):
    """A particle with an infinite velocity and one with a NaN affine matrix: their blocks'
    other nodes, and the other blocks, keep the values they have without them."""
    counts = [70, 300, 40]
    ref = _scene(counts, False)
    bad = _scene(counts, False)
    bad.v[3] = (np.inf, 0.0, 0.0)
    bad.C[75] = np.nan
    out = []
    for sc in (ref, bad):
        st = mpm.MpmState.from_scene(pipeline, sc)
        st.set_debug_grid(True)
        pipeline.step(st)
        grid = st.read_grid(momentum=True)
        order = np.lexsort(st.read_sort_canonical()["vid"].T)   # blocks come in hash order
        out.append((st.read_particles(), {k: v[order] for k, v in grid.items()}))
        st.close()
    (a, ga), (b, gb) = out
    last = slice(370, 410)
    for f in ("x", "v", "C", "F"):
        assert np.array_equal(a[f][last], b[f][last]), f
    good = np.isfinite(gb["mv"]).all(-1)
    assert np.isfinite(ga["mv"]).all() and 27 <= (~good).sum() <= 2 * 27
    assert np.array_equal(ga["m"][good], gb["m"][good])
