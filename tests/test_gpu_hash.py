"""The block hash in scenes that its regions hold awkwardly: a sheet one block thick (a floor
covered with sand uses a quarter of the places of a group of blocks), a line along each axis,
blocks on both sides of the coordinate origin, one particle per block at almost the whole
grid capacity, and the smallest capacities.  The set of active blocks, the canonical sort
and the neighbours (through the substep's result) against the oracle."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

from parity import assert_field_close, compare_sort, oracle_pair

pytestmark = pytest.mark.gpu
H = 1 / 32


def _blocks(kind, n):
    """Block coordinates, one particle each, far enough apart that no two are neighbours."""
    if kind == "sheet":
        s = int(np.ceil(n ** 0.5))
        b = np.stack(np.meshgrid(np.arange(s), [0], np.arange(s)), -1).reshape(-1, 3) - [s // 2, 0, s // 2]
    elif kind == "ball":
        b = np.unique(np.floor(np.random.default_rng(n).normal(0, n ** (1 / 3), (4 * n, 3))).astype(int), axis=0)
        np.random.default_rng(1).shuffle(b)
    else:
        b = np.zeros((n, 3), int)
        b[:, "xyz".index(kind)] = np.arange(n) - n // 2
    return b[:n] * 2


@pytest.mark.parametrize("kind", ["sheet", "ball", "x", "y", "z"])
@pytest.mark.parametrize("capacity", [8, 64, 1024, 4096])
def test_awkward_block_sets(pipeline, kind, capacity):
    # Each particle activates its block and 7 neighbours; along y the domain has 1021 blocks.
    n = min(capacity // 8, 500) if kind == "y" else capacity // 8
    rng = np.random.default_rng([capacity, len(kind)])
    x = (_blocks(kind, n) * 4 + rng.uniform(1.6, 4.4, (n, 3))) * H
    v = rng.normal(0, 0.5, (n, 3))
    sc = scenes.make_scene(scenes.particles(x, H / 4, 1000.0, scenes.model_neo_hookean(1e4, 0.3), velocity=v), H, 1e-3)
    st = mpm.MpmState.from_scene(pipeline, sc, capacity)
    pipeline.step(st)
    x0 = sc.x.copy()
    o32, o64 = oracle_pair(sc, 1)
    can = st.read_sort_canonical()
    assert can["vid"].shape[0] == 8 * n     # the capacity, exactly
    compare_sort(can, o32, x0, sc.cell_width)
    p = st.read_particles()
    for f in ("x", "v", "C", "F"):
        assert_field_close(f, p[f], getattr(o32.s, f), getattr(o64.s, f), o64.s)
    st.close()
