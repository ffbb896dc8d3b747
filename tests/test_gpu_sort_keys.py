"""The canonical sort against block keys worked out from the positions alone: a key pass whose
workgroups meet more different blocks than their set in LDS holds and go on to further rounds,
and, over the sizes of the hash, the keys and slots that the particle update leaves for
the next substep."""
import numpy as np
import pytest

import oracle as O
from nexus_amd import mpm, scenes

from test_gpu_key_pass import _scene as _dense
from test_gpu_slot_scan import _scene as _sparse

pytestmark = pytest.mark.gpu


def _check_sort(can, x, h):
    vid, loc = O.block_keys(np.asarray(x, np.float32), h, 32)
    assert np.array_equal(can["vid"][can["particle_block"]], vid)
    assert np.array_equal(can["particle_cell"], loc[:, 0] + 4 * loc[:, 1] + 16 * loc[:, 2])
    occupied, count = np.unique(vid, axis=0, return_counts=True)
    corners = np.stack(np.unravel_index(np.arange(8), (2, 2, 2)), -1)
    active = np.unique((occupied[:, None, :] + corners).reshape(-1, 3), axis=0)
    order = np.lexsort(can["vid"].T[::-1])
    assert np.array_equal(can["vid"][order], active)
    held = {tuple(v): c for v, c in zip(occupied.tolist(), count.tolist())}
    assert can["np"][order].tolist() == [held.get(tuple(v), 0) for v in active.tolist()]


@pytest.mark.parametrize("n,per_block", [(600_001, 2), (1_100_003, 3)])
def test_key_set_over_rounds(pipeline, n, per_block):
    """Two and three rounds of 512 particles a workgroup, in random order: nearly every one of
    them of a block of its own, so that the second round fills the set of 1024 and the
    third starts with it emptied."""
    sc = _dense(n, per_block, 0)
    st = mpm.MpmState.from_scene(pipeline, sc, 1 << 19)
    pipeline.step(st)
    _check_sort(st.read_sort_canonical(), sc.x, sc.cell_width)
    st.close()


@pytest.mark.parametrize("capacity,n", [(8, 1), (256, 20), (512, 60), (1024, 100), (1 << 18, 900), (1 << 19, 900),
                                        (1 << 19, 1)])
def test_keys_of_the_particle_update(pipeline, capacity, n):
    sc = _sparse(n, 0)
    sc.v[:] = np.random.default_rng(n).normal(0, 0.3 * sc.cell_width / sc.dt, (n, 3))   # many change their block
    st = mpm.MpmState.from_scene(pipeline, sc, capacity)
    seen = []
    for _ in range(4):
        x = st.read_positions()
        pipeline.step(st)
        can = st.read_sort_canonical()
        _check_sort(can, x, sc.cell_width)
        seen.append(can["vid"][can["particle_block"]])
    if n >= 100:
        assert (seen[0] != seen[3]).any(1).sum() > n // 20
    st.close()
