"""Any positive cap on the grid-stride kernels' workgroups: one, a few (a workgroup takes several
chunks of the unsorted count, several tiles of each scan) and caps beyond what any launch
needs, up to the largest word.  The same bits as the default, whose first substep is checked
against the oracle's sort."""
import numpy as np
import pytest

from nexus_amd import mpm

from parity import compare_sort, oracle_pair
from test_gpu_key_pass import _scene

pytestmark = pytest.mark.gpu


def _run(pipeline, sc, groups, substeps):
    st = mpm.MpmState.from_scene(pipeline, sc, 32768)
    batch = mpm.Batch(pipeline)
    batch.add(st)
    if groups:
        batch.set_launch_config(batch.launch_config()[0], 16, groups)
    batch.step()
    sort = st.read_sort_canonical()
    for _ in range(substeps - 1):
        batch.step()
    out = st.read_particles()
    batch.close()
    st.close()
    return sort, out


@pytest.mark.parametrize("n,per_block", [(700, 3), (20_011, 7)])
def test_any_cap(pipeline, n, per_block):
    sc = _scene(n, per_block, 3)
    _, ref = _run(pipeline, sc, 0, 3)
    o32, _ = oracle_pair(sc.copy(), 1)
    for groups in (1, 3, 8, 1 << 24, 1 << 28, (1 << 28) + 1, (1 << 31) - 1, 1 << 31, (1 << 32) - 1):
        sort, out = _run(pipeline, sc, groups, 3)
        compare_sort(sort, o32, sc.x, sc.cell_width)
        for f in ("x", "v", "C", "F", "enabled"):
            assert np.array_equal(ref[f], out[f]), (groups, f)
