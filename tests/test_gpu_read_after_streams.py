"""Readbacks between worlds that come and go: staged uploads into batches that capture graphs
and are closed, their streams destroyed, while other scenes are read from the same context."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

pytestmark = pytest.mark.gpu
H = 1 / 32


def _scene(n, seed):
    rng = np.random.default_rng([n, seed])
    return scenes.make_scene(scenes.particles(rng.random((n, 3)), H / 4, 1000.0, scenes.model_neo_hookean(1e4, 0.3)), H, 5e-4)


@pytest.mark.parametrize("graph", [False, True])
def test_reads_while_streams_go(pipeline, graph):
    ref = None
    for k in range(6):
        batch = mpm.Batch(pipeline)
        if graph:
            batch.set_graph(True)
        member = mpm.MpmState.from_scene(pipeline, _scene(500, 0))
        batch.add(member)
        lone = mpm.MpmState.from_scene(pipeline, _scene(300, k))
        for _ in range(3):
            batch.step()
            pipeline.step(lone)
            lone.read_particles()
        got = member.read_particles()
        if ref is not None:
            for f in ("x", "v", "C", "F"):
                assert np.array_equal(got[f], ref[f]), f
        ref = got
        batch.close()
        for _ in range(3):
            pipeline.step(lone)
            lone.read_particles()
        lone.close()
        member.close()
