"""The tuner's P2G stage tries only launches that differ: a world whose particle count bounds
the launch has one, a larger one three (the first stage times each candidate over three
substeps after an untimed one, the others three and five candidates)."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cpic,launches", [(1000, False, 1), (60_000, False, 1), (60_000, True, 2), (300_000, False, 3),
                                             (1_048_576, False, 3)])
def test_tuner_launches_differ(pipeline, n, cpic, launches):
    h = 1 / 32
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    x = (np.stack(np.unravel_index(np.arange(n), (side,) * 3), -1) + rng.uniform(0.2, 0.8, (n, 3))) * h / 2
    sc = scenes.make_scene(scenes.particles(x, h / 4, 1000.0, scenes.model_neo_hookean(1e4, 0.3)), h, 1e-4, cpic=cpic)
    st = mpm.MpmState.from_scene(pipeline, sc)
    st.set_autotune(True)
    for _ in range(60):
        pipeline.step(st)
        if not st.autotune_state()[0]:
            break
    tuning, substeps = st.autotune_state()
    assert not tuning and substeps == (1 + 3 * launches) + (1 + 9) + (1 + 15)
    st.close()
