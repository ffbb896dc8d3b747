"""The Drucker-Prager projection over the size of the plastic change (its growth factors
switch formula at 1/16) and over its three outcomes (elastic, slip, opened), for both
backbones: one substep of particles with random strains against the oracle."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

from parity import assert_field_close, oracle_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("neo_hookean", [False, True])
@pytest.mark.parametrize("strain", [0.0, 1e-5, 1e-3, 0.03, 0.06, 0.07, 0.3])
def test_sand_projection(pipeline, strain, neo_hookean):
    h, n = 1 / 64, 3000
    rng = np.random.default_rng([int(strain * 1e6), neo_hookean])
    pos = 0.3 + 0.2 * rng.random((n, 3))
    model = scenes.model_sand(3.5e5, 0.3, friction_deg=30.0, neo_hookean=neo_hookean)
    sc = scenes.make_scene(scenes.particles(pos, h / 4, 2200.0, model, velocity=rng.normal(0, 0.2, (n, 3))), h, 5e-5)
    # a third compressed, a third sheared, a third stretched
    F = np.eye(3) + strain * rng.uniform(-1, 1, (n, 3, 3)) + strain * np.repeat([-0.7, 0.0, 0.7], n // 3)[:, None, None] * np.eye(3)
    sc.F = F.reshape(n, 9).astype(np.float32)
    sc.model.view(np.float32)[:, 2] = rng.uniform(-0.1, 0.1, n) * strain      # log volume gain
    st = mpm.MpmState.from_scene(pipeline, sc)
    pipeline.step(st)
    p = st.read_particles()
    o32, o64 = oracle_pair(sc.copy(), 1)
    for f in ("x", "v", "C", "F"):
        assert_field_close(f, p[f], getattr(o32.s, f), getattr(o64.s, f), o64.s)
    assert np.array_equal(p["enabled"], o32.s.enabled)
    assert_field_close("plastic state", p["model"].view(np.float32)[:, :3], o32.s.pstate, o64.s.pstate)
    st.close()
