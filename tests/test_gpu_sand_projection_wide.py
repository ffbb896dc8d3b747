"""The Drucker-Prager projection where singular values of F change by a large factor: one
substep of particles at rest with wide random strains.  The mean relative error of F against
64 bits is at most three times the 32-bit oracle's, and one rounding more (the GPU's SVD runs
on reciprocals of about 1 ulp)."""
import numpy as np
import pytest

from nexus_amd import mpm, scenes

from parity import oracle_pair

pytestmark = pytest.mark.gpu


def _rotations(rng, n):
    q, _ = np.linalg.qr(rng.normal(size=(n, 3, 3)))
    return q * np.sign(np.linalg.det(q))[:, None, None]


@pytest.mark.parametrize("neo_hookean", [False, True])
@pytest.mark.parametrize("strain", [0.2, 0.6, 1.0, 1.5, 2.0])
def test_wide_sand_projection(pipeline, strain, neo_hookean):
    h, n = 1 / 64, 3000
    rng = np.random.default_rng([int(strain * 10), neo_hookean])
    model = scenes.model_sand(3.5e5, 0.3, friction_deg=30.0, neo_hookean=neo_hookean)
    sc = scenes.make_scene(scenes.particles(0.3 + 0.2 * rng.random((n, 3)), h / 4, 2200.0, model), h, 5e-5)
    # a third compressed, a third sheared, a third stretched
    logs = strain * (rng.normal(size=(n, 3)) + np.repeat([-0.7, 0.0, 0.7], n // 3)[:, None])
    F = (_rotations(rng, n) * np.exp(logs)[:, None, :]) @ _rotations(rng, n)
    sc.F = F.transpose(0, 2, 1).reshape(n, 9).astype(np.float32)
    st = mpm.MpmState.from_scene(pipeline, sc)
    pipeline.step(st)
    got = st.read_particles()["F"]
    st.close()
    o32, o64 = oracle_pair(sc.copy(), 1)
    ref = o64.s.F.reshape(n, 9).astype(np.float64)
    norm = np.linalg.norm(ref, axis=1)
    err = np.linalg.norm(got - ref, axis=1) / norm
    mirror = np.linalg.norm(o32.s.F.reshape(n, 9) - ref, axis=1) / norm
    print(f"mean {err.mean():.2e}, 32-bit oracle {mirror.mean():.2e}; largest {err.max():.2e}, {mirror.max():.2e}")
    assert err.mean() <= 3 * mirror.mean() + 2.0 ** -23
