"""Single calls through the batch kernels: the argument block by value (forward, 7
and 8 levels) or in the workspace (sixteen levels, forward + VJP), written by the
level-set launch or, with a given level set, by one of its own.

The fused launch computes the same terms from the same code, so a call given the
level set that the fused call found must agree with it to rounding: 1e-6 of each
field's largest value for the tendencies, 1e-5 for the gradients, whose sums may
contract differently in the two builds."""
import numpy as np
import pytest

from jcm_amd import synthetic
from jcm_amd.physics_interface import PhysicsTendency

pytestmark = pytest.mark.gpu
FIELDS = ("u_wind", "v_wind", "temperature", "specific_humidity")


def _close(a, b, tol):
    a, b = (x.detach().cpu().numpy().astype(np.float64) for x in (a, b))
    assert np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("kx", [7, 8, 16])
@pytest.mark.parametrize("kind", ["plain", "verify", "diagnostics", "vjp"])
def test_given_level_set_equals_the_fused_call(kx, kind):
    import torch
    from jcm_amd.speedy_physics import SpeedyPhysics
    nlon, nlat = 64, 33
    phys = SpeedyPhysics(with_diagnostics=kind == "diagnostics")
    case = synthetic.make_case(nlon, nlat, kx, seed=31, land=True)
    if kind == "vjp":
        rng = np.random.default_rng(32)
        cot = PhysicsTendency(*(rng.standard_normal((kx, nlon, nlat)).astype(np.float32) for _ in range(4)))
        run = lambda *c, **k: phys.compute_tendencies_vjp(*c, cot, **k)  # noqa: E731
    else:
        run = lambda *c, **k: phys.compute_tendencies(*c, verify=kind == "verify", **k)  # noqa: E731
    first = run(*case)
    torch.cuda.synchronize()
    S = phys.level_sets(nlon, nlat, 1)[0]
    given = run(*case, level_set=S)
    for f in FIELDS:
        _close(getattr(given[0], f), getattr(first[0], f), 1e-6)
    if kind == "vjp":
        for f in FIELDS + ("normalized_surface_pressure",):
            _close(getattr(given[1], f), getattr(first[1], f), 1e-5)
