"""Where one level of a column is not usable (a missing value), the gradients that do not
depend on it stay finite: a term that is off at a level adds nothing there, whatever its
other factor is.

A temperature of 0 makes the level's saturation humidity not finite, so every condition
on it is false and its terms are off."""
import numpy as np
import pytest

import helpers as H
from jcm_amd import synthetic
from jcm_amd.physics_interface import PhysicsTendency
from test_host_column import make

FIELDS = dict(u="u_wind", v="v_wind", t="temperature", q="specific_humidity")


def _case(name, field, value):
    """The case with `value` at one level (not the lowest) of every column, and that level."""
    case = make(name)
    kx, ix, il = case[2].nodal_shape
    level = (np.arange(ix * il) % (kx - 1)).reshape(ix, il)
    x = getattr(case[0], FIELDS[field]).copy()
    x[np.arange(kx)[:, None, None] == level] = value
    rng = np.random.default_rng(1)
    cot = [rng.standard_normal((kx, ix, il)).astype(np.float32) for _ in range(4)]
    return (case[0].copy(**{FIELDS[field]: x}),) + case[1:], level, cot


def _check_zero_temperature(level, g):
    kx = g["t"].shape[0]
    other = np.arange(kx)[:, None, None] != level
    for f in "uvtq":
        assert np.isfinite(g[f][other]).all(), f
    assert not np.isfinite(g["t"][~other]).any()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", ["T21_wet", "T21_wet_kx7", "T21_wet_kx16", "T21_wet_swoff"])
def test_a_level_of_zero_temperature_stays_alone(name, dtype):
    case, level, cot = _case(name, "t", 0.0)
    p = synthetic.draw_vjp_parameters(2)
    S = H.run_host_column(make(name), p)[2]
    with np.errstate(all="ignore"):
        g = H.run_host_vjp(case, p, cot, level_set=S, dtype=dtype)[1]
    _check_zero_temperature(level, g)
    assert np.isfinite(g["prm"]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("level_set", [-1, 0b1100])   # the single launch, and the batch kernels
@pytest.mark.parametrize("name", ["T21_wet", "T21_wet_kx7", "T21_wet_kx16"])
def test_a_level_of_zero_temperature_stays_alone_on_the_gpu(name, level_set):
    from jcm_amd.speedy_physics import SpeedyPhysics
    case, level, cot = _case(name, "t", 0.0)
    phys = SpeedyPhysics(parameters=synthetic.draw_vjp_parameters(2))
    _, sg, pg = phys.compute_tendencies_vjp(*case, PhysicsTendency(*cot), level_set=level_set)
    _check_zero_temperature(level, {k: getattr(sg, n).cpu().numpy() for k, n in FIELDS.items()})
    assert all(np.isfinite(v.cpu().numpy()).all() for v in pg.values())
