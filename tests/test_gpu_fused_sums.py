"""Parameter gradients summed inside the forward + VJP launch, by the block counted in
last for each member, at the edges of that rule (62 members; 63 and more are summed
in a launch of their own), with blocks that span two members and members of one block.

Each member's sums equal those of the same member called alone with its level set,
whose sums take a launch of their own: 1e-5 of the member's largest gradient (other
kernels, whose sums may contract differently).  Repeated calls, with calls on another
grid through the same object between them, give the same bits."""
import numpy as np
import pytest

from jcm_amd import synthetic
from jcm_amd.params import VJP_PARAMS
from jcm_amd.physics_interface import PhysicsTendency

pytestmark = pytest.mark.gpu
FIELDS = ("u_wind", "v_wind", "temperature", "specific_humidity")


@pytest.mark.parametrize("kx", [7, 8])
@pytest.mark.parametrize("nlon,nlat,nmember", [(64, 33, 1), (16, 16, 62), (16, 16, 63), (17, 16, 5), (97, 7, 3)])
def test_sums_in_the_launch_equal_their_own(nlon, nlat, nmember, kx):
    import torch
    from jcm_amd.speedy_physics import SpeedyPhysics
    phys = SpeedyPhysics()
    st, fo, ge, da = synthetic.make_case(nlon, nlat, kx, seed=51, land=True, nmember=nmember, member_t_sigma=0.5)
    rng = np.random.default_rng(52)
    cot = [rng.standard_normal(st.temperature.shape).astype(np.float32) for _ in range(4)]
    other = synthetic.make_case(30, 20, kx, seed=53, land=True)
    other_cot = PhysicsTendency(*(rng.standard_normal((kx, 30, 20)).astype(np.float32) for _ in range(4)))

    def grads(state, c, **more):
        g = phys.compute_tendencies_vjp(state, fo, ge, da, PhysicsTendency(*c), **more)[2]
        return np.stack([g[f"{a}.{b}"].cpu().numpy().reshape(-1) for a, b in VJP_PARAMS], axis=-1)

    first = grads(st, cot)
    S = phys.level_sets(nlon, nlat, nmember)
    for _ in range(4):
        phys.compute_tendencies_vjp(*other, other_cot)
        assert np.array_equal(grads(st, cot), first)
    for m in sorted({0, nmember // 2, nmember - 1}):
        one = st if nmember == 1 else st.copy(**{k: np.ascontiguousarray(getattr(st, k)[m]) for k in
                                                  FIELDS + ("geopotential", "normalized_surface_pressure")})
        alone = grads(one, cot if nmember == 1 else [np.ascontiguousarray(c[m]) for c in cot], level_set=S[m])[0]
        assert np.abs(first[m].astype(np.float64) - alone).max() <= 1e-5 * np.abs(alone).max()
