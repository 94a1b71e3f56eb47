"""The single launch with every level-set word formed by the block that needs it
(SPEEDY_FLAG_NO_WAIT, what a block does whose neighbours have not started), in batches
and in the forward + VJP: the same bits as by the exchange of words."""
import numpy as np
import pytest

from jcm_amd import _native, synthetic
from jcm_amd.physics_interface import PhysicsTendency

pytestmark = pytest.mark.gpu
FIELDS = ("u_wind", "v_wind", "temperature", "specific_humidity")
STATE = FIELDS + ("geopotential", "normalized_surface_pressure")


def _bits(tend, sg, pg):
    out = [getattr(tend, f) for f in FIELDS]
    if sg is not None:
        out += [getattr(sg, f) for f in FIELDS + ("normalized_surface_pressure",)] + [pg[k] for k in sorted(pg)]
    return [x.cpu().numpy() for x in out]


@pytest.mark.parametrize("kx", [7, 8])
def test_batches(kx):
    import torch
    from jcm_amd.serving import PhysicsServer, Request
    from jcm_amd.speedy_physics import SpeedyPhysics
    up = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    cases = []
    for i, (nlon, nlat, nm, vjp) in enumerate([(33, 19, 3, True), (17, 16, 2, False), (16, 16, 1, True), (64, 32, 1, True),
                                               (16, 16, 4, False)]):
        st, fo, ge, da = synthetic.make_case(nlon, nlat, kx, seed=71 + i, land=True, nmember=nm, member_t_sigma=0.5)
        st = st.copy(**{k: up(getattr(st, k)) for k in STATE})
        rng = np.random.default_rng(i)
        cot = PhysicsTendency(*(up(rng.standard_normal(st.temperature.shape).astype(np.float32)) for _ in range(4)))
        cases.append((st, fo, ge, da, cot if vjp else None))

    def serve(flag):
        server = PhysicsServer(SpeedyPhysics(), n_streams=1, record_level_sets=True)
        member = server._member
        server._member = lambda req: (lambda h: h[:3] + (h[3] | flag,) + h[4:])(member(req))
        for _ in range(2):   # the second batch finds the words of the first
            reqs = [Request(state=s, forcing=f, geometry=g, date=d, cotangent=c) for s, f, g, d, c in cases]
            server.run(reqs, realtime=False)
        assert max(server.batch_sizes) == len(cases)
        return [(list(r.level_set), _bits(r.tendency, r.state_grads, r.param_grads)) for r in reqs]

    for (s0, a), (s1, b) in zip(serve(0), serve(_native.FLAG_NO_WAIT)):
        assert s0 == s1
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("kx", [7, 8])
@pytest.mark.parametrize("nlon,nlat,nmember", [(64, 32, 1), (33, 19, 3), (256, 128, 1)])
def test_forward_and_vjp(nlon, nlat, nmember, kx):
    from jcm_amd.speedy_physics import SpeedyPhysics
    case = synthetic.make_case(nlon, nlat, kx, seed=81, land=True, nmember=nmember, member_t_sigma=0.5)
    rng = np.random.default_rng(82)
    cot = PhysicsTendency(*(rng.standard_normal(case[0].temperature.shape).astype(np.float32) for _ in range(4)))
    res = []
    for flag in (0, _native.FLAG_NO_WAIT):
        phys = SpeedyPhysics()
        phys._launch_flags = flag
        for _ in range(2):
            out = _bits(*phys.compute_tendencies_vjp(*case, cot))
        res.append((phys.level_sets(nlon, nlat, nmember), out))
        assert phys.barrier_status(nlon, nlat, nmember) == 0
    assert res[0][0] == res[1][0]
    for x, y in zip(res[0][1], res[1][1]):
        assert np.array_equal(x, y)
