"""Batches in one launch (co-resident blocks, 7 and 8 levels, members of a workgroup
or more) and at the edges of that rule: exactly and just above the co-resident grid,
members of exactly one workgroup, blocks that span two members, one narrow member,
sixteen levels.  Every request equals the same request called alone, within 1e-6 of a
tendency's and 1e-5 of a gradient's largest value (the same code in another kernel,
whose sums may contract differently), with the same level set."""
import numpy as np
import pytest

from jcm_amd import synthetic
from jcm_amd.physics_interface import PhysicsTendency

pytestmark = pytest.mark.gpu
FIELDS = ("u_wind", "v_wind", "temperature", "specific_humidity")
T85, T21 = (256, 128, 1), (64, 32, 1)
BATCHES = {"co-resident grid": [T85 + ("vjp",), T85 + ("fwd",), T85 + ("vjp",), T85 + ("fwd",)],
           "above it": [T85 + ("vjp",), T85 + ("fwd",), T85 + ("vjp",), T85 + ("fwd",), T21 + ("vjp",)],
           "ragged members": [(33, 19, 3, "vjp"), (17, 16, 2, "fwd"), (16, 16, 1, "vjp"), (16, 16, 4, "fwd")],
           "one narrow": [(16, 8, 3, "vjp"), T21 + ("fwd",), T21 + ("vjp",)],
           "forward only": [T21 + ("fwd",), (30, 20, 2, "fwd")],
           "adjoint only": [T21 + ("vjp",), (30, 20, 2, "vjp")]}


def _close(a, b, tol):
    a, b = (x.detach().cpu().numpy().astype(np.float64) for x in (a, b))
    assert np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("kx", [7, 8, 16])
@pytest.mark.parametrize("batch", BATCHES)
def test_requests_equal_their_calls_alone(batch, kx):
    import torch
    from jcm_amd.serving import PhysicsServer, Request
    from jcm_amd.speedy_physics import SpeedyPhysics
    dev = torch.device("cuda", 0)
    up = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
    reqs = []
    for i, (nlon, nlat, nm, kind) in enumerate(BATCHES[batch]):
        st, fo, ge, da = synthetic.make_case(nlon, nlat, kx, seed=41 + i, land=True, nmember=nm, member_t_sigma=0.5)
        st = st.copy(**{k: up(getattr(st, k)) for k in FIELDS + ("geopotential", "normalized_surface_pressure")})
        rng = np.random.default_rng(i)
        cot = PhysicsTendency(*(up(rng.standard_normal(st.temperature.shape).astype(np.float32)) for _ in range(4)))
        reqs.append(Request(state=st, forcing=fo, geometry=ge, date=da, cotangent=cot if kind == "vjp" else None, rid=i))
    phys = SpeedyPhysics()
    server = PhysicsServer(phys, n_streams=1, record_level_sets=True)
    server.run(reqs, realtime=False)
    torch.cuda.synchronize()
    alone = SpeedyPhysics()
    for r, (nlon, nlat, nm, kind) in zip(reqs, BATCHES[batch]):
        case = (r.state, r.forcing, r.geometry, r.date)
        out = alone.compute_tendencies(*case) if kind == "fwd" else alone.compute_tendencies_vjp(*case, r.cotangent)
        torch.cuda.synchronize()
        assert list(r.level_set) == list(alone.level_sets(nlon, nlat, nm))
        for f in FIELDS:
            _close(getattr(r.tendency, f), getattr(out[0], f), 1e-6)
        if kind == "vjp":
            for f in FIELDS + ("normalized_surface_pressure",):
                _close(getattr(r.state_grads, f), getattr(out[1], f), 1e-5)
            for k, v in out[2].items():
                _close(r.param_grads[k], v, 1e-5)
