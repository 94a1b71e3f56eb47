"""Edges of the native call preparation (csrc/host_calls.cpp): what the general Python
path accepts, refuses and raises is the same before and after a grid's first call,
which is the one that the native path leaves to it."""
import numpy as np
import pytest

from test_gpu_host_calls import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [True, 1, np.bool_(True), False, 0, None])
def test_diagnostics_are_asked_for_by_truth_value(value):
    from jcm_amd.speedy_physics import SpeedyPhysics
    st, fo, ge, da, _ = _case()
    phys = SpeedyPhysics(with_diagnostics=value)
    for _ in range(3):   # the first call makes the workspace, the others are native
        _, data = phys.compute_tendencies(st, fo, ge, da)
        assert (data is not None) == bool(value)


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("call", ["fwd", "vjp", "d2p", "t2d"])
def test_out_of_memory_keeps_its_type(call, native, monkeypatch):
    """A caller that catches torch.OutOfMemoryError, to free something or to go on with
    fewer members, still can.  The allocator's own limit stands in for a full card."""
    import torch
    from jcm_amd import _native
    from jcm_amd import transforms as T
    from jcm_amd.physics_interface import PhysicsTendency
    from jcm_amd.speedy_physics import SpeedyPhysics
    if call in ("fwd", "vjp"):   # fields of 16 MiB
        st, fo, ge, da, cot = _case(nmember=128, nlon=64, nlat=64)
        phys = SpeedyPhysics()
        run = ((lambda: phys.compute_tendencies(st, fo, ge, da)) if call == "fwd" else
               (lambda: phys.compute_tendencies_vjp(st, fo, ge, da, cot)))
    else:
        grid = T.SpectralGrid.truncation(213)
        z = lambda *s: torch.zeros(s, device="cuda")  # noqa: E731
        dyn = T.PrimitiveEquations(z(16) + 250.0, z(*grid.modal_shape),
                                   T.CoordinateSystem(grid, T.SigmaCoordinates(np.linspace(0, 1, 17))))
        if call == "d2p":
            m = z(16, *grid.modal_shape)
            state = T.DynamicsState(m, m, m, z(*grid.modal_shape), {"specific_humidity": m})
            run = lambda: T.dynamics_state_to_physics_state(state, dyn)  # noqa: E731
        else:
            x = z(16, *grid.nodal_shape)
            tend = PhysicsTendency(x, x, x, x)
            run = lambda: T.physics_tendency_to_dynamics_tendency(tend, dyn)  # noqa: E731
    run()                               # workspaces and plans
    torch.cuda.synchronize()
    if not native:
        monkeypatch.setattr(_native, "host", None)
        monkeypatch.setattr(T, "host", None)
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    held = []
    try:
        for size in (4 << 20, (1 << 20) + 512):   # what the allocator still has
            with pytest.raises(torch.OutOfMemoryError):
                while True:
                    held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        with pytest.raises(torch.OutOfMemoryError):
            run()
    finally:
        del held
        torch.cuda.set_per_process_memory_fraction(1.0)
    run()
    torch.cuda.synchronize()


def test_parameter_types_are_judged_alike_on_every_call():
    """A flag that is not a bool is refused by Parameters.to_abi, so also once the grid's
    workspace exists; values that it converts are taken."""
    from jcm_amd import Parameters
    from jcm_amd.speedy_physics import SpeedyPhysics
    st, fo, ge, da, _ = _case()
    for group, name, value in [("surface_flux", "lscasym", 1), ("surface_flux", "lskineb", 0),
                               ("forcing", "increase_co2", 1)]:
        phys = SpeedyPhysics(parameters=Parameters.default().replace(**{group: {name: value}}))
        for _ in range(3):
            with pytest.raises(TypeError):
                phys.compute_tendencies(st, fo, ge, da)
    for group, name, value in [("forcing", "co2_year_ref", 1960.0), ("forcing", "co2_year_ref", True),
                               ("convection", "rhbl", 1), ("convection", "rhbl", True), ("convection", "rhbl", "0.9")]:
        phys = SpeedyPhysics(parameters=Parameters.default().replace(**{group: {name: value}}))
        for _ in range(2):
            phys.compute_tendencies(st, fo, ge, da)


def test_device_copies_given_back_are_made_again():
    """The cache of device copies of NumPy fields is bounded; after it was emptied, a
    forcing and geometry known from before find their copies again."""
    from jcm_amd import _native, synthetic
    from jcm_amd.speedy_physics import SpeedyPhysics
    st, fo, ge, da, _ = _case()
    fo = fo.copy(**{k: getattr(fo, k).cpu().numpy() for k in ("alb0", "sice_am", "snowc_am", "soilw_am", "stl_am",
                                                              "sea_surface_temperature")})
    phys = SpeedyPhysics()
    native = lambda: _native.host.fwd(phys._consts, phys._workspaces, phys.parameters, *phys._where(), st, fo, ge, da, 0,  # noqa: E731,E501
                                      _native.TERMS_ALL, -1, False)
    phys.compute_tendencies(st, fo, ge, da)
    assert isinstance(native(), tuple)
    keep = []
    for i in range(30):                  # 11 fields each
        other = synthetic.make_case(4, 6, 8, seed=i, land=True)
        keep.append(other)
        phys.compute_tendencies(*other)
        assert len(phys._consts) <= 257
        phys.compute_tendencies(st, fo, ge, da)
        assert isinstance(native(), tuple)


class _Counting:
    """The parameters, counting how often one of their groups is read."""

    def __init__(self, p):
        self.__dict__.update(p=p, reads=0)

    def __getattr__(self, name):
        self.__dict__["reads"] += 1
        return getattr(self.p, name)


@pytest.mark.parametrize("form", ["climatology", "tensor climatology", "new forcing", "new grid", "numpy state"])
def test_refused_calls_have_not_packed_their_parameters(form, monkeypatch):
    """Calls that the native path leaves to the general one are found out by their fields:
    parameters, levels and date are read for the general path alone."""
    import torch
    from jcm_amd import Parameters, _native
    from jcm_amd.speedy_physics import SpeedyPhysics
    st, fo, ge, da, _ = _case()
    host = {k: getattr(fo, k).cpu().numpy() for k in ("sice_am", "stl_am", "sea_surface_temperature")}
    if form == "climatology":
        fo = fo.copy(**{k: np.repeat(v[..., None], 4, -1) for k, v in host.items()})
    elif form == "tensor climatology":
        fo = fo.copy(**{k: torch.as_tensor(np.repeat(v[..., None], 4, -1), device="cuda") for k, v in host.items()})
    elif form == "numpy state":
        st = st.copy(temperature=st.temperature.cpu().numpy())
    phys = SpeedyPhysics(parameters=_Counting(Parameters.default()))
    phys.compute_tendencies(st, fo, ge, da)
    reads = []
    for native in (_native.host, None):
        monkeypatch.setattr(_native, "host", native)
        if form == "new forcing":
            fo = fo.copy(**{k: v.copy() for k, v in host.items()})
        if form == "new grid":
            phys._workspaces.clear()
        phys.parameters.__dict__["reads"] = 0
        phys.compute_tendencies(st, fo, ge, da)
        reads.append(phys.parameters.reads)
    assert reads[0] == reads[1]
