"""The native call preparation (csrc/host_calls.cpp) against the general Python path:
the same outputs bit for bit for the calls it takes, and the general path for every
other form (which it must not take, and which gives the same values)."""
import numpy as np
import pytest

from jcm_amd import synthetic
from jcm_amd.physics_interface import PhysicsTendency

pytestmark = pytest.mark.gpu

STATE = ("u_wind", "v_wind", "temperature", "specific_humidity", "geopotential", "normalized_surface_pressure")
FORCING = ("alb0", "sice_am", "snowc_am", "soilw_am", "stl_am", "sea_surface_temperature")
TEND = STATE[:4]


def _case(kx=8, nmember=1, nlon=24, nlat=14):
    import torch
    st, fo, ge, da = synthetic.make_case(nlon, nlat, kx, seed=4, land=True, nmember=nmember, member_t_sigma=0.5)
    up = lambda o, names: o.copy(**{k: torch.as_tensor(getattr(o, k), device="cuda") for k in names})  # noqa: E731
    g = torch.Generator(device="cuda").manual_seed(3)
    cot = PhysicsTendency(*[torch.randn(st.temperature.shape, generator=g, device="cuda") for _ in range(4)])
    return up(st, STATE), up(fo, FORCING), ge, da, cot


def _calls(phys, case, verify):
    st, fo, ge, da, cot = case
    t, data = phys.compute_tendencies(st, fo, ge, da, verify=verify)
    out = [getattr(t, n) for n in TEND] + ([data._diag] if data is not None else [])
    if data is not None:
        assert data.date is da and len(data._names) == data._diag.shape[-2]
    tv, sg, pg = phys.compute_tendencies_vjp(st, fo, ge, da, cot, verify=verify)
    assert sg.geopotential is None
    return out + [getattr(tv, n) for n in TEND] + [getattr(sg, n) for n in TEND] + [
        sg.normalized_surface_pressure] + [pg[k] for k in sorted(pg)]


def _compare(case, monkeypatch, diagnostics=False, verify=False, params=None, taken=True):
    import torch
    from jcm_amd import _native
    from jcm_amd.speedy_physics import SpeedyPhysics
    assert _native.host is not None, "the native call preparation is not built"
    phys = SpeedyPhysics(parameters=params, with_diagnostics=diagnostics)
    _calls(phys, case, verify)          # workspaces and device copies of NumPy fields
    st, fo, ge, da, cot = case
    r = _native.host.fwd(phys._consts, phys._workspaces, phys.parameters, *phys._where(), st, fo, ge, da, 0,
                         _native.TERMS_ALL, -1, diagnostics)
    assert isinstance(r, tuple) == taken
    fast = _calls(phys, case, verify)
    monkeypatch.setattr(_native, "host", None)
    general = _calls(phys, case, verify)
    torch.cuda.synchronize()
    assert len(fast) == len(general)
    for a, b in zip(fast, general):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("kx,nmember,diagnostics,verify", [(8, 1, False, False), (7, 3, True, True), (16, 1, True, False),
                                                           (8, 5, False, True)])
def test_native_calls_equal_the_general_path(kx, nmember, diagnostics, verify, monkeypatch):
    _compare(_case(kx, nmember), monkeypatch, diagnostics, verify)


def test_native_calls_read_every_parameter_and_date(monkeypatch):
    """Values away from the defaults, changed in place after a first call: nothing of an
    earlier call is reused."""
    p = synthetic.draw_vjp_parameters(5)
    case = _case()
    _compare(case, monkeypatch, params=p)
    monkeypatch.undo()
    rng = np.random.default_rng(0)
    for grp in vars(p).values():
        for k, v in vars(grp).items():
            if isinstance(v, float) and k not in ("co2_scale",):
                setattr(grp, k, v * float(rng.uniform(0.97, 1.03)))
    p.surface_flux.fhum0, p.surface_flux.lscasym, p.forcing.increase_co2 = 0.3, False, True
    case = case[:3] + (case[3].copy(tyear=0.71, model_year=2003, model_step=4, dt_seconds=900.0),) + case[4:]
    _compare(case, monkeypatch, params=p, verify=True)


@pytest.mark.parametrize("form", ["numpy state", "strided", "float64", "wide strides", "numpy forcing", "climatology",
                                  "no land fluxes", "int year"])
def test_forms_of_the_inputs(form, monkeypatch):
    import torch
    st, fo, ge, da, cot = _case()
    taken = False
    if form == "numpy state":
        st = st.copy(temperature=st.temperature.cpu().numpy())
    elif form == "strided":
        st = st.copy(u_wind=st.u_wind.transpose(-1, -2).contiguous().transpose(-1, -2))
    elif form == "float64":
        st = st.copy(specific_humidity=st.specific_humidity.double())
    elif form == "wide strides":
        wide = torch.zeros(st.geopotential.shape[:-1] + (20,), device="cuda")
        wide[..., :14] = st.geopotential
        st = st.copy(geopotential=wide[..., :14])
    elif form == "numpy forcing":
        fo, taken = fo.copy(**{k: getattr(fo, k).cpu().numpy() for k in FORCING}), True
    elif form == "climatology":
        fo = fo.copy(stl_am=torch.stack([fo.stl_am + i for i in range(4)], -1))
    elif form == "no land fluxes":
        fo, taken = fo.copy(lfluxland=False), True
    elif form == "int year":
        da, taken = da.copy(tyear=0, model_year=np.int64(1950)), False
    _compare((st, fo, ge, da, cot), monkeypatch, taken=taken)


def test_what_was_refused_stays_refused(monkeypatch):
    import torch
    from jcm_amd import _native
    from jcm_amd.speedy_physics import SpeedyPhysics
    st, fo, ge, da, cot = _case()
    bad = [st.copy(temperature=st.temperature[:, :-1].contiguous()), st.copy(v_wind=st.v_wind[:-1].contiguous()),
           st.copy(normalized_surface_pressure=st.normalized_surface_pressure[:-1].contiguous())]
    for native in (True, False):
        if not native:
            monkeypatch.setattr(_native, "host", None)
        phys = SpeedyPhysics()
        phys.compute_tendencies(st, fo, ge, da)
        for b in bad:
            with pytest.raises(ValueError):
                phys.compute_tendencies(b, fo, ge, da)
        with pytest.raises(ValueError):
            phys.compute_tendencies_vjp(st, fo, ge, da, cot.copy(u_wind=cot.u_wind[:-1].contiguous()))
        with pytest.raises(_native.SpeedyError):
            phys.compute_tendencies(st, fo, ge, da, term_mask=1 << 20)
    torch.cuda.synchronize()


@pytest.mark.parametrize("kx,nsp", [(8, None), (3, 1), (5, 5)])
def test_native_conversions_equal_the_general_path(kx, nsp, monkeypatch):
    import torch
    from jcm_amd import transforms as T
    from jcm_amd.physics_interface import PhysicsState
    grid = T.SpectralGrid.truncation(21)
    g = torch.Generator(device="cuda").manual_seed(1)
    modal = lambda *lead: torch.randn(*lead, *grid.modal_shape, generator=g, device="cuda") * 1e-3  # noqa: E731
    dyn = T.PrimitiveEquations(torch.linspace(230, 280, kx, device="cuda"), modal(),
                               T.CoordinateSystem(grid, T.SigmaCoordinates(np.linspace(0, 1, kx + 1))))
    st = T.DynamicsState(modal(kx), modal(kx), modal(kx), modal() if nsp is None else modal(nsp),
                         {"specific_humidity": modal(kx)})

    def calls(state):
        y = T.dynamics_state_to_physics_state(state, dyn)
        p = PhysicsState(y.u_wind, y.v_wind, y.temperature, y.specific_humidity, None, y.normalized_surface_pressure)
        x = T.physics_state_to_dynamics_state(p, dyn)
        z = T.physics_tendency_to_dynamics_tendency(PhysicsTendency(*(getattr(p, n) for n in TEND)), dyn)
        assert z.sim_time == 0.0 and x.sim_time is None
        return [getattr(y, n) for n in STATE] + [v for d in (x, z) for v in (
            d.vorticity, d.divergence, d.temperature_variation, d.log_surface_pressure, d.tracers["specific_humidity"])]

    calls(st)
    assert T._native_call("dynamics_to_physics", st.vorticity, dyn, st) is not None
    strided = T.DynamicsState(st.vorticity, st.divergence.transpose(1, 2).contiguous().transpose(1, 2),
                              st.temperature_variation.double(), st.log_surface_pressure.cpu().numpy(), st.tracers)
    assert T._native_call("dynamics_to_physics", strided.vorticity, dyn, strided) is None
    fast, other = calls(st), calls(strided)
    monkeypatch.setattr(T, "host", None)
    general = calls(st)
    torch.cuda.synchronize()
    for a, b, c in zip(fast, general, other):
        assert a.shape == b.shape and torch.equal(a, b) and torch.equal(a, c)
    with pytest.raises(ValueError):
        T.dynamics_state_to_physics_state(T.DynamicsState(st.vorticity[:-1], st.divergence, st.temperature_variation,
                                                          st.log_surface_pressure, st.tracers), dyn)
