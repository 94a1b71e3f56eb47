"""The Legendre stages with the modal operators inside (chunks of eight fields of
one order; operand blocks of 16 l x 16 latitudes) at the sizes where they can go
wrong: counts that leave ragged blocks, one latitude pair, one field and nine,
level counts that leave part of a chunk, more blocks than are staged at a time
and modal rows that do not fit in LDS, against the float64 oracle.

Tolerance as in test_gpu_fourier_fft.py for the transforms, relative in the
2-norm: 6e-8 * (2 log2(nlon) + 2 sqrt(nlat)).  The conversions weigh
neighbouring l with factors of order l and subtract them, at worst another
factor of 4 on random fields, and scale or exponentiate once more."""
import numpy as np
import pytest

from oracle import sht_oracle as so

pytestmark = pytest.mark.gpu


def _tol(dims):
    return 6e-8 * (2 * np.log2(max(dims[2], 2)) + 2 * np.sqrt(dims[3]))


def _check(gpu, ref, tol):
    gpu = gpu.cpu().numpy().astype(np.float64)
    ref = np.asarray(ref, np.float64).reshape(gpu.shape)
    assert np.linalg.norm(gpu - ref) <= tol * np.linalg.norm(ref)


@pytest.mark.parametrize("dims,nfield", [((1, 2, 1, 2), 1), ((3, 17, 8, 18), 9), ((16, 33, 64, 34), 8), ((33, 33, 66, 48), 7),
                                         ((8, 65, 15, 130), 17), ((2, 1001, 4, 1002), 3), ((2, 640, 3, 980), 2)])
def test_transforms_at_the_edges_of_the_blocks(dims, nfield):
    import torch
    from jcm_amd import transforms
    transforms.load()
    gg, og = transforms.SpectralGrid(*dims), so.Grid(*dims)
    rng = np.random.default_rng(sum(dims))
    c = (rng.standard_normal((nfield,) + og.modal_shape) * og.mask).astype(np.float32)
    _check(gg.to_nodal(torch.as_tensor(c, device="cuda")), og.to_nodal(c.astype(np.float64)), _tol(dims))
    x = rng.standard_normal((nfield,) + og.nodal_shape).astype(np.float32)
    modal = gg.to_modal(torch.as_tensor(x, device="cuda"))
    _check(modal, og.to_modal(x.astype(np.float64)), _tol(dims))
    assert not modal.cpu().numpy()[:, ~og.mask].any()


@pytest.mark.parametrize("dims,kx,nsp", [((5, 6, 64, 18), 1, 1), ((16, 18, 64, 34), 5, 2), ((17, 40, 96, 40), 9, 9),
                                         ((3, 18, 8, 18), 16, 1), ((2, 1001, 4, 1002), 5, 1)])
def test_conversions_at_the_edges_of_the_chunks(dims, kx, nsp):
    import torch
    from jcm_amd import transforms as tr
    from jcm_amd.physics_interface import PhysicsState, PhysicsTendency
    tr.load()
    gg, og = tr.SpectralGrid(*dims), so.Grid(*dims)
    rng = np.random.default_rng(kx + sum(dims))
    sigma, reft = np.linspace(0.0, 1.0, kx + 1), np.linspace(220.0, 288.0, kx).astype(np.float32)
    modal = lambda n, scale: (rng.standard_normal((n,) + og.modal_shape) * og.mask * scale).astype(np.float32)
    nodal = lambda n, scale, mean=0.0: (mean + scale * rng.standard_normal((n,) + og.nodal_shape)).astype(np.float32)
    up, wide = lambda a: torch.as_tensor(a, device="cuda"), lambda a: a.astype(np.float64)
    orog = modal(1, 300.0)[0]
    dyn = tr.PrimitiveEquations(reference_temperature=reft, orography=orog,
                                coords=tr.CoordinateSystem(gg, tr.SigmaCoordinates(sigma)))
    ref = so.Dynamics(grid=og, sigma_boundaries=sigma, reference_temperature=wide(reft), orography=wide(orog))
    tol = 4 * _tol(dims)

    s = [modal(kx, 1e-5), modal(kx, 1e-6), modal(kx, 1.0), modal(nsp, 0.002), modal(kx, 1e-3)]
    out = tr.dynamics_state_to_physics_state(tr.DynamicsState(*map(up, s[:4]), {"specific_humidity": up(s[4])}), dyn)
    exp = so.dynamics_state_to_physics_state(so.DynamicsState(*map(wide, s[:4]), {"specific_humidity": wide(s[4])}), ref)
    for name, r in zip(("u_wind", "v_wind", "temperature", "specific_humidity", "geopotential",
                        "normalized_surface_pressure"), exp):
        _check(getattr(out, name), r, tol)

    n = [nodal(kx, 10.0), nodal(kx, 10.0), nodal(kx, 20.0, 250.0), nodal(kx, 1.0, 5.0), nodal(nsp, 0.05, 1.0)]
    n[4] = n[4] if nsp > 1 else n[4][0]
    names = ("vorticity", "divergence", "temperature_variation", "log_surface_pressure")
    out = tr.physics_state_to_dynamics_state(PhysicsState(*map(up, n[:4]), up(np.zeros_like(n[0])), up(n[4])), dyn)
    exp = so.physics_state_to_dynamics_state(*map(wide, n), ref)
    for name in names:
        _check(getattr(out, name), getattr(exp, name), tol)
    _check(out.tracers["specific_humidity"], exp.tracers["specific_humidity"], tol)

    out = tr.physics_tendency_to_dynamics_tendency(PhysicsTendency(*map(up, n[:4])), dyn)
    exp = so.physics_tendency_to_dynamics_tendency(*map(wide, n[:4]), ref)
    for name in names[:3]:
        _check(getattr(out, name), getattr(exp, name), tol)
    assert not out.log_surface_pressure.any()


def test_a_field_that_is_not_finite_stays_its_own():
    """Infinities and NaN in one field leave the others finite, and reach every mode of theirs."""
    import torch
    from jcm_amd import transforms
    gg = transforms.SpectralGrid.truncation(21)
    x = torch.randn((9,) + so.Grid.truncation(21).nodal_shape, device="cuda")
    x[3, 5, 7], x[8, 0, 0] = float("inf"), float("nan")
    finite = torch.isfinite(gg.to_modal(x)).flatten(1)
    assert not finite[[3, 8]].any()
    assert finite[[0, 1, 2, 4, 5, 6, 7]].all()
