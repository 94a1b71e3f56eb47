"""One workspace for calls on several grids (speedy_abi.h allows it): what calls of other
grids and routes left in it is never taken for a word of this call."""
import ctypes

import numpy as np
import pytest

from jcm_amd import _native, synthetic
from jcm_amd.params import VJP_PARAMS
from jcm_amd.physics_interface import PhysicsTendency

pytestmark = pytest.mark.gpu
FIELDS = ("u_wind", "v_wind", "temperature", "specific_humidity")


class Calls:
    """The C entry points on a workspace of the caller's choice."""

    def __init__(self, phys):
        import torch
        self.phys, self.lib = phys, _native.load()
        self.torch = torch

    def workspace(self, *grids):
        n = max(self.lib.speedy_workspace_bytes(*g) for g in grids)
        ws = self.torch.empty(n, dtype=self.torch.uint8, device="cuda")
        _native.check(self.lib.speedy_workspace_init(ws.data_ptr(), n, self.phys._stream()), "init")
        return ws

    def __call__(self, ws, case, cot=None, level_set=-1):
        st, fo, ge, da = case
        keep = []
        p, v = self.phys._params(), ge.to_abi()
        if cot is None:
            f, out, (ix, il, nm), flags = self.phys.prepare_fwd(st, fo, ge, da, keep)
            rc = self.lib.speedy_fwd(ctypes.byref(f), ctypes.byref(v), ctypes.byref(p), ctypes.byref(da.to_abi()), ix, il,
                                     nm, flags, _native.TERMS_ALL, level_set, ws.data_ptr(), ws.numel(), self.phys._stream())
        else:
            f, adj, out, (ix, il, nm), flags = self.phys.prepare_vjp(st, fo, ge, da, cot, keep)
            rc = self.lib.speedy_fwd_vjp(ctypes.byref(f), ctypes.byref(adj), ctypes.byref(v), ctypes.byref(p),
                                         ctypes.byref(da.to_abi()), ix, il, nm, flags, level_set, ws.data_ptr(), ws.numel(),
                                         self.phys._stream())
        _native.check(rc, "call")
        sets = (ctypes.c_uint32 * nm)()
        _native.check(self.lib.speedy_read_level_sets(ws.data_ptr(), ws.numel(), nm, sets, self.phys._stream()), "sets")
        res = [getattr(out["tendency"], n).cpu().numpy() for n in FIELDS]
        if cot is not None:
            res += [getattr(out["state_grads"], n).cpu().numpy() for n in FIELDS]
            res += [out["param_grads"][f"{a}.{b}"].cpu().numpy() for a, b in VJP_PARAMS]
        return res, (list(sets) if level_set < 0 else None)


def _cot(case, seed):
    rng = np.random.default_rng(seed)
    return PhysicsTendency(*(rng.standard_normal(case[0].temperature.shape).astype(np.float32) for _ in range(4)))


def _same(a, b):
    assert a[1] == b[1]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("kx", [7, 8])
def test_words_of_other_grids_are_not_this_call_s(kx):
    """Level sets, chunk words, partials and argument blocks of batch-route calls in a
    workspace, then single launches whose tags equal each integer that lies there."""
    from jcm_amd.speedy_physics import SpeedyPhysics
    run = Calls(SpeedyPhysics())
    small = synthetic.make_case(128, 64, kx, seed=61, land=True)
    cot = _cot(small, 62)
    narrow = synthetic.make_case(8, 8, kx, seed=63, land=True, nmember=300, member_t_sigma=0.5)
    grids = [(128, 64, 1), (8, 8, 300)]
    fresh_f, fresh_v = run(run.workspace(*grids), small), run(run.workspace(*grids), small, cot)
    ws = run.workspace(*grids)
    words = ws.view(run.torch.int32)
    _, sets = run(ws, narrow)
    run(ws, narrow, _cot(narrow, 64))
    for tag in sorted(set(sets))[:6] + [1, kx, 64, 128, 8192]:   # level sets and sizes
        run(ws, narrow)
        words[0] = tag - 1                                       # the generation before a call of this tag
        _same(run(ws, small, cot), fresh_v)
        assert int(words[0]) == tag                              # it was a single launch
        words[0] = tag - 1
        _same(run(ws, small), fresh_f)
        assert int(words[1]) == 0


@pytest.mark.parametrize("kx", [7, 8, 16])
def test_words_of_32768_calls_before_are_not_this_call_s(kx):
    """A smaller grid's calls leave the words of a larger one's later blocks as they were,
    for any number of calls; the generation they reach is set here."""
    from jcm_amd.speedy_physics import SpeedyPhysics
    run = Calls(SpeedyPhysics())
    a = synthetic.make_case(256, 128, kx, seed=65, land=True)
    b = synthetic.make_case(256, 128, kx, seed=66, land=True)
    grid = (256, 128, 1)
    fresh = run(run.workspace(grid), b)
    for ahead in (1, 32767, 32768, 65535, 65536, (1 << 31) - 2):
        ws = run.workspace(grid)
        words = ws.view(run.torch.int32)
        run(ws, a)
        words[0] = ahead
        _same(run(ws, b), fresh)
        assert int(words[0]) == ahead + 1
    words[0] = -2                        # the last generation; the next is the first again
    _same(run(ws, b), fresh)
    assert int(words[0]) == 0
    _same(run(ws, b), fresh)


@pytest.mark.parametrize("nlon,nlat,nmember", [(64, 33, 3), (16, 16, 5), (97, 7, 4), (640, 320, 1), (96, 48, 40)])
def test_budgets_of_blocks_on_two_members(nlon, nlat, nmember):
    """Each member's budgets equal those of the member alone: the float64 sums of float32
    tendencies that another kernel's contractions change by 1e-6 of their largest, and
    ten times that of the largest budget (2e-5 with both sides' share)."""
    from jcm_amd.speedy_physics import SpeedyPhysics
    phys = SpeedyPhysics()
    st, fo, ge, da = synthetic.make_case(nlon, nlat, 8, seed=67, land=True, nmember=nmember, member_t_sigma=0.5)
    phys.compute_tendencies(st, fo, ge, da, budgets=True)
    got = phys.last_budgets.cpu().numpy()
    S = phys.level_sets(nlon, nlat, nmember)
    again = []
    for _ in range(2):
        phys.compute_tendencies(st, fo, ge, da, budgets=True)
        again.append(phys.last_budgets.cpu().numpy())
    assert np.array_equal(again[0], got) and np.array_equal(again[1], got)
    names = FIELDS + ("geopotential", "normalized_surface_pressure")
    for m in range(nmember if nmember < 6 else 3):
        one = st if nmember == 1 else st.copy(**{k: np.ascontiguousarray(getattr(st, k)[m]) for k in names})
        phys.compute_tendencies(one, fo, ge, da, budgets=True, level_set=S[m])
        alone = phys.last_budgets.cpu().numpy()[0]
        # the tendencies of the two routes differ in their last float32 bits
        assert np.all(np.abs(got[m] - alone) <= 2e-5 * np.abs(alone) + 2e-5 * np.abs(got[m]).max())


@pytest.mark.parametrize("kx", [7, 8])
def test_counts_out_of_step_are_reported(kx):
    """Calls that overlap on one workspace can leave the count of arrived blocks where no
    block is the last; such a call ends, and the workspace's status says that its
    results are invalid.  The count is set from the host here."""
    import torch
    from jcm_amd.speedy_physics import SpeedyPhysics
    run = Calls(SpeedyPhysics())
    case = synthetic.make_case(128, 64, kx, seed=68, land=True)
    cot = _cot(case, 69)
    ws = run.workspace((128, 64, 1))
    words = ws.view(torch.int32)
    fresh = run(ws, case, cot)
    status = lambda: (_native.check(run.lib.speedy_workspace_status(  # noqa: E731
        ws.data_ptr(), ws.numel(), ctypes.byref(st), run.phys._stream()), "status"), int(st.value))[1]
    st = ctypes.c_uint32(0)
    assert status() == 0 and int(words[2]) == 0
    words[2] = 32                        # as many as the grid has blocks
    run(ws, case, cot)
    assert status() == 1
    _same(run(ws, case, cot), fresh)     # the query reset the workspace
    assert status() == 0
