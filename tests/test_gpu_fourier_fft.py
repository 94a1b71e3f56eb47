"""The compiled Fourier stages (short FFTs in registers, one kernel pair per
nlon = n1 * n2) at the sizes where they can go wrong: the largest n_m each nlon
admits, single wavenumbers, latitude counts that leave ragged tiles, and the two
longest nlon, against the float64 oracle on the same grid.

Tolerance, relative in the 2-norm: every value passes about 2 log2(nlon)
roundings in the FFT steps and the twiddles and sums nlat products in the
Legendre stage, each rounding at most eps/2 = 6e-8 of its own operand, so the
error is below 6e-8 * (2 log2(nlon) + 2 sqrt(nlat)) with the sums' roundings
adding up at random."""
import numpy as np
import pytest

from oracle import sht_oracle as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(32, 32, 64, 34), (1, 2, 64, 2), (48, 50, 96, 50), (9, 33, 128, 36), (64, 65, 128, 66),
                                  (128, 128, 256, 130), (160, 160, 320, 162), (3, 180, 360, 180), (180, 180, 360, 182),
                                  (17, 19, 512, 20), (33, 40, 640, 42), (100, 101, 1024, 102), (20, 21, 1280, 22),
                                  (130, 131, 1280, 132)])
def test_compiled_fourier_stages_at_their_edges(dims):
    import torch
    from jcm_amd import transforms
    transforms.load()
    gg, og = transforms.SpectralGrid(*dims), so.Grid(*dims)
    tol = 6e-8 * (2 * np.log2(dims[2]) + 2 * np.sqrt(dims[3]))
    rng = np.random.default_rng(dims[2] + dims[0])

    def check(gpu, ref):
        gpu = gpu.cpu().numpy().astype(np.float64)
        assert np.linalg.norm(gpu - ref) <= tol * np.linalg.norm(ref)

    c = (rng.standard_normal((3,) + og.modal_shape) * og.mask).astype(np.float32)
    check(gg.to_nodal(torch.as_tensor(c, device="cuda")), og.to_nodal(c.astype(np.float64)))
    x = rng.standard_normal((2,) + og.nodal_shape).astype(np.float32)
    check(gg.to_modal(torch.as_tensor(x, device="cuda")), og.to_modal(x.astype(np.float64)))
