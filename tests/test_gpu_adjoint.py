"""GPU check of the image adjoint's spectra (scaled, column 0 folded and their
maxima found by the columns pass): scatter_images against the scatter of the
same spectra computed in FP64 and rounded once, for one slab of columns and
several, full and partial chunks.

Bar: fp32 transforms are within a few 1e-7 relative (RMS) of the rounded FP64
spectra, the insertion is the same: 1e-6 rel-L2.
"""
import numpy as np
import pytest

from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nx", [4, 8, 64, 128, 256])
def test_scatter_images_vs_fp64_spectra(nx):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    rng = np.random.default_rng(nx)
    N, m, ip = 2 * nx, 11, nx // 2
    r = rng.standard_normal((m, nx, nx)).astype(np.float32)
    ang = synth.uniform_angles(m, rng)
    g = np.zeros((m, N, N))
    g[:, ip:ip + nx, ip:ip + nx] = r
    R = np.fft.rfft2(g) / N**2
    R[:, :, 1:nx] *= 2.0
    R[:, 1:nx, 0] += np.conj(R[:, :nx:-1, 0])
    R[:, nx + 1:, 0] = 0.0
    sign = 1.0 - 2.0 * (np.add.outer(np.arange(N), np.arange(nx + 1)) % 2)
    bi = torch.from_numpy((sign * np.conj(R)).astype(np.complex64)).cuda()
    with bp.Backprojector(nx, batch=8) as b:
        X1 = b.scatter_images(torch.from_numpy(r).cuda(), ang).cpu().numpy().astype(np.complex128)
        X2 = b.scatter(bi, ang)
        X2 = (X2[0] if isinstance(X2, tuple) else X2).cpu().numpy().astype(np.complex128)
    assert np.linalg.norm(X1 - X2) <= 1e-6 * np.linalg.norm(X2)
