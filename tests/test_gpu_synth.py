"""GPU check of the own image synthesis (gathered sections -> cropped images)
against the hipFFT path: every radix, odd NX, one slab and several, full and
partial chunks.

Bar: the sections are identical, both transforms are fp32 and within a few
1e-7 relative (RMS) of the exact sum: 1e-6 rel-L2 per image set.
"""
import numpy as np
import pytest

from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nx", [4, 5, 8, 9, 16, 21, 35, 49, 64, 75, 96, 128, 150])
def test_images_match_hipfft(nx):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    rng = np.random.default_rng(nx)
    shape = (2 * nx, 2 * nx, nx + 1)
    X = torch.from_numpy((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)).cuda()
    ang = synth.uniform_angles(37, rng)   # a partial chunk
    out = []
    for hipfft in (False, True):
        with bp.Backprojector(nx, hipfft=hipfft, batch=16) as b:
            out.append(b.gather_images(X, ang).cpu().numpy().astype(np.float64))
    assert out[0].shape == (37, nx, nx) and np.isfinite(out[0]).all()
    assert np.linalg.norm(out[0] - out[1]) <= 1e-6 * np.linalg.norm(out[1])
