"""GPU check of the scatter's spectrum conversion, which also finds each
spectrum's largest value: spectra of very different magnitudes in one call (the
insertion's fixed-point units follow the maxima), sizes below, at and above one
block of 2,048 values and not a multiple of it.

Bar: scaling every spectrum by a power of two scales its units and sums
exactly, so the scatter of the scaled set equals the sum of scaled scatters
of each spectrum, up to the fp32 rounding of the global adds: 1e-6 rel-L2.
"""
import numpy as np
import pytest

from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nx", [5, 16, 31, 32, 33, 64])
def test_scatter_of_mixed_magnitudes(nx):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    rng = np.random.default_rng(nx)
    N, H = 2 * nx, nx + 1
    mag = [1.0, 2.0**40, 2.0**-40]
    B = (rng.standard_normal((3, N, H)) + 1j * rng.standard_normal((3, N, H))).astype(np.complex64)
    ang = synth.uniform_angles(3, rng)
    with bp.Backprojector(nx) as b:
        one = [b.scatter(torch.from_numpy(B[k:k + 1]).cuda(), ang[k:k + 1]).cpu().numpy().astype(np.complex128) for k in range(3)]
        for k in range(3):
            s = b.scatter(torch.from_numpy(B[k:k + 1] * np.float32(mag[k])).cuda(), ang[k:k + 1]).cpu().numpy()
            assert np.linalg.norm(s / mag[k] - one[k]) <= 1e-6 * np.linalg.norm(one[k])
        both = b.scatter(torch.from_numpy(B[:2] * np.array(mag[:2], np.float32)[:, None, None]).cuda(), ang[:2])
        want = one[0] * mag[0] + one[1] * mag[1]
        assert np.linalg.norm(both.cpu().numpy() - want) <= 1e-6 * np.linalg.norm(want)
