"""GPU check of the re-summed weights at the smallest sizes, where both squares
of samples around a target (its own and its mirror image's) reach most voxels
and are cut by every border: every voxel equals the FP32-faithful oracle's
serial sum bit for bit."""
import numpy as np
import pytest

import oracle
from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m", [1, 17, 120])
@pytest.mark.parametrize("nx", [4, 5, 9, 12])
def test_reference_weights_small(nx, m):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    rng = np.random.default_rng(100 * nx + m)
    imgs = rng.standard_normal((m, nx, nx)).astype(np.float32)
    ang = synth.uniform_angles(m, rng)
    ang[0] = 0.0   # axis-aligned: ties of the squares' borders
    with bp.Backprojector(nx) as b:
        b.insert(torch.from_numpy(imgs).cuda(), ang)
        w = b.reference_weights(np.arange((nx + 1) * (2 * nx) ** 2, dtype=np.int64))
    ref = oracle.bp(imgs, ang, prec="f32", want_xw=True)["W"]
    np.testing.assert_array_equal(w.astype(np.float32), np.asarray(ref, np.float32).ravel())
