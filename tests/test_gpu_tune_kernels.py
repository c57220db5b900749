"""GPU check that the tuner times the unit-cell plan by its faster kernel.

1,024 sections of 270^2 into one half are past the unit cells' threshold for a
context of one half (540) and below it for one of two (1,080); the tuner's
sample lies in one half either way, so it is the same work, and the plan's
time has to be the same.  The nearest-voxel kernel takes ~1.2 times the unit
cells' here; 1.1 leaves half of that for the noise of a millisecond's timing.
"""
import numpy as np
import pytest

from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_both_kernels_of_the_cell_plan_are_timed():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    nx, m = 270, 1024
    rng = np.random.default_rng(270)
    imgs = torch.randn(m, nx, nx, generator=torch.Generator("cuda").manual_seed(1), device="cuda")
    ang = synth.uniform_angles(m, rng)
    best = []
    for two in (False, True):
        with bp.Backprojector(nx, two_halves=two) as b:
            best.append(b.tune(imgs, ang)["ms_per_proj"][7].min())
            print(f"two_halves={two}: {best[-1] * m:.3f} ms", flush=True)
    assert 0 < best[1] <= 1.1 * best[0]
