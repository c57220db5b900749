"""GPU check of the unit-cell insertion's weight precision: every weight term
is rounded to units of 2^-50, as in the other insertion kernels, so a voxel's
weight is within 2^-51 per term (and the fp32 rounding of its one or two
flushes, 2^-24 each) of the exact sum of the fp32 terms.

Sections whose lightest voxels show it: of 4,000 random rotations the eight
with the smallest weight in any voxel, each inserted 2 NX times (the fewest
sections the kernel takes, all in the one brick of an NX = 5 box).
"""
import numpy as np
import pytest

import oracle
from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_light_voxels_keep_their_bits():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    nx, m = 5, 10
    ang = synth.uniform_angles(4000, np.random.default_rng(0))
    tab, fltb = oracle.kb_table(2 * nx, "f32")
    assert tab.max() <= 1.0   # the fixed-point range of a weight term
    flat = oracle.spectrum(np.zeros((nx, nx), np.float32), "f32")

    def weights(a, table):
        X, W = oracle.empty_grid(nx, "f64")
        oracle.insert_f32_acc64(X, W, flat, oracle.cang(a[2], a[1], a[0], prec="f32"), table, fltb)
        return W

    def least(W):
        return W[W > 0].min()

    small = [least(weights(a, tab)) for a in ang]
    imgs = torch.from_numpy(np.random.default_rng(1).standard_normal((m, nx, nx)).astype(np.float32)).cuda()
    for k in np.argsort(small)[:8]:
        ref = m * weights(ang[k], tab)
        terms = m * weights(ang[k], (tab > 0).astype(np.float32))   # every nonzero term counted as 1
        with bp.Backprojector(nx) as b:
            b.insert(imgs, np.repeat(ang[k][None], m, axis=0))
            W = b.export_raw(0)[1].cpu().numpy().astype(np.float64)
        err = np.abs(W - ref)
        print(f"rotation {k}: least weight {small[k]:.3e}", flush=True)
        np.testing.assert_array_equal(W > 0, ref > 0)
        assert np.all(err <= terms * 2.0**-51 + 2.0**-23 * ref)
