"""GPU checks of batches whose jobs lie on both sides of the insertion
kernels' section threshold (2 NX per half): each kind in a launch of its own
where the round repays it, else one kernel for all.  Sums against the oracle's
terms summed in FP64 (bars as in test_gpu_cells.py), eager and replayed from a
graph with eager work in between; the launches counted by the contexts that
lead them.
"""
import numpy as np
import pytest

import oracle
from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def rel(a, b):
    a = np.asarray(a).astype(np.complex128).ravel()
    b = np.asarray(b).astype(np.complex128).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def exact_sums(imgs, ang, nx):
    X, W = oracle.empty_grid(nx, "f64")
    tab, fltb = oracle.kb_table(2 * nx, "f32")
    for img, a in zip(imgs, ang):
        oracle.insert_f32_acc64(X, W, oracle.spectrum(img, "f32"), oracle.cang(a[2], a[1], a[0], prec="f32"), tab, fltb)
    return X, W


# (box, sections) per job, and the jobs that lead a launch
@pytest.mark.parametrize("spec,leads", [
    # 1.5 M pixels of few-section jobs, 4.2 M pixels past the threshold: two launches
    ([(64, 127), (64, 1152), (64, 127), (64, 127)], [0, 1]),
    # the few-section job rides with the cells
    ([(16, 20), (48, 700)], [0]),
    # hardly past the threshold: the nearest-voxel bricks for all
    ([(24, 100), (16, 10)], [0]),
    ([(33, 64), (33, 64), (64, 120), (64, 120), (33, 66)], [0])])
def test_mixed_batch(spec, leads):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import _lib, bp
    rng = np.random.default_rng(len(spec))
    data = [(rng.standard_normal((m, nx, nx)).astype(np.float32), synth.uniform_angles(m, rng)) for nx, m in spec]
    ref = [exact_sums(imgs, ang, nx) for (nx, _), (imgs, ang) in zip(spec, data)]
    ctxs = [bp.Backprojector(nx, timing=True) for nx, _ in spec]
    items = [(c, torch.from_numpy(imgs).cuda(), ang) for c, (imgs, ang) in zip(ctxs, data)]
    print(f"case {spec}", flush=True)

    def check():
        for c, (X, W) in zip(ctxs, ref):
            Xg, Wg = (t.cpu().numpy() for t in c.export_raw(0))
            np.testing.assert_array_equal(Wg > 0, W > 0)
            assert rel(Xg, X) <= 1e-6 and rel(Wg, W) <= 1e-6

    bp.insert_batch(items)
    check()
    assert [c.kernel_stats(_lib.K_INSERT)[1] for c in ctxs] == [int(j in leads) for j in range(len(spec))]
    g = bp.BatchGraph(items, reset_first=True)
    for _ in range(3):
        g.launch()
        torch.cuda.synchronize()
        check()
        ctxs[0].finalize()
    g.close()
    for c in ctxs:
        c.close()
