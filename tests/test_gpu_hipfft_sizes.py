"""GPU checks of the paths hipFFT still serves: padded sizes with a prime
factor above 7 (NX = 11, 13, 22: N = 22, 26, 44).  Insertion of full and
partial chunks and finalisation against the oracle, failed allocations, and
what a live batch graph refuses and replays, whose captured transforms are
hipFFT's there.

Bars as elsewhere for these paths: accumulators rel-L2 1e-6, volumes 1e-5 of
the FP32-faithful oracle.
"""
import numpy as np
import pytest

import oracle
from spider_amd import synth
from test_gpu_failure import bpmod  # noqa: F401
from test_gpu_failure import test_failed_allocation_leaves_context_usable as failed_allocations
from test_gpu_mixed_batch import exact_sums, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dataset(nx, m, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((m, nx, nx)).astype(np.float32), synth.uniform_angles(m, rng)


def export(b):
    X, W = b.export_raw(0)
    return X.cpu().numpy(), W.cpu().numpy()


@pytest.mark.parametrize("nx", [11, 13, 22])
def test_insert_and_finalize(bpmod, nx):  # noqa: F811
    imgs, ang = dataset(nx, 41, nx)
    with bpmod.Backprojector(nx, batch=16) as b:   # chunks of 16, 16 and 9
        b.insert(torch.from_numpy(imgs).cuda(), ang)
        X, W = export(b)
        vol = b.finalize()["full"].cpu().numpy()
    Xo, Wo = exact_sums(imgs, ang, nx)
    np.testing.assert_array_equal(W > 0, Wo > 0)
    assert rel(X, Xo) <= 1e-6 and rel(W, Wo) <= 1e-6
    ref = oracle.bp(imgs, ang, prec="f32")["full"]
    assert np.linalg.norm(vol - ref) <= 1e-5 * np.linalg.norm(ref)


def test_failed_allocations(bpmod):  # noqa: F811
    failed_allocations(bpmod, 22)


def test_live_graph_refuses_a_new_plan_and_replays(bpmod):  # noqa: F811
    from spider_amd import _lib
    imgs, ang = dataset(22, 100, 91)
    t = torch.from_numpy(imgs).cuda()
    Xo, Wo = exact_sums(imgs, ang, 22)
    with bpmod.Backprojector(22, batch=64) as c:   # a chunk of 64 and a partial one of 36
        g = bpmod.BatchGraph([(c, t, ang)], reset_first=True)
        try:
            for r in range(3):
                g.launch()
                torch.cuda.synchronize()
                X, W = export(c)
                np.testing.assert_array_equal(W > 0, Wo > 0)
                assert rel(X, Xo) <= 1e-6 and rel(W, Wo) <= 1e-6
                with pytest.raises(bpmod.SpbpError) as e:
                    c.insert(t[:50], ang[:50])     # its transforms would replace the captured plan of 36
                assert e.value.code == _lib.ERR_ARG and "captured batch graph" in str(e.value)
                c.insert(t[:64], ang[:64])         # the graph's own sizes run
                c.insert(t[:36], ang[:36])
                torch.cuda.synchronize()
        finally:
            g.close()
        c.reset()
        c.insert(t[:50], ang[:50])
        X, W = export(c)
    Xo, Wo = exact_sums(imgs[:50], ang[:50], 22)
    assert rel(X, Xo) <= 1e-6 and rel(W, Wo) <= 1e-6
