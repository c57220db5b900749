"""GPU checks of the own forward transforms for padded sizes 2^a 3^b 5^c 7^d
that are no power of two: every radix alone and mixed, odd NX (a last row
without a partner), one to many rows and columns per block, and the first
size of each kind.

Bars: as for the powers of two -- weights with the same support and within
1e-6 relative per voxel (independent of the spectra; fp32 sums in another
order), X within rel-L2 1e-6 of the hipFFT path, and within 4e-7 of FP64 sums
of the oracle's FP64 spectra rounded once.
"""
import numpy as np
import pytest

import oracle
from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def bpmod():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    return bp


def rel(a, b):
    a = np.asarray(a).astype(np.complex128).ravel()
    b = np.asarray(b).astype(np.complex128).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("nx", [5, 6, 7, 9, 10, 14, 15, 21, 35, 48, 49, 54, 75, 81, 96, 105, 125, 147, 192, 300])
def test_own_transforms_match_hipfft(bpmod, nx, bf16):
    rng = np.random.default_rng(1000 + nx)
    m = 21   # a partial chunk
    imgs = torch.from_numpy(rng.standard_normal((m, nx, nx)).astype(np.float32)).cuda()
    if bf16:
        imgs = imgs.to(torch.bfloat16)
    ang = synth.uniform_angles(m, rng)
    out = []
    for hipfft in (False, True):
        with bpmod.Backprojector(nx, hipfft=hipfft, batch=16) as b:
            b.insert(imgs, ang)
            X, W = b.export_raw(0)
            out.append((X.cpu().numpy(), W.cpu().numpy()))
    W0, W1 = out[0][1], out[1][1]
    np.testing.assert_array_equal(W0 != 0, W1 != 0)
    nz = W1 != 0
    assert np.max(np.abs(W0[nz] - W1[nz]) / W1[nz]) <= 1e-6
    assert rel(out[0][0], out[1][0]) <= 1e-6


@pytest.mark.parametrize("nx", [7, 15, 49, 75, 96])
def test_own_spectrum_vs_fp64(bpmod, nx):
    rng = np.random.default_rng(nx)
    m = 6
    imgs = rng.standard_normal((m, nx, nx)).astype(np.float32)
    ang = synth.uniform_angles(m, rng)
    tab, fltb = oracle.kb_table(2 * nx, "f32")
    X64, W64 = oracle.empty_grid(nx, "f64")
    for p in range(m):
        dm = oracle.cang(ang[p][2], ang[p][1], ang[p][0], prec="f32")
        oracle.insert_f32_acc64(X64, W64, oracle.spectrum(imgs[p], "f64").astype(np.complex64), dm, tab, fltb)
    with bpmod.Backprojector(nx) as b:
        b.insert(torch.from_numpy(imgs).cuda(), ang)
        X, _ = b.export_raw(0)
    assert rel(X.cpu().numpy(), X64) <= 4e-7
