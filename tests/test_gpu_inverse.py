"""GPU checks of the own inverse transform (normalisation, three cropped passes,
window) against the hipFFT path from the same imported grids: every radix, odd
NX (a last row pair of one row), one slab and several, one and many row pairs
per block, one and two halves, plain and compensated weights.

Bar: both paths are fp32 transforms of identical normalised values, each
within a few 1e-7 relative (RMS) of the exact sum, so 1e-6 rel-L2 apart; a
batch of contexts of several sizes gives bit-identical volumes to single
finalisations (the same blocks in another launch).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def bpmod():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    from spider_amd import bp
    return bp


def rel(a, b):
    a = np.asarray(a).astype(np.float64).ravel()
    b = np.asarray(b).astype(np.float64).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def partial(nx, seed):
    """A Hermitian-free half grid with weights on both sides of the threshold."""
    rng = np.random.default_rng(seed)
    shape = (2 * nx, 2 * nx, nx + 1)
    X = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    W = rng.uniform(0.0, 2.0, shape).astype(np.float32)
    return torch.from_numpy(X).cuda(), torch.from_numpy(W).cuda()


@pytest.mark.parametrize("twosum", [False, True])
@pytest.mark.parametrize("nx", [4, 5, 7, 8, 9, 15, 16, 21, 32, 35, 49, 64, 75, 96, 105, 128, 150])
def test_volumes_match_hipfft(bpmod, nx, twosum):
    parts = [partial(nx, 10 * nx + h) for h in (0, 1)]
    vols = []
    for hipfft in (False, True):
        with bpmod.Backprojector(nx, two_halves=True, twosum=twosum, plain_threshold=True, hipfft=hipfft) as b:
            for h, (X, W) in enumerate(parts):
                b.import_partial(X, W, half=h, accumulate=False)
            out = b.finalize(full=True, halves=True)
            vols.append({k: v.cpu().numpy() for k, v in out.items()})
    assert vols[0].keys() == vols[1].keys() and len(vols[0]) == 3
    for k in vols[0]:
        assert np.isfinite(vols[0][k]).all()
        assert rel(vols[0][k], vols[1][k]) <= 1e-6, k


def test_batch_of_sizes_matches_single(bpmod):
    """Contexts of several sizes, own and hipFFT transforms mixed (22 = 2 * 11),
    finalised in one call."""
    sizes = [16, 11, 25, 32, 13, 9]
    ctxs = [bpmod.Backprojector(nx, plain_threshold=True) for nx in sizes]
    try:
        for nx, c in zip(sizes, ctxs):
            c.import_partial(*partial(nx, nx), half=0, accumulate=False)
        single = [{k: v.cpu().numpy() for k, v in c.finalize().items()} for c in ctxs]
        batch = bpmod.finalize_batch([(c, True, False) for c in ctxs])
        for s, t in zip(single, batch):
            for k in s:
                np.testing.assert_array_equal(s[k], t[k].cpu().numpy())
    finally:
        for c in ctxs:
            c.close()
