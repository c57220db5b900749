"""GPU checks that the projector's gather carries ONELINE's own fp32 weights
(TABI(X) * (TABI(Y) * TABI(Z)), each product rounded to fp32), whichever
kernel a call's size takes: by bricks of unit cells or sample by sample.

Both sum in FP64 and round once, so a value is within 2^-24 of itself of the
oracle's FP64 sum over the same weights, and the two kernels are within one
fp32 unit (2^-23) of each other; 2^-40 covers the FP64 sums (64 products of
at most ~5, in any order).  Unrounded weights differ from these by up to
2^-23 of a tap, which values smaller than their taps show.
"""
import numpy as np
import pytest

import oracle
from spider_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def grid(nx, rng):
    N = 2 * nx
    return (rng.standard_normal((N, N, nx + 1)) + 1j * rng.standard_normal((N, N, nx + 1))).astype(np.complex64)


def parts(a):
    return np.asarray(a, np.complex128).view(np.float64)


# 2^19 pixels and more go by bricks (from 2^20 for NX 32 to 45); cases just below
@pytest.mark.parametrize("nx,m", [(9, 6473), (16, 2048), (16, 2047), (33, 963), (33, 962), (75, 94)])
def test_gather_carries_oneline_weights(nx, m):
    from spider_amd import _lib, bp
    rng = np.random.default_rng(200 + nx)
    X = grid(nx, rng)
    dm = _lib.rotations(synth.uniform_angles(m, rng)).reshape(m, 9)
    print(f"case nx={nx} m={m}", flush=True)
    with bp.Backprojector(nx) as b:
        out = b.gather(torch.from_numpy(X).cuda(), dm=dm).cpu().numpy()
    pick = np.unique(np.r_[0:24, rng.integers(0, m, 24), m - 1])
    got, ref = parts(out[pick]), parts(oracle.gather(X.astype(np.complex128), dm[pick]))
    assert np.all(np.abs(got - ref) <= 2.0**-24 * np.abs(ref) + 2.0**-40)


@pytest.mark.parametrize("geom_f64", [False, True])
@pytest.mark.parametrize("nx,m", [(10, 5243), (16, 2100), (40, 700)])
def test_both_gathers_agree(nx, m, geom_f64):
    from spider_amd import bp
    rng = np.random.default_rng(300 + nx)
    X = torch.from_numpy(grid(nx, rng)).cuda()
    ang = synth.uniform_angles(m, rng)
    print(f"case nx={nx} m={m} geom_f64={geom_f64}", flush=True)
    with bp.Backprojector(nx, geom_f64=geom_f64) as b:
        bricks = parts(b.gather(X, angles=ang).cpu().numpy())
        samples = parts(np.concatenate([b.gather(X, angles=a).cpu().numpy() for a in np.array_split(ang, 3)]))
    assert np.all(np.abs(bricks - samples) <= 2.0**-23 * np.abs(samples) + 2.0**-40)
    assert np.any(samples != 0)


@pytest.mark.parametrize("nx,m,bricks", [(16, 2048, True), (16, 2047, False), (31, 546, True), (32, 1024, True),
                                         (32, 1023, False), (36, 405, False), (45, 518, True), (45, 517, False),
                                         (46, 248, True), (75, 74, False)])
def test_gather_route(nx, m, bricks):
    """Where the bricks' lists and regions are not repaid a call goes sample by
    sample: it builds no lists."""
    from spider_amd import _lib, bp
    rng = np.random.default_rng(400 + nx)
    X = torch.from_numpy(grid(nx, rng)).cuda()
    with bp.Backprojector(nx, timing=True) as b:
        b.gather(X, angles=synth.uniform_angles(m, rng))
        torch.cuda.synchronize()
        assert b.kernel_stats(_lib.K_BIN)[1] == (1 if bricks else 0)
        assert b.kernel_stats(_lib.K_GATHER)[1] == 1


@pytest.mark.parametrize("nx,m,batch,launches", [(16, 100, 16, 1), (16, 5000, 1024, 1), (16, 5000, 2048, 3), (16, 2100, 0, 1)])
def test_gather_chunks(nx, m, batch, launches):
    """A context's chunk size splits the gather where the chunks go by bricks;
    sample by sample all sections go at once."""
    from spider_amd import _lib, bp
    rng = np.random.default_rng(500 + batch)
    X = grid(nx, rng)
    dm = _lib.rotations(synth.uniform_angles(m, rng)).reshape(m, 9)
    with bp.Backprojector(nx, batch=batch, timing=True) as b:
        out = b.gather(torch.from_numpy(X).cuda(), dm=dm).cpu().numpy()
        assert b.kernel_stats(_lib.K_GATHER)[1] == launches
    pick = np.unique(np.r_[0:20, rng.integers(0, m, 20), m - 1])
    got, ref = parts(out[pick]), parts(oracle.gather(X.astype(np.complex128), dm[pick]))
    assert np.all(np.abs(got - ref) <= 2.0**-24 * np.abs(ref) + 2.0**-40)
