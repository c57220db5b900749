"""GPU checks of the unit-cell insertion kernel (plan 7 from 2 NX sections per
half up) against the oracle's terms summed in FP64: identical weight support,
raw sums equal up to the kernel's fp32 flush (rel-L2 <= 1e-6, the bar of every
other plan).  (The serial fp32 sums themselves are further off than that where
many equal terms meet, as the axis-aligned rotations here make them.)"""
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


def exact_sums(imgs, ang, nx, geom_f64):
    """(X, W) of the oracle's per-tap terms, summed in FP64."""
    X, W = oracle.empty_grid(nx, "f64")
    tab, fltb = oracle.kb_table(2 * nx, "f64" if geom_f64 else "f32")
    for img, a in zip(imgs, ang):
        if geom_f64:
            dm = oracle.cang(a[2], a[1], a[0], prec="f64", exact_pi=False)
            oracle.insert(X, W, oracle.spectrum(img, "f64"), dm, tab, fltb, "f64")
        else:
            dm = oracle.cang(a[2], a[1], a[0], prec="f32")
            oracle.insert_f32_acc64(X, W, oracle.spectrum(img, "f32"), dm, tab, fltb)
    return X, W


def angles(m, rng):
    """Uniform orientations; the first ones axis-aligned and diagonal (lattice
    lines along the grid, matrix entries of exactly 0)."""
    ang = synth.uniform_angles(m, rng)
    special = [(p, t, f) for p in (0, 45, 90, 180) for t in (0, 45, 90, 180) for f in (0, 90, 270)]
    k = min(len(special), m)
    ang[:k] = special[:k]
    return ang


# smallest boxes; edges and remainders of the 9-cell bricks; odd boxes; a pool
# that fills many times (thousands of sections through the few bricks of a
# small box); sections just at and just below the kernel's threshold
@pytest.mark.parametrize("nx,m,opts", [
    (4, 60, {}), (5, 40, {}), (9, 18, {}), (10, 19, {}), (13, 300, {"two_halves": True}), (16, 3000, {}),
    (18, 400, {"geom_f64": True}), (27, 200, {"twosum": True}), (32, 64, {}), (32, 63, {}),
    (40, 400, {"two_halves": True, "geom_f64": True}), (75, 150, {})])
def test_cells_match_oracle(nx, m, opts):
    from spider_amd import bp
    rng = np.random.default_rng(7 * nx + m)
    imgs = rng.standard_normal((m, nx, nx)).astype(np.float32)
    ang = angles(m, rng)
    half = (np.arange(m) % 2).astype(np.int8) if opts.get("two_halves") else np.zeros(m, np.int8)
    print(f"case cells nx={nx} m={m} {opts}", flush=True)
    with bp.Backprojector(nx, **opts) as b:
        b.insert(torch.from_numpy(imgs).cuda(), ang, half=half if opts.get("two_halves") else None)
        out = [[t.cpu().numpy() for t in b.export_raw(h)] for h in range(int(half.max()) + 1)]
    for h, (X, W) in enumerate(out):
        Xo, Wo = exact_sums(imgs[half == h], ang[half == h], nx, opts.get("geom_f64", False))
        np.testing.assert_array_equal(W > 0, Wo > 0)
        assert rel(X, Xo) <= 1e-6
        assert rel(W, Wo) <= 1e-6


@pytest.mark.parametrize("nx,m", [(16, 500), (33, 66)])
def test_cells_scatter_without_weights(nx, m):
    """The adjoint's weight-less kernel, with and without a weight grid."""
    from spider_amd import _lib, bp
    rng = np.random.default_rng(nx)
    N = 2 * nx
    dm = _lib.rotations(angles(m, rng))
    B = torch.from_numpy((rng.standard_normal((m, N, nx + 1)) + 1j * rng.standard_normal((m, N, nx + 1)))
                         .astype(np.complex64)).cuda()
    Xo, Wo = oracle.scatter(B.cpu().numpy().astype(np.complex128), dm, nx)
    with bp.Backprojector(nx) as b:
        W = torch.zeros(b.grid_shape, dtype=torch.float32, device="cuda")
        X, X2 = b.scatter(B, dm=dm, W=W).cpu().numpy(), b.scatter(B, dm=dm).cpu().numpy()
        W = W.cpu().numpy()
    assert rel(X, Xo) <= 1e-6
    assert rel(X2, Xo) <= 1e-6
    assert rel(W, Wo) <= 1e-6


def test_cells_batch_and_graph_replays():
    """Several boxes in one launch (the LDS table changes with the job), the
    batch replayed from a graph with eager work in between."""
    from spider_amd import bp
    rng = np.random.default_rng(3)
    sets = []
    for nx, m in ((16, 200), (24, 90), (9, 30)):
        sets.append((nx, torch.from_numpy(rng.standard_normal((m, nx, nx)).astype(np.float32)).cuda(), angles(m, rng)))
    ref = [exact_sums(imgs.cpu().numpy(), ang, nx, False) for nx, imgs, ang in sets]
    ctxs = [bp.Backprojector(nx) for nx, _, _ in sets]
    items = [(c, imgs, ang) for c, (_, imgs, ang) in zip(ctxs, sets)]

    def check():
        for c, (X, W) in zip(ctxs, ref):
            Xg, Wg = (t.cpu().numpy() for t in c.export_raw(0))
            np.testing.assert_array_equal(Wg > 0, W > 0)
            assert rel(Xg, X) <= 1e-6 and rel(Wg, W) <= 1e-6

    bp.insert_batch(items)
    check()
    g = bp.BatchGraph(items, reset_first=True)
    for _ in range(3):
        g.launch()
        torch.cuda.synchronize()
        check()
        ctxs[0].finalize()
    g.close()
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("nx,m", [(9, 6473), (16, 2048), (16, 2047), (33, 482), (75, 94)])
def test_gather_by_bricks_matches_oracle(nx, m):
    """The projector's gather through the unit-cell bricks (from NX sections
    and 2^19 pixels up; one case just below) against the oracle's, FP64 sums
    of the same taps: the bar of the sample-by-sample gather, 2e-7, and exact
    zeros where ONELINE has no sample."""
    from spider_amd import _lib, bp
    rng = np.random.default_rng(nx + m)
    N = 2 * nx
    dm = _lib.rotations(angles(m, rng)).reshape(m, 9)
    X = (rng.standard_normal((N, N, nx + 1)) + 1j * rng.standard_normal((N, N, nx + 1))).astype(np.complex64)
    print(f"case gather nx={nx} m={m}", flush=True)
    with bp.Backprojector(nx) as b:
        out = b.gather(torch.from_numpy(X).cuda(), dm=dm).cpu().numpy()
    pick = np.unique(np.r_[0:48, rng.integers(0, m, 40), m - 1])
    ref = oracle.gather(X, dm[pick])
    np.testing.assert_array_equal(out[pick][ref == 0], 0)
    for g, r in zip(out[pick], ref):
        assert rel(g, r) <= 2e-7


def test_gather_by_bricks_transposes_the_scatter_with_fp64_geometry():
    """<G x, b> = <x, S b> over 2,100 sections with FP64 geometry, both through
    the unit-cell bricks (bar as test_adjoint_identity's)."""
    from spider_amd import bp
    rng = np.random.default_rng(5)
    nx, m = 16, 2100
    N = 2 * nx
    ang = angles(m, rng)
    X = (rng.standard_normal((N, N, nx + 1)) + 1j * rng.standard_normal((N, N, nx + 1))).astype(np.complex64)
    B = (rng.standard_normal((m, N, nx + 1)) + 1j * rng.standard_normal((m, N, nx + 1))).astype(np.complex64)
    with bp.Backprojector(nx, geom_f64=True) as c:
        GX = c.gather(torch.from_numpy(X).cuda(), angles=ang).cpu().numpy().astype(np.complex128)
        SB = c.scatter(torch.from_numpy(B).cuda(), angles=ang).cpu().numpy().astype(np.complex128)
    lhs = np.sum(GX.real * B.real + GX.imag * B.imag)
    rhs = np.sum(X.real * SB.real + X.imag * SB.imag)
    assert abs(lhs - rhs) <= 1e-6 * np.sqrt(np.sum(np.abs(GX) ** 2) * np.sum(np.abs(B.astype(np.complex128)) ** 2))
