"""Brute force at the edges of its tiles and of the matrix filter: triangle
and ray counts around 32 and 128, scenes far from the origin, very small and
very large ones, degenerate, flat and non-finite triangles, rays with zero,
huge or non-finite components.  Bar: bit-exact records against the oracle's
sequential loop, which has no filter."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


def check(pm, orc, torch, tris, org, dirs, label, test=None, cap=0):
    tests = (pm.MOELLER, pm.WOOP) if test is None else (test,)
    ctx = pm.Context(0)
    P = [dev(torch, t) for t in tris]
    ctx.set_geometry(*P)
    for k in tests:
        want = orc.trace(None, tris, org, dirs, orc.BRUTE, brute_cap=cap, intersection=k, threads=8)
        cnt = torch.zeros((org.shape[0], 4), dtype=torch.int32, device="cuda:0")
        tp = pm.trace_params(intersection=k, brute_cap=cap)
        h = pm.hits_to_numpy(ctx.trace(pm.BRUTE, dev(torch, org), dev(torch, dirs), tp))
        assert_same_hits(h, want, f"{label} test {k}")
        h = pm.hits_to_numpy(ctx.trace(pm.BRUTE, dev(torch, org), dev(torch, dirs), tp, counters=cnt))
        assert_same_hits(h, want, f"{label} test {k}, counted")
        n = tris[0].shape[0]
        assert (cnt.cpu().numpy() == [0, 0, min(n, cap) if cap else n, 0]).all()
    ctx.close()
    return want


@pytest.mark.parametrize("ntris", [1, 31, 32, 33, 511, 512, 513, 2000])
@pytest.mark.parametrize("nrays", [1, 33, 129, 16385, 32769])
def test_counts_bit_exact(pm, orc, scenes, torch, ntris, nrays):
    tris = scenes.random_soup(ntris, seed=ntris, size=0.4)
    org, dirs = scenes.random_rays(nrays, seed=nrays)
    want = check(pm, orc, torch, tris, org, dirs, f"{ntris} x {nrays}")
    if ntris >= 32 and nrays > 1000:
        assert (want["id"] >= 0).mean() > 0.05
    check(pm, orc, torch, tris, org, dirs, "cap", cap=40)


@pytest.mark.parametrize("shift", [0.0, 1e3, 1e6])
@pytest.mark.parametrize("scale", [1e-18, 1e-6, 1.0, 1e6, 1e15])
def test_frames_bit_exact(pm, orc, scenes, torch, shift, scale):
    """scenes moved and scaled: hits, grazing rays, and rays aimed at edges and
    vertices, where the filter is closest to the test"""
    rng = np.random.default_rng(11)
    tris = tuple(t.copy() for t in scenes.random_soup(700, seed=8, size=0.3))
    org, dirs = (a.copy() for a in scenes.random_rays(6000, seed=9))
    k = rng.integers(0, 700, 3000)
    b = rng.dirichlet((1, 1, 1), 3000)
    b[:1000, 0] = 0.0                          # on an edge
    b[1000:1500] = [1.0, 0.0, 0.0]             # at a vertex
    b[:1000] /= b[:1000].sum(1, keepdims=True)
    aim = sum(b[:, i:i + 1] * tris[i][k, :3] for i in range(3))
    dirs[:3000, :3] = aim - org[:3000, :3]
    # in the triangle's plane
    dirs[3000:3500, :3] = tris[1][k[:500], :3] - tris[0][k[:500], :3]
    org[3000:3500, :3] = tris[0][k[:500], :3] - 0.5 * dirs[3000:3500, :3]
    for t in tris:
        t[:, :3] = t[:, :3] * np.float32(scale) + np.float32(shift * scale)
    org[:, :3] = org[:, :3] * np.float32(scale) + np.float32(shift * scale)
    check(pm, orc, torch, tris, org, dirs, f"shift {shift} scale {scale}")


def test_degenerate_and_non_finite_bit_exact(pm, orc, scenes, torch):
    tris = tuple(t.copy() for t in scenes.random_soup(300, seed=21, size=0.5))
    p0, p1, p2 = tris
    p1[5] = p0[5]; p2[5] = p0[5]               # a point
    p2[6] = p1[6]                              # a segment
    p2[7, :3] = 2 * p1[7, :3] - p0[7, :3]      # collinear
    p0[8, 0] = np.nan; p1[9, 1] = np.inf; p2[10, 2] = -np.inf
    p0[11, :3] = 3e38; p1[12, :3] = -3e38
    p1[13, :3] = p0[13, :3] + np.float32(1e-30)
    org, dirs = (a.copy() for a in scenes.random_rays(2000, seed=22))
    dirs[0, :3] = 0; dirs[1, :3] = np.nan; dirs[2, 0] = np.inf; dirs[3, :3] *= np.float32(1e30)
    dirs[4, :3] *= np.float32(1e-30); org[5, :3] = 3e38; org[6, 1] = np.nan; org[7, 0] = -np.inf
    dirs[8, :3] = [1, 0, 0]; dirs[9, :3] = [0, -1, 0]; dirs[10, :3] = [0, 0, 1]
    check(pm, orc, torch, tris, org, dirs, "odd triangles")
    # the frame's own vertex is not finite
    q = tuple(t[8:].copy() for t in tris)
    check(pm, orc, torch, q, org, dirs, "first vertex NaN")
    # all triangles coincide in one vertex, and ties between copies
    r = tuple(np.repeat(t[:40], 3, 0) for t in tris)
    r[0][:] = r[0][0]
    check(pm, orc, torch, r, org, dirs, "fan of copies")
