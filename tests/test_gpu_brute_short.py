"""Brute force where lengths are too short for their squares to be floats:
directions and edges from 2^-56 down to 2^-76 in scenes large enough that the
filter's scales still lie in its range.  Records bit-exact against the oracle's
sequential loop; rays aimed at edges and vertices among them."""
import numpy as np
import pytest

from test_gpu_brute import check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.mark.parametrize("extent", [33, 35, 38])
@pytest.mark.parametrize("length", [-56, -60, -64, -70, -73, -74, -75, -76])
def test_short_directions(pm, orc, scenes, torch, extent, length):
    """a hit lies within 2^31 lengths of the origin: triangles in the plane
    z = 0, origins on it or just above"""
    rng = np.random.default_rng(extent - length)
    tris = tuple(t.copy() for t in scenes.random_soup(600, seed=8, size=0.4))
    for t in tris:
        t[:, :3] *= np.float32(2.0 ** extent)
        t[:, 2] = 0.0
    n = 6000
    k = rng.integers(0, 600, n)
    b = rng.dirichlet((1, 1, 1), n)
    b[::2, 0] = 0.0                            # on an edge
    b[1::7] = [1.0, 0.0, 0.0]                  # at a vertex
    b /= b.sum(1, keepdims=True)
    org, dirs = np.ones((n, 4), np.float32), np.zeros((n, 4), np.float32)
    org[:, :3] = sum(b[:, i:i + 1] * tris[i][k, :3] for i in range(3))
    org[::3, 2] = np.float32(2.0 ** (length + 29))
    # of lengths whose squares round worst: sums of squares 2.47, 2.5, 3.49
    d = rng.normal(size=(n, 3))
    d[:2000] = rng.permuted(np.tile(np.sqrt([1.495, 0.495, 0.495]), (2000, 1)), axis=1)
    d *= (np.sqrt(rng.choice([1.0, 2.47, 2.5, 3.49], n)) * 2.0 ** (length + 0.5) / np.linalg.norm(d, axis=1))[:, None]
    d[:, 2] = -abs(d[:, 2])
    dirs[:, :3] = d.astype(np.float32)
    want = check(pm, orc, torch, tris, org, dirs, f"2^{length} in 2^{extent}", test=pm.MOELLER)
    assert (want["id"] >= 0).mean() > 0.2


@pytest.mark.parametrize("length", [-56, -60, -64, -70, -74])
def test_short_edges_far_from_the_frame(pm, orc, scenes, torch, length):
    """tiny triangles about the origin, the others (the first among them, and
    every one of the sample that sizes the frame) 2^36 away"""
    rng = np.random.default_rng(-length)
    far = tuple(t.copy() for t in scenes.random_soup(4096, seed=8, size=0.3))
    for t in far:
        t[:, :3] = t[:, :3] * np.float32(2.0 ** 10) + np.float32(2.0 ** 36)
    small = rng.normal(size=(3, 64, 3)) * 2.0 ** length
    at = 5 + 64 * np.arange(64)
    for i in range(3):
        far[i][at, :3] = small[i].astype(np.float32)
    assert not np.isin(at, np.arange(64) * 4096 // 64).any()
    org = np.ones((3000, 4), np.float32)
    org[:, :3] = rng.normal(size=(3000, 3)) * 2.0 ** (length + 3)
    dirs = np.zeros((3000, 4), np.float32)
    k = rng.integers(0, 64, 3000)
    b = rng.dirichlet((1, 1, 1), 3000)
    b[::2, 0] = 0.0
    b /= b.sum(1, keepdims=True)
    d = sum(b[:, i:i + 1] * small[i][k] for i in range(3)) - org[:, :3]
    dirs[:, :3] = d / np.linalg.norm(d, axis=1, keepdims=True)
    want = check(pm, orc, torch, far, org, dirs, f"edges 2^{length}", test=pm.MOELLER)
    if length >= -60:
        assert (want["id"] >= 0).mean() > 0.2
