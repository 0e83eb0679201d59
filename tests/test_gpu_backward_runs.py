"""Per-vertex gradient sums over long runs: a few large triangles under many
rays, so that a vertex's entries end inside a block of the sum, cross into the
next, or span several; bit-exact against the oracle's sequential sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


@pytest.mark.parametrize("grid", [1, 2, 5, 9])
@pytest.mark.parametrize("n", [1, 2, 85, 86, 171, 257, 1000, 5000, 20011])
def test_long_runs_bit_exact(pm, orc, torch, grid, n):
    g = grid + 1
    y, x = np.meshgrid(np.linspace(0, 1, g), np.linspace(0, 1, g), indexing="ij")
    V = np.stack([x.reshape(-1), y.reshape(-1), 0.1 * np.sin(7 * x.reshape(-1))], 1).astype(np.float32)
    i = np.arange(g * g).reshape(g, g)
    a, b, c, d = i[:-1, :-1].ravel(), i[:-1, 1:].ravel(), i[1:, 1:].ravel(), i[1:, :-1].ravel()
    F = np.concatenate([np.stack([a, b, c], 1), np.stack([a, c, d], 1)]).astype(np.int32)
    tris = []
    for k in range(3):
        p = np.ones((F.shape[0], 4), np.float32)
        p[:, :3] = V[F[:, k]]
        tris.append(p)
    rng = np.random.default_rng(n)
    org = np.ones((n, 4), np.float32)
    org[:, :2] = rng.uniform(-0.05, 1.05, (n, 2)); org[:, 2] = 2.0
    dirs = np.zeros((n, 4), np.float32)
    dirs[:, :2] = rng.uniform(-0.05, 0.05, (n, 2)); dirs[:, 2] = -1.0
    dev = "cuda:0"
    P, O, D = ([torch.from_numpy(t).to(dev) for t in tris], torch.from_numpy(org).to(dev),
               torch.from_numpy(dirs).to(dev))
    ctx = pm.Context(0)
    ctx.set_geometry(*P)
    H = ctx.trace(pm.BRUTE, O, D)
    h = pm.hits_to_numpy(H)
    if n > 50:
        assert 0.5 < (h["id"] >= 0).mean()
    up = [rng.normal(size=n).astype(np.float32) for _ in range(3)]
    got = ctx.trace_backward(O, D, H, *[torch.from_numpy(u).to(dev) for u in up],
                             torch.from_numpy(F.reshape(-1).copy()).to(dev), V.shape[0], tris=P)
    want = orc.trace_backward(tuple(tris), org, dirs, h, *up, F, V.shape[0])
    for p, q in zip(got, want):
        assert np.array_equal(p.cpu().numpy().view(np.int32), q.view(np.int32))
    ctx.close()
