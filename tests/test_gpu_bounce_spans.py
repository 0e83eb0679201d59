"""Photon bounces at the edges of the survivor counting: rays that fill a wave,
a block and a span less, exactly and plus one, all or none of them surviving,
and every ray of a call long enough for several iterations a wave.  The
survivors' order and count are whole numbers, compared exactly with numpy; the
rays with the same rays bounced in one call of their own size, whose values
depend on the ray's index and inputs only."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _setup(scenes, n, seed):
    tris = scenes.random_soup(500, 3)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in tris]
    g = np.random.default_rng(seed)
    org = np.ones((n, 4), np.float32)
    org[:, :3] = g.random((n, 3), np.float32)
    d = np.zeros((n, 4), np.float32)
    d[:, :3] = g.random((n, 3), np.float32) - 0.5
    hits = np.zeros((n, 4), np.float32)
    hits[:, 1] = g.random(n, np.float32)
    return dev, org, d, hits, g


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 524287, 524288, 524289, 1048577, 1700001])
@pytest.mark.parametrize("share", [0.0, 0.6, 1.0])
def test_survivors_in_order(pm, scenes, n, share):
    (p0, p1, p2), org, d, hits, g = _setup(scenes, n, n)
    ids = np.where(g.random(n) < share, g.integers(0, 480, n), np.where(g.random(n) < 0.5, -1, 490)).astype(np.int32)
    hits[:, 0] = ids.view(np.float32)
    ctx = pm.Context()
    ctx.set_geometry(p0, p1, p2)
    O, D, H = (torch.from_numpy(a).cuda() for a in (org, d, hits))
    o2, d2, src, cnt = ctx.photon_bounce(O, D, H, 480, seed=5)
    want = np.nonzero((ids >= 0) & (ids < 480))[0]
    assert int(cnt) == len(want)
    got = src[:len(want)].cpu().numpy()
    assert np.array_equal(got, want)
    if len(want) == 0:
        return
    # the last rays once more with every ray before them dead: same values
    k = max(0, n - 200)
    dead = hits.copy()
    dead[:k, 0] = np.full(k, -1, np.int32).view(np.float32)
    o3, d3, src3, c3 = ctx.photon_bounce(O, D, torch.from_numpy(dead).cuda(), 480, seed=5)
    tail = want[want >= k]
    assert int(c3) == len(tail) and np.array_equal(src3[:len(tail)].cpu().numpy(), tail)
    assert torch.equal(o3[:len(tail)].view(torch.int32), o2[len(want) - len(tail):len(want)].view(torch.int32))
    assert torch.equal(d3[:len(tail)].view(torch.int32), d2[len(want) - len(tail):len(want)].view(torch.int32))
