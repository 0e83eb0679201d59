"""Brute force on both sides of the lines between its kernels (a lane per ray
for few triangles and many rays, else the matrix filter or the split Woop
kernel): records bit-exact against the oracle's sequential loop, with and
without counters, under a cap on the triangles; and that many rays against one
triangle cost about what moving the rays costs."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_hits, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as T
    assert T.cuda.is_available(), "these tests need the GPU"
    return T


def cases():
    out = []
    # 30 triangles (Woop 8) per 128 rays of each of the 256 CUs; 192 (384) at most
    for n in (32768, 40001, 131072):
        out += [("MOELLER", t, n) for t in (30 * n // 32768, 30 * n // 32768 + 1)]
        out += [("WOOP", t, n) for t in (8 * n // 32768, 8 * n // 32768 + 1)]
    out += [("MOELLER", t, 262147) for t in (1, 192, 193)]
    out += [("WOOP", t, 1600003) for t in (1, 384, 385)]
    out += [("MOELLER", 0, 70000), ("WOOP", 0, 70000)]
    return out


@pytest.mark.parametrize("test,ntris,nrays", cases())
def test_both_sides_bit_exact(pm, orc, scenes, torch, test, ntris, nrays):
    tris = tuple(t[:ntris].copy() for t in scenes.random_soup(max(ntris, 1), seed=ntris, size=0.5))
    org, dirs = scenes.random_rays(nrays, seed=nrays % 1000)
    dirs[:5, :3] = 0.0
    ix = getattr(pm, test)
    ctx = pm.Context(0)
    P = [dev(torch, t if ntris else np.zeros((1, 4), np.float32))[:ntris] for t in tris]
    ctx.set_geometry(*P)
    O, D = dev(torch, org), dev(torch, dirs)
    pick = np.unique(np.concatenate([np.arange(0, nrays, 1 + nrays // 60000), np.arange(nrays - 300, nrays)]))
    for cap in (0, 7):
        want = orc.trace(None, tris, org[pick], dirs[pick], orc.BRUTE, brute_cap=cap, intersection=ix, threads=8)
        tp = pm.trace_params(intersection=ix, brute_cap=cap)
        cnt = torch.full((nrays, 4), -7, dtype=torch.int32, device="cuda:0")
        H = torch.full((nrays, 4), -7.0, device="cuda:0")
        assert_same_hits(pm.hits_to_numpy(ctx.trace(pm.BRUTE, O, D, tp, out=H))[pick], want, f"cap {cap}")
        H.fill_(-7.0)
        assert_same_hits(pm.hits_to_numpy(ctx.trace(pm.BRUTE, O, D, tp, out=H, counters=cnt))[pick], want, "counted")
        assert (cnt.cpu().numpy() == [0, 0, min(ntris, cap) if cap else ntris, 0]).all()
    ctx.close()


def test_one_triangle_costs_the_rays_bytes(pm, scenes, torch):
    """2M rays read (64 MB) and their records written (32 MB): within six times
    a copy of the rays"""
    org, dirs = scenes.random_rays(2_000_000, seed=1)
    ctx = pm.Context(0)
    P = [dev(torch, t) for t in scenes.random_soup(1, seed=1, size=0.5)]
    ctx.set_geometry(*P)
    O, D = dev(torch, org), dev(torch, dirs)
    H, O2, D2 = torch.empty_like(O), torch.empty_like(O), torch.empty_like(D)

    def ms(f):
        f()
        t = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                f()
            b.record()
            b.synchronize()
            t.append(a.elapsed_time(b) / 5)
        return sorted(t)[4]

    copy = ms(lambda: (O2.copy_(O), D2.copy_(D)))
    for ix in (pm.MOELLER, pm.WOOP):
        tp = pm.trace_params(intersection=ix)
        assert ms(lambda: ctx.trace(pm.BRUTE, O, D, tp, out=H)) < 6 * copy, ix
    ctx.close()
