"""Buffers that grow while a build runs keep what they hold and nothing past
it: the host class (with stubbed runtime calls, CPU), and forests whose
subtrees' first level writes more empty-space nodes than the level before it
had room for, built after a tiny build in the same context (GPU)."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_growth_keeps_no_more_than_held(tmp_path):
    exe = str(tmp_path / "test_devbuf")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-o", exe, os.path.join(HERE, "cpp", "test_devbuf.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "DevBuf OK" in r.stdout, r.stdout + r.stderr


def corner_pairs(n: int, depth: int, seed: int, ext: float = 0.3):
    """n tiny triangles in 2^depth cells: every box holds two boxes of `ext` of
    its size in opposite corners, so that a split leaves three sides of either
    child empty"""
    rng = np.random.default_rng(seed)
    lo, size = np.zeros((1, 3)), 1.0
    for _ in range(depth):
        lo = np.concatenate([lo, lo + size * (1.0 - ext)])
        size *= ext
    lo = np.repeat(lo, n // lo.shape[0], 0)
    c = lo + 0.9 * size * rng.random(lo.shape)
    v = [c + 0.02 * size * rng.random(lo.shape) for _ in range(3)]
    return tuple(np.concatenate([x, np.ones((n, 1))], 1).astype(np.float32) for x in v)


@pytest.mark.gpu
@pytest.mark.parametrize("meshes,n,depth", [(8, 16384, 7), (4, 32768, 7), (2, 65536, 7), (8, 16384, 5)])
def test_subtrees_with_more_empty_nodes_than_the_level_before(pm, orc, scenes, meshes, n, depth):
    import torch

    from test_gpu_parity import assert_same_tree, dev, orc_params

    bp = pm.build_params("default")
    ctx = pm.Context(0)
    small = scenes.random_soup(100, seed=1, size=0.05)
    ctx.build(*[dev(torch, t) for t in small], bp)
    parts = [corner_pairs(n, depth, m) for m in range(meshes)]
    tris = tuple(np.concatenate([p[k] for p in parts]) for k in range(3))
    off = (np.arange(meshes + 1) * n).astype(np.int32)
    print(f"forest of {meshes} x {n}, {depth} deep", flush=True)
    ctx.build_batched(*[dev(torch, t) for t in tris], off, bp)
    ref = orc.build_batched(tris, off, orc_params(orc, bp))
    assert_same_tree(ctx.tree_arrays(), ref.arrays(), f"{meshes} x {n}")
    assert ctx.stats()["upper_levels"] == ref.stats()["upper_levels"]
    ctx.close()
