"""A context's first build on a GPU with little memory left: its buffers are
not sized ahead then, and it builds what a build sized level by level builds."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_tree

pytestmark = pytest.mark.gpu


def test_first_build_in_little_memory(pm):
    """8M small triangles: 386 bytes each level by level, 795 sized ahead; 600 free"""
    import torch
    n = 8_000_000
    g = torch.Generator(device="cuda:0")
    g.manual_seed(1)
    c = torch.rand((n, 3), device="cuda:0", generator=g)
    one = torch.ones((n, 1), device="cuda:0")
    P = [torch.cat([c + 0.0005 * torch.rand((n, 3), device="cuda:0", generator=g), one], 1) for _ in range(3)]
    small = [p[:100].contiguous() for p in P]
    bp = pm.build_params("default")
    del c, one
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    ctx = pm.Context(0)
    ctx.build(*small, bp)
    ctx.build(*P, bp)                    # not its first: sized level by level
    want = ctx.tree_arrays()
    ctx.close()
    free = torch.cuda.mem_get_info()[0]
    fill = torch.empty(free - 600 * n, dtype=torch.uint8, device="cuda:0")
    ctx = pm.Context(0)
    ctx.build(*P, bp)
    got = ctx.tree_arrays()
    ctx.close()
    del fill
    torch.cuda.empty_cache()
    assert_same_tree(got, want, "little memory")
    ctx = pm.Context(0)
    ctx.build(*P, bp)                    # with room: sized ahead
    assert_same_tree(ctx.tree_arrays(), want, "room")
    ctx.close()
    assert np.isin([np.int32(n - 1)], got["prim_indices"]).all()
