"""The gathers of launches of few workgroups (64 or 32 rows per wave) against
those that fill the GPU (128 rows per wave), and the scatters (32 rows per wave) of
both: the same heads once a few at a time and once repeated past the line between
the two, bit for bit.
Every candidate shape, grids with padding, a valid mask, chunks of 64 and 128
tokens with row padding (an odd number of 64-row tiles)."""
import numpy as np
import pytest
import torch

from tests.test_gpu_parity import bits_equal, host, say

pytestmark = pytest.mark.gpu


def _both(x, dot, gather, scatter, units, dtype):
    """(few, many) outputs of head 0 .. H-1."""
    B, H, S, D = x.shape
    reps = -(-1100 // (units * H))
    out = []
    for n in (1, reps):
        xs, ds = x.repeat(1, n, 1, 1), dot.repeat(1, n, 1, 1)
        pooled, plain, dotted = gather(xs, None), gather(xs, False), gather(xs, ds)
        back = scatter(plain["rows"], dtype)
        keep = [pooled["rows"], pooled["block_mean"], plain["rows"], dotted["rows"], dotted["rowdot"], back]
        out.append([host(t[:, :H]) for t in keep] + [host(pooled[k]) for k in ("block_count", "tile_count", "valid_re")])
    return out


@pytest.mark.parametrize("D,dtype", [(64, torch.float32), (128, torch.bfloat16), (128, torch.float32),
                                     (64, torch.bfloat16)], ids=str)
def test_zone_gather_few_equals_many(D, dtype):
    from prism_amd import ops
    say("zone gather", D, dtype)
    g = torch.Generator(device="cuda").manual_seed(1)
    grid, box, H = (16, 8, 56), (13, 7, 50), 2
    sid = torch.arange(14, device="cuda") % 13
    lay = ops.ZoneLayout(sid, grid, box)
    S = box[0] * box[1] * box[2]
    x = torch.randn((1, H, S, D), device="cuda", generator=g).to(dtype)
    dot = torch.randn((1, H, lay.S, D), device="cuda", generator=g).to(torch.bfloat16)
    valid = torch.rand((S,), device="cuda", generator=g) < 0.7

    def gather(t, how):
        if how is None:
            return ops.gather_pool(t, lay, valid, pool=True, counts=True)
        return ops.gather_pool(t, lay, None, dot_with=None if how is False else how)

    few, many = _both(x, dot, gather, lambda r, dt: ops.scatter_rows(r, lay, dt), 14, dtype)
    for i, (a, b) in enumerate(zip(few, many)):
        assert bits_equal(a, b), i
    xb = x.to(torch.bfloat16).to(dtype)
    assert np.array_equal(few[5], host(xb))  # scattered back: the input's bf16 values


@pytest.mark.parametrize("chunk,grid", [((4, 4, 4), (7, 9, 30)), ((2, 8, 8), (5, 9, 24)), ((1, 1, 64), (1, 1, 1000)),
                                        ((1, 1, 128), (1, 1, 1000)), ((64, 1, 1), (70, 2, 3))], ids=str)
def test_chunk_gather_few_equals_many(chunk, grid):
    from prism_amd import ops
    say("chunk gather", chunk, grid)
    g = torch.Generator(device="cuda").manual_seed(2)
    H, D, dtype = 2, 128, torch.bfloat16
    lay = ops.ChunkLayout(grid, chunk, "cuda")
    x = torch.randn((1, H, lay.S_in, D), device="cuda", generator=g).to(dtype)
    dot = torch.randn((1, H, lay.rows, D), device="cuda", generator=g).to(torch.bfloat16)
    valid = torch.rand((lay.S_in,), device="cuda", generator=g) < 0.7

    def gather(t, how):
        if how is None:
            return ops.chunk_gather_pool(t, lay, valid, pool=True, counts=True)
        return ops.chunk_gather_pool(t, lay, None, dot_with=None if how is False else how)

    few, many = _both(x, dot, gather, lambda r, dt: ops.chunk_scatter_rows(r, lay, dt), -(-lay.rows // 512), dtype)
    for i, (a, b) in enumerate(zip(few, many)):
        assert bits_equal(a, b), i
    assert np.array_equal(few[5], host(x))
