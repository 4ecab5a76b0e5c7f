"""Permutations through the transpose tiles, on rows that start on cache lines
(tiles in launch order) and rows that do not (contiguous tile ranges per XCD),
at the edges of the 64- and 128-wide tiles. Exact."""

import pytest
import torch

import trntensor_amd as tt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("sub", ["ijk->kji", "ijk->ikj", "ijk->jki", "ijk->kij"])
@pytest.mark.parametrize("shape", [(64, 128, 64), (65, 127, 130), (3, 200, 201), (131, 5, 257), (32, 96, 128), (129, 64, 33)])
def test_permute_edges(hip, dt, sub, shape):
    g = torch.Generator().manual_seed(sum(shape))
    lhs, out = sub.split("->")
    order = [lhs.index(c) for c in out]
    x = torch.randn(shape, generator=g, dtype=torch.float64).to(dt)
    for off in (0, 1):  # base on and off a cache line
        buf = torch.full((x.numel() + off,), float("nan"), dtype=dt, device="cuda")
        buf[off:] = x.reshape(-1).cuda()
        v = buf[off:].view(shape)
        assert torch.equal(tt.einsum(sub, v).cpu(), x.permute(order))
        c = torch.randn([shape[k] for k in order], generator=g, dtype=torch.float64).to(dt)
        got = tt.einsum(sub, v, alpha=2.0, beta=0.5, out=c.cuda())
        assert torch.equal(got.cpu(), 2.0 * x.permute(order) + 0.5 * c)


def test_permute_more_tiles_than_a_grid(hip):
    """One small transpose per batch entry, 2^24 and more of them: their tiles
    do not fit one launch."""
    import trntensor_amd as tt

    x = torch.arange(6 * (2**24 + 5), dtype=torch.float32, device="cuda").view(2**24 + 5, 2, 3)
    assert torch.equal(tt.einsum("aij->aji", x), x.transpose(1, 2).contiguous())
