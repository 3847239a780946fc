"""The chained scatter-back around the groups of 64 workgroups that hand their query counts along: a workgroup's place among
the next block's packed rows is what the counts of all workgroups before it add up to, at the edges of a group, past the
64 groups whose sums a wave reads in one go, and at the most regions a launch takes.  Whole numbers: exact."""
import pytest
import torch

from util import SPLITS, random_indices

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.mark.parametrize("B,Hr,Wr,extra", [(63, 2, 2, 0), (1, 16, 16, 2), (65, 2, 2, 1), (1, 12, 43, 0), (128, 2, 2, 1),
                                           (4097, 2, 2, 0), (2, 68, 241, 1), (1, 256, 256, 1)])
def test_places_across_groups_of_workgroups(dev, B, Hr, Wr, extra):
    from vtpack_amd import ops
    H, W, C = 4 * Hr, 4 * Wr, 264
    g = torch.Generator(dev).manual_seed(B + Wr)
    idx = torch.from_numpy(random_indices(B + Wr, B, Hr, Wr)).to(dev)
    splits = torch.tensor(SPLITS, dtype=torch.int64, device=dev)
    x = torch.randn(B, extra + H * W, C, generator=g, device=dev).bfloat16()
    assert ops.fits_pack_next(x, H, W, 4, SPLITS)
    offsets = ops.index_to_patch(idx, splits, 4, extra)[1]
    q = torch.randn(int(offsets[B]), C, generator=g, device=dev).bfloat16()
    wgt = torch.randn(3, C, generator=g, device=dev).bfloat16()
    bias = torch.zeros(3, device=dev).bfloat16()
    out, _, nidx, _, cnt, packed = ops.decompress_router(q, idx, splits, offsets, x, H, W, 4, next_weight=wgt, next_bias=bias,
                                                         stats_eps=EPS, next_splits=splits, pack_next=True, pack_eps=EPS)
    assert int(packed["workspace"][0]) == 0
    per = splits[nidx.reshape(B, -1)] ** 2
    lengths = per.sum(1) + extra
    want_off = torch.cat([torch.zeros(1, dtype=torch.int64, device=dev), lengths.cumsum(0)])
    assert torch.equal(packed["offsets"], want_off)
    rows = (want_off[:B, None] + extra + per.cumsum(1) - per).reshape(-1)
    assert torch.equal(packed["region_rows"].long(), rows)
    assert len(set(nidx.reshape(-1).tolist())) == 3
    total = int(want_off[B])
    w_comp, w_rec = ops.compress_regions(out, nidx, splits, H, W, 4, counts=cnt, stats_eps=EPS)[:2]
    assert torch.equal(packed["comp"][:total], w_comp[:total]) and torch.equal(packed["records"][:total], w_rec[:total])
