"""The scatter-back by region where several regions share a wave: their first packed rows are found by the whole wave
where a sample's regions fill it evenly, by each group where they do not, and every token fetches its packed row by
itself.  Against the two separate operators, bit for bit (stored values and indices are the same sums in the same
order)."""
import pytest
import torch

from util import SPLITS, random_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,C,gs", [(torch.bfloat16, 64, 8), (torch.bfloat16, 8, 8), (torch.bfloat16, 128, 16),
                                        (torch.bfloat16, 72, 16), (torch.bfloat16, 256, 32), (torch.bfloat16, 768, 64),
                                        (torch.float32, 64, 16), (torch.float32, 128, 32), (torch.float32, 260, 64)])
@pytest.mark.parametrize("held", [True, False])
def test_regions_that_share_a_wave(dev, dtype, C, gs, held):
    from vtpack_amd import _lib, ops
    splits = torch.tensor(SPLITS, dtype=torch.int64, device=dev)
    per_group = 4 * (64 // gs)                           # regions a workgroup takes
    for Hr, Wr, extra in ((8, 8, 0), (10, 12, 2), (5, 7, 1), (1, 1, 1), (9, 16, 0)):
        n = Hr * Wr
        B = min(3, max(1, 255 * per_group // n)) if held else 256 * per_group // n + 1
        H, W = 4 * Hr, 4 * Wr
        g = torch.Generator(dev).manual_seed(n + C)
        mixed = torch.from_numpy(random_indices(n + C, B, Hr, Wr)).to(dev)
        for idx in (mixed, torch.zeros_like(mixed), torch.full_like(mixed, len(SPLITS) - 1)):
            patches, offsets, _ = ops.index_to_patch(idx, splits, 4, extra)
            L = int(offsets[-1])
            q, comp = (torch.randn(L, C, generator=g, device=dev).to(dtype) for _ in range(2))
            x = torch.randn(B, extra + H * W, C, generator=g, device=dev).to(dtype)
            wgt = (torch.randn(3, C, generator=g, device=dev) / C ** 0.5).to(dtype)
            bias = (torch.randn(3, generator=g, device=dev) * 0.1).to(dtype)
            for sub in ((comp,) if held else (comp, None)):
                got, gate, nidx = ops.decompress_router(q, idx, splits, offsets, x, H, W, 4, sub=sub, next_weight=wgt, next_bias=bias)
                name = _lib.last_kernel()
                assert f", {gs}, " in name and name.split(">")[0].endswith("true" if held else "false"), name
                want = ops.decompress(q, patches[:L], x, W, extra, add_ref=True, sub=sub)
                want_gate, want_idx = ops.router(want, wgt, bias, H, W, 4)
                assert torch.equal(got, want), (Hr, Wr, extra)
                assert torch.equal(nidx, want_idx) and torch.equal(gate, want_gate), (Hr, Wr, extra)
