"""The largest launches that vtdge_region_step is taken for, class of rows by class, against the separate operators bit for bit;
one sample more is refused."""
import pytest
import torch

import test_gpu_region_step as step
from util import random_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,dtype,mode", [(640, 384, "bf16", "records"), (700, 192, "bf16", "norm"), (320, 768, "bf16", "norm"),
                                            (192, 64, "bf16", "norm"), (128, 128, "f32", "norm"), (800, 192, "f32", "norm"), (200, 384, "f32", "norm"), (80, 768, "f32", "norm")])
def test_the_most_regions(dev, B, C, dtype, mode):
    from vtpack_amd import _lib
    step.test_against_the_separate_operators(dev, B, 4, 4, C, 1, dtype, mode, B % 32 == 0)
    code = _lib.BF16 if dtype == "bf16" else _lib.F32
    assert _lib.load().vtdge_region_step_fits(B + 1, 16, 16, C, 1, code) == 0


@pytest.mark.parametrize("C,dtype", [(64, "bf16"), (384, "bf16"), (768, "bf16"), (1536, "bf16"), (192, "f32"), (384, "f32"), (768, "f32")])
@pytest.mark.parametrize("choices", [(4, 2), (1, 2, 4, 4), (2, 4, 1, 2, 1), (4, 1, 2, 2, 4, 1, 1, 4)])
def test_choices_of_the_router(dev, C, dtype, choices):
    """Two to eight splits to choose from, some of them more than once: up to four have their weights read ahead."""
    from vtpack_amd import _lib, ops
    from vtpack_amd._lib import ptr
    dt, code = (torch.bfloat16, _lib.BF16) if dtype == "bf16" else (torch.float32, _lib.F32)
    B, Hr, Wr, extra, S = 9, 3, 4, 1, len(choices)
    H, W, regions = 4 * Hr, 4 * Wr, B * Hr * Wr
    N = extra + H * W
    g = torch.Generator(dev).manual_seed(C + S)
    splits = torch.tensor(choices, dtype=torch.int64, device=dev)
    idx = torch.from_numpy(random_indices(C + S, B, Hr, Wr)).to(dev) % S
    patches, offsets, _ = ops.index_to_patch(idx, splits, 4, extra)
    L = int(offsets[-1])
    q, comp, x = (torch.randn(*s, C, generator=g, device=dev).to(dt) for s in ((L,), (L,), (B, N)))
    wgt, bias = torch.randn(S, C, generator=g, device=dev).to(dt), (torch.randn(S, generator=g, device=dev) * 0.1).to(dt)
    out, gate, nidx = torch.empty_like(x), torch.empty((B, Hr, Wr, S), dtype=dt, device=dev), torch.empty_like(idx)
    ncnt, ncomp = torch.empty((regions,), dtype=torch.uint8, device=dev), torch.empty((B * N, C), dtype=dt, device=dev)
    npat, noff = torch.empty((B * N, 4), dtype=torch.int64, device=dev), torch.empty((B + 1,), dtype=torch.int64, device=dev)
    nrr = torch.empty((regions,), dtype=torch.int32, device=dev)
    ws = torch.zeros((_lib.load().vtdge_region_step_workspace(B, H, W) // 8,), dtype=torch.int64, device=dev)
    _lib.call("vtdge_region_step", ptr(q), ptr(comp), ptr(idx), ptr(splits), ptr(offsets), None, None, ptr(x), ptr(out), ptr(wgt),
              ptr(bias), ptr(gate), ptr(nidx), ptr(splits), ptr(ncnt), None, None, None, None, 1e-6, ptr(ncomp), None, None, ptr(npat),
              B * N, ptr(noff), ptr(nrr), ptr(ws), ws.numel() * 8, B, H, W, C, extra, S, S, code, _lib.stream_ptr())
    want = ops.decompress(q, patches[:L], x, W, extra, add_ref=True, sub=comp)
    want_gate, want_idx = ops.router(want, wgt, bias, H, W, 4)
    wpat, woff, _ = ops.index_to_patch(want_idx, splits, 4, extra)
    n = int(woff[-1])
    assert torch.equal(out, want) and torch.equal(gate, want_gate) and torch.equal(nidx, want_idx)
    assert torch.equal(noff, woff) and torch.equal(npat[:n], wpat[:n]) and torch.equal(ncomp[:n], ops.compress(want, wpat[:n], W, extra))
