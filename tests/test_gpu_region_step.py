"""A block's scatter-back, the next router, index -> patch, compress and LayerNorm as one launch (vtdge_region_step) against the
separate operators, bit for bit: region counts around the groups of 64 that hand their query counts along, rows of one to three vectors a lane, every split."""
import pytest
import torch

from util import SPLITS, random_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hr,Wr,C,extra,dtype,mode", [
    (1, 1, 1, 264, 0, "bf16", "records"), (3, 4, 4, 384, 1, "bf16", "records"), (4, 4, 4, 512, 2, "bf16", "records"),
    (5, 5, 13, 384, 3, "bf16", "records"), (96, 4, 4, 384, 1, "bf16", "records"), (1, 8, 8, 384, 1, "bf16", "plain"),
    (2, 4, 4, 512, 9, "bf16", "norm"), (7, 3, 3, 768, 1, "bf16", "norm"), (1, 4, 4, 1536, 1, "bf16", "norm"),
    (65, 1, 1, 192, 1, "f32", "norm"), (128, 4, 4, 192, 1, "f32", "norm"), (3, 4, 4, 132, 0, "f32", "plain"),
    (2, 6, 4, 320, 0, "f32", "norm"), (3, 4, 4, 768, 64, "f32", "norm"), (2, 4, 4, 8, 0, "bf16", "norm"),
    (1, 16, 16, 64, 0, "bf16", "norm"), (3, 4, 4, 64, 1, "f32", "norm"), (96, 4, 4, 192, 1, "bf16", "norm"),
    (2, 3, 5, 12, 0, "f32", "plain"), (5, 8, 8, 128, 0, "bf16", "plain"), (2, 4, 4, 256, 1, "bf16", "norm"),
    (192, 4, 4, 192, 1, "bf16", "norm"), (12, 16, 16, 64, 0, "bf16", "norm"),
    (192, 4, 4, 192, 1, "f32", "norm"), (80, 4, 4, 768, 1, "bf16", "norm"), (48, 4, 4, 384, 1, "f32", "norm")])
@pytest.mark.parametrize("placed", [False, True])
def test_against_the_separate_operators(dev, B, Hr, Wr, C, extra, dtype, mode, placed):
    from vtpack_amd import _lib, ops
    from vtpack_amd._lib import ptr
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    code, eps, H, W = _lib.BF16 if dtype == "bf16" else _lib.F32, 1e-6, 4 * Hr, 4 * Wr
    N, regions = extra + H * W, B * Hr * Wr
    lib = _lib.load()
    assert lib.vtdge_region_step_fits(B, H, W, C, extra, code) == 1
    g = torch.Generator(dev).manual_seed(B + C)
    idx = torch.from_numpy(random_indices(B + C, B, Hr, Wr)).to(dev)
    splits = torch.tensor(SPLITS, dtype=torch.int64, device=dev)
    patches, offsets, _ = ops.index_to_patch(idx, splits, 4, extra)
    L = int(offsets[-1])
    q, comp, x = (torch.randn(*s, C, generator=g, device=dev).to(dt) for s in ((L,), (L,), (B, N)))
    x[:, :, 5] = -0.0
    wgt, bias = (torch.randn(3, C, generator=g, device=dev) / C ** 0.5).to(dt), (torch.randn(3, generator=g, device=dev) * 0.1).to(dt)
    lw, lb = (torch.randn(C, generator=g, device=dev).to(dt) for _ in range(2))
    cur = rr = None
    if placed:
        per = splits[idx.reshape(B, -1)] ** 2
        cur = per.reshape(-1).to(torch.uint8)
        rr = (offsets[:B, None] + extra + per.cumsum(1) - per).reshape(-1).to(torch.int32)

    out, gate = torch.empty_like(x), torch.empty((B, Hr, Wr, 3), dtype=dt, device=dev)
    nidx, ncnt = torch.empty_like(idx), torch.empty((regions,), dtype=torch.uint8, device=dev)
    rec = nrec = oln = cln = None
    ncomp, npat = torch.empty((B * N, C), dtype=dt, device=dev), torch.empty((B * N, 4), dtype=torch.int64, device=dev)
    if mode == "records":
        rec, nrec = (torch.empty((B * N, 16), dtype=dt, device=dev) for _ in range(2))
    elif mode == "norm":
        oln, cln = torch.empty((B * N, C), dtype=dt, device=dev), torch.empty((B * N, C), dtype=dt, device=dev)
    noff, nrr = torch.empty((B + 1,), dtype=torch.int64, device=dev), torch.empty((regions,), dtype=torch.int32, device=dev)
    ws = torch.zeros((lib.vtdge_region_step_workspace(B, H, W) // 8,), dtype=torch.int64, device=dev)
    _lib.call("vtdge_region_step", ptr(q), ptr(comp), ptr(idx), ptr(splits), ptr(offsets), ptr(rr), ptr(cur), ptr(x), ptr(out),
              ptr(wgt), ptr(bias), ptr(gate), ptr(nidx), ptr(splits), ptr(ncnt), ptr(rec), ptr(oln), ptr(lw if oln is not None else None),
              ptr(lb if oln is not None else None), eps, ptr(ncomp), ptr(nrec), ptr(cln), ptr(npat), B * N, ptr(noff), ptr(nrr),
              ptr(ws), ws.numel() * 8, B, H, W, C, extra, 3, 3, code, _lib.stream_ptr())

    want = ops.decompress(q, patches[:L], x, W, extra, add_ref=True, sub=comp)
    want_gate, want_idx = ops.router(want, wgt, bias, H, W, 4)
    wpat, woff, _ = ops.index_to_patch(want_idx, splits, 4, extra)
    n = int(woff[-1])
    wcomp = ops.compress(want, wpat[:n], W, extra)
    assert int(ws[0]) == 0 and torch.equal(out, want) and torch.equal(gate, want_gate) and torch.equal(nidx, want_idx)
    assert torch.equal(noff, woff) and torch.equal(npat[:n], wpat[:n])
    assert torch.equal(ncomp[:n].view(torch.int16), wcomp.view(torch.int16))       # the sign of zero too
    per = splits[want_idx.reshape(B, -1)] ** 2
    assert torch.equal(ncnt.long(), per.reshape(-1))
    assert torch.equal(nrr.long(), (woff[:B, None] + extra + per.cumsum(1) - per).reshape(-1))
    if mode == "records":
        twice = ops.decompress_router(q, idx, splits, offsets, x, H, W, 4, sub=comp, next_weight=wgt, next_bias=bias, stats_eps=eps)
        assert torch.equal(rec, twice[3])
        counts = ops.region_counts_buffer(B, Hr * Wr, dev)
        counts[:regions] = ncnt
        assert torch.equal(nrec[:n], ops.compress_regions(want, nidx, splits, H, W, counts=counts, stats_eps=eps)[1][:n])
    elif mode == "norm":
        assert torch.equal(oln, ops.layernorm(want, lw, lb, eps).view(-1, C))
        assert torch.equal(cln[:n], ops.layernorm(wcomp, lw, lb, eps))
