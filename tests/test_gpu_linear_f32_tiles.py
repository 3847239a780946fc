"""The fp32 Linear around the edges of its 64x64 tiles: live rows just under, at and over one and two tiles, output
widths that end inside a tile, and enough tiles that a workgroup walks several; and of the 256x128 tiles of large products."""
import pytest
import torch

from util import FP32_REL, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("live,cap", [(0, 70), (1, 70), (63, 70), (64, 64), (65, 200), (129, 200), (25000, 25061)])
@pytest.mark.parametrize("N,K", [(60, 64), (64, 32), (68, 192), (192, 96)])
@pytest.mark.parametrize("act,res", [("none", True), ("gelu", False)])
def test_tile_edges(dev, live, cap, N, K, act, res):
    from vtpack_amd import ops
    g = torch.Generator().manual_seed(live + N)
    a, w = torch.randn(cap, K, generator=g), torch.randn(N, K, generator=g)
    bias, r = torch.randn(N, generator=g), torch.randn(cap, N, generator=g)
    out = torch.full((cap, N), 7.0, device=dev)
    ops.linear(a.to(dev), w.to(dev), bias.to(dev), r.to(dev) if res else None, act=act,
               rows_dev=torch.tensor([live], dtype=torch.int64, device=dev), out=out)
    if live:
        want = a[:live].double() @ w.double().T + bias.double()
        want = torch.nn.functional.gelu(want) if act == "gelu" else want
        want = want + r[:live].double() if res else want
        assert rel_err(out[:live], want) <= FP32_REL
    assert bool((out[live:] == 7.0).all())


@pytest.mark.parametrize("act,res", [("none", True), ("gelu", False)])
def test_large_tiles(dev, act, res):
    """2048 tiles of 256x128 and more: the larger tile, with live rows and output columns that end inside one."""
    from vtpack_amd import _lib, ops
    cap, live, N, K = 256 * 512, 256 * 301 + 77, 452, 64
    g = torch.Generator(dev).manual_seed(3)
    a, w, r = (torch.randn(*s, generator=g, device=dev) for s in ((cap, K), (N, K), (cap, N)))
    bias = torch.randn(N, generator=g, device=dev)
    out = torch.full((cap, N), 7.0, device=dev)
    ops.linear(a, w, bias, r if res else None, act=act, rows_dev=torch.tensor([live], dtype=torch.int64, device=dev), out=out)
    assert "linear_dma_kernel<float, 256, 128" in _lib.last_kernel()
    want = a[:live].double() @ w.double().T + bias.double()
    want = torch.nn.functional.gelu(want) if act == "gelu" else want
    want = want + r[:live].double() if res else want
    assert rel_err(out[:live], want.cpu()) <= FP32_REL
    assert bool((out[live:] == 7.0).all())
