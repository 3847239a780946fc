"""The Linear over blocks of tokens around the edges of its tiles: few rows (walked either way), 64x64, 128x64 and 128x128
tiles, with rows and output widths that end inside one."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N", [(1, 136), (1, 784), (1, 1000), (5, 136), (5, 64), (9, 136), (9, 200), (9, 1280), (19, 64)])
@pytest.mark.parametrize("C", [64, 192])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_tile_edges(dev, B, N, C, dtype):
    from vtpack_amd import ops
    side, k = 56, 2
    g = torch.Generator(dev).manual_seed(B + N)
    x = torch.randn(B, side * side, C, generator=g, device=dev).to(dtype)
    w = (torch.randn(N, k * k * C, generator=g, device=dev) * (k * k * C) ** -0.5).to(dtype)
    bias = torch.randn(N, generator=g, device=dev).to(dtype)
    got = ops.patch_linear(x, side, side, k, w, bias)
    rows = x.view(B, side // k, k, side // k, k, C).permute(0, 1, 3, 2, 4, 5).reshape(-1, k * k * C)
    want = rows.double() @ w.double().T + bias.double()
    # one rounding of the result: 2^-9 of values up to about 6, against the largest of them; fp32: sums of at most 768
    # products, sqrt(768) * 2^-24 of their size
    assert rel_err(got, want.cpu()) <= (2 ** -8 if dtype == torch.bfloat16 else 4e-6)
