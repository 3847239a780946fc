"""The bf16 Linear around the edges of its tiles, for each of its three shapes (128x256, 128x128 with two or three stages):
live rows around a tile of a larger capacity, output widths that end inside a tile, one K slab and several."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,N", [(5600, 1536), (5600, 1544), (11000, 768), (13200, 648), (300, 1544), (300, 72)])
@pytest.mark.parametrize("live", [0, 1, 127, 128, 129, 260, None])
@pytest.mark.parametrize("K", [64, 192, 2048])
@pytest.mark.parametrize("act,res", [("none", False), ("gelu", False), ("none", True)])
def test_tile_edges(dev, cap, N, live, K, act, res):
    from vtpack_amd import ops
    live = cap if live is None else live
    g = torch.Generator(dev).manual_seed(live + N)
    a, w, bias, r = ((torch.randn(*s, generator=g, device=dev) * s[-1] ** -0.5 * k).bfloat16() for s, k in (
        ((cap, K), K ** 0.5), ((N, K), 1), ((N,), N ** 0.5), ((cap, N), N ** 0.5)))
    out = torch.full((cap, N), 7.0, device=dev, dtype=torch.bfloat16)
    ops.linear(a, w, bias, r if res else None, act=act, rows_dev=torch.tensor([live], device=dev), out=out)
    if live:
        want = a[:live].double() @ w.double().T + bias.double()
        want = torch.nn.functional.gelu(want) if act == "gelu" else want
        want = want + r[:live].double() if res else want
        # one rounding of the result: 2^-9 of values up to about 6, against the largest of them
        assert rel_err(out[:live], want.cpu()) <= 2 ** -8
    assert bool((out[live:] == 7.0).all())
