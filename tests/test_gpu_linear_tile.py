"""The bf16 Linear over long rows (K and N from 768 on) around the edges of its tiles: live rows at the ends of its 64-row units
and of rounds of large tiles, each shape of the rest, output widths that end inside a tile, one slab of K more than twelve."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("live", [0, 1, 63, 64, 65, 511, 513, 1700, 4200, 5500, 8190, 8193, 10700, 16390, 23000, None])
@pytest.mark.parametrize("N,K", [(768, 768), (776, 832), (1664, 768), (3072, 768), (768, 3072)])
@pytest.mark.parametrize("act,res", [("none", False), ("gelu", False), ("none", True)])
def test_long_rows(dev, live, N, K, act, res):
    from vtpack_amd import _lib, ops
    cap = 25443
    K = max(K, 1600) if res else K                                 # residuals behind a shorter K are linear_dma.hip's
    live = cap if live is None else live
    g = torch.Generator(dev).manual_seed(live + N)
    a, r = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((cap, K), (cap, N)))
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    bias = torch.randn(N, generator=g, device=dev).bfloat16() if live % 2 else None
    out = torch.full((cap, N), 7.0, device=dev, dtype=torch.bfloat16)
    ops.linear(a, w, bias, r if res else None, act=act, rows_dev=torch.tensor([live], device=dev), out=out)
    assert "linear_tile_kernel" in _lib.last_kernel()
    if live:
        want = a[:live].float() @ w.float().T + (bias.float() if bias is not None else 0)
        want = torch.nn.functional.gelu(want) if act == "gelu" else want
        want = want + r[:live].float() if res else want
        # one rounding of the result: 2^-9 of values up to about 6, against the largest of them
        assert rel_err(out[:live], want) <= 2 ** -8
    assert bool((out[live:] == 7.0).all())


def test_rows_apart_and_a_result_in_the_residuals_place(dev):
    from vtpack_amd import _lib, ops
    g = torch.Generator(dev).manual_seed(1)
    wide = torch.randn(6000, 2432, generator=g, device=dev).bfloat16()
    w = (torch.randn(768, 1600, generator=g, device=dev) * 1600 ** -0.5).bfloat16()
    r = torch.randn(6000, 768, generator=g, device=dev).bfloat16()
    a = wide[:, 832:]
    want = a.float() @ w.float().T + r.float()
    ops.linear(a, w, None, r, out=r)
    assert "linear_tile_kernel" in _lib.last_kernel()
    assert rel_err(r, want) <= 2 ** -8


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("live", [24576, 25000, 25443])
def test_rows_that_are_not_finite_stay_by_themselves(dev, bad, live):
    """Rows of an infinity or NaN beside rows of another XCD's share of the live ones (whole 64-row units),
    at tiles' edges and past the live rows: only their own results are not finite."""
    from vtpack_amd import _lib, ops
    g = torch.Generator(dev).manual_seed(live)
    a = torch.randn(25443, 768, generator=g, device=dev).bfloat16()
    w = (torch.randn(776, 768, generator=g, device=dev) * 768 ** -0.5).bfloat16()
    units = -(-live // 64)
    rows = {live - 1}
    for share in range(8):
        at = units * share // 8 * 64
        rows |= {r for r in (at, at - 1, at + 255, at + 256) if 0 <= r < live}
    rows = sorted(rows)
    ops.linear(a, w, None, rows_dev=torch.tensor([live], device=dev), out=(want := torch.zeros(25443, 776, device=dev, dtype=a.dtype)))
    a[rows, 5] = bad
    a[live:] = bad
    out = torch.full_like(want, 7.0)
    ops.linear(a, w, None, rows_dev=torch.tensor([live], device=dev), out=out)
    assert "linear_tile_kernel" in _lib.last_kernel()
    assert not bool(out[rows].isfinite().any())
    out[rows], want[rows] = 0, 0
    assert torch.equal(out[:live], want[:live]) and bool((out[live:] == 7.0).all())


@pytest.mark.parametrize("rows,N,K,act,res,tile", [
    (2048, 1536, 768, "none", False, True), (2047, 1536, 768, "none", False, False),
    (10922, 768, 768, "none", False, False), (10923, 768, 768, "none", False, True),
    (25443, 768, 1472, "none", True, False), (25443, 768, 1600, "none", True, True),
    (2730, 768, 3072, "none", True, True), (2731, 768, 3072, "none", True, None),
    (5461, 768, 3072, "none", True, None), (5462, 768, 3072, "none", True, True),
    (2730, 1536, 2048, "none", False, None), (2731, 1536, 2048, "none", False, True),
    (3413, 1536, 768, "none", False, True), (3414, 1536, 768, "none", False, False),
    (5120, 1536, 768, "none", False, False), (5121, 1536, 768, "none", False, True), (4096, 1536, 1024, "none", False, True),
    (2048, 3072, 768, "gelu", False, True), (4096, 2048, 832, "gelu", True, False)])
@pytest.mark.parametrize("packed", [False, True])
def test_calls_that_take_it(dev, rows, N, K, act, res, packed, tile):
    """Each line of the rule from both sides, with the result of either kernel."""
    from vtpack_amd import _lib, ops
    g = torch.Generator(dev).manual_seed(rows)
    a, r = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((rows, K), (rows, N)))
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    rows_dev = torch.tensor([rows - 1], device=dev) if packed else None
    out = ops.linear(a, w, None, r if res else None, act=act, rows_dev=rows_dev)
    tile = packed if tile is None else tile      # None: packed rows only
    assert ("linear_tile_kernel" if tile else "linear_dma_kernel") in _lib.last_kernel()
    want = a.float() @ w.float().T
    want = torch.nn.functional.gelu(want) if act == "gelu" else want
    want = want + r.float() if res else want
    # one rounding of the result, as above (two with an activation in front of the residual)
    assert rel_err(out[:rows - packed], want[:rows - packed]) <= 2 ** -8
