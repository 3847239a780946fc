"""The fp32 Linear on the bf16 matrix instructions (a weight split into three bf16 parts): live rows and widths around the
edges of its three tile shapes, its error beside the fp32 instructions', and values that the split does not cover."""
import pytest
import torch

from util import FP32_REL, rel_err

pytestmark = pytest.mark.gpu


def _run(a, w, bias, res, act, live, split, dev):
    """`ops.linear` with and without the split copy; rows behind the live ones keep what was in them."""
    from vtpack_amd import ops
    out = torch.full((a.shape[0], w.shape[0]), 7.0, device=dev)
    ops.linear(a, w, bias, res, act=act, rows_dev=torch.tensor([live], dtype=torch.int64, device=dev), out=out, keep_split=split)
    assert bool((out[live:] == 7.0).all())
    return out[:live]


@pytest.mark.parametrize("cap,N,K,tile", [(20000, 64, 32, "64, 64"), (8300, 192, 192, "64, 64"), (33000, 384, 96, "128, 64"),
                                          (16500, 1024, 384, "128, 128"), (65600, 256, 416, "128, 128")])
@pytest.mark.parametrize("act,res", [("none", False), ("none", True), ("gelu", False)])
def test_tile_edges(dev, cap, N, K, tile, act, res):
    from vtpack_amd import _lib
    g = torch.Generator(dev).manual_seed(cap + K)
    a, w, r = (torch.randn(*s, generator=g, device=dev) for s in ((cap, K), (N, K), (cap, N)))
    bias = torch.randn(N, generator=g, device=dev)
    for live in (0, 1, 63, 64, 65, 127, 129, 4097, cap):
        got = _run(a, w, bias, r if res else None, act, live, True, dev)
        assert f"linear_dma_split_kernel<{'64, 64' if res else tile}" in _lib.last_kernel()
        if live == 0:
            continue
        want = a[:live].double() @ w.double().T + bias.double()
        want = torch.nn.functional.gelu(want) if act == "gelu" else want
        want = want + r[:live].double() if res else want
        assert rel_err(got, want) <= FP32_REL
        if live >= 4097:            # no less exact than the fp32 instructions (0.85 of their error at these sizes)
            plain = _run(a, w, bias, r if res else None, act, live, False, dev)
            assert "linear_dma_kernel" in _lib.last_kernel()
            assert float((got - want).norm()) <= float((plain - want).norm()) * 1.02


@pytest.mark.parametrize("scale_a,scale_w", [(1e-30, 1.0), (1e-18, 1e-18), (1e30, 1e-3), (1.0, 1e-35), (1e18, 1e18),
                                             (2.0 ** -120, 2.0 ** 60), (2.0 ** 60, 2.0 ** -120)])
def test_magnitudes(dev, scale_a, scale_w):
    """Every magnitude whose product is an fp32 number comes out with fp32's relative error, also where the smaller bf16
    parts of the operands fall below the smallest bf16 numbers."""
    g = torch.Generator(dev).manual_seed(5)
    a, w = torch.randn(8300, 192, generator=g, device=dev) * scale_a, torch.randn(192, 192, generator=g, device=dev) * scale_w
    got = _run(a, w, None, None, "none", 8300, True, dev)
    want = a.double() @ w.double().T
    assert float((got.double() - want).norm() / want.norm()) <= 1e-6


@pytest.mark.parametrize("K", [192, 768])
def test_partial_products_left_out_add_up(dev, K):
    """All operands just below 1 + 2^-8, where the second and third part are largest and of opposite signs: the three partial
    products that are left out are 2^-24 of every product, all on one side.  Beside them one rounding of the sum for each of
    the 6 K / 16 instructions that make it."""
    x = 1.0038986
    a, w = torch.full((16500, K), x, device=dev), torch.full((192, K), x, device=dev)
    got = _run(a, w, None, None, "none", 16500, True, dev)
    want = K * float(a[0, 0].double()) ** 2
    assert float((got.double() - want).abs().max()) <= (1 + 6 * K / 16) * 2.0 ** -24 * want


def test_values_outside_the_split(dev):
    """Infinities, NaN and numbers that round to infinity in bf16: the same results as on the fp32 instructions, in the
    rows and columns that hold them and beside them."""
    g = torch.Generator(dev).manual_seed(6)
    a, w = torch.randn(8300, 192, generator=g, device=dev), torch.randn(192, 192, generator=g, device=dev)
    a[5, 7], a[70, 0], a[71, 191], a[4000, 3] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[:, 3] *= 1e-3
    w[100, 9] = float("inf")
    w[130, :] = 0.0
    got, plain = (_run(a, w, None, None, "none", 8300, s, dev) for s in (True, False))
    assert torch.equal(got.isnan(), plain.isnan()) and torch.equal(got.isinf(), plain.isinf())
    assert torch.equal(got[got.isinf()], plain[plain.isinf()])
    ok = got.isfinite()
    # sums of 192 products in another order: 192 roundings of the largest partial sum either way
    assert bool(((got - plain).abs()[ok] <= 2 * 192 * 2 ** -24 * (a.abs().clamp_max(3.4e38).nan_to_num().double()
                                                                  @ w.abs().clamp_max(3.4e38).double().T)[ok]).all())


def test_gelu_of_special_values(dev):
    """The fp32 GELU at zero, infinities, NaN and the ends of its polynomial, against float64 (a relative error of 2e-6, which
    exp(-x^2/2) has at |x| = 6 from the rounding of its argument)."""
    from vtpack_amd import ops
    x = torch.tensor([0.0, -0.0, 1e-30, -1e-30, 0.5, -0.5, 1.0, -1.0, 3.0, -3.0, 6.0, -6.0, 12.0, 20.0, 3e38, float("inf"),
                      float("nan"), -20.0, -3e38, float("-inf")], device=dev)
    a = torch.zeros(x.numel(), 4, device=dev)
    a[:, 0] = x
    got = ops.linear(a, torch.eye(4, device=dev), act="gelu")[:, 0]
    want = torch.nn.functional.gelu(x.double())
    assert bool(got[15].isinf()) and bool(got[16].isnan()) and bool(got[19].isnan())
    assert bool(((got - want)[:15].abs() <= 2e-6 * want[:15].abs()).all())
    assert bool((got[17:19].abs() <= 1e-30).all())
