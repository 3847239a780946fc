"""The Linear for few rows (32x32 tiles, K split over the waves of a workgroup) at its edges: rows and columns around a
tile, one slab of K up to more than the ring holds, and the LayerNorm inside it for every way a row can lie in a wave
(8 to 128 16-byte vectors).  Each against fp64 and, with the LayerNorm, bit for bit against the LayerNorm kernel followed
by the same Linear."""
import pytest
import torch
import torch.nn.functional as F

from util import FP32_REL, rel_err

pytestmark = pytest.mark.gpu
# bf16 results are rounded once (2^-9 of the value, against the largest one of the result)
TOL = {torch.float32: FP32_REL, torch.bfloat16: 2.0 ** -8}


def _make(dev, dtype, seed, *shapes):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(s, generator=g).to(dtype).to(dev) for s in shapes]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("live,cap", [(0, 40), (1, 1), (31, 40), (32, 32), (33, 70), (65, 300)])
@pytest.mark.parametrize("N", [4, 32, 36, 1000])
@pytest.mark.parametrize("slabs", [1, 3, 8, 9, 24, 40])
def test_linear_edges(dev, dtype, live, cap, N, slabs):
    from vtpack_amd import _lib, ops
    K = slabs * 128 // torch.empty((), dtype=dtype).element_size()
    a, w, b, r = _make(dev, dtype, live + N + slabs, (cap, K), (N, K), (N,), (cap, N))
    w = w / K ** 0.5
    rd = torch.tensor([live], dtype=torch.int64, device=dev)
    for act, bias, res in (("none", b, r), ("gelu", b, None), ("none", None, None)):
        out = torch.full((cap, N), 7.0, device=dev, dtype=dtype)
        ops.linear(a, w, bias, residual=res, act=act, rows_dev=rd, out=out)
        assert "linear_small" in _lib.last_kernel()
        want = a[:live].double() @ w.double().T + (0 if bias is None else bias.double())
        want = F.gelu(want) if act == "gelu" else want
        want = want + r[:live].double() if res is not None else want
        if live:
            assert rel_err(out[:live], want) <= TOL[dtype]
        assert bool((out[live:] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("vecs", [8, 16, 24, 32, 40, 64, 96, 128])
@pytest.mark.parametrize("rows,live", [(1, 1), (37, 33), (129, 64)])
def test_layernorm_inside(dev, dtype, vecs, rows, live):
    from vtpack_amd import _lib, ops
    C = vecs * 16 // torch.empty((), dtype=dtype).element_size()
    x, c, wk, wq, w1, bk, bq, b1, g, b = _make(dev, dtype, vecs + rows, (rows, C), (rows, C), (2 * C, C), (C, C), (256, C),
                                               (2 * C,), (C,), (256,), (C,), (C,))
    x = x + 3                                       # a mean that is not small beside the spread
    rd = torch.tensor([live], dtype=torch.int64, device=dev)
    assert ops.fits_layernorm_linear(x, wk, c, wq) and ops.fits_layernorm_linear(c, w1)
    k, q = ops.layernorm_linear(x, wk, bk, g, b, 1e-6, second=(c, wq, bq, rd))
    f = ops.layernorm_linear(c, w1, b1, g, b, 1e-6, act="gelu", rows_dev=rd)
    assert "linear_small" in _lib.last_kernel()
    xn, cn = ops.layernorm(x, g, b, 1e-6), ops.layernorm(c, g, b, 1e-6)
    assert torch.equal(k, ops.linear(xn, wk, bk))
    assert torch.equal(q[:live], ops.linear(cn, wq, bq)[:live])
    assert torch.equal(f[:live], ops.linear(cn, w1, b1, act="gelu")[:live])
    ref = F.layer_norm(x.double(), (C,), g.double(), b.double(), 1e-6).to(dtype).double() @ wk.double().T + bk.double()
    assert rel_err(k, ref) <= TOL[dtype] + (2.0 ** -8 if dtype == torch.bfloat16 else 0)   # LayerNorm(x) rounded first


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N0,N1", [(64, 128, 64), (192, 36, 192), (512, 1024, 512)])
@pytest.mark.parametrize("rows,live", [(1, 1), (37, 0), (129, 64)])
def test_two_products_in_one_launch(dev, dtype, K, N0, N1, rows, live):
    from vtpack_amd import _lib, ops
    x, c, w0, w1, b0 = _make(dev, dtype, K + rows, (rows, K), (rows, K), (N0, K), (N1, K), (N0,))
    rd = torch.tensor([live], dtype=torch.int64, device=dev)
    k, q = (torch.full((rows, n), 7.0, device=dev, dtype=dtype) for n in (N0, N1))
    _lib.call("vtdge_linear_pair", x.data_ptr(), K, w0.data_ptr(), b0.data_ptr(), k.data_ptr(), 0, rows, N0, c.data_ptr(), K,
              w1.data_ptr(), 0, q.data_ptr(), rd.data_ptr(), rows, N1, K, _lib.dtype_code(x), _lib.stream_ptr())
    assert "linear_small" in _lib.last_kernel()
    assert torch.equal(k, ops.linear(x, w0, b0))
    assert torch.equal(q[:live], ops.linear(c, w1)[:live])
    assert bool((q[live:] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,C,k,N", [(1, 8, 64, 2, 32), (3, 8, 64, 8, 64), (2, 4, 128, 1, 8), (5, 12, 64, 4, 40)])
def test_strided_convolution_of_few_rows(dev, dtype, B, H, C, k, N):
    from vtpack_amd import _lib, ops
    x, w, b = _make(dev, dtype, C + k, (B, H * H, C), (N, C, k, k), (N,))
    w = w / (C * k * k) ** 0.5
    got = ops.patch_linear(x, H, H, k, w.permute(0, 2, 3, 1).reshape(N, -1).contiguous(), b)
    assert "linear_small" in _lib.last_kernel()
    want = F.conv2d(x.double().cpu().transpose(1, 2).reshape(B, C, H, H), w.double().cpu(), b.double().cpu(), stride=k)
    assert rel_err(got, want.flatten(2).transpose(1, 2).reshape(-1, N)) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,P,N,extra", [(1, 64, 16, 96, 1), (3, 32, 8, 64, 2), (2, 48, 16, 36, 0)])
def test_patch_embedding_of_few_rows(dev, dtype, B, S, P, N, extra):
    from vtpack_amd import _lib, ops
    N = N // 8 * 8
    G = S // P
    img, w, b, pos = _make(dev, dtype, S + P, (B, 3, S, S), (N, 3, P, P), (N,), (extra + G * G, N))
    w = w / (3 * P * P) ** 0.5
    out = torch.full((B, extra + G * G, N), 7.0, device=dev, dtype=dtype)
    ops.patch_embed(img, w, b, pos, P, extra, out=out)
    assert "linear_small" in _lib.last_kernel()
    want = F.conv2d(img.double().cpu(), w.double().cpu(), b.double().cpu(), stride=P).flatten(2).transpose(1, 2)
    assert rel_err(out[:, extra:], want + pos[extra:].double().cpu()) <= TOL[dtype]
    assert bool((out[:, :extra] == 7.0).all())


@pytest.mark.parametrize("dtype,rows,N,K,small", [
    (torch.bfloat16, 257, 1536, 384, True), (torch.bfloat16, 1339, 1536, 384, False), (torch.bfloat16, 1285, 768, 768, True),
    (torch.bfloat16, 2715, 768, 768, False), (torch.bfloat16, 4091, 320, 1280, False), (torch.float32, 1339, 768, 768, True),
    (torch.float32, 7451, 192, 192, False)])
def test_packed_rows_are_counted_as_if_all_were_live(dev, dtype, rows, N, K, small):
    """An untrained router leaves every row live: the rule must not count on half of them being absent."""
    from vtpack_amd import _lib, ops
    a, w, b = _make(dev, dtype, rows, (rows, K), (N, K), (N,))
    w = w / K ** 0.5
    live = rows - 3
    out = torch.full((rows, N), 7.0, device=dev, dtype=dtype)
    ops.linear(a, w, b, rows_dev=torch.tensor([live], device=dev), out=out)
    assert ("linear_small" if small else "linear_dma") in _lib.last_kernel()
    assert rel_err(out[:live], a[:live].double() @ w.double().T + b.double()) <= TOL[dtype]
    assert bool((out[live:] == 7.0).all())
