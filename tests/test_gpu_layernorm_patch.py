"""LayerNorm inside the Linear over blocks of tokens, against the two operators it stands for: the normalised tokens are the
LayerNorm's bit for bit, so what is left is the order of fp32 sums and one rounding, bounded beside the comparison.  Sizes
around a workgroup's 32 rows, with steps of two and four tokens, two steps in all and many."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W,C,P", [(1, 8, 8, 64, 8), (31, 8, 8, 64, 8), (33, 8, 8, 64, 8), (3, 24, 20, 64, 4),
                                       (2, 36, 24, 64, 12), (2, 12, 8, 128, 4), (5, 12, 14, 128, 2), (1, 16, 16, 128, 8),
                                       (8, 32, 32, 128, 4), (96, 64, 64, 64, 8)])
def test_layernorm_inside_the_spatial_reduction(dev, B, H, W, C, P):
    from vtpack_amd import _lib
    lib = _lib.load()
    assert lib.vtdge_layernorm_patch_linear_fits(B, H, W, C, P, _lib.BF16) == 1
    g = torch.Generator(dev).manual_seed(B + H + P)
    K, rows = P * P * C, B * (H // P) * (W // P)
    x = (torch.randn(B, H * W, C, generator=g, device=dev) * 2 + 3 * torch.randn(B, H * W, 1, generator=g, device=dev)).bfloat16()
    x[0, 0] = 1.5                                                        # a token without variance
    nw, nb = ((torch.randn(C, generator=g, device=dev) * 0.3 + i).bfloat16() for i in (1, 0))
    w = (torch.randn(C, K, generator=g, device=dev) / K ** 0.5).bfloat16()
    b = torch.randn(C, generator=g, device=dev).bfloat16()
    out, norm = (torch.full((rows + 1, C), 7.0, device=dev, dtype=torch.bfloat16) for _ in range(2))
    packed = torch.full((2 * w.numel() + 8,), 7.0, device=dev, dtype=torch.bfloat16)
    two = (ctypes.c_void_p * 2)(torch.zeros_like(w).data_ptr(), w.data_ptr())
    _lib.call("vtdge_layernorm_patch_pack", ctypes.cast(two, ctypes.c_void_p), 2, packed.data_ptr(), C, P, _lib.stream_ptr())
    for to, n2 in ((out, (0, 0)), (norm, (nw.data_ptr(), nb.data_ptr()))):
        _lib.call("vtdge_layernorm_patch_linear", x.data_ptr(), nw.data_ptr(), nb.data_ptr(), 1e-6,
                  packed.data_ptr() + w.numel() * 2, b.data_ptr(), *n2, 1e-5, to.data_ptr(), B, H, W, C, P, _lib.BF16,
                  _lib.stream_ptr())
    assert (out[rows:] == 7).all() and (norm[rows:] == 7).all() and (packed[2 * w.numel():] == 7).all()    # nothing past the end
    # the rows' own LayerNorm: the operator's on the rows it stands for, bit for bit
    want = torch.empty_like(out[:rows])
    _lib.call("vtdge_layernorm", out.data_ptr(), nw.data_ptr(), nb.data_ptr(), want.data_ptr(), None, rows, C, 1e-5, _lib.BF16,
              _lib.stream_ptr())
    assert torch.equal(norm[:rows], want)
    ln = torch.empty_like(x)
    _lib.call("vtdge_layernorm", x.data_ptr(), nw.data_ptr(), nb.data_ptr(), ln.data_ptr(), None, B * H * W, C, 1e-6, _lib.BF16,
              _lib.stream_ptr())
    a = ln.reshape(B, H // P, P, W // P, P, C).permute(0, 1, 3, 2, 4, 5).reshape(rows, K).double().cpu()
    w64 = w.double().cpu()
    want = a @ w64.t() + b.double().cpu()
    # K fp32 sums in any order, each within 2^-24 of the sum of magnitudes so far, and one rounding to 8 bits
    bound = K * 2.0 ** -24 * (a.abs() @ w64.abs().t()) + want.abs() * 2.0 ** -8
    assert ((out[:rows].double().cpu() - want).abs() <= bound).all()


@pytest.mark.parametrize("args,fits", [((4, 64, 64, 64, 8), 1), ((4, 64, 64, 64, 2), 0), ((4, 64, 64, 320, 2), 0),
                                       ((4, 60, 64, 64, 8), 0), ((4, 12, 12, 128, 3), 0)])
def test_what_it_takes(args, fits):
    from vtpack_amd import _lib
    lib = _lib.load()
    assert lib.vtdge_layernorm_patch_linear_fits(*args, _lib.BF16) == fits
    assert lib.vtdge_layernorm_patch_linear_fits(*args, _lib.F32) == 0
    assert lib.vtdge_layernorm_patch_linear_wanted(*args, _lib.BF16) == 0            # few rows
    assert lib.vtdge_layernorm_patch_linear_wanted(256, *args[1:], _lib.BF16) == fits
