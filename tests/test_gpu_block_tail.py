"""Projection, LayerNorm and MLP of the packed queries as one kernel, against the same steps in float64 with the roundings the
modules make: row counts around a wave's 32 rows and a workgroup's, live counts below the capacity, biases present or not."""
import pytest
import torch

from util import randn

pytestmark = pytest.mark.gpu


def _bf(t):
    return t.to(torch.bfloat16).double()


@pytest.mark.parametrize("C", [64, 128, 192])
@pytest.mark.parametrize("hidden", [64, 192, 512])
@pytest.mark.parametrize("rows,live", [(1, 1), (31, 31), (33, 32), (128, 127), (129, 129), (700, 0), (3000, 1025)])
@pytest.mark.parametrize("bias", [True, False])
def test_against_float64(dev, C, hidden, rows, live, bias):
    from vtpack_amd import ops
    g = [torch.from_numpy(randn(i, *s)).to(torch.bfloat16) for i, s in enumerate(
        [(rows, C), (rows, C), (C, C), (C,), (C,), (C,), (hidden, C), (hidden,), (C, hidden), (C,)])]
    for i, k in ((2, C), (6, C), (8, hidden)):
        g[i] = (g[i].float() * k ** -0.5).to(torch.bfloat16)
    o, comp, wp, bp, lw, lb, w1, b1, w2, b2 = [t.to(dev) for t in g]
    nb = [None] * 3 if not bias else [bp, b1, b2]
    got = torch.full_like(o, 7.0)
    ops.block_tail(o, comp, (wp, nb[0]), (lw, lb), 1e-5, (w1, nb[1]), (w2, nb[2]),
                   rows_dev=torch.tensor([live], device=dev), out=got)
    assert bool((got[live:] == 7.0).all())                 # rows past the live ones are not written
    o, comp, wp, bp, lw, lb, w1, b1, w2, b2 = [t.double() for t in g]
    if not bias:
        bp, b1, b2 = bp * 0, b1 * 0, b2 * 0
    q1 = _bf(o @ wp.T + bp + comp)
    ln = _bf(torch.nn.functional.layer_norm(q1, (C,), lw, lb, 1e-5))
    want = q1 + _bf(torch.nn.functional.gelu(ln @ w1.T + b1)) @ w2.T + b2
    if live == 0:
        return
    # q1, the normalised rows and the hidden rows may round the other way (2^-8 of one of them): a term of that size in sums
    # of products that are about one
    err = (got.double().cpu() - want)[:live].abs().max()
    assert float(err) <= 2e-2 * float(want.abs().max())
    rms = ((got.double().cpu() - want)[:live].pow(2).mean() / want[:live].pow(2).mean()).sqrt()
    assert float(rms) <= 4e-3


def test_what_it_does_not_take(dev):
    from vtpack_amd import _lib, ops
    lib = _lib.load()
    assert [lib.vtdge_block_tail_fits(64, c, h, _lib.BF16) for c, h in ((64, 64), (128, 4096), (96, 64), (64, 96), (64, 4160))] \
        == [1, 1, 0, 0, 0]
    assert [lib.vtdge_block_tail_wanted(r, c, 64, _lib.BF16) for r, c in ((1023, 64), (1024, 64), (8191, 192), (8192, 192))] == [
        0, 1, 0, 1]
    t = torch.zeros(2048, 64, dtype=torch.bfloat16, device=dev)
    w = torch.zeros(64, 64, dtype=torch.bfloat16, device=dev)
    v = torch.zeros(65, dtype=torch.bfloat16, device=dev)
    assert ops.fits_block_tail(t, (w, None), (v[:64], v[:64]), (w, None), (w, None))
    assert not ops.fits_block_tail(t, (w, v[1:]), (v[:64], v[:64]), (w, None), (w, None))
    with pytest.raises(RuntimeError):
        ops.block_tail(t, t, (w, v[1:]), (v[:64], v[:64]), 1e-5, (w, None), (w, None))
