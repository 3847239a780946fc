"""fp32 attention of many pairs, on the bf16 matrix instructions with operands split in three: at the sizes where its tiling
turns, against float64, and with what the split does not cover, which the fp32 instructions have to give as before."""
import math

import pytest
import torch

from util import randn

pytestmark = pytest.mark.gpu

LENGTHS = [1, 0, 16, 17, 32, 33, 47, 48, 49, 63, 64, 65, 96, 97, 113, 128, 129, 200]
HEADS = 20                                 # 360 pairs of up to four workgroups: beyond the line from 34 keys on


def _inputs(dev, n, lengths, h=HEADS):
    L, B = sum(lengths), len(lengths)
    return [torch.from_numpy(randn(950 + i, *shape)).to(dev) for i, shape in enumerate([(L, h * 64), (B, n, h * 64), (B, n, h * 64)])]


def _run(q, k, v, lengths, h=HEADS, scale=0.125, split=True):
    from vtpack_amd import _lib, ops
    offsets, _ = ops.lengths_to_offsets(torch.tensor(lengths), q.device)
    out = ops.sparse_attention(q, k, v, offsets, scale, h, max(lengths))
    assert ("attention_f32_split_kernel<" if split else "attention_f32_kernel<64") in _lib.last_kernel()
    return out


def _alone(q, k, v, lengths, sample, h=HEADS):
    """One sample by itself: few pairs, so the fp32 instructions."""
    at = sum(lengths[:sample])
    return _run(q[at:at + lengths[sample]].contiguous(), k[sample:sample + 1].contiguous(), v[sample:sample + 1].contiguous(),
                lengths[sample:sample + 1], h, split=False)


def _float64(q, k, v, lengths, h=HEADS, scale=0.125):
    out, at = [], 0
    for b, m in enumerate(lengths):
        qb, kb, vb = (t.cpu().double().reshape(-1, h, 64).transpose(0, 1) for t in (q[at:at + m], k[b], v[b]))
        out.append((torch.softmax(qb @ kb.transpose(1, 2).contiguous() * scale, -1) @ vb).transpose(0, 1).reshape(m, h * 64))
        at += m
    return torch.cat(out)


@pytest.mark.parametrize("n", [34, 48, 63, 64, 65, 96, 97, 128, 129, 144, 257])
def test_tiles_and_stages(dev, n):
    q, k, v = _inputs(dev, n, LENGTHS)
    got, want = _run(q, k, v, LENGTHS).cpu().double(), _float64(q, k, v, LENGTHS)
    # the scores' fp32 sums (64 products of unit normals, 2^-24 each) in the exponent and the sums behind it: 4.1e-7 over 257
    # keys with the fp32 instructions, 3.7e-7 here
    assert float((got - want).norm() / want.norm()) <= 6e-7


def test_long_chain_of_few_pairs(dev):
    lengths = [70, 3, 130]
    q, k, v = _inputs(dev, 515, lengths, 1)
    got, want = _run(q, k, v, lengths, 1).cpu().double(), _float64(q, k, v, lengths, 1)
    assert float((got - want).norm() / want.norm()) <= 1.2e-6      # 5e-7 over as many keys with the fp32 instructions


def test_short_workgroups_are_those_of_the_fp32_instructions(dev):
    lengths = [32, 20, 64, 1] * 6
    q, k, v = _inputs(dev, 200, lengths)
    got = _run(q, k, v, lengths)
    for b in (0, 1, 3):
        at = sum(lengths[:b])
        assert torch.equal(got[at:at + lengths[b]], _alone(q, k, v, lengths, b))


def _spoil(what, q, k, v, rows, b):
    """Puts into sample b what the split is not exact for."""
    if what == "infinite value":
        v[b, 40, 3] = float("inf")
    elif what == "nan key":
        k[b, 7, 70] = float("nan")
    elif what == "scores of -infinity":
        q[rows, 0], k[b, :70, 0] = 1.0, -float("inf")
    elif what == "key beyond bf16":
        q[rows, 64], k[b, 5, 64] = 1e-38, 3.4e38                   # 3.4e38 rounds to infinity in bf16
    elif what == "tiny values":
        v[b] *= 1e-36
    elif what == "huge values":
        v[b] *= 1e30
    elif what == "tiny queries, huge keys":
        q[rows] *= 1e-36
        k[b] *= 1e36


@pytest.mark.parametrize("what", ["infinite value", "nan key", "scores of -infinity", "key beyond bf16", "tiny values",
                                  "huge values", "tiny queries, huge keys"])
def test_what_the_split_does_not_cover(dev, what):
    lengths = [113, 70, 200, 64] * 5
    q, k, v = _inputs(dev, 130, lengths)
    clean = _run(q, k, v, lengths)
    b, at = 2, 183
    rows = slice(at, at + 200)
    _spoil(what, q, k, v, rows, b)
    got, want = _run(q, k, v, lengths), _alone(q, k, v, lengths, b)
    assert torch.equal(got[:at], clean[:at]) and torch.equal(got[at + 200:], clean[at + 200:])
    # heads without anything odd in them stay on the bf16 instructions
    finite = want.isfinite()
    assert torch.equal(got[rows].isnan(), want.isnan()) and torch.equal(got[rows].isinf(), want.isinf())
    err = (got[rows] - want)[finite].double()
    assert float(err.norm()) <= 1.5e-6 * float(want[finite].double().norm())


@pytest.mark.parametrize("below", [90, 104, 112, 118, 124])
@pytest.mark.parametrize("size", [2.0 ** 30, 2.0 ** 60, 2.0 ** 100])
def test_large_values_of_improbable_keys(dev, below, size):
    """Probabilities of 2^-`below` lose parts under the smallest bf16 number, which shows where the keys that matter have no
    values to add.  The rounding of scores of some 80 in the exponent leaves 4e-6 of each probability, over 129 of them less."""
    lengths = [113, 70, 200, 64] * 5
    q, k, v = _inputs(dev, 130, lengths)
    q.zero_()
    q[:, ::64] = 1.0
    k[:, :, ::64] = -8 * math.log(2) * (below + torch.rand(20, 130, HEADS, generator=torch.Generator().manual_seed(below))).to(dev)
    k[:, 0, ::64] = 0.0
    v *= size
    v[:, 0] = 0.0
    got, want = _run(q, k, v, lengths).cpu().double(), _float64(q, k, v, lengths)
    assert float((got - want).norm() / want.norm()) <= 4e-6


def test_keys_far_apart_and_in_reverse(dev):
    """Token strides of 2^23 values and negative ones, for both kinds of workgroups: the same bytes as from dense operands."""
    from vtpack_amd import _lib, ops
    n, lengths, h = 70, [113, 20, 64] * 6, HEADS
    q, k, v = _inputs(dev, n, lengths)
    v[0, 30, 2] = float("inf")                          # and for a workgroup that starts again
    want = _run(q, k, v, lengths)
    far = [torch.empty_strided(t.shape, (h * 64, 1 << 23, 1), device=dev).copy_(t) for t in (k, v)]
    got = _run(q, *far, lengths)
    assert "attention_f32_split_kernel<true>" in _lib.last_kernel()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    offsets, _ = ops.lengths_to_offsets(torch.tensor(lengths), dev)
    back = [t.flip(1).contiguous() for t in (k, v)]
    _lib.call("vtdge_sparse_attention", q.data_ptr(), h * 64, 64, *(t[0, n - 1].data_ptr() for t in back), n * h * 64, -h * 64, 64,
              offsets.data_ptr(), got.data_ptr(), h * 64, 64, len(lengths), h, 64, n, max(lengths), 0.125, _lib.F32,
              _lib.stream_ptr())
    assert "attention_f32_split_kernel<true>" in _lib.last_kernel()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
