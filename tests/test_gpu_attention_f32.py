"""fp32 attention of packed queries (16-query tiles, four a workgroup, waves that share a tile splitting its keys) at
the sizes where its tiling turns: key counts around a block of 16 and a stage of 32, query counts around a tile, a pair
of tiles and a workgroup of four, and key counts that leave some parts of a split without a key."""
import numpy as np
import pytest
import torch

from oracle import dge_oracle as orc
from util import assert_close, randn, rng

pytestmark = pytest.mark.gpu

LENGTHS = [1, 0, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 97, 128, 200]


def _run(dev, q, k, v, lengths, scale):
    from vtpack_amd import _C
    got = _C.batched_sparse_attention_forward(*(torch.from_numpy(t).to(dev) for t in (q, k, v)),
                                              torch.from_numpy(lengths), scale)
    return got.cpu()


@pytest.mark.parametrize("d", [64, 32])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 48, 63, 64, 65, 128, 129, 257, 300])
def test_tiles_and_key_stages(dev, n, d):
    h = 3
    lengths = rng(900 + n).permutation(np.array(LENGTHS, dtype=np.int64))
    L, B = int(lengths.sum()), len(lengths)
    q, k, v = randn(901, h, L, d), randn(902, h, B, n, d), randn(903, h, B, n, d)
    assert_close(_run(dev, q, k, v, lengths, d ** -0.5), orc.attention(q, k, v, lengths, d ** -0.5), torch.float32,
                 f"fp32 attention over {n} keys")


@pytest.mark.parametrize("shape", ["ramp", "late spike", "early spike", "steps", "stage"])
def test_scores_far_above_the_first_stage(dev, shape):
    """Running maxima that keep rising, one key hundreds above the rest, and jumps of 60 between every second and the
    next stage or from one stage of 32 keys to the next, for tiles of a wave each (200 rows: three
    workgroups of four) and tiles whose keys two waves split (its last 8 rows, 20 and 5)."""
    h, d, n = 2, 64, 257
    lengths = np.array([200, 20, 5], dtype=np.int64)
    q, k, v = 0.05 * randn(910, h, 225, d), 0.05 * randn(911, h, 3, n, d), randn(912, h, 3, n, d)
    j = np.arange(n, dtype=np.float32)
    q[..., 0] = 8.0
    k[..., 0] = {"ramp": 0.25 * j, "late spike": np.where(j == n - 7, 300.0, 0.0),
                 "early spike": np.where(j == 5, 300.0, 0.0), "steps": 60.0 * np.floor(j / 64),
                 "stage": np.where(j < 32, -60.0, 0.0)}[shape]
    got = _run(dev, q, k, v, lengths, 0.125)
    assert bool(torch.isfinite(got).all())
    # scores reach 300: their fp32 rounding (300 x 2^-24 in the exponent, both sides) is 4e-5 of a probability
    want = orc.attention(q, k, v, lengths, 0.125)
    assert float((got - torch.from_numpy(want)).abs().max()) <= 4e-5 * np.abs(want).max()


@pytest.mark.parametrize("scale", [0.0, -0.5])
def test_scale_zero_and_negative(dev, scale):
    lengths = np.array([30, 70], dtype=np.int64)
    q, k, v = randn(920, 1, 100, 64), randn(921, 1, 2, 40, 64), randn(922, 1, 2, 40, 64)
    assert_close(_run(dev, q, k, v, lengths, scale), orc.attention(q, k, v, lengths, scale), torch.float32, "scale")


@pytest.mark.parametrize("rows", [1, 20, 64])
def test_first_stages_without_a_finite_score(dev, rows):
    """Scores that overflow to -infinity over the first 70 keys (more than two stages): probability zero, the rest as usual."""
    n = 150
    q, k, v = randn(930, 1, rows, 64), randn(931, 1, 1, n, 64), randn(932, 1, 1, n, 64)
    q[:, ::2, 0], k[:, :, :, 0] = 1e30, 0.0
    k[:, :, :70, 0] = -1e30
    q[:, 1::2, 0] = 0.0                                     # every other query sees all keys
    got = _run(dev, q, k, v, np.array([rows], dtype=np.int64), 0.125)
    s = np.einsum("hld,hnd->hln", q[..., 1:].astype(np.float64), k[:, 0, :, 1:].astype(np.float64)) * 0.125
    s[:, ::2, :70] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    want = (p / p.sum(-1, keepdims=True)) @ v[:, 0].astype(np.float64)
    assert float(np.abs(got.numpy() - want).max()) <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("d", [64, 32])
def test_keys_far_apart_and_in_reverse(dev, d):
    """Token strides of 2^23 values and more, and negative ones: the same bytes as from dense keys and values."""
    from vtpack_amd import _lib, ops
    h, n, lengths = 2, 37, [20, 70]
    L, B = sum(lengths), len(lengths)
    q, k, v = (torch.from_numpy(randn(940 + i, *s, h * d)).to(dev) for i, s in enumerate([(L,), (B, n), (B, n)]))
    offsets, _ = ops.lengths_to_offsets(torch.tensor(lengths), dev)
    want = ops.sparse_attention(q, k, v, offsets, 0.2, h, max(lengths))
    far = [torch.empty_strided(t.shape, (h * d, 1 << 23, 1), device=dev).copy_(t) for t in (k, v)]
    assert torch.equal(ops.sparse_attention(q, *far, offsets, 0.2, h, max(lengths)), want)
    back = [t.flip(1).contiguous() for t in (k, v)]
    got = torch.empty_like(want)
    _lib.call("vtdge_sparse_attention", q.data_ptr(), h * d, d, *(t[0, n - 1].data_ptr() for t in back), n * h * d, -h * d, d,
              offsets.data_ptr(), got.data_ptr(), h * d, d, B, h, d, n, max(lengths), 0.2, _lib.F32, _lib.stream_ptr())
    assert torch.equal(got, want)
