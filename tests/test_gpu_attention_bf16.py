"""bf16 attention of packed queries, head_dim 64, at the key counts and pair counts where its kernels turn."""
import numpy as np
import pytest
import torch

from oracle import dge_oracle as orc
from util import assert_close, bf16_round, randn, rng

pytestmark = pytest.mark.gpu


def _few(n):
    """The kernel of few pairs: a wave for each block of 32 keys up to nine, else eight in turn."""
    return f"sparse_attention_bf16_d64_split_kernel<{-(-n // 32) if n <= 288 else 8}, {str(n > 288).lower()}>"


def _check(dev, h, n, lengths, what, kernel):
    from vtpack_amd import _C, _lib
    lengths = np.array(lengths, dtype=np.int64)
    L, B = int(lengths.sum()), len(lengths)
    q, k, v = (bf16_round(randn(seed, *shape)) for seed, shape in ((801, (h, L, 64)), (802, (h, B, n, 64)), (803, (h, B, n, 64))))
    got = _C.batched_sparse_attention_forward(*(torch.from_numpy(t).to(dev, torch.bfloat16) for t in (q, k, v)),
                                              torch.from_numpy(lengths), 0.125)
    assert kernel in _lib.last_kernel()
    assert_close(got.float(), orc.attention(q, k, v, lengths, 0.125), torch.bfloat16, what)


@pytest.mark.parametrize("n", [352, 353, 383, 384, 385, 416, 417, 448, 449, 480, 481, 484, 511, 512, 1000])
def test_last_stage_of_streamed_keys(dev, n):
    """The streaming kernel's last stage of one to four blocks of 32 keys, whole and partial."""
    lengths = rng(800 + n).choice([0, 1, 32, 33, 128, 129, 150], size=60)
    _check(dev, 5, n, lengths, f"300 pairs of {n} keys", "sparse_attention_bf16_d64_stream_kernel")


# (sample, head) pairs that few workgroups take: the kernel whose waves split the keys.  Every number of blocks (1 .. 9), whole
# and partial, then rounds of eight blocks with a last one that some waves sit out; empty samples, a query more and less than
# a tile, more tiles than a workgroup takes at once.
@pytest.mark.parametrize("lengths,h", [([1, 0, 33], 2), ([257, 32, 96, 0, 31, 150], 3), ([300], 1), ([64] * 85, 1)])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 96, 128, 129, 160, 192, 197, 224, 256, 257, 288, 289, 511, 512, 513, 1025])
def test_few_pairs(dev, n, lengths, h):
    _check(dev, h, n, lengths, f"{h} x {len(lengths)} pairs of {n} keys", _few(n))


def test_few_pairs_many_tiles(dev):
    _check(dev, 2, 144, [1500], "two pairs of 47 tiles", _few(144))


@pytest.mark.parametrize("n", [1, 33, 64, 257, 288])
@pytest.mark.parametrize("h,most,lengths", [(41, 1300, [1300, 0, 257]), (40, 512, [511, 256, 1]), (150, 4000, [3000, 300])])
def test_queries_dealt_out_in_chunks(dev, h, most, lengths, n):
    """The resident kernel with a pair's queries in chunks, some of them empty, and in one piece (the same pairs among so many
    that they fill the chip): a tile's arithmetic is the same, so the results are equal."""
    from vtpack_amd import _C, _lib, ops
    resident = f"sparse_attention_bf16_d64_pipelined_kernel<{-(-n // 32)}, "
    lengths = torch.tensor(lengths, dtype=torch.int64)
    L, B = int(lengths.sum()), len(lengths)
    g = torch.Generator(dev).manual_seed(n)
    q, k, v = (torch.randn(s, generator=g, device=dev).to(torch.bfloat16) for s in ((h, L, 64), (h, B, n, 64), (h, B, n, 64)))
    off, _ = ops.lengths_to_offsets(lengths, q.device)
    got = ops.sparse_attention_heads(q, k, v, off, 0.125, most)
    assert resident + "true>" in _lib.last_kernel()
    times = 1 + 512 // (h * B)
    whole = _C.batched_sparse_attention_forward(q.repeat(times, 1, 1), k.repeat(times, 1, 1, 1), v.repeat(times, 1, 1, 1),
                                                lengths, 0.125)
    assert resident + "false>" in _lib.last_kernel()
    assert torch.equal(got, whole.view(times, h, L, 64)[0]) and torch.equal(whole[-h:], whole[:h])
    want = orc.attention(*(t[:2].float().cpu().numpy() for t in (q, k, v)), lengths.numpy(), 0.125)
    assert_close(got[:2].float(), want, torch.bfloat16, f"{h} x {B} pairs of {n} keys in chunks")


@pytest.mark.parametrize("n", [33, 257])
@pytest.mark.parametrize("lengths", [[511, 512], [512, 512], [0, 1], [4000, 1]])
def test_pairs_of_few_live_rows_stay_whole(dev, lengths, n):
    """300 pairs that may have 4000 rows each, in two chunks from 1024 live rows on, on either side of that: the bits of the same pairs
    among 600, which no rule deals out."""
    from vtpack_amd import _lib, ops
    h, L = 150, sum(lengths)
    g = torch.Generator(dev).manual_seed(n)
    q, k, v = (torch.randn(s, generator=g, device=dev).to(torch.bfloat16) for s in ((h, L, 64), (h, 2, n, 64), (h, 2, n, 64)))
    off, _ = ops.lengths_to_offsets(torch.tensor(lengths), q.device)
    got = ops.sparse_attention_heads(q, k, v, off, 0.125, 4000)
    assert f"pipelined_kernel<{-(-n // 32)}, true>" in _lib.last_kernel()
    twice = ops.sparse_attention_heads(*(torch.cat((t, t)) for t in (q, k, v)), off, 0.125, 4000)
    assert "false>" in _lib.last_kernel() and torch.equal(got, twice[:h]) and torch.equal(got, twice[h:])
    want = orc.attention(*(t[:2].float().cpu().numpy() for t in (q, k, v)), np.array(lengths), 0.125)
    assert_close(got[:2].float(), want, torch.bfloat16, f"{lengths} of {n} keys")


@pytest.mark.parametrize("n", [65, 145, 257, 401, 577])
@pytest.mark.parametrize("size", [1.0, 4.0])
def test_few_pairs_are_as_exact_as_many(dev, n, size):
    """The same pairs alone and among many, which other kernels take: each wave has its own reference for its probabilities, so
    the results differ, and are no further from float64 (0.92 to 0.99 of the distance: 2.6e-3 against 2.8e-3 over 257 keys)."""
    from vtpack_amd import _C, _lib
    h, B, L, times = 3, 2, 64, 50
    q, k, v = (torch.from_numpy(randn(830 + i, *s)).to(dev, torch.bfloat16)
               for i, s in enumerate([(h, B, L, 64), (h, B, n, 64), (h, B, n, 64)]))
    q = q * size
    want = (torch.softmax(q.double() @ k.double().transpose(2, 3).contiguous() * 0.125, -1) @ v.double()).view(h, B * L, 64)
    lengths = torch.full((B,), L, dtype=torch.int64)
    few = _C.batched_sparse_attention_forward(q.view(h, B * L, 64), k, v, lengths, 0.125)
    assert _few(n) in _lib.last_kernel()
    many = _C.batched_sparse_attention_forward(q.repeat(1, times, 1, 1).view(h, -1, 64), k.repeat(1, times, 1, 1),
                                               v.repeat(1, times, 1, 1), lengths.repeat(times), 0.125)[:, :B * L]
    assert "split" not in _lib.last_kernel()
    assert float((few.double() - want).norm()) <= 1.02 * float((many.double() - want).norm())


@pytest.mark.parametrize("n", [257, 700])
@pytest.mark.parametrize("place", [3, 40, 250, 256])
def test_few_pairs_one_key_above_all(dev, n, place):
    """A key hundreds above the others: every wave but its own adds nothing, whichever wave that is."""
    from vtpack_amd import _C
    q, k, v = 0.05 * randn(811, 2, 70, 64), 0.05 * randn(812, 2, 1, n, 64), randn(813, 2, 1, n, 64)
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, :, place, 0] = 300.0
    q, k, v = bf16_round(q), bf16_round(k), bf16_round(v)
    lengths = np.array([70], dtype=np.int64)
    got = _C.batched_sparse_attention_forward(*(torch.from_numpy(t).to(dev, torch.bfloat16) for t in (q, k, v)),
                                              torch.from_numpy(lengths), 0.125)
    assert_close(got.float(), orc.attention(q, k, v, lengths, 0.125), torch.bfloat16, "one key above all")


def test_few_pairs_infinities(dev):
    """Keys whose scores are -infinity count for nothing, in a block of their own too; all of them make NaN, as a softmax of
    nothing does; one of +infinity makes its query NaN."""
    from vtpack_amd import _C
    n, h = 257, 1
    q, k, v = torch.zeros(h, 40, 64), torch.zeros(h, 2, n, 64), torch.from_numpy(randn(821, h, 2, n, 64))
    q[..., 0] = 1.0
    k[:, 0, :100, 0] = -float("inf")
    k[:, 1, :, 0] = -float("inf")
    q[:, 3, 0] = -1.0                                 # sample 0: +infinity
    lengths = torch.tensor([20, 20])
    got = _C.batched_sparse_attention_forward(*(t.to(dev, torch.bfloat16) for t in (q, k, v)), lengths, 0.125).float().cpu()
    want = v.to(torch.bfloat16).float()[:, 0, 100:].mean(1)
    rows = [i for i in range(20) if i != 3]
    assert float((got[:, rows] - want).abs().max()) <= 4e-3 * float(want.abs().max())
    assert bool(got[:, 3].isnan().all()) and bool(got[:, 20:].isnan().all())
