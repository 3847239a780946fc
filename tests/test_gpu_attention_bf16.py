"""bf16 attention of packed queries, head_dim 64, at the key counts and pair counts where its kernels turn."""
import numpy as np
import pytest
import torch

from oracle import dge_oracle as orc
from util import assert_close, bf16_round, randn, rng

pytestmark = pytest.mark.gpu


def _check(dev, h, n, lengths, what):
    from vtpack_amd import _C
    lengths = np.array(lengths, dtype=np.int64)
    L, B = int(lengths.sum()), len(lengths)
    q, k, v = (bf16_round(randn(seed, *shape)) for seed, shape in ((801, (h, L, 64)), (802, (h, B, n, 64)), (803, (h, B, n, 64))))
    got = _C.batched_sparse_attention_forward(*(torch.from_numpy(t).to(dev, torch.bfloat16) for t in (q, k, v)),
                                              torch.from_numpy(lengths), 0.125)
    assert_close(got.float(), orc.attention(q, k, v, lengths, 0.125), torch.bfloat16, what)


@pytest.mark.parametrize("n", [352, 353, 383, 384, 385, 416, 417, 448, 449, 480, 481, 484, 511, 512, 1000])
def test_last_stage_of_streamed_keys(dev, n):
    """The streaming kernel's last stage of one to four blocks of 32 keys, whole and partial."""
    lengths = rng(800 + n).choice([0, 1, 32, 33, 128, 129, 150], size=60)
    _check(dev, 5, n, lengths, f"300 pairs of {n} keys")
