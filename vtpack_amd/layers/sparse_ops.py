"""Variable-length batched operators (mirror of vtpack/layers/sparse_ops.py:11-78)."""
import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable

from .. import _C, ops


class _SparseGEMM(Function):
    # vtpack/layers/sparse_ops.py:11-54; the backward is four more forward calls, as in the reference.
    @staticmethod
    def forward(ctx, a, b, a_lengths, b_lengths, is_a_transposed, is_b_transposed):
        a, b = a.contiguous(), b.contiguous()
        a_lengths, b_lengths = a_lengths.contiguous(), b_lengths.contiguous()
        ctx.flags = (is_a_transposed, is_b_transposed)
        ctx.save_for_backward(a, b, a_lengths, b_lengths)
        return _C.batched_sparse_gemm_forward(a, b, a_lengths, b_lengths, is_a_transposed, is_b_transposed)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad):
        grad = grad.contiguous()
        a, b, la, lb = ctx.saved_tensors
        ta, tb = ctx.flags
        f = _C.batched_sparse_gemm_forward
        g_a = f(grad, b, la, lb, ta, not tb) if not ta else f(b, grad, lb, la, tb, ta)
        g_b = f(a, grad, la, la, not ta, tb) if not tb else f(grad, a, la, la, tb, ta)
        return g_a, g_b, None, None, None, None


class _SparseAttention(Function):
    # vtpack/layers/sparse_ops.py:60-73 (forward only there as well)
    @staticmethod
    def forward(ctx, q, k, v, q_lengths, scale):
        return _C.batched_sparse_attention_forward(q, k, v, q_lengths, scale)

    @staticmethod
    def backward(ctx, grad):
        raise NotImplementedError("Backward is not implemented.")


batched_sparse_gemm = _SparseGEMM.apply
batched_sparse_attention = _SparseAttention.apply


class _SparseAttentionTrain(Function):
    """Attention of packed queries with gradients, without score-sized tensors: scores are worked out from q and k forward
    and again backward.  q [h, L, d], k and v [h, B, n, d] -> [L, h * d]."""

    @staticmethod
    def forward(ctx, q, k, v, q_lengths, scale, max_rows):
        ops._need_gpu(q, k, v)
        q, k, v = (ops.on_boundary(t) for t in (ops.vector_rows(q), k.contiguous(), v.contiguous()))
        h, L, d = q.shape
        offsets, _ = ops.lengths_to_offsets(q_lengths, q.device)
        out = torch.empty((L, h * d), dtype=q.dtype, device=q.device)
        ctx.scale, ctx.max_rows = scale, max_rows
        ops.sparse_attention_heads(q, k, v, offsets, scale, ctx.max_rows, out=out.view(L, h, d).transpose(0, 1), train=True)
        ctx.save_for_backward(q, k, v, offsets)      # not the result: a caller may change that in place
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, grad):
        q, k, v, offsets = ctx.saved_tensors
        h, L, d = q.shape
        # k and v share their strides in the kernel; a saved-tensor hook may lay them out anew
        q, k, v, grad = (ops.on_boundary(t) for t in (ops.vector_rows(q), *(t.contiguous() for t in (k, v, grad))))
        grad = grad.view(L, h, d).transpose(0, 1)
        dq, dk, dv = ops.sparse_attention_backward(q, k, v, None, grad, offsets, ctx.scale, ctx.max_rows)
        return dq, dk, dv, None, None, None


def sparse_attention_train(q, k, v, q_lengths, scale):
    """Differentiable attention of packed queries for the training branch of the models
    (vtpack/models/dge/deit_dge.py:79-95): q [h, L, d]; k, v [h, B, n, d]; -> [L, h*d].

    Equal query counts (dense training: every granularity for every sample) use one batched matmul.  Otherwise, on the GPU
    with head dim 64, one attention kernel forward and two backward; other operands, and a scale that is a tensor (it may want
    a gradient or differ by head), compose two `batched_sparse_gemm` calls around a softmax over the keys."""
    h, L, d = q.shape
    B, n = k.shape[1], k.shape[2]
    counts = q_lengths.flatten().tolist()
    if max(counts) == min(counts):
        scores = torch.matmul(q.reshape(h, B, -1, d), k.transpose(-1, -2)) * scale
        ctx = torch.matmul(scores.softmax(dim=-1, dtype=v.dtype), v)              # [h, B, Lq, d]
        return ctx.permute(1, 2, 0, 3).reshape(-1, h * d)
    if (d == 64 and not torch.is_tensor(scale) and q.is_cuda and q.dtype in (torch.float32, torch.bfloat16)
            and q.dtype == k.dtype == v.dtype and k.shape == v.shape and k.shape[0] == h and k.shape[3] == d
            and len(counts) == B and sum(counts) == L):
        return _SparseAttentionTrain.apply(q, k, v, q_lengths, float(scale), int(max(counts)))
    kv_lengths = q_lengths.new_full([B], n)
    scores = batched_sparse_gemm(q, k.reshape(h, -1, d), q_lengths, kv_lengths, False, True) * scale
    ctx = batched_sparse_gemm(scores.softmax(dim=-1, dtype=v.dtype), v.reshape(h, -1, d), q_lengths, kv_lengths,
                              False, False)
    return ctx.transpose(0, 1).reshape(-1, h * d)
