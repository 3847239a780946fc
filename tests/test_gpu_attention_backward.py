"""Gradients of the packed-query attention against float64 autograd through the same composition: query counts around a
tile of 16, a stage of 32 and a workgroup of 64, samples without queries, key counts with a partial last tile and stage."""
import numpy as np
import pytest
import torch

from util import randn

pytestmark = pytest.mark.gpu
# fp32: sums of a few hundred products, 4e-6 of the largest gradient seen; bf16: P and dS are rounded to bf16 (2^-9 each)
# and the operands of delta too
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2}


def _reference(q, k, v, lengths, scale, g):
    q, k, v = (t.double().requires_grad_(True) for t in (q, k, v))
    outs, at = [], 0
    for b, n in enumerate(lengths):
        qb = q[:, at:at + n]
        p = torch.softmax(qb @ k[:, b].transpose(1, 2).contiguous() * scale, dim=-1)
        outs.append((p @ v[:, b]).permute(1, 0, 2).reshape(n, q.shape[0] * q.shape[2]))
        at += n
    out = torch.cat(outs)
    return out.detach(), torch.autograd.grad(out, (q, k, v), g.double())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 15, 33, 64, 65, 257])
@pytest.mark.parametrize("lengths", [[1, 2], [16, 0, 17, 31], [64, 65, 33, 5, 130]])
@pytest.mark.parametrize("scale,dense", [(0.125, False), (-0.3, True)])
def test_against_float64(dev, dtype, n, lengths, scale, dense):
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, d, L, B = 3, 64, sum(lengths), len(lengths)
    packed = torch.from_numpy(randn(n, L, h, d)).to(dtype)
    q = packed.transpose(0, 1).contiguous() if dense else packed.transpose(0, 1)
    k, v = (torch.from_numpy(randn(s + n, h, B, n, d)).to(dtype) for s in (1, 2))
    g = torch.from_numpy(randn(3 + n, L, h * d)).to(dtype)
    want, grads = _reference(q, k, v, lengths, scale, g)
    args = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    got = sparse_attention_train(*args, torch.tensor(lengths), scale)
    again = torch.autograd.grad(got, args, g.to(dev), retain_graph=True)
    assert float((got.detach().double().cpu() - want).abs().max()) <= TOL[dtype] * float(want.abs().max())
    for name, a, b in zip("qkv", torch.autograd.grad(got, args, g.to(dev)), grads):
        # dS is P (dP - delta) scale: two sums of 64 products of unit normals (3 sigma: 24) that cancel, entirely where
        # there is one key; what their rounding leaves is relative to them, not to what remains
        size = max(float(b.abs().max()), 24 * abs(scale) if name != "v" else 0)
        assert float((a.double().cpu() - b).abs().max()) <= TOL[dtype] * size, name
    assert all(torch.equal(a, b) for a, b in zip(again, torch.autograd.grad(sparse_attention_train(
        *args, torch.tensor(lengths), scale), args, g.to(dev))))                      # the same bytes on every call


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("common", [1.0, 2.0])
def test_keys_and_values_with_a_common_component(dev, dtype, common):
    """What a kv bias gives: every key and every value shifted by the same vector.  A row of dS adds up to zero, so the
    gradients do not see the shift; an error in delta would reach dQ times the mean key.  bf16: dS is rounded once, 2^-9 at
    most and 2^-9 / sqrt(3) rms, and multiplies keys sqrt(1 + common^2) times as large as what remains of them: 2.5e-3 of
    dQ at common = 2; bound: four times that."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, n, lengths = 3, 257, [113, 17, 64]
    L, B = sum(lengths), len(lengths)
    q, g = (torch.from_numpy(randn(s, L, h * 64)).to(dtype) for s in (1, 4))
    q = q.view(L, h, 64).transpose(0, 1)
    k, v = (torch.from_numpy(randn(s, h, B, n, 64) + common * randn(s + 7, h, 1, 1, 64)).to(dtype) for s in (2, 3))
    want, grads = _reference(q, k, v, lengths, 0.125, g)
    args = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    got = sparse_attention_train(*args, torch.tensor(lengths), 0.125)
    for name, a, b in zip("qkv", torch.autograd.grad(got, args, g.to(dev)), grads):
        assert float((a.double().cpu() - b).norm()) <= (1e-5 if dtype == torch.float32 else 1e-2) * float(b.norm()), name


@pytest.mark.parametrize("size,common", [(1.0, 0.0), (4.0, 0.0), (16.0, 0.0), (1.0, 2.0)])
def test_fp32_gradients_are_as_exact_as_the_composition(dev, size, common):
    """Against float64, beside a softmax and products in fp32 on the same operands.  Rounding m + log2(s) at its own size would
    put 2e-7 into every P of a row, 1.4 times the composition's error of dV at size = 1; an exponent that is rounded before the
    subtraction in one pass and not in the other, as much at size = 16; sums of e dP key by key, 1.6 times its error of dQ at
    common = 2.  Bound: a tenth above the composition, for the spread of two rms errors over 324 rows, 1 / sqrt(2 * 324) each."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, n, lengths = 3, 257, [113, 17, 64, 130]
    L, B = sum(lengths), len(lengths)
    q, g = (torch.from_numpy(f * randn(s, L, h * 64)) for s, f in ((1, size), (4, 1.0)))
    q = q.view(L, h, 64).transpose(0, 1)
    k, v = (torch.from_numpy(randn(s, h, B, n, 64) + common * randn(s + 7, h, 1, 1, 64)) for s in (2, 3))
    want, grads = _reference(q, k, v, lengths, 0.125, g)
    args = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    lens = torch.tensor(lengths)
    got = [torch.autograd.grad(sparse_attention_train(*args, lens, scale), args, g.to(dev))
           for scale in (0.125, torch.tensor(0.125, device=dev))]      # a scale that is a tensor: the composition
    for name, ours, theirs, b in zip("qkv", *got, grads):
        err, ref = (float((a.double().cpu() - b).norm() / b.norm()) for a in (ours, theirs))
        assert err <= 1.1 * ref, (name, err, ref)


@pytest.mark.parametrize("which", ["q", "k", "v", "grad", "hook"])
def test_operands_off_a_16_byte_boundary(dev, which):
    """Operands that start 4 bytes behind a boundary, and saved tensors that come back from a hook that way."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, n, lengths = 2, 33, [5, 17]
    L, B = sum(lengths), len(lengths)

    def shifted(t):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        flat[1:] = t.reshape(-1)
        return flat[1:].view(t.shape)

    host = {name: torch.from_numpy(randn(i, *s)) for i, (name, s) in enumerate(
        {"q": (h, L, 64), "k": (h, B, n, 64), "v": (h, B, n, 64), "grad": (L, h * 64)}.items())}
    on = {name: shifted(t.to(dev)) if name == which else t.to(dev) for name, t in host.items()}
    args = [on[name].requires_grad_(True) for name in "qkv"]
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: t, (lambda t: shifted(t) if t.is_floating_point() else t) if which == "hook" else lambda t: t):
        got = sparse_attention_train(*args, torch.tensor(lengths), 0.125)
    grads = torch.autograd.grad(got, args, on["grad"])
    want, wants = _reference(host["q"], host["k"], host["v"], lengths, 0.125, host["grad"])
    for a, b in zip((got.detach(),) + grads, (want,) + wants):
        assert float((a.double().cpu() - b).abs().max()) <= 1e-5 * float(b.abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("first", [1, 32, 40])
def test_first_scores_of_minus_infinity(dev, dtype, first):
    """Keys whose scores overflow to -infinity have probability zero, also where they are the first of their sample."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, n, lengths = 2, 65, [5, 17]
    L, B = sum(lengths), len(lengths)
    q, k, v = (torch.from_numpy(randn(i, *s)) for i, s in enumerate([(h, L, 64), (h, B, n, 64), (h, B, n, 64)]))
    q[..., 3], k[..., 3] = 1e20, 0
    k[:, :, :first, 3] = -1e20                               # -1e40: past the range of fp32
    q, k, v, g = (t.to(dtype) for t in (q, k, v, torch.from_numpy(randn(3, L, h * 64))))
    want, grads = _reference(q, k, v, lengths, 0.125, g)
    args = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    got = sparse_attention_train(*args, torch.tensor(lengths), 0.125)
    pairs = list(zip((got.detach(),) + torch.autograd.grad(got, args, g.to(dev)), (want,) + grads))
    keep = [c for c in range(64) if c != 3]                  # (the gradient of the huge channel is as huge)
    pairs[2] = tuple(t[..., keep] for t in pairs[2])
    for a, b in pairs:
        assert float((a.double().cpu() - b).abs().max()) <= TOL[dtype] * float(b.abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("length", [5, 32, 45])
def test_an_infinite_gradient_of_the_last_query(dev, dtype, length):
    """dV takes it with the query's probabilities: infinite in its channel, finite in the others (rows past the last query,
    which repeat it, have probability zero, and zero times infinity is NaN)."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    lengths = [length, 7]
    L = sum(lengths)
    q, k, v, g = (torch.from_numpy(randn(i, *s)).to(dtype)
                  for i, s in enumerate([(1, L, 64), (1, 2, 33, 64), (1, 2, 33, 64), (L, 64)]))
    g[length - 1, 3] = float("inf")
    _, grads = _reference(q, k, v, lengths, 0.125, g)
    args = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    dv = torch.autograd.grad(sparse_attention_train(*args, torch.tensor(lengths), 0.125), args, g.to(dev))[2].double().cpu()
    inf = torch.isinf(grads[2])
    assert int(inf.sum()) == 33 and torch.equal(torch.isinf(dv), inf) and bool((dv[inf] > 0).all())
    assert float((dv - grads[2])[~inf].abs().max()) <= TOL[dtype] * float(grads[2][~inf].abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("n", [5, 64, 257])
def test_a_key_or_value_that_is_nan(dev, dtype, which, n):
    """A NaN in the last key or value (at 5 keys the only one some lanes hold) is NaN in every gradient of its sample
    that it is in for the composition, and in none of the other sample's."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, lengths = 2, [19, 7]
    L = sum(lengths)
    t = {name: torch.from_numpy(randn(i, *s)).to(dtype)
         for i, (name, s) in enumerate({"q": (h, L, 64), "k": (h, 2, n, 64), "v": (h, 2, n, 64), "g": (L, h * 64)}.items())}
    t[which][:, 0, n - 1, 7] = float("nan")
    want, grads = _reference(t["q"], t["k"], t["v"], lengths, 0.125, t["g"])
    args = [t[name].to(dev).requires_grad_(True) for name in "qkv"]
    got = sparse_attention_train(*args, torch.tensor(lengths), 0.125)
    for a, b in zip((got.detach(),) + torch.autograd.grad(got, args, t["g"].to(dev)), (want,) + grads):
        a, nan = a.double().cpu(), torch.isnan(b)
        assert torch.equal(torch.isnan(a), nan)
        assert float((a - b)[~nan].abs().max()) <= TOL[dtype] * float(b[~nan].abs().max())


def test_scores_are_those_of_the_queries_as_given(dev):
    """Scores of spread 8 in bf16: a query rounded once more, times the scale, would be off by 2^-9 / sqrt(3) of its score,
    i.e. 9e-3 of a probability.  What remains are the roundings of the probabilities and of the result, 1.1e-3 each."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    h, n, lengths = 3, 257, [113, 64]
    L, B = sum(lengths), len(lengths)
    q, k, v = (torch.from_numpy(randn(i, *s)).bfloat16()
               for i, s in enumerate([(h, L, 64), (h, B, n, 64), (h, B, n, 64)]))
    want, _ = _reference(q, k, v, lengths, 0.9, torch.ones(L, h * 64))
    got = sparse_attention_train(*(t.to(dev) for t in (q, k, v)), torch.tensor(lengths), 0.9)
    assert float((got.double().cpu() - want).norm()) <= 2.5 * 1.6e-3 * float(want.norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("h,B,n,step", [(1, 2, 33, 64), (1, 1, 1, 64), (2, 1, 33, 64), (1, 2, 3, 1 << 23)])
def test_strides_of_single_heads_samples_and_keys(dev, dtype, h, B, n, step):
    """Dimensions of size one may carry any stride, queries may lie far apart: the same bytes as from dense operands."""
    from vtpack_amd import _C
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    lengths = [3, 5][:B]
    L = sum(lengths)

    def odd(t, row=None):
        st = [3 if s == 1 else d for s, d in zip(t.shape, t.stride())]
        if row is not None:
            st[-2], st[0] = row, (3 if t.shape[0] == 1 else t.stride(0))
        out = torch.empty_strided(t.shape, st, dtype=t.dtype, device=dev)
        return out.copy_(t)

    q, k, v, g = (torch.from_numpy(randn(i, *s)).to(dtype).to(dev)
                  for i, s in enumerate([(h, L, 64), (h, B, n, 64), (h, B, n, 64), (L, h * 64)]))
    runs = []
    for a in ((q, k, v), (odd(q, step if step > 64 else None), odd(k), odd(v))):
        a = [t.detach().requires_grad_(True) for t in a]
        out = _C.batched_sparse_attention_forward(*(t.detach() for t in a), torch.tensor(lengths), 0.125)
        res = sparse_attention_train(*a, torch.tensor(lengths), 0.125)
        runs.append((out, res.detach()) + torch.autograd.grad(res, a, g))
    assert all(torch.equal(x, y) for x, y in zip(*runs))


@pytest.mark.parametrize("shape", [(), (2, 1, 1)])
def test_a_scale_that_is_a_tensor(dev, shape):
    """One for all heads or one each, with a gradient of its own."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    lengths = [5, 17]
    q, k, v = (torch.from_numpy(randn(i, *s)) for i, s in enumerate([(2, 22, 64), (2, 2, 33, 64), (2, 2, 33, 64)]))
    g = torch.from_numpy(randn(3, 22, 128))
    scale = (torch.arange(1, 1 + int(np.prod(shape))) * 0.1).view(shape).double().requires_grad_(True)
    outs = [torch.softmax(q[:, a:b].double() @ k[:, i].double().transpose(1, 2) * scale, -1) @ v[:, i].double()
            for i, (a, b) in enumerate([(0, 5), (5, 22)])]
    want, = torch.autograd.grad(torch.cat(outs, 1).permute(1, 0, 2).reshape(22, 128), scale, g.double())
    got = scale.detach().float().to(dev).requires_grad_(True)
    out = sparse_attention_train(*(t.to(dev) for t in (q, k, v)), torch.tensor(lengths), got)
    gs, = torch.autograd.grad(out, got, g.to(dev))
    assert float((gs.double().cpu() - want).abs().max()) <= 1e-4 * float(want.abs().max())


def test_the_result_may_be_changed_in_place(dev):
    """As the composition's could: the backward pass does not need it."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    lengths = [5, 17]
    args = [torch.from_numpy(randn(i, *s)).to(dev).requires_grad_(True)
            for i, s in enumerate([(2, 22, 64), (2, 2, 33, 64), (2, 2, 33, 64)])]
    g = torch.from_numpy(randn(3, 22, 128)).to(dev)
    want = torch.autograd.grad(sparse_attention_train(*args, torch.tensor(lengths), 0.125), args, g)
    out = sparse_attention_train(*args, torch.tensor(lengths), 0.125)
    out -= 1
    out *= 1
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(out, args, g), want))


@pytest.mark.parametrize("B", [1, 3, 447, 448, 449, 1000])
def test_offsets_of_lengths(dev, B):
    from vtpack_amd import ops
    lengths = torch.from_numpy(np.random.RandomState(B).randint(0, 300, size=B))
    if B > 448:
        lengths[:448] = 0
    got, _ = ops.lengths_to_offsets(lengths, dev)
    assert torch.equal(got.cpu(), torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_from_a_workspace_of_two_floats_a_row(dev, dtype):
    """The C entry whose workspace holds m + log2(s) and delta only; nothing is written behind it.  In bf16 both entries keep
    these two and agree to the last bit."""
    from vtpack_amd import _lib, ops
    h, n, lengths = 2, 65, [17, 0, 64]
    L, B = sum(lengths), len(lengths)
    q, g = (torch.from_numpy(randn(s, h, L, 64)).to(dtype) for s in (1, 4))
    k, v = (torch.from_numpy(randn(s, h, B, n, 64)).to(dtype) for s in (2, 3))
    _, grads = _reference(q, k, v, lengths, 0.125, g.transpose(0, 1).reshape(L, h * 64))
    q, k, v, g = (t.to(dev) for t in (q, k, v, g))
    offsets, _ = ops.lengths_to_offsets(torch.tensor(lengths), dev)
    work = torch.full((2 * h * L + 64,), 7.0, device=dev)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    q_st, kv_st = (64, L * 64), (n * 64, 64, B * n * 64)
    _lib.call("vtdge_sparse_attention_backward", q.data_ptr(), *q_st, k.data_ptr(), v.data_ptr(), *kv_st, 0, g.data_ptr(), *q_st,
              offsets.data_ptr(), dq.data_ptr(), *q_st, dk.data_ptr(), dv.data_ptr(), *kv_st, work.data_ptr(), L, B, h, 64, n,
              64, 0.125, _lib.dtype_code(q), _lib.stream_ptr())
    assert (work[2 * h * L:] == 7).all()
    for name, a, b, c in zip("qkv", (dq, dk, dv), ops.sparse_attention_backward(q, k, v, None, g, offsets, 0.125, 64), grads):
        assert float((a.double().cpu() - c).abs().max()) <= TOL[dtype] * float(c.abs().max()), name
        assert dtype == torch.float32 or torch.equal(a, b), name


@pytest.mark.parametrize("n", [32, 63, 95, 96, 97, 128, 160, 161, 256, 288, 289, 320])
def test_scores_kept_between_the_walks(dev, n):
    """fp32: whole and partial last stages at the edges of three, five and nine kept ones, and one beyond."""
    from vtpack_amd import _lib, ops
    lengths = [64, 0, 65, 33, 5, 130]
    test_against_float64(dev, torch.float32, n, lengths, 0.125, False)
    q, g = (torch.ones(3, sum(lengths), 64, device=dev) for _ in range(2))
    k, v = (torch.ones(3, len(lengths), n, 64, device=dev) for _ in range(2))
    offsets, _ = ops.lengths_to_offsets(torch.tensor(lengths), dev)
    ops.sparse_attention_backward(q, k, v, None, g, offsets, 0.125, max(lengths))
    held = next((stages for stages in (3, 5, 9) if n <= 32 * stages), 0)
    assert f"attention_dq_kernel<float, {held}>" in _lib.last_kernel(1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,h", [(2051, 1), (1023, 8), (1025, 8), (4, 12)])
@pytest.mark.parametrize("n", [20, 65, 130])       # searched for from 128 keys on; key chunks pair by pair and chunk by chunk
def test_workgroups_find_their_queries(dev, dtype, B, h, n):
    """Ragged batches whose workgroups look through several steps of pairs for theirs, or through none: the bits of the same
    samples in calls of 16 (of 2), whose pairs are found in the first step, and a few samples, longest and last, against float64."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    d = 64
    g = torch.Generator(dev).manual_seed(B)
    lengths = torch.randint(0, 9, (B,), generator=torch.Generator().manual_seed(h))
    lengths[::97] = 130
    lengths[-1] = 65
    L = int(lengths.sum())
    q, go = (torch.randn(L, h, d, generator=g, device=dev).to(dtype) for _ in range(2))
    k, v = (torch.randn(h, B, n, d, generator=g, device=dev).to(dtype) for _ in range(2))

    def run(q, k, v, lengths, go):
        args = [q.transpose(0, 1).requires_grad_(True), k.contiguous().requires_grad_(True), v.contiguous().requires_grad_(True)]
        out = sparse_attention_train(*args, lengths, 0.125)
        return out.detach(), *torch.autograd.grad(out, args, go.reshape(out.shape))
    out, dq, dk, dv = run(q, k, v, lengths, go)
    first = torch.cumsum(lengths, 0) - lengths
    some = sorted({0, 1, min(97, B - 1), B // 2, B - 2, B - 1})
    rows = torch.cat([torch.arange(first[b], first[b] + lengths[b]) for b in some])
    want, grads = _reference(q[rows].cpu().transpose(0, 1), k[:, some].cpu(), v[:, some].cpu(), lengths[some].tolist(), 0.125,
                             go[rows].cpu().reshape(len(rows), h * d))
    assert float((out[rows].double().cpu() - want).abs().max()) <= TOL[dtype] * float(want.abs().max())
    for name, a, b in zip("qkv", (dq[:, rows], dk[:, some], dv[:, some]), grads):
        size = max(float(b.abs().max()), 24 * 0.125 if name != "v" else 0)       # as in test_against_float64
        assert float((a.double().cpu() - b).abs().max()) <= TOL[dtype] * size, name
    part = 16 if B > 16 else 2
    for b in range(0, B, max(part, B // 8 // 16 * 16)):
        e = min(b + part, B)
        at = int(lengths[:b].sum())
        to = at + int(lengths[b:e].sum())
        if int(lengths[b:e].max()) == int(lengths[b:e].min()):
            continue
        o, q1, k1, v1 = run(q[at:to], k[:, b:e], v[:, b:e], lengths[b:e], go[at:to])
        # (fp32: few workgroups have a forward kernel of their own, whose sums are in another order: a few roundings of 2^-24)
        assert torch.equal(o, out[at:to]) if dtype == torch.bfloat16 else float((o - out[at:to]).abs().max()) <= 2 ** -19
        assert torch.equal(q1, dq[:, at:to]) and torch.equal(k1, dk[:, b:e]) and torch.equal(v1, dv[:, b:e])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("low,high", [(1, 66), (60, 66), (128, 131)])
def test_a_grid_with_holes_and_one_without(dev, dtype, low, high):
    """As many pairs as the forward pass of bf16 searches for, too, with lengths that leave half the grid empty or none of it: the bits of
    the same samples fifteen at a time, which the grid as it stands serves."""
    from vtpack_amd.layers.sparse_ops import sparse_attention_train
    B, h, n = 360, 8, 129
    g = torch.Generator(dev).manual_seed(high)
    lengths = torch.randint(low, high, (B,), generator=torch.Generator().manual_seed(low))
    lengths[::90] = high - 1
    L = int(lengths.sum())
    q, go = (torch.randn(L, h, 64, generator=g, device=dev).to(dtype) for _ in range(2))
    k, v = (torch.randn(h, B, n, 64, generator=g, device=dev).to(dtype) for _ in range(2))

    def run(at, to, b, e):
        args = [q[at:to].transpose(0, 1).requires_grad_(True), k[:, b:e].clone().requires_grad_(True), v[:, b:e].clone().requires_grad_(True)]
        out = sparse_attention_train(*args, lengths[b:e], 0.125)
        return out.detach(), *torch.autograd.grad(out, args, go[at:to].reshape(out.shape))
    out, dq, dk, dv = run(0, L, 0, B)
    for b in range(0, B, 15):
        at, to = int(lengths[:b].sum()), int(lengths[:b + 15].sum())
        o, q1, k1, v1 = run(at, to, b, b + 15)
        # (fp32: few workgroups have a forward kernel of their own, as above)
        assert torch.equal(o, out[at:to]) if dtype == torch.bfloat16 else float((o - out[at:to]).abs().max()) <= 2 ** -19
        assert torch.equal(q1, dq[:, at:to]) and torch.equal(k1, dk[:, b:b + 15]) and torch.equal(v1, dv[:, b:b + 15])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("which", ["q", "k"])
def test_sums_near_the_largest_number(dev, dtype, which):
    """64 queries with the same score for each of 64 keys, dP of +-2^120: dS is 2^111 behind the scale, and dQ (of keys of 2^4) and dK
    (of queries of 2^9) are 2^121 and 2^126 where dP's own products would add up to 2^130 and 2^129.  Powers of two: exact."""
    from vtpack_amd import ops
    sign = torch.tensor([1.0, -1.0]).repeat(32)[:, None].expand(64, 64)
    q = torch.zeros(1, 64, 64) if which == "q" else torch.full((1, 64, 64), 2.0 ** 9)
    k = (sign * 2.0 ** 4)[None, None] if which == "q" else torch.zeros(1, 1, 64, 64)
    v, g = torch.zeros(1, 1, 64, 64), torch.zeros(1, 64, 64)
    v[..., 0], g[..., 0] = sign[:, 0] * 2.0 ** 60, 2.0 ** 60
    offsets, _ = ops.lengths_to_offsets(torch.tensor([64]), dev)
    dq, dk, dv = ops.sparse_attention_backward(*(t.to(dev, dtype).contiguous() for t in (q, k, v)), None, g.to(dev, dtype), offsets,
                                               0.125, 64)
    assert torch.equal(dq.cpu().float(), torch.full((1, 64, 64), 2.0 ** 121 if which == "q" else 0.0))
    assert torch.equal(dk.cpu().float()[0, 0], sign * 2.0 ** 126 if which == "k" else torch.zeros(64, 64))
    assert torch.equal(dv.cpu().float()[0, 0], g[0])
