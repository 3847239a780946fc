"""The fp32 gradients of the packed-query attention on the bf16 matrix instructions: stages and tiles around their edges against
float64, and operands that a sum of three bf16 values does not cover, which the fp32 instructions have to give as before."""
import pytest
import torch

from util import randn

pytestmark = pytest.mark.gpu

LENGTHS = [1, 0, 16, 17, 32, 33, 47, 48, 63, 64, 65, 97, 128, 129, 200]
HEADS = 20                                 # 300 pairs, about 440 live workgroups: more than there are compute units


def _reference(q, k, v, g, lengths, scale):
    """-> gradients of q, g [h, L, 64] and k, v [h, B, n, 64] in float64 on the CPU."""
    q, k, v, g = (t.cpu().double() for t in (q, k, v, g))
    dq, dk, dv, at = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v), 0
    for b, m in enumerate(lengths):
        qb, gb = q[:, at:at + m], g[:, at:at + m]
        p = torch.softmax(qb @ k[:, b].transpose(1, 2) * scale, -1)
        dp = gb @ v[:, b].transpose(1, 2)
        ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
        dq[:, at:at + m] = ds @ k[:, b]
        dk[:, b], dv[:, b] = ds.transpose(1, 2) @ qb, p.transpose(1, 2) @ gb
        at += m
    return dq, dk, dv


def _operands(dev, n, lengths=LENGTHS, h=HEADS):
    L, B = sum(lengths), len(lengths)
    return [torch.from_numpy(randn(n + i, *s)).to(dev) for i, s in enumerate([(h, L, 64), (h, B, n, 64), (h, B, n, 64), (h, L, 64)])]


def _run(q, k, v, g, lengths=LENGTHS, scale=0.125, kernel="attention_dq_split_kernel<"):
    from vtpack_amd import _lib, ops
    offsets, _ = ops.lengths_to_offsets(torch.tensor(lengths), q.device)
    out = ops.sparse_attention_backward(q, k, v, None, g, offsets, scale, max(lengths))
    if kernel is None:
        assert "split" not in _lib.last_kernel(1) + _lib.last_kernel()
    else:
        assert kernel in _lib.last_kernel(1) and "attention_dkv_split_kernel" in _lib.last_kernel()
    return out


@pytest.mark.parametrize("n", [161, 176, 177, 192, 193, 256, 257, 288, 289, 320, 321, 515])
def test_tiles_and_stages(dev, n):
    """As far off as the fp32 instructions at most, 4.2e-7 of dQ at 257 keys (2.9e-7 here), growing with the square root of the
    keys (6.7e-7 at 1025, 5.2e-7 here)."""
    q, k, v, g = _operands(dev, n)
    kernel = f"attention_dq_split_kernel<{9 if n <= 288 else 0}>"
    got = _run(q, k, v, g, kernel=kernel)
    for name, a, b in zip("qkv", got, _reference(q, k, v, g, LENGTHS, 0.125)):
        assert float((a.cpu().double() - b).norm() / b.norm()) <= 4.2e-7 * max(1.0, n / 257) ** 0.5, name
    assert all(torch.equal(a, b) for a, b in zip(got, _run(q, k, v, g, kernel=kernel)))      # the same bytes on every call


@pytest.mark.parametrize("samples,n", [(1, 161), (2, 257), (63, 193), (64, 257), (65, 257)])
def test_samples_in_any_order(dev, samples, n):
    """Up to 64 samples are taken with the longest first, equal ones and empty ones among them; of more as they come.  The bound
    of test_tiles_and_stages, dK and dV being fp32 sums over the queries as dQ is over the keys: an rms that grows with the
    square root of the longer."""
    lengths = [2000] if samples == 1 else [3 * LENGTHS[(7 * b) % 15] + (700 if samples == 2 else 0) for b in range(samples)]
    h = {1: 20, 2: 20}.get(samples, 6)
    q, k, v, g = _operands(dev, n, lengths, h)
    for name, a, b in zip("qkv", _run(q, k, v, g, lengths), _reference(q, k, v, g, lengths, 0.125)):
        assert float((a.cpu().double() - b).norm() / b.norm()) <= 4.2e-7 * max(1.0, n / 257, max(lengths) / 257) ** 0.5, name


@pytest.mark.parametrize("size,common", [(1.0, 0.0), (4.0, 0.0), (16.0, 0.0), (1.0, 2.0)])
def test_as_exact_as_the_fp32_instructions(dev, size, common):
    """Large scores, and keys and values with a common component, beside the same samples in calls that are too small for the
    split.  A twentieth is allowed for the spread of two rms errors over 940 rows, 1 / sqrt(2 * 940) each."""
    q, k, v, g = _operands(dev, 257)
    q, k, v = q * size, k + common * k[:, :1, :1], v + common * v[:, :1, :1]
    got, at, parts = _run(q, k, v, g), 0, []
    for b, m in enumerate(LENGTHS):
        if m > 0:
            parts.append(_run(q[:, at:at + m].contiguous(), k[:, b:b + 1].contiguous(), v[:, b:b + 1].contiguous(), g[:, at:at + m].contiguous(),
                              [m], kernel=None))
        at += m
    plain = [torch.cat([p[i] for p in parts], dim=1) for i in range(3)]
    some = [b for b, m in enumerate(LENGTHS) if m > 0]
    for name, a, c, w in zip("qkv", got, plain, _reference(q, k, v, g, LENGTHS, 0.125)):
        a, w = (t if name == "q" else t[:, some] for t in (a, w))
        assert float((a.cpu().double() - w).norm()) <= 1.05 * float((c.cpu().double() - w).norm()), name


@pytest.mark.parametrize("scale", [-0.3, 0.0, 0.9])
def test_other_scales(dev, scale):
    """A scale that is not positive goes to the fp32 instructions for dQ; at zero every key has the same probability."""
    q, k, v, g = _operands(dev, 257)
    for a, b in zip(_run(q, k, v, g, scale=scale), _reference(q, k, v, g, LENGTHS, scale)):
        assert float((a.cpu().double() - b).norm()) <= 2e-6 * float(b.norm())


@pytest.mark.parametrize("of_k,of_v,of_g", [(1.0, 1.0, 1e-12), (1.0, 1.0, 1e-20), (1.0, 1e-30, 1e-5), (1.0, 1e7, 1e-10), (1.0, 1e20, 1e-20),
                                            (1e-3, 1e-25, 1e25), (1.0, 1.0, 65536.0)])
def test_magnitudes(dev, of_k, of_v, of_g):
    """Gradients of every magnitude that fp32 holds come out with its relative error, also where bf16 parts would fall below the
    smallest bf16 numbers."""
    q, k, v, g = _operands(dev, 257)
    k, v, g = k * of_k, v * of_v, g * of_g
    for name, a, b in zip("qkv", _run(q, k, v, g), _reference(q, k, v, g, LENGTHS, 0.125)):
        assert float((a.cpu().double() - b).norm() / b.norm()) <= 6e-7, name


@pytest.mark.parametrize("which,value", [(w, x) for x in (float("inf"), float("nan")) for w in "qkvg"] + [("v", 1e30), ("g", 1e30)])
def test_values_outside_the_split(dev, which, value):
    """One such value in a long sample: NaN where the composition has one, and everything else as it was.  (A query or key of
    1e30 makes scores whose last fp32 bit is more than any exponent, on either instructions.)"""
    t = dict(zip("qkvg", _operands(dev, 257)))
    first = sum(LENGTHS[:12])
    if which in "qg":
        t[which][3, first + 100, 7] = value
    else:
        t[which][3, 12, 256, 7] = value
    got, want = _run(*t.values()), _reference(*t.values(), LENGTHS, 0.125)
    for name, a, b in zip("qkv", got, want):
        a = a.cpu().double()
        assert torch.equal(a.isnan() | a.isinf(), b.isnan() | b.isinf()), name
        # what the large value multiplies and the rest, each in its own 2-norm (three times the 3.5e-7 of a whole gradient of unit
        # normals: a few elements are left; one that cancels is off by its terms' last bits, not its own)
        huge = b.abs() >= 1e9
        for part in (b.isfinite() & huge, b.isfinite() & ~huge):
            assert float((a - b)[part].norm()) <= 1e-6 * float(b[part].norm()), name


@pytest.mark.parametrize("odd", [None, "q", "k", "g"])
@pytest.mark.parametrize("kind", ["x100", "x1000", "point"])
def test_as_exact_where_few_keys_take_all(dev, kind, odd):
    """Large scores, of which the largest key's P is 1 only if it comes from the scores that m and s are of: queries a hundred and a
    thousand times as large, and queries that point at one key each (dV is then a copy of dO and all but exact: one rounding, 2^-24, is
    allowed).  `odd`: a value too small for the split in one sample of a head, whose rows, or for a key all rows of the sample, take the
    fp32 instructions while the rest of that sample does not.  Else the bound of test_as_exact_as_the_fp32_instructions."""
    t = dict(zip("qkvg", _operands(dev, 257)))
    at = [sum(LENGTHS[:b]) for b in range(len(LENGTHS))]
    if kind == "point":
        pick = torch.Generator().manual_seed(3)
        for b, m in enumerate(LENGTHS):
            t["q"][:, at[b]:at[b] + m] += 8 * t["k"][:, b, torch.randint(0, 257, (m,), generator=pick)]
    else:
        t["q"] *= float(kind[1:])
    if odd in ("q", "g"):
        for head in range(HEADS):
            t[odd][head, at[14] + 70, 5] = 1e-25
    elif odd == "k":
        t["k"][:, 14, 7, 3] = 1e-25
    got, parts = _run(*t.values()), []
    some = [b for b, m in enumerate(LENGTHS) if m > 0]
    for b in some:
        rows = slice(at[b], at[b] + LENGTHS[b])
        one = (t["q"][:, rows], t["k"][:, b:b + 1], t["v"][:, b:b + 1], t["g"][:, rows])
        parts.append(_run(*(x.contiguous() for x in one), [LENGTHS[b]], kernel=None))
    plain = [torch.cat([p[i] for p in parts], dim=1) for i in range(3)]
    for name, a, c, w in zip("qkv", got, plain, _reference(*t.values(), LENGTHS, 0.125)):
        a, w = (x if name == "q" else x[:, some] for x in (a, w))
        off = float((a.cpu().double() - w).norm())
        allowed = 2.0 ** -24 * float(w.norm()) if name == "v" and kind == "point" else 0.0
        assert off <= max(allowed, 1.05 * float((c.cpu().double() - w).norm())), name
