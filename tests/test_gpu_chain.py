"""A chain of blocks issued by one call into the library against the same blocks composed launch by launch: the same
kernels in the same order, so every output and every value of `states` is the same bit for bit."""
import copy
import threading

import pytest
import torch

from vtpack_amd import engine
from vtpack_amd.models.dge.deit_dge import VisionTransformer
from vtpack_amd.models.dge.pvt_dge import PyramidVisionTransformer
from vtpack_amd.synthetic import set_synthetic_router, synthetic_images

pytestmark = pytest.mark.gpu
KEYS = ("comp", "input", "patches", "batches", "batches_device", "offsets_device", "gate", "queries", "size",
        "num_extra_tokens")


def _deit(dev, dtype, dim, img=128, depth=3, **kw):
    torch.manual_seed(dim + depth)
    m = VisionTransformer(img_size=img, patch_size=16, embed_dim=dim, depth=depth, num_heads=dim // 64, num_classes=40,
                          split_sizes=[4, 2, 1], **kw)
    return set_synthetic_router(m, 3).eval().to(dev).to(dtype)


def _pvt(dev, dtype, img=128):
    torch.manual_seed(9)
    m = PyramidVisionTransformer(img_size=img, patch_size=4, embed_dims=[64, 128, 320, 512], num_heads=[1, 2, 5, 8],
                                 mlp_ratios=[2, 2, 2, 2], qkv_bias=True, depths=[2, 1, 2, 1], sr_ratios=[8, 4, 2, 1],
                                 split_sizes=[[4, 2, 1]] * 4, num_classes=30)
    return set_synthetic_router(m, 4).eval().to(dev).to(dtype)


def _blocks(m):
    return list(m.blocks) if hasattr(m, "blocks") else [b for i in range(4) for b in getattr(m, f"block{i + 1}")]


def _run(m, images, native):
    engine.NATIVE_CHAIN = native
    try:
        with torch.no_grad():
            out = m(images).clone()
        return out, [{k: b.dge.states[k] for k in KEYS} for b in _blocks(m)]
    finally:
        engine.NATIVE_CHAIN = True


def _same(a, b):
    return torch.equal(a, b) if torch.is_tensor(a) else a == b


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim,batch,kw", [(64, 1, {}), (192, 3, {}), (384, 1, {}), (384, 33, {}), (384, 40, {"img": 192}),
                                          (768, 2, {}), (192, 130, {}), (384, 31, {"distilled": True}), (192, 2, {"cls_token": False}),
                                          (384, 32, {"depth": 1})])
@pytest.mark.parametrize("two_streams", [False, True])
def test_deit(dev, dtype, dim, batch, kw, two_streams):
    kw = dict(kw)
    img = kw.get("img", 128)
    m = _deit(dev, dtype, dim, **kw)
    images = synthetic_images(batch, img, seed=5, dtype=dtype, device=dev)
    before = engine.OVERLAP_FROM
    engine.OVERLAP_FROM = 0 if two_streams else 1 << 62
    try:
        got, st = _run(m, images, True)
    finally:
        engine.OVERLAP_FROM = before
    assert getattr(m.blocks[0], "_vtdge_chain").common is not None
    want, wst = _run(m, images, False)
    assert torch.equal(got, want)
    for i, (a, b) in enumerate(zip(st, wst)):
        for k in KEYS:
            assert _same(a[k], b[k]), (i, k)


@pytest.mark.parametrize("dtype,batch", [(torch.float32, 1), (torch.bfloat16, 3), (torch.bfloat16, 9), (torch.bfloat16, 33)])
def test_pvt(dev, dtype, batch):
    m = _pvt(dev, dtype)
    images = synthetic_images(batch, 128, seed=6, dtype=dtype, device=dev)
    got, st = _run(m, images, True)
    want, wst = _run(m, images, False)
    assert torch.equal(got, want)
    assert all(_same(a[k], b[k]) for a, b in zip(st, wst) for k in KEYS)


@pytest.mark.parametrize("two_streams", [False, True])
@pytest.mark.parametrize("batch,img,depths,kernels", [
    (48, 256, [3, 2, 1, 1], 4),       # 3072 rows: of 64 channels every block, of 128 (3072 regions too) the first, the second from region_step
    (47, 256, [2, 2, 1, 1], 0), (52, 256, [18, 3, 1, 1], 21),          # a row short; more blocks than one launch packs weights for
    (193, 128, [1, 2, 1, 1], 3)])
def test_pvt_with_norm1_inside_the_reduction(dev, batch, img, depths, kernels, two_streams):
    from vtpack_amd import _lib
    torch.manual_seed(10)
    m = PyramidVisionTransformer(img_size=img, patch_size=4, embed_dims=[64, 128, 320, 512], num_heads=[1, 2, 5, 8], mlp_ratios=[2] * 4,
                                 qkv_bias=True, depths=depths, sr_ratios=[8, 4, 2, 1], split_sizes=[[4, 2, 1]] * 4, num_classes=30)
    m = set_synthetic_router(m, 4).eval().to(dev).bfloat16()
    with torch.no_grad():
        for blk in _blocks(m):                   # no block's parameters like another's
            for t in blk.parameters():
                t += 0.02 * torch.randn_like(t) if t.is_floating_point() else 0
    images = synthetic_images(batch, img, seed=6, dtype=torch.bfloat16, device=dev)
    before, calls = engine.OVERLAP_FROM, []
    engine.OVERLAP_FROM = 0 if two_streams else 1 << 62
    whole = engine.ops.layernorm_patch_linear
    engine.ops.layernorm_patch_linear = lambda *a: calls.append(a) or whole(*a)
    try:
        got, st = _run(m, images, True)
        assert not calls
        want, wst = _run(m, images, False)
    finally:
        engine.OVERLAP_FROM = before
        engine.ops.layernorm_patch_linear = whole
    assert len(calls) == kernels
    assert torch.equal(got, want)
    assert all(_same(a[k], b[k]) for a, b in zip(st, wst) for k in KEYS)


def test_changes_of_the_parameters_are_seen(dev):
    """In-place edits, a parameter or a module replaced, another data type, a copy of the model: each call works with
    the parameters as they are then."""
    m = _deit(dev, torch.bfloat16, 384)
    images = synthetic_images(33, 128, seed=7, dtype=torch.bfloat16, device=dev)
    first, _ = _run(m, images, True)
    other = copy.deepcopy(m)
    assert torch.equal(_run(other, images, True)[0], first)

    def check(model, im=images, changed=True):
        got = _run(model, im, True)[0]
        assert torch.equal(got, _run(model, im, False)[0])
        assert torch.equal(got, first) != changed

    with torch.no_grad():
        m.blocks[1].norm2.weight.mul_(1.5)
    check(m)
    check(other, changed=False)
    other.blocks[2].attn.kv.weight = torch.nn.Parameter(other.blocks[2].attn.kv.weight.detach() * 2)
    check(other)
    fresh = torch.nn.Linear(384, 768)
    with torch.no_grad():
        fresh.weight.mul_(0.1)
    m.blocks[0].mlp.fc1, m.blocks[0].mlp.fc2 = fresh.to(dev).bfloat16(), torch.nn.Linear(768, 384).to(dev).bfloat16()
    check(m)                                     # the blocks are no longer alike: composed
    # numbers of the modules, and a parameter that keeps its storage and its version but not its shape
    other.blocks[1].norm1.eps = 0.5
    check(other)
    first = _run(other, images, True)[0]
    for blk in other.blocks:
        blk.attn.scale, blk.attn.num_heads = 0.3, 12
    check(other)
    first = _run(other, images, True)[0]
    with pytest.raises(ValueError):
        short = copy.deepcopy(other)
        _run(short, images, True)
        short.blocks[1].mlp.fc2.bias.data = short.blocks[1].mlp.fc2.bias.data[:192]
        _run(short, images, True)
    m32 = copy.deepcopy(other).float()
    assert torch.equal(_run(m32, images.float(), True)[0], _run(m32, images.float(), False)[0])


def test_outputs_and_states_belong_to_their_call(dev):
    m = _deit(dev, torch.bfloat16, 384)
    a, b = (synthetic_images(n, 128, seed=8 + n, dtype=torch.bfloat16, device=dev) for n in (33, 40))
    with torch.no_grad():
        first = m(a)
        kept, gate = first.clone(), m.blocks[1].dge.states["gate"]
        gate_kept = gate.clone()
        m(b)
        m(b)
    assert torch.equal(first, kept) and torch.equal(gate, gate_kept)


@pytest.mark.parametrize("dtype,batch", [(torch.float32, 2), (torch.bfloat16, 33)])
def test_a_kept_value_keeps_no_more_than_itself(dev, dtype, batch):
    """The chain's blocks share buffers; a caller who collects one block's values over many batches must not hold those."""
    m = _deit(dev, dtype, 384)
    images = synthetic_images(batch, 128, seed=5, dtype=dtype, device=dev)
    with torch.no_grad():
        m(images)
    assert getattr(m.blocks[0], "_vtdge_chain").common is not None
    for blk in m.blocks:
        for key in ("comp", "input", "patches", "queries", "gate", "offsets_device", "batches_device"):
            t = blk.dge.states[key]
            held, wanted = t.untyped_storage().nbytes(), t.numel() * t.element_size()
            assert held <= 2 * wanted, key
    # captured, `input`, `gate` and the offsets are the graph's own memory: its replays show in them
    static_in = images.clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(g):
        m(static_in)
    held = {key: m.blocks[1].dge.states[key] for key in ("input", "gate", "offsets_device")}
    for seed in (5, 6, 5):
        static_in.copy_(synthetic_images(batch, 128, seed=seed, dtype=dtype, device=dev))
        with torch.no_grad():
            m(static_in)
        want = {key: m.blocks[1].dge.states[key] for key in held}
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(held[key], want[key]) for key in held), seed


def test_values_read_on_another_stream(dev):
    """The reader's stream has not waited for the forward, which is still queued behind a long kernel."""
    m = _deit(dev, torch.bfloat16, 384)
    images = synthetic_images(33, 128, seed=5, dtype=torch.bfloat16, device=dev)
    with torch.no_grad():
        m(images)
        want = [{k: b.dge.states[k].clone() for k in ("queries", "comp", "gate", "batches")} for b in m.blocks]
        m(torch.zeros_like(images))
        torch.cuda.synchronize()
        reader = torch.cuda.Stream()
        torch.cuda._sleep(20_000_000)
        m(images)
        with torch.cuda.stream(reader):
            got = [{k: b.dge.states[k] + 0 for k in w} for b, w in zip(m.blocks, want)]
        m(torch.zeros_like(images))             # may take the buffers that the values were read from
    torch.cuda.synchronize()
    assert all(torch.equal(a[k], b[k]) for a, b in zip(got, want) for k in a)


def _two_stream_models(dev):
    return [(_deit(dev, torch.float32, 192), torch.float32, 40), (_deit(dev, torch.bfloat16, 768), torch.bfloat16, 40),
            (_pvt(dev, torch.bfloat16), torch.bfloat16, 9)]


def test_two_streams_of_a_chain_captured_in_a_graph(dev, monkeypatch):
    """Fork and join of the side stream inside a capture: every replay gives what the eager forward gives for its images,
    with eager work and synchronisations between the replays."""
    monkeypatch.setattr(engine, "OVERLAP_FROM", 0)
    for m, dtype, batch in _two_stream_models(dev):
        static_in = synthetic_images(batch, 128, seed=20, dtype=dtype, device=dev)
        side = torch.cuda.Stream()
        with torch.no_grad():
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                m(static_in)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                static_out = m(static_in)
            for seed in (20, 21, 22, 20):
                img = synthetic_images(batch, 128, seed=seed, dtype=dtype, device=dev)
                eager = m(img).clone()
                torch.cuda.synchronize()
                static_in.copy_(img)
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(static_out, eager), (dtype, seed)


def test_host_threads_with_streams_of_their_own(dev, monkeypatch):
    """One model called from four threads at once, each on a stream of its own (and its side stream)."""
    monkeypatch.setattr(engine, "OVERLAP_FROM", 0)
    for m, dtype, batch in _two_stream_models(dev):
        images = [synthetic_images(batch, 128, seed=30 + i, dtype=dtype, device=dev) for i in range(4)]
        with torch.no_grad():
            want = [m(im).clone() for im in images]
        torch.cuda.synchronize()
        got, errors = [None] * 4, []

        def work(i):
            try:
                with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream()):
                    for _ in range(5):
                        got[i] = m(images[i])
                    torch.cuda.current_stream().synchronize()
            except Exception as e:      # noqa: BLE001
                errors.append(e)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors
        assert all(torch.equal(a, b) for a, b in zip(got, want)), dtype
