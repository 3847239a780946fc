"""What a Linear makes of its weight is never older than the weight: a weight used first on two streams at once, changed between
calls in every way there is, captured without a warm-up, replayed after a change, made in inference mode."""
import pytest
import torch

from vtpack_amd import _lib, engine
from vtpack_amd.models.dge.deit_dge import VisionTransformer
from vtpack_amd.models.dge.pvt_dge import PyramidVisionTransformer
from vtpack_amd.synthetic import set_synthetic_router, synthetic_images

pytestmark = pytest.mark.gpu
BATCH, GRID = 32, 16


def _blocks(dev, dim=192, dtype=torch.float32, seed=0):
    torch.manual_seed(seed)
    m = VisionTransformer(img_size=256, patch_size=16, embed_dim=dim, depth=2, num_heads=dim // 64, num_classes=10, qkv_bias=True,
                          split_sizes=[4, 2, 1])
    return list(set_synthetic_router(m, 3).eval().to(dev).to(dtype).blocks)


def _tokens(dev, dim=192, dtype=torch.float32):
    assert dtype != torch.float32 or _lib.load().vtdge_linear_split_wanted(BATCH * (GRID * GRID + 1), dim, dim) == 1
    return torch.randn(BATCH, GRID * GRID + 1, dim, generator=torch.Generator(dev).manual_seed(1), device=dev).to(dtype)


def _run(blocks, x):
    with torch.no_grad():
        return engine._run_blocks(blocks, x, GRID, GRID)


def _fresh(blocks, x):
    """What blocks with these weights give that have never run before, with nothing else on the GPU."""
    other = _blocks(x.device, x.shape[-1], x.dtype)
    for mine, theirs in zip(other, blocks):
        mine.load_state_dict(theirs.state_dict())
    torch.cuda.synchronize()
    out = _run(other, x).clone()
    torch.cuda.synchronize()
    return out


@pytest.fixture(params=[True, False], ids=["native", "composed"])
def native(request, monkeypatch):
    monkeypatch.setattr(engine, "NATIVE_CHAIN", request.param)
    return request.param


def test_f32_first_use_on_two_streams(dev, native):
    blocks, x = _blocks(dev), _tokens(dev)
    want = _fresh(blocks, x)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for change in (None, 0.5):
        if change is not None:
            with torch.no_grad():
                for p in blocks[0].mlp.parameters():
                    p.mul_(change)
            want = _fresh(blocks, x)
        with torch.cuda.stream(a):
            torch.cuda._sleep(100_000_000)          # some 40 ms in front of whatever is made of the weights
            one = _run(blocks, x)
        with torch.cuda.stream(b):
            two = _run(blocks, x)
        torch.cuda.synchronize()
        assert torch.equal(two, want) and torch.equal(one, want)


def test_f32_weights_changed_between_calls(dev, native):
    blocks, x = _blocks(dev), _tokens(dev)
    last = _run(blocks, x).clone()
    other = _blocks(dev, seed=5)

    def in_place():
        with torch.no_grad():
            blocks[1].attn.kv.weight.mul_(1.5)

    def behind_the_counter():
        blocks[0].mlp.fc2.weight.data.mul_(0.5)

    def optimiser_step():
        for p in blocks[1].parameters():
            p.grad = torch.ones_like(p) if p.is_floating_point() else None
        torch.optim.SGD([p for p in blocks[1].parameters() if p.grad is not None], 1e-2).step()

    def loaded():
        for mine, theirs in zip(blocks, other):
            mine.load_state_dict(theirs.state_dict())

    for change in (in_place, behind_the_counter, optimiser_step, loaded):
        change()
        got = _run(blocks, x).clone()
        assert torch.equal(got, _fresh(blocks, x)) and not torch.equal(got, last), change.__name__
        last = got


def test_f32_captured_without_a_warm_up(dev, native):
    blocks, x = _blocks(dev), _tokens(dev)
    want = _fresh(blocks, x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = _run(blocks, x)
    assert torch.equal(_run(blocks, x), want)       # before the first replay
    for step in range(4):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), step
        if step == 1:
            blocks[0].attn.proj.weight.data.mul_(2.0)
        else:
            with torch.no_grad():
                blocks[1].mlp.fc1.weight.add_(0.01)
        want = _fresh(blocks, x)


def test_f32_parameters_made_in_inference_mode(dev):
    """Such parameters have no version to tell a change by: prepare() and the composed blocks take them as they are."""
    x = _tokens(dev)
    want = _fresh(_blocks(dev), x)
    with torch.inference_mode():
        torch.manual_seed(0)
        m = VisionTransformer(img_size=256, patch_size=16, embed_dim=192, depth=2, num_heads=3, num_classes=10, qkv_bias=True,
                              split_sizes=[4, 2, 1])
        m = set_synthetic_router(m, 3).eval().to(dev)
        assert m.blocks[0].attn.q.weight.is_inference()
        engine.prepare(m)
        got = _run(list(m.blocks), x)
    assert torch.equal(got, want)


def _model(kind, dtype, dev):
    torch.manual_seed(2)
    if kind == "pvt":
        m = PyramidVisionTransformer(img_size=128, patch_size=4, embed_dims=[64, 128, 320, 512], num_heads=[1, 2, 5, 8],
                                     mlp_ratios=[2, 2, 2, 2], qkv_bias=True, depths=[2, 1, 2, 1], sr_ratios=[8, 4, 2, 1],
                                     split_sizes=[[4, 2, 1]] * 4, num_classes=30)
    else:
        m = VisionTransformer(img_size=128, patch_size=16, embed_dim=384, depth=2, num_heads=6, num_classes=30, qkv_bias=True,
                              split_sizes=[4, 2, 1])
    return set_synthetic_router(m, 3).eval().to(dev).to(dtype)


@pytest.mark.parametrize("kind,dtype", [("deit", torch.bfloat16), ("pvt", torch.bfloat16), ("pvt", torch.float32)])
def test_copies_that_are_kept(dev, kind, dtype, native):
    """Packed, folded and reordered weights and the class-token rows, which stay between calls: first used on two streams at
    once, and in a capture that no call came before."""
    images = synthetic_images(48, 128, seed=6, dtype=dtype, device=dev)

    def forward(m):
        with torch.no_grad():
            return m(images)

    def fresh():
        m = _model(kind, dtype, dev)
        torch.cuda.synchronize()
        return m

    want = forward(fresh()).clone()
    m = fresh()
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda._sleep(100_000_000)
        one = forward(m)
    with torch.cuda.stream(torch.cuda.Stream()):
        two = forward(m)
    torch.cuda.synchronize()
    assert torch.equal(one, want) and torch.equal(two, want)

    m = fresh()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = forward(m)
    assert torch.equal(forward(m), want)            # before the first replay
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(forward(m), want)
