"""Host-side logic of the package: API surface, state-dict names, error behaviour, complexity counter."""
import contextlib
import math
import types

import pytest
import torch


def test_layer_api_surface():
    import vtpack_amd.layers as L
    for name in ["DynamicGrainedEncoder", "grained_sample_compress", "grained_sample_decompress",
                 "grained_sample_index_to_patch", "batched_sparse_gemm", "batched_sparse_attention"]:
        assert hasattr(L, name)          # vtpack/layers/__init__.py:1-10
    from vtpack_amd import _C
    for name in ["grained_sample_compress", "grained_sample_decompress", "grained_sample_index_to_patch",
                 "grained_sample_index_to_patch_dense", "batched_sparse_gemm_forward",
                 "batched_sparse_gemm_v2_forward", "batched_sparse_attention_forward"]:
        assert callable(getattr(_C, name))   # vtpack/layers/csrc/vision.cpp:11-21


def test_install_as_vtpack_registers_operator_module():
    import sys
    import vtpack_amd
    saved = {k: sys.modules.get(k) for k in ("vtpack", "vtpack._C")}
    try:
        c = vtpack_amd.install_as_vtpack()
        from vtpack import _C
        assert _C is c and callable(_C.grained_sample_compress)
    finally:
        for k, v in saved.items():
            if v is None:
                sys.modules.pop(k, None)
            else:
                sys.modules[k] = v


def test_state_dict_keys_follow_the_reference():
    from vtpack_amd.models.dge import deit_dge_s124_tiny_patch16_256
    m = deit_dge_s124_tiny_patch16_256()
    keys = set(m.state_dict().keys())
    want = {"cls_token", "pos_embed", "patch_embed.proj.weight", "patch_embed.proj.bias", "norm.weight",
            "norm.bias", "head.weight", "head.bias"}
    for i in range(12):
        for k in ["norm1.weight", "norm1.bias", "attn.q.weight", "attn.q.bias", "attn.kv.weight", "attn.kv.bias",
                  "attn.proj.weight", "attn.proj.bias", "norm2.weight", "norm2.bias", "mlp.fc1.weight",
                  "mlp.fc1.bias", "mlp.fc2.weight", "mlp.fc2.bias", "dge.splits", "dge.router.gate.weight",
                  "dge.router.gate.bias"]:
            want.add(f"blocks.{i}.{k}")
    assert keys == want
    assert m.blocks[0].dge.splits.dtype == torch.int64 and m.blocks[0].dge.splits.tolist() == [4, 2, 1]
    assert m.bfloat16().blocks[0].dge.splits.dtype == torch.int64      # integer data survives dtype casts
    assert m.pos_embed.shape == (1, 257, 192) and m.blocks[0].norm1.eps == 1e-6


def test_router_initialisation():
    # vtpack/layers/dge.py:129-138: bias = +-1/2 ln 38 in favour of the finest split
    from vtpack_amd.layers import DynamicGrainedEncoder
    d = DynamicGrainedEncoder(64, [4, 2, 1])
    b = 0.5 * math.log(38.0)
    assert torch.allclose(d.router.gate.bias, torch.tensor([b, -b, -b]), atol=1e-6)
    assert 0.005 < float(d.router.gate.weight.std()) < 0.015 and d.region_size == 4
    assert torch.allclose(DynamicGrainedEncoder(64, [1]).router.gate.bias, torch.zeros(1))


def test_operators_refuse_cpu_tensors_and_training():
    from vtpack_amd import _C
    from vtpack_amd.layers import DynamicGrainedEncoder
    x = torch.zeros(1, 17, 8)
    patches = torch.zeros(2, 4, dtype=torch.int64)
    with pytest.raises(RuntimeError, match="GPU only"):
        _C.grained_sample_compress(x, patches, 4, 4, 1)
    with pytest.raises(RuntimeError, match="GPU only"):
        _C.batched_sparse_attention_forward(torch.zeros(1, 2, 64), torch.zeros(1, 1, 3, 64), torch.zeros(1, 1, 3, 64),
                                            torch.tensor([2]), 1.0)
    with pytest.raises(ValueError):
        DynamicGrainedEncoder(8, [4, 3])           # 3 does not divide the region size 4
    d = DynamicGrainedEncoder(8, [4, 2, 1], sparse_train=True).train()
    with pytest.raises(RuntimeError, match="GPU only"):
        d.compress(x, 4, 4)                        # sparse training uses the kernels: no CPU path either
    with pytest.raises(TypeError):
        _C.grained_sample_index_to_patch(torch.zeros(1, 1, 1, dtype=torch.int32), torch.tensor([4, 2, 1]), 4, 1)


def _fake_states(model, gate_index):
    B, N, C = 2, 257, model.embed_dim
    for blk in model.blocks:
        gate = torch.zeros(B, 4, 4, 3)
        gate[..., gate_index] = 1.0
        blk.dge.states.update({"input": torch.zeros(B, N, C), "gate": gate, "num_extra_tokens": 1})


@pytest.mark.parametrize("away", ["k", "v"])
def test_sparse_training_attention_refuses_keys_that_are_not_on_the_gpu(monkeypatch, away):
    """Queries on the GPU, keys or values on the CPU: refused, as the composition of products does, before any kernel."""
    from vtpack_amd import ops
    from vtpack_amd.layers.sparse_ops import sparse_attention_train

    class OnGpu(torch.Tensor):          # stands for a tensor on the GPU
        is_cuda = property(lambda self: True)
        device = property(lambda self: torch.device("cuda", 0))

    def launched(*args, **kw):
        raise AssertionError("a kernel was handed an address of host memory")
    for name in ("lengths_to_offsets", "sparse_attention_heads"):
        monkeypatch.setattr(ops, name, launched)
    t = {"q": torch.zeros(2, 5, 64), "k": torch.zeros(2, 2, 7, 64), "v": torch.zeros(2, 2, 7, 64)}
    args = [x if name == away else x.as_subclass(OnGpu) for name, x in t.items()]
    with pytest.raises(RuntimeError, match="GPU only"):
        sparse_attention_train(*args, torch.tensor([2, 3]), 0.125)


@pytest.mark.parametrize("factory,macs", [("deit_dge_s124_small_patch16_256", 6.1e9),
                                          ("deit_dge_s124_tiny_patch16_256", 1.7e9)])
def test_complexity_counter_reproduces_published_macs(factory, macs):
    """Static MACs of DeiT-S / DeiT-Ti at 256 px: 6.1 G / 1.7 G (README.md:59,61 of the reference)."""
    from vtpack_amd.models import dge as zoo
    m = getattr(zoo, factory)().eval()
    img = torch.zeros(2, 3, 256, 256)
    _fake_states(m, 0)                       # all-fine gate: every token is its own query
    c = m.complexity(img)
    assert abs(float(c["static"]) - macs) / macs < 0.03
    assert float(c["dynamic"]) == pytest.approx(float(c["static"]))
    _fake_states(m, 2)                       # all-coarse gate: 17 queries per image
    c2 = m.complexity(img)
    assert float(c2["static"]) == pytest.approx(float(c["static"]))
    assert 0.1 < float(c2["dynamic"]) / float(c2["static"]) < 0.4


def test_dense_training_branch_equals_the_sparse_statement_on_cpu():
    """Training without sparse_train is plain torch (vtpack/layers/dge.py:68-72, :91-95): with its hard one-hot
    gate it must give what the sparse operators give for the sampled granularity, and pass gradients to the
    input and to the router."""
    from oracle import torch_ref
    from vtpack_amd.layers import DynamicGrainedEncoder
    torch.manual_seed(3)
    B, H, W, C, extra = 2, 8, 12, 16, 1
    d = DynamicGrainedEncoder(C, [4, 2, 1]).train()
    with torch.no_grad():
        d.router.gate.bias.zero_()
        d.router.gate.weight.normal_(0, 1.0)
    x = torch.randn(B, extra + H * W, C, requires_grad=True)
    comp = d.compress(x, H, W)
    assert comp.shape[0] == B * (extra + H * W + H * W // 4 + H * W // 16) and d.states["patches"] is None
    gate = d.states["gate"]
    assert torch.equal(gate.sum(-1), torch.ones_like(gate.sum(-1))) and set(gate.unique().tolist()) <= {0.0, 1.0}
    out = d.decompress(torch.tanh(comp) * 2)
    idx = gate.argmax(-1)
    assert len(idx.unique()) > 1
    patches, _ = torch_ref.index_to_patch(idx, d.splits, 4, extra)
    xd = x.detach()
    c_ref = torch_ref.compress(xd, patches, H, W, extra)
    want = torch_ref.decompress(torch.tanh(c_ref) * 2 - c_ref, patches, xd, H, W, extra, True)
    assert float((out - want).abs().max()) <= 1e-5
    out.square().sum().backward()
    assert x.grad is not None and float(x.grad.abs().max()) > 0
    assert float(d.router.gate.weight.grad.abs().max()) > 0


def test_checkpoint_round_trip(tmp_path):
    """A checkpoint written the way the reference's training loop writes it ({"model": state_dict, ...}) loads
    through a loader that executes nothing from the file, into the same keys and values (main.py:372-379)."""
    from vtpack_amd import harness
    from vtpack_amd.models.dge import deit_dge_s124_tiny_patch16_256
    torch.manual_seed(0)
    a = deit_dge_s124_tiny_patch16_256(num_classes=10)
    with torch.no_grad():
        for p in a.parameters():
            if p.is_floating_point():
                p.add_(0.01 * torch.randn_like(p))
    path = tmp_path / "checkpoint.pth"
    torch.save({"model": a.state_dict(), "epoch": 7, "args": {"dge_budget": 0.5}}, path)
    torch.manual_seed(1)
    b = deit_dge_s124_tiny_patch16_256(num_classes=10)
    rest = harness.load_checkpoint(b, path)
    assert rest == {"epoch": 7, "args": {"dge_budget": 0.5}}
    sa, sb = a.state_dict(), b.state_dict()
    assert list(sa) == list(sb) and all(torch.equal(sa[k], sb[k]) for k in sa)
    assert sb["blocks.0.dge.splits"].dtype == torch.int64
    # a bare state dict and a DistributedDataParallel-style wrapper are accepted as well
    torch.save(a.state_dict(), path)

    class Wrapped(torch.nn.Module):
        def __init__(self, m):
            super().__init__()
            self.module = m

    torch.manual_seed(2)
    c = Wrapped(deit_dge_s124_tiny_patch16_256(num_classes=10))
    assert harness.load_checkpoint(c, path) == {}
    assert all(torch.equal(sa[k], v) for k, v in c.module.state_dict().items())
    # a checkpoint of another architecture is refused, not half-loaded
    with pytest.raises(RuntimeError):
        harness.load_checkpoint(deit_dge_s124_tiny_patch16_256(num_classes=10, distilled=True), path)


def test_evaluate_meters_on_a_plain_model():
    """The evaluation loop's meters (vtpack/engine/engine.py:102-147): per-batch means of the loss, accuracies
    weighted by the batch size, against a direct computation."""
    from vtpack_amd import harness
    torch.manual_seed(0)
    net = torch.nn.Sequential(torch.nn.Flatten(), torch.nn.Linear(3 * 8 * 8, 7))
    batches = [(torch.randn(5, 3, 8, 8), torch.randint(0, 7, (5,))), (torch.randn(3, 3, 8, 8), torch.randint(0, 7, (3,)))]
    stats = harness.evaluate(batches, net, "cpu")
    assert set(stats) == {"loss", "acc1", "acc5"}
    with torch.no_grad():
        outs = [net(x) for x, _ in batches]
    losses = [float(torch.nn.functional.cross_entropy(o, t)) for o, (_, t) in zip(outs, batches)]
    assert stats["loss"] == pytest.approx(sum(losses) / 2)
    hits1 = sum(int((o.argmax(1) == t).sum()) for o, (_, t) in zip(outs, batches))
    hits5 = sum(int((o.topk(5, 1).indices == t[:, None]).any(1).sum()) for o, (_, t) in zip(outs, batches))
    assert stats["acc1"] == pytest.approx(100.0 * hits1 / 8) and stats["acc5"] == pytest.approx(100.0 * hits5 / 8)


def test_budget_loss_from_planted_gates():
    """loss_dge = scale * (dynamic / static - budget)^2 (vtpack/engine/engine.py:58-63) on the counter's output."""
    from vtpack_amd import harness
    from vtpack_amd.models.dge import deit_dge_s124_tiny_patch16_256
    m = deit_dge_s124_tiny_patch16_256().eval()
    img = torch.zeros(2, 3, 256, 256)
    _fake_states(m, 2)
    loss, ratio, comp = harness.budget_loss(m, img, dge_budget=0.5, dge_lr_scale=3.0)
    assert float(ratio) == pytest.approx(float(comp["dynamic"]) / float(comp["static"]))
    assert float(loss) == pytest.approx(3.0 * (float(ratio) - 0.5) ** 2)
    _fake_states(m, 0)
    loss, ratio, _ = harness.budget_loss(m, img, dge_budget=1.0)
    assert float(ratio) == pytest.approx(1.0) and float(loss) == pytest.approx(0.0, abs=1e-12)
    # the per-encoder ratio of engine.py:20-32 on the same states
    assert float(harness.get_complexity(m)) == pytest.approx(1.0)


def test_states_resolve_deferred_values_on_every_read_and_on_every_way_out():
    """`states` hands out what the reference's plain dict would hold, however it is read, and a deferred value is
    worked out again on every read (a graph replay rewrites the tensors behind it without running Python)."""
    from vtpack_amd.layers.dge import Deferred, States
    box = {"n": 3}
    st = States({"plain": 7, "batches": Deferred(lambda: box["n"]), "comp": Deferred(lambda: list(range(box["n"])))})
    assert st["batches"] == 3 and st.get("comp") == [0, 1, 2] and st.get("missing", 5) == 5
    box["n"] = 2                                   # what a replay does: new counts, no Python
    assert st["batches"] == 2 and st["comp"] == [0, 1]
    assert isinstance(dict.__getitem__(st, "batches"), Deferred)       # nothing was stored back
    for view in (dict(st), {**st}, st.copy(), st.snapshot(), dict(st.items()), dict(zip(st.keys(), st.values()))):
        assert type(view) is dict and view == {"plain": 7, "batches": 2, "comp": [0, 1]}
    snap = st.copy()
    box["n"] = 4
    assert snap["batches"] == 2 and st["batches"] == 4                 # a snapshot does not follow
    assert st.setdefault("batches", 0) == 4 and st.setdefault("new", 9) == 9
    assert st.pop("comp") == [0, 1, 2, 3] and "comp" not in st and st.pop("comp", None) is None
    with pytest.raises(KeyError):
        st.pop("comp")
    seen = {}
    while st:
        k, v = st.popitem()
        seen[k] = v
    assert seen == {"plain": 7, "batches": 4, "new": 9}


def test_fused_forward_refuses_a_distillation_token_without_a_class_token():
    """The reference never builds that token order (deit_dge.py:270-275); layer mode raises in embed_tokens and the
    fused forward must not run with the distillation token in the class token's place."""
    from vtpack_amd import engine
    from vtpack_amd.models.dge.deit_dge import VisionTransformer
    m = VisionTransformer(img_size=32, patch_size=16, embed_dim=16, depth=1, num_heads=1, distilled=True,
                          split_sizes=[2, 1]).eval()
    m.cls_token = None
    img = torch.zeros(1, 3, 32, 32)
    with pytest.raises(ValueError, match="class token"):
        engine.model_forward(m, img)
    with pytest.raises(ValueError, match="class token"):
        m.embed_tokens(img)


def test_parameters_made_in_inference_mode_have_no_chain_plan():
    """Such parameters carry no version to check a plan against: their blocks are composed one by one."""
    from vtpack_amd import engine
    from vtpack_amd.models.dge.deit_dge import VisionTransformer
    args = dict(img_size=64, patch_size=16, embed_dim=64, depth=2, num_heads=1, qkv_bias=True, split_sizes=[4, 2, 1])
    blocks = list(VisionTransformer(**args).eval().blocks)
    assert engine._chain_plan(blocks, torch.float32, torch.device("cpu"), 64, 1) is not None
    with torch.inference_mode():
        blocks = list(VisionTransformer(**args).eval().blocks)
        assert engine._chain_plan(blocks, torch.float32, torch.device("cpu"), 64, 1) is None


def test_a_parameter_replaced_at_the_same_address_has_a_new_chain_plan():
    """An allocator hands the storage of a parameter that is gone to the one that replaces it: same address, version and
    shape, other values - and packed copies of the weights of before."""
    from vtpack_amd import engine
    from vtpack_amd.models.dge.deit_dge import VisionTransformer
    blocks = list(VisionTransformer(img_size=64, patch_size=16, embed_dim=64, depth=2, num_heads=1, qkv_bias=True,
                                    split_sizes=[4, 2, 1]).eval().blocks)

    def plan():
        return engine._chain_plan(blocks, torch.float32, torch.device("cpu"), 64, 1)

    for module in (blocks[1].attn.proj, blocks[0].mlp.fc2):    # as load_state_dict(assign=True) leaves them: version 0
        module.weight = torch.nn.Parameter(module.weight.detach().clone())
    first = plan()
    assert first is not None and plan() is first
    for module in (blocks[1].attn.proj, blocks[0].mlp.fc2):
        values, version = module.weight.detach().numpy(), module.weight._version      # the storage outlives the parameter
        module.weight = torch.nn.Parameter(torch.from_numpy(values))
        values += 1
        assert module.weight.data_ptr() == values.ctypes.data and module.weight._version == version
        second = plan()
        assert second is not first and plan() is second
        first = second


@pytest.mark.parametrize("captured", [False, True])
def test_values_of_a_native_chain_are_copied_on_the_readers_stream(monkeypatch, captured):
    """A copy made on the forward's stream would not be ordered before what the reader does with it on another one: the
    reader's stream waits for the forward's and copies itself, and the buffers are kept for it."""
    from vtpack_amd import engine
    log = []

    class Stream:
        def wait_stream(self, other):
            log.append(("wait", self, other))

    reader, forward = Stream(), Stream()
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: reader)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: log.append(("on", s)) or contextlib.nullcontext())
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: log.append(("record", t.data_ptr(), s)))
    monkeypatch.setattr(torch.Tensor, "clone", lambda t: log.append(("clone",)) or t + 0)
    x, ints, big = torch.zeros(2, 17, 64), torch.zeros(4096, dtype=torch.uint8), torch.arange(255, dtype=torch.uint8).repeat(400)
    desc = types.SimpleNamespace(H=4, W=4, S=3)
    ints[:24].view(torch.int64)[:3] = torch.tensor([0, 5, 9])
    layout = [0] * 8 + [512, 0, -1, -1, 0, 1024, 1024, 1024]          # gate, offsets, lengths, status, input, comp, queries, patches
    view = engine._ChainBlock((x, ints, big, (desc, layout), forward, captured), 0)
    for key, rows in (("comp", 9), ("queries", 9), ("patches", 9), ("gate", 2), ("input", 2), ("offsets_device", 3)):
        log.clear()
        assert view.get(key).shape[0] == rows
        held = captured and key in ("gate", "input", "offsets_device")
        assert not any(e[0] == "on" for e in log) and (("clone",) in log) == (not held), key
        if not captured:
            assert log[0] == ("wait", reader, forward), key
            assert {e[1] for e in log if e[0] == "record"} == {x.data_ptr(), ints.data_ptr(), big.data_ptr()}


def test_layernorm_linear_is_wanted_where_it_fits_and_not_beyond_its_lead():
    from vtpack_amd import _lib
    lib = _lib.load()
    for rows, C, hidden, dtype, pair, fc1 in [
            (257, 384, 1536, _lib.BF16, 1, 1), (514, 384, 1536, _lib.BF16, 1, 0), (514, 768, 3072, _lib.BF16, 1, 0),
            (771, 768, 3072, _lib.BF16, 0, 0), (771, 320, 1280, _lib.BF16, 1, 0), (1285, 192, 768, _lib.BF16, 1, 1),
            (514, 192, 768, _lib.F32, 1, 1), (771, 192, 768, _lib.F32, 1, 0), (3000, 192, 768, _lib.F32, 0, 0)]:
        both, one = (rows, 2 * C, rows, C, C, dtype), (rows, hidden, 0, 0, C, dtype)
        assert (lib.vtdge_layernorm_linear_wanted(*both), lib.vtdge_layernorm_linear_wanted(*one)) == (pair, fc1), (rows, C)
        assert lib.vtdge_layernorm_linear_fits(*both) >= pair and lib.vtdge_layernorm_linear_fits(*one) >= fc1
    assert lib.vtdge_layernorm_linear_fits(771, 1536, 771, 768, 768, _lib.BF16)      # what was taken before still is


def test_region_step_is_planned_wherever_it_is_said_to_fit():
    """A chain's status words, eight bytes a region where its blocks are joined by vtdge_region_step and a fourth of that by the
    chained scatter-back: by the one rule of vtdge_region_step_fits, with no sizes of a chain's own in between."""
    import ctypes
    from vtpack_amd import _lib
    lib = _lib.load()
    for C, grid, batches in ((384, 16, (13, 192, 240, 241, 247, 250, 256, 257, 300, 511, 512, 640, 641, 700)),
                             (384, 32, (60, 61, 63, 64, 65, 128, 160, 161))):
        for B in batches:
            desc = _lib.Chain(B=B, H=grid, W=grid, C=C, heads=C // 64, hidden=4 * C, extra=1, S=3, depth=3, dtype=_lib.BF16, sr=1,
                              splits_124=1, eps1=1e-6, eps2=1e-6, sr_eps=0.0, scale=0.125)
            words = (ctypes.c_int64 * (_lib.CHAIN_LAYOUT_HEAD + 3 * _lib.CHAIN_LAYOUT_BLOCK))()
            assert lib.vtdge_chain_layout(ctypes.addressof(desc), ctypes.addressof(words)) == 0
            regions = B * (grid // 4) ** 2
            step = lib.vtdge_region_step_fits(B, grid, grid, C, 1, _lib.BF16)
            assert step == (regions <= 10240)
            want = lib.vtdge_region_step_workspace(B, grid, grid) if step else \
                lib.vtdge_decompress_router_compress_workspace(B, grid, grid, 4)
            assert words[3] == want, (grid, B)
