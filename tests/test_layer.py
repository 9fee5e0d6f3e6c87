"""A decoder layer as one autograd node against the four nodes it stands for: the same kernels in the same order, so the same
bits -- but for the gradient of the embeddings, where the first layer's two summands are rounded once instead of twice."""
import pytest
import torch

import tritonformer_amd.transformer as TM
from tests.util import rel_l2
from tritonformer_amd import layer
from tritonformer_amd.transformer import Transformer, TransformerConfig

pytestmark = pytest.mark.gpu


def build(dev, bias=False, alibi=False, param_dtype=torch.float32, layers=3, d=128, heads=2):
    torch.manual_seed(5)
    m = Transformer(TransformerConfig(512, d, 64, heads, d // heads, 3 * d, layers, bias, alibi), device=dev, param_dtype=param_dtype)
    with torch.no_grad():
        m.logits_out.weight.normal_(0, 0.02)
        for p in m.parameters():
            if p.ndim == 1:
                p.add_(torch.randn_like(p) * 0.05)
    return m


def step(m, fused, amp=None, passes=1, retain=False):
    ids = torch.randint(0, 512, (2, 64), generator=torch.Generator().manual_seed(7)).to(m.embed_tokens.weight.device)
    m.zero_grad(set_to_none=True)
    TM.FUSE_LAYER = fused
    try:
        for _ in range(passes):
            with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
                logits, loss = m(ids, ids)
            if retain:
                (loss * 256).backward(retain_graph=True)
            (loss * 256).backward()
    finally:
        TM.FUSE_LAYER = True
    return logits, loss, {n: None if p.grad is None else p.grad.clone() for n, p in m.named_parameters()}


def assert_same(one, four, dtype):
    assert torch.equal(one[0], four[0]) and torch.equal(one[1], four[1])
    assert one[2].keys() == four[2].keys()
    for name, g in four[2].items():
        if g is None:
            assert one[2][name] is None, name
        elif name.startswith("embed"):  # a rounding to 16 bits more or less: half a unit of the last place per element
            assert rel_l2(one[2][name], g) < (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7), name
        else:
            assert torch.equal(one[2][name], g), name


@pytest.mark.parametrize("bias,alibi", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("param_dtype,amp", [(torch.float32, torch.float16), (torch.float32, torch.bfloat16), (torch.float16, None)])
def test_one_node_gives_the_bits_of_four(bias, alibi, param_dtype, amp, dev):
    m = build(dev, bias, alibi, param_dtype)
    assert_same(step(m, True, amp), step(m, False, amp), amp or param_dtype)
    with torch.no_grad():
        ids = torch.arange(64, device=dev)[None]
        one = m(ids, None) if amp is None else None
        TM.FUSE_LAYER = False
        try:
            assert one is None or torch.equal(one, m(ids, None))
        finally:
            TM.FUSE_LAYER = True


def test_accumulated_and_repeated_passes(dev):
    m = build(dev, bias=True)
    assert_same(step(m, True, torch.float16, passes=2), step(m, False, torch.float16, passes=2), torch.float16)
    assert_same(step(m, True, torch.float16, retain=True), step(m, False, torch.float16, retain=True), torch.float16)


@pytest.mark.parametrize("train", ["mlp.", "attention.v_proj", "layernorm", "layer_list.2", "layer_list.0.input_layernorm",
                                   "layer_list.1.mlp.dense_4h_to_h.bias", "embed"])
def test_frozen_parameters(train, dev):
    m = build(dev, bias=True)
    for name, p in m.named_parameters():
        p.requires_grad_(train in name)
    assert_same(step(m, True, torch.float16), step(m, False, torch.float16), torch.float16)


def test_gradients_without_the_queue(dev):
    m = build(dev)
    TM.DEFER_DW = False
    try:
        assert_same(step(m, True, torch.float16), step(m, False, torch.float16), torch.float16)
    finally:
        TM.DEFER_DW = True


def test_saved_tensor_hooks_see_what_the_layer_keeps(dev):
    m = build(dev)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.clone())[1], lambda t: t):
        hooked = step(m, True, torch.float16)
    assert len(seen) > 3 * 12
    assert_same(hooked, step(m, True, torch.float16), torch.float16)


def test_watched_or_replaced_modules_are_called(dev):
    m = build(dev)
    plain = step(m, False, torch.float16)
    calls = []
    hooks = [m.layer_list[0].input_layernorm.register_forward_hook(lambda *_: calls.append("ln")),
             m.layer_list[1].attention.register_forward_pre_hook(lambda *_: calls.append("attention")),
             m.layer_list[2].mlp.register_full_backward_hook(lambda *_: calls.append("mlp"))]
    assert_same(step(m, True, torch.float16), plain, torch.float16)
    assert sorted(calls) == ["attention", "ln", "mlp"]
    for h in hooks:
        h.remove()

    class Doubled(TM.MLPBlock):
        def forward(self, x):
            return 2 * super().forward(x)

    m.layer_list[1].mlp.__class__ = Doubled
    assert not torch.equal(step(m, True, torch.float16)[0], plain[0])


def test_a_backward_pass_holds_no_more_than_that_of_four_nodes(dev, monkeypatch):
    """What a part of the layer kept goes when its gradients are there."""
    m = build(dev, param_dtype=torch.float16, layers=1, d=256, heads=4)
    monkeypatch.setattr(TM, "DEFER_DW", False)
    peaks = []
    for fused in (True, False):
        monkeypatch.setattr(TM, "FUSE_LAYER", fused)
        for _ in range(2):
            m.zero_grad(set_to_none=True)
            x, pending = (torch.randn(128, 64, 256, device=dev).half().requires_grad_() for _ in range(2))
            out = m.layer_list[0].forward_deferred(x, pending)
            grads = [torch.ones_like(t) for t in out]
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            torch.autograd.backward(out, grads)
            peaks.append(torch.cuda.max_memory_allocated() - before)
            del x, pending, out, grads
    assert peaks[1] <= peaks[3], peaks


def test_saved_tensors_that_were_packed_away_come_back_a_part_at_a_time(dev):
    """Bytes that live at once between their unpacking and the release by the engine."""
    m = build(dev, layers=1, d=256, heads=4)
    x = torch.randn(128, 64, 256, device=dev).half().requires_grad_()
    peaks = []
    for fused in (True, False):
        TM.FUSE_LAYER = fused
        try:
            m.zero_grad(set_to_none=True)
            with torch.autograd.graph.save_on_cpu(), torch.autocast("cuda", dtype=torch.float16):
                out = m.layer_list[0].forward_deferred(x, x)
        finally:
            TM.FUSE_LAYER = True
        grads = [torch.ones_like(t) for t in out]
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        torch.autograd.backward(out, grads)
        peaks.append(torch.cuda.max_memory_allocated() - before)
    assert peaks[0] <= peaks[1], peaks


@pytest.mark.parametrize("train", ["", "mlp", "post_attention_layernorm", "attention", "input_layernorm"])
@pytest.mark.parametrize("used", [0, 1])
def test_one_output_used(train, used, dev):
    """Of an output that nobody reads no gradient comes: parameters behind it alone have none, where zeros would be one."""
    m = build(dev, bias=True, layers=1)
    for name, p in m.named_parameters():
        p.requires_grad_(train in name)
    results = []
    for fused in (True, False):
        TM.FUSE_LAYER = fused
        m.zero_grad(set_to_none=True)
        torch.manual_seed(3)
        x, pending = (torch.randn(2, 64, 128, device=dev).half().requires_grad_(not train) for _ in range(2))
        try:
            with torch.autocast("cuda", dtype=torch.float16):
                out = m.layer_list[0].forward_deferred(x, pending)[used]
        finally:
            TM.FUSE_LAYER = True
        if not out.requires_grad or (used == 0 and train in ("mlp", "post_attention_layernorm")):
            continue  # nothing to train stands before this output (of one node all outputs require a gradient)
        out.backward(torch.randn_like(out))
        results.append([out] + [t.grad for t in (x, pending)] + [p.grad for p in m.layer_list[0].parameters()])
    for one, four in zip(*results) if results else ():
        assert (one is None) == (four is None)
        assert one is None or torch.equal(one, four)


def test_a_pass_without_a_graph_holds_no_more_than_four_nodes(dev, monkeypatch):
    m = build(dev, layers=1, d=256, heads=4)
    x, pending = torch.randn(2, 128, 64, 256, device=dev).half().unbind(0)
    peaks = []
    for fused in (True, False):
        monkeypatch.setattr(TM, "FUSE_LAYER", fused)
        for _ in range(2):
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
                torch.cuda.reset_peak_memory_stats()
                before = torch.cuda.memory_allocated()
                out = m.layer_list[0].forward_deferred(x, pending)
            peaks.append(torch.cuda.max_memory_allocated() - before)
            del out
    assert peaks[1] <= peaks[3], peaks


def test_attention_with_nothing_to_train_before_it_is_not_differentiated(dev, monkeypatch):
    m = build(dev, bias=True, layers=1)
    for name, p in m.named_parameters():
        p.requires_grad_("mlp" in name or "post_attention_layernorm" in name)
    monkeypatch.setattr(layer, "_ATTENTION", (layer._ATTENTION[0], None))
    assert step(m, True, torch.float16)[2]["layer_list.0.post_attention_layernorm.weight"] is not None


@pytest.mark.parametrize("kind,name,calls_per_pass", [(TM.CausalAttention, "forward", 3), (TM.MLPBlock, "forward", 3), (TM.tnn.LayerNorm, "forward", 1),
                                                      (torch.nn.Module, "__call__", 8)])
def test_classes_patched_by_the_caller_are_called(kind, name, calls_per_pass, dev, monkeypatch):
    m = build(dev)
    ids = torch.zeros((2, 64), dtype=torch.long, device=dev)
    plain = step(m, False, torch.float16)
    own, calls = getattr(kind, name), []
    monkeypatch.setattr(kind, name, lambda self, *a, **k: (calls.append(type(self)), own(self, *a, **k))[1])
    assert_same(step(m, True, torch.float16), plain, torch.float16)
    assert len(calls) == calls_per_pass
    calls.clear()
    m.half()
    with torch.no_grad():
        m(ids, ids)
    assert len(calls) == calls_per_pass


def test_graph_of_a_step_goes_with_its_outputs(dev):
    """An output that the node held beside its saved tensors would keep the whole pass alive."""
    m = build(dev)
    step(m, True, torch.float16)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for _ in range(3):
        ids = torch.zeros((2, 64), dtype=torch.long, device=dev)
        with torch.autocast("cuda", dtype=torch.float16):
            out = m(ids, ids)
        del out, ids
    assert torch.cuda.memory_allocated() == before
