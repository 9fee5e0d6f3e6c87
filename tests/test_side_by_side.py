"""A product over matrices that lie apart against the product over their copy side by side, and a layer of which nothing is kept
against the graph nodes it stands for: the same bits."""
import pytest
import torch

import tritonformer_amd.transformer as TM
from tests.test_layer import build
from tritonformer_amd import _lib, linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,each,K,count", [(1, 64, 64, 3), (65, 128, 192, 3), (128, 1024, 1024, 3), (300, 256, 2048, 2), (960, 768, 768, 3),
                                            (8192, 256, 64, 3), (64, 192, 4096, 1), (700, 64, 128, 3)])
def test_side_by_side_gives_the_bits_of_the_copy(M, each, K, count, dtype, dev):
    lib = _lib.load()
    g = torch.Generator().manual_seed(11)
    a = torch.randn(M, K, generator=g).to(dtype).to(dev)
    parts = [(torch.randn(K, each, generator=g) / K ** 0.5).to(dtype).to(dev) for _ in range(count)]
    n, code, st = each * count, _lib.dtype_code(dtype), _lib.stream_ptr()
    nb = lib.tf_gemm_workspace_bytes(0, 1, M, n, K)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device=dev)
    whole, apart = torch.empty(M, n, dtype=dtype, device=dev), torch.full((M, n), float("nan"), dtype=dtype, device=dev)
    copy = torch.cat(parts, 1)
    _lib.check(lib.tf_gemm(st, code, 0, 1, M, n, K, a.data_ptr(), K, copy.data_ptr(), n, whole.data_ptr(), n, None, 0, ws.data_ptr(), nb))
    ptrs = (_lib._vp * count)(*[p.data_ptr() for p in parts])
    rc = lib.tf_gemm_side_by_side(st, code, M, each, count, K, a.data_ptr(), K, ptrs, each, apart.data_ptr(), n, ws.data_ptr(), nb)
    _lib.check(rc)  # tiles that divide each part: all of these are served
    assert torch.equal(apart, whole)


def test_side_by_side_refuses_what_it_does_not_serve(dev):
    lib = _lib.load()
    a = torch.randn(128, 128, device=dev).half()
    w = torch.randn(128, 128, device=dev).half()
    c = torch.empty(128, 384, device=dev).half()
    st = _lib.stream_ptr()

    def run(each=128, K=128, off=0, count=3, ldb=128):
        ptrs = (_lib._vp * 3)(w.data_ptr() + off, w.data_ptr(), w.data_ptr())
        return lib.tf_gemm_side_by_side(st, 0, 128, each, count, K, a.data_ptr(), 128, ptrs, ldb, c.data_ptr(), 384, None, 0)

    assert run() == 0
    assert run(each=96) == run(each=60) == run(K=96) == run(off=2) == run(ldb=64) == -4
    assert run(count=4) == run(count=0) == -1


@pytest.mark.parametrize("bias,alibi", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,heads", [(128, 2), (96, 3), (256, 4)])
def test_a_layer_in_one_call_gives_the_bits_of_its_nodes(bias, alibi, dtype, d, heads, dev, monkeypatch):
    m = build(dev, bias, alibi, dtype, d=d, heads=heads)
    ids = torch.arange(128, device=dev).view(2, 64) * 3
    calls = []
    native = _lib.launch().layer

    class Counting:
        def __getattr__(self, name):
            if name == "layer":
                return lambda *a: (calls.append(1), native(*a))[1]
            return getattr(_lib.launch(), name)

    monkeypatch.setattr(TM, "launch", lambda: Counting())
    with torch.no_grad():
        one = m(ids, None)
        assert len(calls) == 3
        TM.FUSE_LAYER = False
        try:
            nodes = m(ids, None)
        finally:
            TM.FUSE_LAYER = True
    assert torch.equal(one, nodes) and len(calls) == 3
    assert torch.equal(m(ids, None).detach(), nodes) and len(calls) == 3     # a graph is built: its nodes run
    with torch.inference_mode():
        assert torch.equal(m(ids, None), nodes)


def test_a_layer_in_one_call_leaves_other_forms_to_the_nodes(dev):
    """Tangents, traces, autocast and weights of another type: the graph nodes decide."""
    m = build(dev, param_dtype=torch.float16)
    ids = torch.arange(64, device=dev)[None]
    with torch.no_grad():
        plain = m(ids, None)
        layer = m.layer_list[0]
        x = torch.randn(1, 64, 128, device=dev).half()
        args = (x, None, layer.input_layernorm.weight, layer.input_layernorm.bias, 1e-5,
                [getattr(layer.attention, n).weight for n in ("q_proj", "k_proj", "v_proj", "out_proj")], 2, None,
                layer.post_attention_layernorm.weight, layer.post_attention_layernorm.bias, 1e-5,
                layer.mlp.dense_h_to_4h.weight, None, layer.mlp.dense_4h_to_h.weight, None)
        call = _lib.launch().layer
        assert call(*args) is not None
        for i, other in ((0, x.float()), (0, x.transpose(1, 2)), (0, x[0]), (1, x[:, :32]), (2, args[2][:64]), (6, 3), (11, args[13]),
                         (12, torch.zeros(128, device=dev)), (7, torch.zeros(2, 8, 8, device=dev).half())):
            assert call(*args[:i], other, *args[i + 1:]) is None, i
        import torch.autograd.forward_ad as fwAD

        with fwAD.dual_level():
            assert call(fwAD.make_dual(x, torch.ones_like(x)), *args[1:]) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert torch.equal(m(ids, None), plain)
        traced = torch.jit.trace(lambda t: t * (1.0 if call(t, *args[1:]) is None else 0.0), (x,), check_trace=False)
        assert torch.equal(traced(x), x)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,heads,batch", [(2048, 16, 1), (2048, 16, 4), (1024, 16, 2)])
def test_few_tokens_of_a_wide_layer_give_the_bits_of_the_nodes(d, heads, batch, bias, dtype, dev):
    """The first MLP product of these (2048 wide): two slices of the contraction without sign bits, one with them."""
    m = build(dev, bias, False, dtype, layers=2, d=d, heads=heads)
    ids = (torch.arange(64 * batch, device=dev) * 7 % 512).view(batch, 64)
    with torch.no_grad():
        one = m(ids, None)
        TM.FUSE_LAYER = False
        try:
            nodes = m(ids, None)
        finally:
            TM.FUSE_LAYER = True
    assert torch.equal(one, nodes)
    assert torch.equal(m(ids, None).detach(), nodes)


def test_products_without_sign_bits_are_left_to_the_nodes(dev, monkeypatch):
    """With RELU_BITS off the nodes take the product that may split its contraction."""
    m = build(dev, False, False, torch.float16, layers=2, d=2048, heads=16)
    ids = torch.arange(64, device=dev)[None]
    monkeypatch.setattr(linear, "RELU_BITS", False)
    with torch.no_grad():
        one = m(ids, None)
        monkeypatch.setattr(TM, "FUSE_LAYER", False)
        assert torch.equal(one, m(ids, None))


@pytest.mark.parametrize("first", [False, True])
def test_a_layer_in_one_call_holds_no_more_than_its_nodes(first, dev, monkeypatch):
    m = build(dev, False, False, torch.float16, layers=1, d=256, heads=4)
    x, pending = torch.randn(2, 128, 64, 256, device=dev).half().unbind(0)
    peaks = []
    for fused in (True, False):
        monkeypatch.setattr(TM, "FUSE_LAYER", fused)
        for _ in range(2):
            with torch.no_grad():
                torch.cuda.reset_peak_memory_stats()
                before = torch.cuda.memory_allocated()
                out = m.layer_list[0].forward_deferred(x, None if first else pending)
            peaks.append(torch.cuda.max_memory_allocated() - before)
            del out
    assert peaks[1] <= peaks[3], peaks


@pytest.mark.parametrize("odd", range(4))
def test_projections_at_odd_addresses_are_left_to_the_nodes(odd, dev, monkeypatch):
    """Views of one flat buffer, as optimizers and checkpoints make them: the nodes copy such weights to an aligned matrix."""
    m = build(dev, False, False, torch.float16, layers=1, d=2048, heads=16)
    att = m.layer_list[0].attention
    weight = getattr(att, ("q_proj", "k_proj", "v_proj", "out_proj")[odd]).weight
    flat = torch.empty(weight.numel() + 1, dtype=torch.float16, device=dev)
    flat[1:] = weight.detach().flatten()
    weight.data = flat[1:].view_as(weight)
    ids = torch.arange(128, device=dev).view(2, 64)
    answers = []
    native = _lib.launch().layer

    class Watching:
        def __getattr__(self, name):
            if name == "layer":
                return lambda *a: (answers.append(native(*a)), answers[-1])[1]
            return getattr(_lib.launch(), name)

    monkeypatch.setattr(TM, "launch", lambda: Watching())
    with torch.no_grad():
        one = m(ids, None)
        assert answers == [None]
        monkeypatch.setattr(TM, "FUSE_LAYER", False)
        assert torch.equal(one, m(ids, None))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,biased", [(1, 64, 64, True), (128, 6144, 2048, False), (300, 1000, 512, True), (2048, 8192, 2048, True),
                                          (1024, 37376, 128, False)])
def test_relu_without_its_bits_gives_the_bits_of_the_one_with(M, N, K, biased, dtype, dev):
    """The last two: whole rounds of large tiles, and columns that are cut off."""
    lib, st, code = _lib.load(), _lib.stream_ptr(), _lib.dtype_code(dtype)
    a, b = torch.randn(M, K, device=dev).to(dtype), (torch.randn(K, N, device=dev) / K ** 0.5).to(dtype)
    bias = torch.randn(N, device=dev).to(dtype) if biased else None
    ptr = bias.data_ptr() if biased else None
    c = [torch.full((M, N), float("nan"), dtype=dtype, device=dev) for _ in range(2)]
    bits = torch.empty(M, N // 8, dtype=torch.uint8, device=dev)
    _lib.check(lib.tf_gemm_relu_bits(st, code, code, 0, 1, M, N, K, a.data_ptr(), K, b.data_ptr(), N, c[0].data_ptr(), N, ptr, bits.data_ptr(),
                                     None, N // 8))
    _lib.check(lib.tf_gemm_relu(st, code, 0, 1, M, N, K, a.data_ptr(), K, b.data_ptr(), N, c[1].data_ptr(), N, ptr))
    assert torch.equal(*c)
    # where the one with bits is refused, so is this one
    for n, k in ((N, K - 8), (N - 4, K)):
        got = [f(n, k) for f in (
            lambda n, k: lib.tf_gemm_relu_bits(st, code, code, 0, 1, M, n, k, a.data_ptr(), K, b.data_ptr(), N, c[0].data_ptr(), N, ptr,
                                               bits.data_ptr(), None, N // 8),
            lambda n, k: lib.tf_gemm_relu(st, code, 0, 1, M, n, k, a.data_ptr(), K, b.data_ptr(), N, c[1].data_ptr(), N, ptr))]
        assert got[0] == got[1] != 0
