"""The native launch path against the Python launchers it stands in for: the same call with the native functions
answering None (the general path) gives the same bits, for operands of every form -- contiguous ones, which the
native path takes, and strided, misaligned or empty ones, which it hands back."""
import sys

import pytest
import torch

import tritonformer_amd
from tritonformer_amd import _lib
from tritonformer_amd import kernels as K


class HandsBack:
    def __getattr__(self, name):
        return lambda *args: None


def both(monkeypatch, call):
    outcomes = []
    for general in (False, True):
        with monkeypatch.context() as m:
            if general:
                m.setattr(K, "launch", HandsBack)
            try:
                out = call()
                outcomes.append([t for t in (out if isinstance(out, tuple) else (out,)) if isinstance(t, torch.Tensor)])
            except (ValueError, TypeError) as e:
                outcomes.append(type(e))
    native, general = outcomes
    if isinstance(general, type):
        assert native is general
        return
    assert len(native) == len(general)
    for a, b in zip(native, general):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


def forms(t):
    """`t`, and tensors equal to it: other strides, an odd start, every second column of a wider one."""
    wide = torch.zeros(t.shape[:-1] + (2 * t.shape[-1],), dtype=t.dtype, device=t.device)
    wide[..., ::2] = t
    odd = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)
    out = {"plain": t, "strided": wide[..., ::2], "odd": odd}
    if t.ndim >= 2:
        out["transposed"] = t.transpose(-1, -2).contiguous().transpose(-1, -2)
    return out


def randn(*shape, dtype=torch.float16):
    return torch.randn(*shape, device="cuda").to(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "strided", "odd", "transposed"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,k,n", [(1, 64, 64), (77, 128, 264), (130, 67, 33)])
def test_products(m, k, n, dtype, form, dev, monkeypatch):
    torch.manual_seed(m + k)
    a, b, bias, g = randn(2, m, k, dtype=dtype), randn(k, n, dtype=dtype), randn(n, dtype=dtype), randn(2, m, n, dtype=dtype)
    af, bf, gf, biasf = forms(a)[form], forms(b)[form], forms(g)[form], forms(bias).get(form, bias)
    both(monkeypatch, lambda: K.gemm(af, b, biasf, True))
    both(monkeypatch, lambda: K.gemm(a, bf, None))
    both(monkeypatch, lambda: K.gemm_relu_bits(af, bf, biasf))
    both(monkeypatch, lambda: K.mm_dw(af, gf, torch.float32))
    both(monkeypatch, lambda: K.mm_dw(a, gf))
    both(monkeypatch, lambda: K.unbroadcast_leading(gf))
    both(monkeypatch, lambda: K.mask_grad(gf, g))
    both(monkeypatch, lambda: K.mask_grad_sums(gf, g, torch.float32))
    both(monkeypatch, lambda: K.cast_pack([bf.float(), b.float()], dtype))
    act, bits = K.gemm_relu_bits(a, b, bias)
    if bits is not None:
        both(monkeypatch, lambda: K.mm_masked_bits(af, bf, bits, act))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "strided", "odd", "transposed"])
@pytest.mark.parametrize("d", [64, 129])
def test_rows(d, form, dev, monkeypatch):
    torch.manual_seed(d)
    x, r, g = (randn(2, 19, d) for _ in range(3))
    al, be = randn(d).float(), randn(d).float()
    xf, gf, alf = forms(x)[form], forms(g)[form], forms(al).get(form, al)
    both(monkeypatch, lambda: K.layernorm_fwd(xf, alf, be, 1e-5))
    both(monkeypatch, lambda: K.add_layernorm_fwd(xf, r, alf, be, 1e-5))
    y, mean, rstd = K.layernorm_fwd(x, al, be, 1e-5)
    for leave in (False, True):  # partial sums: the buffer's unused tail is whatever memory held
        both(monkeypatch, lambda: K.layernorm_bwd(gf, xf, alf, mean, rstd, leave)[: 1 if leave else 3])
        both(monkeypatch, lambda: K.add_layernorm_bwd(gf, r, xf, alf, mean, rstd, leave)[: 1 if leave else 3])
    for dtype in (torch.float32, torch.bfloat16):
        both(monkeypatch, lambda: K.softmax_fwd(xf.to(dtype)))
        both(monkeypatch, lambda: K.softmax_bwd(gf.to(dtype), x.to(dtype)))


@pytest.mark.gpu
@pytest.mark.parametrize("bias", ["none", "dense", "dense-odd-pitch", "alibi"])
@pytest.mark.parametrize("s,hd", [(64, 32), (192, 64), (96, 128)])
def test_attention(s, hd, bias, dev, monkeypatch):
    torch.manual_seed(s)
    b, nh = 2, 3
    extra = {"none": None, "dense": randn(nh, s + 8, s + 8), "dense-odd-pitch": randn(nh, s + 3, s + 3),
             "alibi": torch.tensor([0.5, 0.25, 0.125], device="cuda", dtype=torch.float16)}[bias]
    qkv, g = randn(b, s, 3, nh, hd), randn(b, s, nh * hd)
    out, lse = K.flash_packed_fwd(qkv, extra)
    both(monkeypatch, lambda: K.flash_packed_fwd(qkv, extra))
    for gf in forms(g).values():
        both(monkeypatch, lambda: K.flash_packed_bwd(gf, out, qkv, lse, extra))
    for q, k, v, go in [tuple(randn(b, s, nh, hd).transpose(1, 2) for _ in range(4)),
                        tuple(randn(b, nh, s, hd) for _ in range(4)),
                        (randn(b, nh, s, hd),) + tuple(randn(b, s, nh, hd).transpose(1, 2) for _ in range(3))]:
        both(monkeypatch, lambda: K.flash_wrapper_fwd(q, k, v, extra))
        o, l = K.flash_wrapper_fwd(q, k, v, extra)
        both(monkeypatch, lambda: K.flash_wrapper_bwd(go, o, q, k, v, l, extra))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "odd"])
def test_products_without_sign_bits_are_tried_once(form, dev, monkeypatch):
    """A contraction that no kernel writes or reads sign bits for (not a multiple of 64; operands at odd elements): the
    plain product follows the native refusal, without a second attempt through the general launcher."""
    torch.manual_seed(0)
    k = 72 if form == "plain" else 128
    a, b, bias, act = (forms(t)[form] for t in (randn(2, 77, k), randn(k, 264), randn(264), randn(2, 77, 264).relu()))
    bits = torch.zeros(2 * 77, 33, dtype=torch.uint8, device="cuda")
    want, masked = K.gemm(a, b, bias, True), K.gemm(a, b, None, False, act)
    monkeypatch.setattr(K, "_gemm_bits", lambda *args: pytest.fail("tried a second time"))
    out, none = K.gemm_relu_bits(a, b, bias)
    assert none is None and torch.equal(out, want)
    assert torch.equal(K.mm_masked_bits(a, b, bits, act), masked)
    with pytest.raises(ValueError):
        K.mm_masked_bits(a, b, bits)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(3, 1), (1, 4), (3, 4)])
def test_attention_of_expanded_operands(dims, dev, monkeypatch):
    """Batches or heads that share their memory: every one has results of its own."""
    torch.manual_seed(1)
    b, nh, s, hd = 3, 4, 128, 64
    small = [randn(b // dims[0], nh // dims[1], s, hd) for _ in range(3)]
    q, k, v = (t.expand(b, nh, s, hd) for t in small)
    g = randn(b, nh, s, hd)
    full = [t.contiguous() for t in (q, k, v)]
    want, lse = K.flash_wrapper_fwd(*full)
    grads = K.flash_wrapper_bwd(g, want, *full, lse)
    out, lse2 = K.flash_wrapper_fwd(q, k, v)
    assert torch.equal(out, want) and torch.equal(lse2, lse) and out.stride() == want.stride()
    for a, e in zip(K.flash_wrapper_bwd(g, out, q, k, v, lse), grads):
        assert torch.equal(a, e)
    both(monkeypatch, lambda: K.flash_wrapper_fwd(q, k, v))
    both(monkeypatch, lambda: K.flash_wrapper_bwd(g, out, q, k, v, lse))


@pytest.mark.gpu
def test_refused_calls_are_refused_alike(dev, monkeypatch):
    x, w = randn(2, 8, 64), randn(64, 64)
    for call in [lambda: K.gemm(x[0], w), lambda: K.gemm(x, w[:32]), lambda: K.gemm(x.float(), w.float()),
                 lambda: K.gemm(x, w.bfloat16()), lambda: K.gemm(x, w.cpu()), lambda: K.gemm(x, w, w[0, :32]),
                 lambda: K.layernorm_fwd(x[0], w[0], w[0], 1e-5), lambda: K.layernorm_fwd(x, w[0, :8], w[0, :8], 1e-5),
                 lambda: K.add_layernorm_fwd(x, x[:1], w[0], w[0], 1e-5), lambda: K.softmax_fwd(w),
                 lambda: K.mask_grad(x, x.bfloat16()), lambda: K.mm_dw(x, x[:1]), lambda: K.cast_pack([w, w[:32]], torch.float16),
                 lambda: K.flash_wrapper_fwd(*(randn(1, 1, 64, 48) for _ in range(3))),
                 lambda: K.flash_wrapper_fwd(*(randn(1, 1, 80, 64) for _ in range(3)))]:
        with pytest.raises((ValueError, TypeError)):
            call()
        both(monkeypatch, call)


@pytest.mark.gpu
def test_attention_bias_without_dimensions_is_refused_alike(dev, monkeypatch):
    qkv = randn(1, 64, 3, 2, 64)
    bias = qkv.new_zeros(())
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    for call in (lambda: K.flash_wrapper_fwd(q, k, v, bias), lambda: K.flash_packed_fwd(qkv, bias)):
        with pytest.raises(ValueError):
            call()
        both(monkeypatch, call)


def test_tensors_off_the_gpu_are_handed_back():
    native = K.launch()
    x, w = torch.zeros(1, 8, 64, dtype=torch.float16), torch.zeros(64, 64, dtype=torch.float16)
    assert native.linear(x, w, None, False) is None
    assert native.layernorm(x, None, w[0], w[0], 1e-5) is None
    assert native.softmax_fwd(x) is None and native.cast_pack([w], torch.bfloat16) is None
    assert native.linear("x", w, None, False) is None
    with pytest.raises(ValueError):
        K.gemm(x, w)
    with pytest.raises(TypeError):
        native.linear(x, w)


def test_a_module_of_another_torch_is_refused(monkeypatch):
    monkeypatch.setattr(_lib, "_launch", None)
    assert _lib.launch().host_abi.startswith(f"torch {torch.__version__} ")
    monkeypatch.setattr(_lib, "_launch", None)
    with monkeypatch.context() as m:  # it loads, but was compiled against another torch
        m.setattr(torch, "__version__", "0.0.0")
        with pytest.raises(ImportError, match="rebuild"):
            _lib.launch()
    assert _lib._launch is None
    with monkeypatch.context() as m:  # it does not load at all
        m.delattr(tritonformer_amd, "_launch", raising=False)
        m.setitem(sys.modules, "tritonformer_amd._launch", None)
        with pytest.raises(ImportError, match="rebuild"):
            _lib.launch()


# ------------------------------------------------------------------------------------------ several launches in one call
class _OneByOne:
    """The extension module without the functions that run a whole block."""

    def __init__(self, native):
        self._native = native

    def __getattr__(self, name):
        return (lambda *a: None) if name in ("attn_block", "attn_block_dqkv", "mlp") else getattr(self._native, name)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("batch,seq,d,heads,ffn,bias", [(2, 64, 128, 2, 512, False), (3, 192, 96, 3, 200, True),
                                                        (1, 96, 128, 1, 129, True)])
def test_blocks_in_one_call_give_the_bits_of_their_launches(dtype, autocast, batch, seq, d, heads, ffn, bias, dev, monkeypatch):
    """Attention and MLP blocks, forward and backward: weights in 16 bits and fp32 masters, contractions that no sign bits
    are served for (96 columns), widths that no row of chunks fits (129)."""
    import tritonformer_amd as T
    from tritonformer_amd import kernels as K

    g = torch.Generator().manual_seed(5)
    wt = torch.float32 if autocast else dtype
    rnd = lambda *s: (torch.randn(s, generator=g) * 0.1).to(dev)
    x = rnd(batch, seq, d).to(dtype)
    wa = [rnd(d, d).to(wt) for _ in range(4)]
    wm = [rnd(d, ffn).to(wt), rnd(ffn).to(wt) if bias else None, rnd(ffn, d).to(wt), rnd(d).to(wt) if bias else None]
    slopes = torch.tensor([2.0 ** -(i + 1) for i in range(heads)], device=dev, dtype=torch.float16) if bias else None

    def run():
        leaves = [None if t is None else t.clone().requires_grad_(True) for t in [x, *wa, *wm]]
        with torch.autocast("cuda", dtype=dtype, enabled=autocast):
            out = T.mlp_fused_relu.apply(T.attention_block.apply(*leaves[:5], heads, slopes), *leaves[5:])
            assert torch.is_autocast_enabled("cuda") == autocast
        out.backward(torch.ones_like(out))
        return [out] + [t.grad for t in leaves if t is not None]

    together = run()
    native = K.launch()
    monkeypatch.setattr(K, "launch", lambda: _OneByOne(native))
    for a, b in zip(together, run()):
        assert torch.equal(a, b)


class _Counted:
    """The extension module; counts the answers of the functions that run a whole block, and those that are None."""

    def __init__(self, native):
        self._native, self.answers = native, {}

    def __getattr__(self, name):
        fn = getattr(self._native, name)
        if name not in ("attn_block", "attn_block_dqkv", "mlp", "adamw"):
            return fn

        def counted(*args):
            out = fn(*args)
            served, declined = self.answers.get(name, (0, 0))
            self.answers[name] = (served + (out is not None), declined + (out is None))
            return out

        return counted


@pytest.mark.gpu
@pytest.mark.parametrize("autocast,cache", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("form", ["plain", "strided", "odd", "transposed"])
def test_blocks_serve_plain_operands_and_hand_back_the_others(form, autocast, cache, dev, monkeypatch):
    """Inputs, weights and biases of every form, kept 16-bit weights: the bits of the launches one by one, and the block
    functions are the ones that ran wherever every operand is plain (the weights that the cache holds in 16 bits are, whatever
    form they were converted from)."""
    import tritonformer_amd as T
    from tritonformer_amd import kernels as K

    torch.manual_seed(11)
    dtype, wt = torch.float16, torch.float32 if autocast else torch.float16
    shape = lambda t: forms(t).get(form, t)
    x = shape(randn(2, 64, 128))
    ws = [torch.nn.Parameter(shape(torch.randn(s, device=dev) * 0.1).to(wt)) for s in
          [(128, 128)] * 4 + [(128, 512), (512,), (512, 128), (128,)]]
    grad = shape(randn(2, 64, 128))
    T.set_weight_cast_cache(cache)

    def run():
        T.clear_weight_cast_cache()
        for w in ws:
            w.grad = None
        leaf = x.detach().requires_grad_(True)
        with torch.autocast("cuda", dtype=dtype, enabled=autocast):
            out = T.mlp_fused_relu.apply(T.attention_block.apply(leaf, *ws[:4], 2, None), *ws[4:])
        out.backward(grad)
        return [out.detach(), leaf.grad] + [w.grad for w in ws]

    try:
        native = K.launch()
        counted = _Counted(native)
        monkeypatch.setattr(K, "launch", lambda: counted)
        together = run()
        monkeypatch.setattr(K, "launch", lambda: _OneByOne(native))
        for a, b in zip(together, run()):
            assert torch.equal(a, b)
    finally:
        T.set_weight_cast_cache(False)
    assert set(counted.answers) >= {"attn_block", "attn_block_dqkv"}
    if form == "plain":
        assert all(declined == 0 for _, declined in counted.answers.values()) and ("mlp" in counted.answers) == (not cache)


@pytest.mark.gpu
@pytest.mark.parametrize("shadow_dtype", [None, torch.float16, torch.bfloat16])
def test_adamw_takes_its_tensors_natively_or_one_by_one(shadow_dtype, dev, monkeypatch):
    """The native hand-over of the tensors against the ctypes one: the same parameters, moments and copies; an empty parameter
    goes the second way, with every other of its step."""
    from tritonformer_amd import optim

    native, counted = optim.launch(), []

    def steps(launch, sizes):
        monkeypatch.setattr(optim, "launch", launch)
        g = torch.Generator().manual_seed(2)
        params = [torch.randn(s, generator=g).to(dev).requires_grad_(True) for s in sizes]
        opt = optim.AdamW(params, lr=3e-3, weight_decay=0.1, shadow_dtype=shadow_dtype)
        for step in range(3):
            for i, p in enumerate(params):
                p.grad = torch.randn(p.shape, generator=g).to(dev) if (step, i) != (1, 0) else None  # steps of their own from here
            versions = [p._version for p in params]
            opt.step()
            assert all((p._version > v) == (p.grad is not None) for p, v in zip(params, versions))
        return [t for p in params for t in (p.detach(), opt.state[p]["exp_avg"], opt.state[p]["exp_avg_sq"], opt.shadow(p))]

    def through():
        counted.append(_Counted(native))
        return counted[-1]

    for sizes in ([(7,), (64, 33), (1000,)], [(7,), (0,), (64, 33)]):
        del counted[:]
        for a, b in zip(steps(through, sizes), steps(HandsBack, sizes)):
            assert a is b is None or torch.equal(a, b)
        served = sum(c.answers.get("adamw", (0, 0))[0] for c in counted)
        assert served == (3 + 1 if (0,) not in sizes else 1)


def test_a_body_that_raises_leaves_autocast_as_it_was():
    """The node's body runs with autocast off, and the flag is back on whichever way the body ends."""
    from tritonformer_amd._amp import amp_fwd

    seen = []

    class Ctx:
        pass

    @amp_fwd
    def body(ctx, fail):
        seen.append(torch.is_autocast_enabled("cuda"))
        if fail:
            raise RuntimeError("body")
        return 1

    was = torch.is_autocast_enabled("cuda")
    try:
        torch.set_autocast_enabled("cuda", True)
        assert body(Ctx(), False) == 1 and torch.is_autocast_enabled("cuda")
        with pytest.raises(RuntimeError, match="body"):
            body(Ctx(), True)
        assert torch.is_autocast_enabled("cuda")
        torch.set_autocast_enabled("cuda", False)
        with pytest.raises(RuntimeError, match="body"):
            body(Ctx(), True)
        assert not torch.is_autocast_enabled("cuda")
    finally:
        torch.set_autocast_enabled("cuda", was)
    assert seen == [False, False, False]


def test_pick_takes_what_the_exhaustive_search_takes():
    """The packing of pending weight gradients against the search over ways to reach a sum, written out."""
    import random

    from tritonformer_amd import _deferred as D

    class Item:
        def __init__(self, tiles, key):
            self.tiles, self.key = tiles, key

    def search(items, cus, split):
        reach = {0: ()}
        for i, it in enumerate(items):
            if it.key == items[0].key:
                for s, sub in list(reach.items()):
                    if len(sub) < D._MAX_GROUP:
                        reach.setdefault(s + it.tiles, sub + (i,))
        best, best_rank = None, None
        for s, sub in reach.items():
            if sub:
                f = 0.9 * s * (cus // s) / cus if split and 2 * s <= cus else s / (-(-s // cus) * cus)
                rank = (min(f, D._FILL), 0 in sub, s)
                if best_rank is None or rank > best_rank:
                    best, best_rank = sub, rank
        return best, best_rank[0]

    rng = random.Random(3)
    for _ in range(200):
        items = [Item(rng.choice([1, 3, 9, 27, 36, 64, 200, 432]), rng.random() < 0.9) for _ in range(rng.randint(1, 26))]
        for split in (False, True):
            assert D._pick(items, 256, split) == search(items, 256, split)
