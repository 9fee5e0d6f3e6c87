"""A decoder layer as one node of the autograd graph."""
from torch.autograd import Function

from ._amp import amp_bwd, amp_fwd
from .attention import AttentionBlock
from .layernorm import AddLayerNorm, LayerNorm
from .linear import MLPReLU


class _Part:
    """Stands in for the context of one of the Functions whose bodies make up the layer.  It holds no tensor of the forward pass
    beyond it (an output held by the node that made it would keep itself alive): these go through the layer's own
    ``save_for_backward``, in the order of the parts."""

    def __init__(self, arg_dtypes, amp_active):
        self.arg_dtypes, self.amp_active = arg_dtypes, amp_active

    def save_for_backward(self, *tensors):
        self.saved_tensors = tensors

    def set_materialize_grads(self, value):
        pass

    def release(self):
        tensors, self.saved_tensors = self.saved_tensors, None
        return tensors

    def restored(self, tensors, input_needs_grad):
        part = object.__new__(_Part)
        part.__dict__.update(self.__dict__)
        part.saved_tensors, part.needs_input_grad = tensors, (input_needs_grad,)
        return part


# the bodies, without the autocast wrapper: the layer's own has done its work
_LN, _ADD_LN, _ATTENTION, _MLP = [(f.forward.__wrapped__, f.backward.__wrapped__)
                                  for f in (LayerNorm, AddLayerNorm, AttentionBlock, MLPReLU)]


class DecoderLayer(Function):
    """``apply(x, pending | None, g1, b1, eps1, Wq, Wk, Wv, Wo, heads, attn_bias | None, g2, b2, eps2, W1, c1 | None, W2,
    c2 | None) -> (stream, MLP output)``: with x + pending as the incoming residual stream, ``stream = x + pending +
    attention_block(layernorm(x + pending))`` and the MLP of its LayerNorm, still to be added (the reference's TransformerLayer,
    transformer.py:240-251, up to its last addition).  The kernels of AddLayerNorm (LayerNorm without ``pending``),
    AttentionBlock, AddLayerNorm and MLPReLU, in their order in both directions, and the same bits; in the first layer
    the two gradients of the stream are summed before their rounding, in the LayerNorm kernel, not after it.

    One node for the four: at a few hundred tokens a pass is bound by the host, and a node costs 20 us of it forward and
    20 us backward beside its launches."""

    @staticmethod
    @amp_fwd(keep=tuple(range(2, 18)))
    def forward(ctx, x, pending, g1, b1, eps1, wq, wk, wv, wo, heads, attn_bias, g2, b2, eps2, w1, c1, w2, c2):
        dt, amp = ctx.arg_dtypes, ctx.amp_active
        ln1, attn, ln2, mlp = parts = [_Part(dt[:1] + dt[2:5], amp), _Part(dt[:1] + dt[5:11], amp), _Part(dt[:2] + dt[11:14], amp),
                                       _Part(dt[:1] + dt[14:], amp)]
        ctx.first = pending is None
        if pending is None:
            normed = _LN[0](ln1, x, g1, b1, eps1)
        else:
            x, normed = _ADD_LN[0](ln1, x, pending, g1, b1, eps1)
        branch = _ATTENTION[0](attn, normed, wq, wk, wv, wo, heads, attn_bias)
        stream, normed = _ADD_LN[0](ln2, x, branch, g2, b2, eps2)
        out = _MLP[0](mlp, normed, w1, c1, w2, c2)
        saved = [part.release() for part in parts]
        ctx.parts, ctx.counts = parts, [len(t) for t in saved]
        ctx.save_for_backward(*[t for tensors in saved for t in tensors])
        return stream, out

    @staticmethod
    @amp_bwd
    def backward(ctx, grad_stream, grad_out):
        need = ctx.needs_input_grad
        need1 = need[0] or need[1] or need[2] or need[3]              # the LayerNorm ahead of the attention
        need2 = need1 or any(need[5:9]) or need[11] or need[12]       # the one ahead of the MLP
        tensors, parts, at = ctx.saved_tensors, [], 0
        for part, count, needed in zip(ctx.parts, ctx.counts, (True, need1, True, need2)):
            parts.append(part.restored(tensors[at:at + count], needed))
            at += count
        # what the parts kept goes with each of them, as it does from node to node: the gradients of a part take its place
        ctx.maybe_clear_saved_tensors()
        del tensors, part
        d_normed, d_w1, d_c1, d_w2, d_c2 = _MLP[1](parts.pop(), grad_out)
        mlp_grads = (d_w1, d_c1, d_w2, d_c2)
        if not need2:
            return (None,) * 14 + mlp_grads
        dx, _, d_g2, d_b2, _ = _ADD_LN[1](parts.pop(), grad_stream, d_normed)
        d_normed = None
        d_normed, d_wq, d_wk, d_wv, d_wo, _, _ = _ATTENTION[1](parts.pop(), dx)
        grads = (d_wq, d_wk, d_wv, d_wo, None, None, d_g2, d_b2, None) + mlp_grads
        if not need1:
            return (None,) * 5 + grads
        # LayerNorm keeps what AddLayerNorm keeps: in the first layer this adds the gradient that x has beside its LayerNorm
        dx, _, d_g1, d_b1, _ = _ADD_LN[1](parts.pop(), dx, d_normed)
        return (dx, None if ctx.first else dx, d_g1, d_b1, None) + grads
