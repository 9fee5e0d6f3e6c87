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

    def __init__(self, arg_dtypes, amp_active, keep):
        self.arg_dtypes, self.amp_active, self.keep = arg_dtypes, amp_active, keep

    def save_for_backward(self, *tensors):
        self.saved_tensors = tensors if self.keep else ()

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
        # the node has its edges by now: none where no graph is built, and nothing is then kept beyond its last reader
        ln1, attn, ln2, mlp = parts = [_Part(types, amp, bool(ctx.next_functions))
                                       for types in (dt[:1] + dt[2:5], dt[:1] + dt[5:11], dt[:2] + dt[11:14], dt[:1] + dt[14:])]
        ctx.set_materialize_grads(False)  # an unused output arrives as None, not as zeros
        ctx.first = pending is None
        if pending is None:
            normed = _LN[0](ln1, x, g1, b1, eps1)
        else:
            x, normed = _ADD_LN[0](ln1, x, pending, g1, b1, eps1)
        branch = _ATTENTION[0](attn, normed, wq, wk, wv, wo, heads, attn_bias)
        stream, normed = _ADD_LN[0](ln2, x, branch, g2, b2, eps2)
        del x, branch
        out = _MLP[0](mlp, normed, w1, c1, w2, c2)
        saved = [part.release() for part in parts]
        ctx.parts, ctx.counts = parts, [len(t) for t in saved]
        ctx.save_for_backward(*[t for tensors in saved for t in tensors])
        return stream, out

    @staticmethod
    @amp_bwd
    def backward(ctx, grad_stream, grad_out):
        need = ctx.needs_input_grad
        need1 = any(need[:4])                         # the LayerNorm ahead of the attention
        attended = need1 or any(need[5:9])            # the attention
        need2 = attended or need[11] or need[12]      # the LayerNorm ahead of the MLP
        tensors, parts, at = ctx.saved_tensors, [], 0
        for part, count, needed in zip(ctx.parts, ctx.counts, (True, need1, True, need2)):
            parts.append(part.restored(tensors[at:at + count], needed))
            at += count
        # what the parts kept goes with each of them, as it does from node to node: the gradients of a part take its place
        ctx.maybe_clear_saved_tensors()
        del tensors, part
        grads, d_normed, mlp = [None] * 18, None, parts.pop()
        if grad_out is not None:
            d_normed, *grads[14:] = _MLP[1](mlp, grad_out)
        del mlp, grad_out
        if need2:
            dx, _, *grads[11:14] = _ADD_LN[1](parts.pop(), grad_stream, d_normed)
            d_normed = None
        if attended:
            d_normed, *grads[5:11] = _ATTENTION[1](parts.pop(), dx)
        if need1:
            # LayerNorm keeps what AddLayerNorm keeps: in the first layer this adds the gradient that x has beside its LayerNorm
            dx, _, *grads[2:5] = _ADD_LN[1](parts.pop(), dx, d_normed)
            grads[:2] = dx, None if ctx.first else dx
        return tuple(grads)
