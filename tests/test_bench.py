"""The benchmark's instrumented steps: every launch of a training step is seen, whichever way it reaches the library."""
import pytest
import torch

import bench
from tritonformer_amd import kernels as K


def test_every_native_launcher_is_accounted_for():
    native = K.launch()
    names = {n for n in dir(native) if callable(getattr(native, n)) and not n.startswith("__")} - {"set_check"}
    assert set(bench.NATIVE_CALLS) == names


@pytest.mark.gpu
@pytest.mark.parametrize("workload", ["gpt2-tiny-ctx256-bs2"])
def test_instrumented_step_sees_every_launch(workload, dev):
    L, d, nh, hd, f, S, B, lin_bias, alibi = bench.WORKLOADS[workload]
    model, tokens = bench.make_model(workload, dev, torch.float16)
    timer, launch = bench.GemmTimer(512), K.launch
    bench.run_steps(model, tokens, 1, torch.float16)
    with timer:
        bench.run_steps(model, tokens, 2, torch.float16)
    assert K.launch is launch
    seen = sum(c * bench.key_flop(key) for key, (c, _) in timer.by_shape.items())
    assert seen == pytest.approx(2 * bench.gemm_flops(L, d, f, S, B), rel=1e-9)
    calls = {family: cnt // 2 for family, (cnt, _, _) in timer.by_family.items()}
    # attention: forward and backward of each layer; LayerNorm: two per layer and the last, forward and backward, and
    # the sums of all their parameter gradients; the loss with its gradient
    assert calls == {"attention": 2 * L, "layernorm": 2 * (2 * L + 1) + 1, "cross_entropy": 1}
    flop = 7.0 * L * B * S * S * nh * hd
    assert timer.by_family["attention"][2] == pytest.approx(2 * flop, rel=1e-9)
    assert all(ms > 0 for _, ms in timer.by_shape.values())
