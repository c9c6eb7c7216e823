"""The input gradient's route: what follows a gradient beside its values
(forward mode, dispatch modes, tracers) gets the torch product, the weights
from an operator."""
import ctypes

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fw
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import _disable_current_modes

from distributed_gptq_amd import _ops
from distributed_gptq_amd.models import layers

M, N, K = 8, 64, 96


def fill(t, values):
    """Values into ``t``'s memory as a kernel writes them: by its address."""
    src = np.ascontiguousarray(values)
    ctypes.memmove(t.data_ptr(), src.ctypes.data, src.nbytes)


@pytest.fixture
def grad_input(monkeypatch):
    """layers._grad_input on the CPU, the kernels stood in for by numpy, and
    how often each ran."""
    W = np.random.default_rng(0).standard_normal((N, K)).astype(np.float32)
    ran = {"dequant": 0, "planes": 0}

    def dequant(packed, bits, scales, zeros, k, g_idx=None, group_size=0, dtype=torch.float32):
        ran["dequant"] += 1
        out = torch.empty(N, K, dtype=dtype)
        fill(out, W)
        return out

    def planes(grad, packed, bits, scales, zeros, k, group_size, perm=None):
        ran["planes"] += 1
        out = torch.empty(grad.shape[0], K, dtype=grad.dtype)
        with _disable_current_modes():
            values = (grad.detach().float() @ torch.from_numpy(W)).to(grad.dtype).view(torch.int16).numpy()
        fill(out, values)
        return out

    monkeypatch.setattr(_ops, "dequant", dequant)
    monkeypatch.setattr(_ops, "linear_grad_input", planes)
    monkeypatch.setattr(layers, "_planes_backward", lambda *a: True)
    q = (torch.zeros(N, K // 2, dtype=torch.uint8), torch.ones(N, 1).half(), torch.zeros(N, 1).half(),
         torch.zeros(K, dtype=torch.int32))

    def run(grad):
        return layers._grad_input(grad, *q, None, torch.bfloat16)
    run.ran, run.W = ran, torch.from_numpy(W)
    return run


def grads():
    g = torch.Generator().manual_seed(1)
    return torch.randn(M, N, generator=g).bfloat16(), torch.randn(M, N, generator=g).bfloat16()


def product(run, g):
    return (g.float() @ run.W).bfloat16()


def test_plain_gradient_takes_the_planes(grad_input):
    g, _ = grads()
    assert torch.equal(grad_input(g), product(grad_input, g))
    assert grad_input.ran == {"dequant": 0, "planes": 1}


def test_forward_mode_tangent(grad_input):
    g, t = grads()
    with fw.dual_level():
        y = fw.unpack_dual(grad_input(fw.make_dual(g, t)))
        assert y.tangent is not None and torch.equal(y.tangent, product(grad_input, t))
        assert torch.equal(y.primal, product(grad_input, g))
        # a level is open, but this gradient has no tangent
        assert fw.unpack_dual(grad_input(g)).tangent is None
    assert grad_input.ran["planes"] == 1


@pytest.mark.parametrize("trace", [lambda f, g: make_fx(f)(g),
                                   lambda f, g: torch.jit.trace(f, (g,), check_trace=False)])
def test_traces_hold_the_computation(grad_input, trace):
    g, other = grads()
    traced = trace(grad_input, g)
    assert grad_input.ran["planes"] == 0
    keep = [torch.full((N, K), float("nan")) for _ in range(8)]  # memory freed by the trace is not its result
    del keep
    before = grad_input.ran["dequant"]
    assert torch.equal(traced(other), product(grad_input, other))
    assert grad_input.ran["dequant"] == before + 1


def test_function_mode_sees_the_product(grad_input):
    from torch.overrides import TorchFunctionMode

    class Seen(TorchFunctionMode):
        names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    g, _ = grads()
    with Seen() as m:
        y = grad_input(g)
    assert grad_input.ran["planes"] == 0 and any("matmul" in n for n in m.names), m.names
    assert torch.equal(y, product(grad_input, g))
