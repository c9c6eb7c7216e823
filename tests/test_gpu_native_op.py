"""The native gptq::linear_rows behind the modules: the same bits as
gptq::linear over the forms a call can take, and the calls it leaves to it."""
import warnings

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


def layer(N, K, bits, gs, act=False, bias=True, packed=True):
    from distributed_gptq_amd.models import QuantizedLinear
    g = torch.Generator(device="cuda").manual_seed(N + K + bits)
    ng = -(-K // gs)
    codes = torch.randint(0, 2 ** bits, (N, K), generator=g, device="cuda", dtype=torch.uint8)
    s = torch.rand(N, ng, generator=g, device="cuda") * 1e-2 + 1e-3
    z = torch.randint(0, 2 ** bits, (N, ng), generator=g, device="cuda").half()
    gi = torch.arange(K, dtype=torch.int32, device="cuda") // gs
    if act:
        gi = gi[torch.randperm(K, generator=g, device="cuda")]
    q = QuantizedLinear(bits, gs, K, N, bias=bias, packed=packed).cuda()
    q.pack_weights(codes, s, z, gi)
    if bias:
        q.bias.data = torch.randn(N, generator=g, device="cuda")
    return q


def general(q, x):
    args = (x, q.qweight, q.scales, q.zeros, q.g_idx, q.bias)
    return torch.ops.gptq.linear(*args, q.perm) if q.perm.numel() else torch.ops.gptq.linear(*args)


class Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,bits,gs,act,bias,packed", [
    (256, 512, 4, 128, False, True, True),
    (261, 384, 3, 128, True, False, True),     # odd rows, act-order
    (128, 1000, 4, 100, False, True, True),    # ragged columns: the generic kernels
    (96, 256, 8, 256, False, True, False),     # one code per byte, per channel
    (4096, 10240, 4, 128, False, False, True),  # split-K partials in the workspace at M = 16
])
def test_same_bits(N, K, bits, gs, act, bias, packed, dtype):
    q = layer(N, K, bits, gs, act, bias, packed)
    xs = [torch.randn(*shape, K, device="cuda").to(dtype) for shape in ((1,), (2, 3), (16,), (33,))]
    xs.append(torch.randn(4, 2 * K, device="cuda").to(dtype)[:, ::2])
    xs.append(torch.randn(K, device="cuda").to(dtype))
    with torch.no_grad():
        for x in xs:
            y = q(x)
            assert y.shape == (*x.shape[:-1], N) and torch.equal(y, general(q, x))
    with torch.inference_mode():
        assert torch.equal(q(xs[2]), general(q, xs[2]))


def test_calls_left_to_the_operator():
    q = layer(256, 512, 4, 128)
    x = torch.randn(8, 512, device="cuda").half()
    with torch.no_grad(), Names() as m:
        y = q(x)
    assert any("gptq.linear.default" in n for n in m.seen), m.seen
    assert torch.equal(q(x.clone().requires_grad_(True)).detach(), y)
    assert q(x).requires_grad  # through the bias
    with torch.no_grad():
        v = torch.func.vmap(q)(x.unsqueeze(1))
    assert torch.equal(v.squeeze(1), torch.cat([general(q, r[None]) for r in x]).detach())
    with torch.no_grad():
        with pytest.raises(TypeError):
            q(x.double())
        with pytest.raises(ValueError):
            q(x[:0])
        for shape in ((8, 1024), (8, 256), (1024,)):  # whole rows of K, but not K wide
            with pytest.raises(RuntimeError):
                q(torch.zeros(shape, device="cuda").half())
        q.qweight.data = q.qweight[:, :-1].contiguous()
        with pytest.raises(ValueError):
            q(x)


@pytest.mark.parametrize("error", [ImportError("not built"), OSError("undefined symbol"), None])
def test_without_the_native_library(monkeypatch, error, tmp_path):
    """An install with libgptq_hip.so alone serves through gptq::linear."""
    from distributed_gptq_amd import _lib
    from distributed_gptq_amd.models import layers

    def load(path=None):
        raise error
    monkeypatch.setattr(layers, "_rows_op", None)
    if error is not None:
        monkeypatch.setattr(_lib, "load_torch_ops", load)
    else:  # the loader's own answer to a missing file
        monkeypatch.setattr(_lib, "_torch_ops", False)
        loader, missing = _lib.load_torch_ops, str(tmp_path / "libgptq_torch.so")
        monkeypatch.setattr(_lib, "load_torch_ops", lambda: loader(missing))
    q = layer(256, 512, 4, 128)
    x = torch.randn(8, 512, device="cuda").half()
    with torch.no_grad():
        with pytest.warns(RuntimeWarning, match="native operator is not available"):
            y = q(x)
        assert torch.equal(y, general(q, x)) and torch.equal(q(x), y)
    assert layers._rows_op is False


def test_failures_are_raised_and_refusals_left(monkeypatch):
    """A failure of the native operator is not run again through gptq::linear;
    a status is the library's own error type."""
    from distributed_gptq_amd import _lib
    from distributed_gptq_amd.models import layers
    q = layer(256, 512, 4, 128)
    x = torch.randn(8, 512, device="cuda").half()
    with torch.no_grad():
        y = q(x)
        for error in (ValueError("refused"), TypeError("refused")):
            def refuse(*a, error=error):
                raise error
            monkeypatch.setattr(layers, "_rows_op", refuse)
            assert torch.equal(q(x), y)
        monkeypatch.setattr(torch.ops.gptq, "linear", None)  # not called from here on
        for error, kind, text in (
                (torch.OutOfMemoryError("no memory"), torch.OutOfMemoryError, "no memory"),
                (RuntimeError("a device error"), RuntimeError, "a device error"),
                (RuntimeError("gptq_linear_ws failed (status 5): launch"), _lib.GPTQLibraryError, "launch")):
            def fail(*a, error=error):
                raise error
            monkeypatch.setattr(layers, "_rows_op", fail)
            with pytest.raises(kind, match=text) as got:
                q(x)
            assert kind is not _lib.GPTQLibraryError or got.value.status == _lib.ERR_LAUNCH


def test_tensors_on_two_devices_are_refused():
    q = layer(256, 512, 4, 128)
    q.scales.data = q.scales.cpu()
    with torch.no_grad(), pytest.raises(RuntimeError, match="GPU tensor"):
        q(torch.randn(8, 512, device="cuda").half())


def test_scales_that_require_a_gradient():
    """No gradient reaches them, but the call is part of the graph, and its
    backward is gptq::linear's (the native operator has none: it would warn)."""
    q = layer(256, 512, 4, 128, bias=False)
    x = torch.randn(8, 512, device="cuda").half()
    assert not q(x).requires_grad
    for t in (q.scales, q.zeros):
        t.requires_grad_(True)
        y = q(x)
        assert y.requires_grad
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            y.float().sum().backward()
        assert t.grad is None
        with torch.no_grad():
            assert not q(x).requires_grad
        t.requires_grad_(False)
