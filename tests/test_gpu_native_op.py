"""The native gptq::linear_rows behind the modules: the same bits as
gptq::linear over the forms a call can take, and the calls it leaves to it."""
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
