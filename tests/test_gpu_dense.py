"""The dense MFMA product, the transposed weight planes and the row-wise
dequantisation, at the edges of their tiles, against fp64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.bfloat16]


def half_ulp(ref, dtype):
    """Half a unit in the last place of ``dtype`` at |ref| (fp64)."""
    p, emin = (11, -14) if dtype == torch.float16 else (8, -126)
    e = torch.floor(torch.log2(ref.abs().clamp(min=2.0 ** emin))).clamp(min=emin)
    return torch.exp2(e - p)


def check(y, ref, mag, depth):
    """|y - ref| within half an ulp of y's type plus the worst case of an fp32
    sum of ``depth`` roundings over terms of total magnitude ``mag``."""
    acc = depth * 2.0 ** -24 * mag
    bound = half_ulp(ref.abs() + acc, y.dtype) + acc
    worst = ((y.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 64),           # one row, the smallest N and K
    (255, 136, 128),      # inside one half tile and past it
    (257, 264, 192),      # one row and one chunk into the next tiles, an odd stage count
    (513, 1000, 4096),
    (4096, 4096, 64),     # 256 whole tiles
    (4300, 4096, 128),    # a whole round and 16 tiles as halves
    (6200, 4104, 64),     # a whole round and more than 128 tiles
])
def test_matmul_nt(M, N, K, dtype):
    from distributed_gptq_amd import _ops
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(dtype)
    bias = torch.randn(N, generator=g, device="cuda")
    xd, wd = x.double(), w.double()
    ref, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    check(_ops.matmul_nt(x, w), ref, mag, K)
    for b in (bias, bias.to(dtype)):
        check(_ops.matmul_nt(x, w, b), ref + b.double(), mag + b.double().abs(), K + 1)


def test_matmul_nt_misaligned_and_strided():
    from distributed_gptq_amd import _ops
    g = torch.Generator(device="cuda").manual_seed(1)
    flat = torch.randn(300 * 64 + 1, generator=g, device="cuda").half()
    w = torch.randn(64, 72, generator=g, device="cuda").half().t()
    x = flat[1:].view(300, 64)
    ref = x.double() @ w.double().t()
    check(_ops.matmul_nt(x, w), ref, x.double().abs() @ w.double().abs().t(), 64)


def make_layer(N, K, bits, gs, act, seed, packed=True, fractional=False):
    from distributed_gptq_amd.models import QuantizedLinear
    rng = np.random.default_rng(seed)
    ng = -(-K // gs)
    codes = torch.from_numpy(rng.integers(0, 2 ** bits, (N, K)).astype(np.uint8)).cuda()
    scales = torch.from_numpy(rng.uniform(1e-3, 1e-2, (N, ng))).half().cuda()
    zeros = rng.integers(0, 2 ** bits, (N, ng)).astype(np.float64)
    if fractional:
        zeros[N // 2, ng - 1] += 0.375  # one zero point off the integers
    zeros = torch.from_numpy(zeros).half().cuda()
    gi = torch.arange(K, dtype=torch.int32, device="cuda") // gs
    if act:
        gi = gi[torch.from_numpy(rng.permutation(K)).cuda()]
    q = QuantizedLinear(bits, gs, K, N, bias=False, packed=packed).cuda()
    q.pack_weights(codes, scales, zeros, gi)
    W = (codes.double() - zeros.double()[:, gi.long()]) * scales.double()[:, gi.long()]
    return q, W


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,K,bits,gs,act,packed,fractional", [
    (64, 32, 4, 32, False, True, False),      # the smallest
    (192, 160, 3, 32, True, True, False),     # columns past a 128-column block
    (576, 1056, 2, 96, False, True, False),
    (128, 288, 8, 288, False, True, False),   # three planes
    (128, 288, 8, 96, True, False, False),    # one code per byte
    (320, 416, 4, 32, True, True, True),      # a fractional zero: three planes
])
def test_input_gradient_planes(N, K, bits, gs, act, packed, fractional, dtype):
    from distributed_gptq_amd import _ops
    q, W = make_layer(N, K, bits, gs, act, N + K + bits, packed, fractional)
    g = torch.Generator(device="cuda").manual_seed(N)
    perm = q.perm if q.perm.numel() else None
    for M in (1, 130, 300):
        go = (torch.randn(M, N, generator=g, device="cuda") * 1e-2).to(dtype)
        gx = _ops.linear_grad_input(go, q.qweight, bits if packed else 0, q.scales, q.zeros, K, gs, perm)
        # (the fp32 weight rounds (q - z) s once, the planes hold that value)
        check(gx, go.double() @ W, go.double().abs() @ W.abs(), 6 * N)


@pytest.mark.parametrize("dtype", DTYPES)
def test_input_gradient_of_infinities(dtype):
    """An infinite or NaN gradient gives what the unsplit product gives: the
    weights' zero low planes are no terms of the sum."""
    from distributed_gptq_amd import _ops
    q, W = make_layer(128, 256, 4, 64, False, 5)
    go = torch.randn(70, 128, device="cuda").to(dtype)
    go[3, 17] = float("inf")
    go[40, 5] = float("nan")
    go[66, 100] = -float("inf")
    gx = _ops.linear_grad_input(go, q.qweight, 4, q.scales, q.zeros, 256, 64)
    ref = (go.float() @ W.float()).to(dtype)
    assert torch.equal(torch.isnan(gx), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert inf.any() and torch.equal(gx[inf], ref[inf]) and torch.equal(torch.isinf(gx), inf)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(300, 192, 544), (2304, 192, 3840)])  # tiles as halves; 135 whole tiles
def test_tiles_with_infinities(M, N, K, dtype):
    """Infinite and NaN gradients and scales, and sums that are too large for
    the type, in some tiles: the unsplit product's infinities and NaNs there,
    every other value as without them."""
    from distributed_gptq_amd import _ops
    q, _ = make_layer(N, K, 4, 32, True, 6)
    go = (torch.randn(M, N, device="cuda") * 1e-2).to(dtype)
    clean = _ops.linear_grad_input(go, q.qweight, 4, q.scales, q.zeros, K, 32, q.perm)
    go[5, 7], go[6], go[M - 1, N - 1], go[M // 2, 3] = float("inf"), -float("inf"), float("inf"), float("nan")
    go[M // 2, :2] = 0
    q.scales[N // 2, 2], q.scales[1, 3] = float("inf"), float("-inf")
    go[9] = torch.finfo(dtype).max if dtype == torch.float16 else 1e30  # (bf16 has fp32's range)
    W = q.unpack_weights()
    ref32 = go.float() @ W
    # (row 9's sums next to the largest value round to it or past it)
    edge = (ref32[9].abs() / torch.finfo(dtype).max - 1).abs() < 0.01
    gx = _ops.linear_grad_input(go, q.qweight, 4, q.scales, q.zeros, K, 32, q.perm)
    ref = ref32.to(dtype)
    gx[9, edge], ref[9, edge] = 0, 0
    assert torch.equal(torch.isnan(gx), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert inf[5].any() and inf[:, 64:].any() and torch.equal(torch.isinf(gx), inf) and torch.equal(gx[inf], ref[inf])
    if dtype == torch.float16:
        assert (inf[9] & torch.isfinite(ref32[9])).any()
    same = torch.isfinite(ref)
    same[9] = False
    # (a group's third plane is used now: its zeros change no sum)
    assert same.any() and torch.equal(gx[same], clean[same])


@pytest.mark.parametrize("dtype", DTYPES)
def test_infinite_gradients_cost_no_more_than_a_second_product(dtype):
    from distributed_gptq_amd import _ops
    M, N, K = 1024, 2048, 4096
    q, _ = make_layer(N, K, 4, 128, False, 7)

    def us(go):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            _ops.linear_grad_input(go, q.qweight, 4, q.scales, q.zeros, K, 128)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return min(times)

    go = (torch.randn(M, N, device="cuda") * 1e-2).to(dtype)
    finite = us(go)
    go[:, 5] = float("inf")
    one = us(go)
    go[:] = float("nan")
    every = us(go)
    assert max(one, every) <= 2 * finite, (finite, one, every)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("act", [False, True])
def test_operator_routes(dtype, act):
    """Forward on the dense kernel, backward on the planes, through the
    operator, and the routes a differentiated or batched gradient takes."""
    from distributed_gptq_amd.models import layers
    N, K, M = 4096, 128, 1536
    assert layers._dense_forward(M, N, K) and layers._planes_backward(M, 256, 4096, 4, dtype, None)
    q, W = make_layer(N, K, 4, 64, act, 9)
    x = torch.randn(M, K, device="cuda").to(dtype)
    with torch.no_grad():
        y = q(x)
    Wr = W.to(dtype).double()
    check(y, x.double() @ Wr.t(), x.double().abs() @ Wr.abs().t(), K)
    q, W = make_layer(256, 4096, 4, 64, act, 10)
    x = torch.randn(M, 4096, device="cuda").to(dtype).requires_grad_(True)
    go = (torch.randn(M, 256, device="cuda") * 1e-2).to(dtype)
    y = q(x)
    gx, = torch.autograd.grad(y, x, go, retain_graph=True)
    check(gx, go.double() @ W, go.double().abs() @ W.abs(), 6 * 256)
    # the gradient of the gradient: gx is linear in go
    gr = go.clone().requires_grad_(True)
    gx2, = torch.autograd.grad(y, x, gr, create_graph=True, retain_graph=True)
    gg, = torch.autograd.grad(gx2.float().sum(), gr)
    assert torch.isfinite(gg).all() and gg.shape == gr.shape
    both, = torch.autograd.grad(y, x, torch.stack([go, go]), is_grads_batched=True)
    assert both.shape == (2, M, 4096)


@pytest.mark.parametrize("act", [False, True])
def test_gradient_that_is_followed(act):
    """Forward over reverse, and a trace of a call that takes the gradient."""
    import torch.autograd.forward_ad as fw
    from torch.fx.experimental.proxy_tensor import make_fx
    from distributed_gptq_amd.models import layers
    N, K, M = 256, 4096, 1536
    assert layers._planes_backward(M, N, K, 4, torch.float16, None)
    q, W = make_layer(N, K, 4, 64, act, 12)
    x = torch.randn(M, K, device="cuda").half()
    go, t = ((torch.randn(M, N, device="cuda") * 1e-2).half() for _ in range(2))

    def grad(x, go):
        x = x.detach().requires_grad_(True)
        return torch.autograd.grad(q(x), x, go)[0]

    with fw.dual_level():
        gx = fw.unpack_dual(grad(x, fw.make_dual(go, t)))
        assert gx.tangent is not None
        check(gx.primal, go.double() @ W, go.double().abs() @ W.abs(), 6 * N)
        check(gx.tangent, t.double() @ W, t.double().abs() @ W.abs(), 6 * N)
    traced = make_fx(grad)(x, go)
    del gx
    keep = [torch.full((N, K), float("nan"), device="cuda") for _ in range(4)]  # freed memory holds no weights
    del keep
    check(traced(x, t), t.double() @ W, t.double().abs() @ W.abs(), 6 * N)


def test_biases_of_the_library_product():
    """Biases that the dense kernel does not read as N values of its types
    keep the library product: its broadcast, its conversion and its errors."""
    from distributed_gptq_amd.models import layers
    N, K, M = 4096, 128, 1536
    assert layers._dense_forward(M, N, K)
    q, W = make_layer(N, K, 4, 64, False, 11)
    x = torch.randn(M, K, device="cuda").half()
    args = (x, q.qweight, q.scales, q.zeros, q.g_idx)
    Wr, b = W.half().double(), torch.randn(N, device="cuda", dtype=torch.float64)
    ref, mag = x.double() @ Wr.t(), x.double().abs() @ Wr.abs().t()
    for bias in (b, b[:1]):
        # the bias itself is rounded to fp32 once
        check(torch.ops.gptq.linear(*args, bias), ref + bias, mag + bias.abs(), K + 2)
    for bias in (b[:-1].float(), b.float().cpu()):
        with pytest.raises(RuntimeError):
            torch.ops.gptq.linear(*args, bias)


@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("N,K,gs", [(1, 32, 32), (5, 96, 32), (7, 2080, 64), (66, 4096, 4096)])
def test_dequant_rows(N, K, gs, bits):
    """One rounding of (q - z) s, bit for bit, past a row's last workgroup and
    the last group of four rows."""
    from distributed_gptq_amd import _ops
    rng = np.random.default_rng(N + K)
    ng = -(-K // gs)
    codes = torch.from_numpy(rng.integers(0, 2 ** bits, (N, K)).astype(np.uint8)).cuda()
    s = torch.from_numpy(rng.uniform(1e-3, 1e-2, (N, ng))).half().cuda()
    z = torch.from_numpy(rng.uniform(0, 2 ** bits, (N, ng))).half().cuda()
    gi = torch.arange(K, device="cuda") // gs
    ref = (codes.float() - z.float()[:, gi]) * s.float()[:, gi]
    for dt in (torch.float32, torch.float16, torch.bfloat16):
        assert torch.equal(_ops.dequant(_ops.pack(codes, bits), bits, s, z, K, group_size=gs, dtype=dt), ref.to(dt))
