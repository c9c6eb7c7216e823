"""The bf16 planes that the input gradient multiplies: what they hold, when a
third one is needed, and that the product uses all of them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def planes_of(codes, bits, s, z, gs, perm=None, packed=True):
    """(hi, mid, lo) of shape (K, N) and the flags; the memory held NaNs, and
    the rows before and after it are checked."""
    from distributed_gptq_amd import _lib as L, _ops
    N, K = codes.shape
    q = _ops.pack(codes, bits) if packed else codes
    rows = torch.full((K + 2, 3 * N), float("nan"), dtype=torch.bfloat16, device="cuda")
    out = rows[1:-1]
    flags = torch.full((256,), -1, dtype=torch.int32, device="cuda")
    L.call("gptq_dequant_planes_t", _ops._p(q), bits if packed else 0, _ops._p(s), _ops._p(z),
           _ops.dtype_code(s.dtype), gs, s.shape[1], N, K, _ops._p(perm), _ops._p(flags), _ops._p(out),
           _ops._stream(q.device))
    assert rows[0].isnan().all() and rows[-1].isnan().all()
    W = _ops.dequant(q, bits if packed else 0, s, z, K, group_size=gs)
    return out.view(K, 3, N).unbind(1), flags, W


def params(N, K, bits, gs, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    codes = torch.randint(0, 2 ** bits, (N, K), generator=g, device="cuda", dtype=torch.uint8)
    s = (torch.rand(N, K // gs, generator=g, device="cuda") * 1e-2 + 1e-3).to(dtype)
    z = torch.randint(0, 2 ** bits, s.shape, generator=g, device="cuda").to(dtype)
    return codes, s, z, g


@pytest.mark.parametrize("what,bits,dtype,packed,three", [
    ("plain", 4, torch.float16, True, False),
    ("plain", 3, torch.float16, True, False),
    ("plain", 2, torch.float16, True, False),
    ("outside", 4, torch.float16, True, False),       # zeros below 0 and above 15, |q - z| <= 31 still
    ("plain", 8, torch.float16, True, True),          # |q - z| > 31
    ("plain", 4, torch.float16, False, True),         # one code per byte: could be up to 255
    ("far", 4, torch.float16, True, True),            # one zero point of 32
    ("fraction", 4, torch.float16, True, True),       # one zero point off the integers
    ("infinite", 4, torch.float16, True, True),       # one infinite and one NaN scale
    ("plain", 4, torch.bfloat16, True, True),
    ("plain", 3, torch.float32, True, True),
])
@pytest.mark.parametrize("act", [False, True])
def test_planes_hold_the_weight(what, bits, dtype, packed, three, act):
    N, K, gs = 192, 416, 32  # columns past a 128-column block
    codes, s, z, g = params(N, K, bits, gs, dtype, bits)
    if what == "outside":
        z[3, 2], z[5, 4] = -16, 31
    elif what == "far":
        z[N - 1, K // gs - 1] = 32
    elif what == "fraction":
        z[17, 5] += 0.375
    elif what == "infinite":
        s[9, 1], s[10, 2] = float("inf"), float("nan")
    perm = torch.randperm(K, generator=g, device="cuda").int() if act else None
    (hi, mid, lo), flags, W = planes_of(codes, bits, s, z, gs, perm, packed)
    assert bool(flags.any()) is three
    if not three:
        assert lo.isnan().all()  # not written
        lo = torch.zeros_like(lo)
    if act:
        W = W[:, torch.argsort(perm.long())]  # row perm[k] holds column k
    W = W.t()
    total = hi.double() + mid.double() + lo.double()
    finite = torch.isfinite(W)
    assert finite.any() and torch.equal(total[finite], W.double()[finite])
    # an infinite or NaN weight is in the first plane alone
    assert torch.equal(hi[~finite].isnan(), W[~finite].isnan())
    inf = torch.isinf(W)
    assert torch.equal(hi[inf].float(), W[inf])
    assert (mid[~finite] == 0).all() and (lo[~finite] == 0).all()
    if three and what == "plain" and bits == 8:
        assert (lo != 0).sum() > 1000  # the third plane holds something


def test_columns_out_of_range_stay_inside():
    """A perm that is none (a damaged file): the rows around the planes keep
    their values, those of its good entries are right."""
    N, K, gs = 64, 160, 32
    codes, s, z, g = params(N, K, 4, gs, torch.float16, 1)
    perm = torch.randperm(K, generator=g, device="cuda").int()
    good = torch.ones(K, dtype=torch.bool, device="cuda")
    for at, value in ((3, K), (40, -1), (90, 2 ** 31 - 1), (159, -2 ** 31)):
        perm[at], good[at] = value, False
    good &= (perm > 0) & (perm < K - 1)  # (the first and last row are written more than once)
    (hi, mid, _), flags, W = planes_of(codes, 4, s, z, gs, perm)
    at = perm[good].long()
    assert torch.equal((hi.double() + mid.double())[at], W.t().double()[good])


def test_split_planes_of_every_half():
    from distributed_gptq_amd import _lib as L, _ops
    x = torch.arange(65536, device="cuda").to(torch.int32).to(torch.int16).view(torch.float16).view(256, 256)
    out = torch.empty(256, 512, dtype=torch.bfloat16, device="cuda")
    L.call("gptq_split_planes", _ops._p(x), 256, 256, _ops._p(out), _ops._stream(x.device))
    hi, lo = out[:, :256], out[:, 256:]
    finite = torch.isfinite(x)
    assert torch.equal((hi.double() + lo.double())[finite], x.double()[finite])
    assert torch.equal(hi.isnan(), x.isnan()) and torch.equal(hi[x.isinf()].float(), x[x.isinf()].float())
    assert (lo[~finite] == 0).all()


@pytest.mark.parametrize("aplanes,out", [(1, torch.bfloat16), (2, torch.float16)])
@pytest.mark.parametrize("M,N,K", [(40, 64, 32), (2304, 128, 3840)])  # a half tile; whole tiles
def test_every_plane_meets_every_plane(M, N, K, aplanes, out):
    """Planes whose other products cancel: each of them alone decides a part
    of the result, and the flags say whether the third is read."""
    from distributed_gptq_amd import _lib as L, _ops
    g = torch.Generator(device="cuda").manual_seed(M)
    half = torch.randint(-3, 4, (aplanes, M, N // 2), generator=g, device="cuda").float()
    A = torch.stack([half, half], -1).view(aplanes, M, N)  # equal pairs along the contraction
    A[-1, :, 0] += 1
    B = torch.randint(1, 9, (3, K, N // 2), generator=g, device="cuda").float()
    B = torch.stack([B, -B], -1).view(3, K, N)             # opposite pairs: the products cancel
    for p, w in enumerate((1.0, 2.0 ** -3, 2.0 ** -6)):    # (sums of whole multiples of 2^-6: exact in fp32)
        B[p, :, 1] = 0
        B[p] *= w
    a, b = (t.transpose(0, 1).reshape(t.shape[1], -1).bfloat16().contiguous() for t in (A, B))
    for flag in (0, 1):
        flags = torch.zeros(256, dtype=torch.int32, device="cuda")
        flags[255] = flag
        y = torch.empty(M, K, dtype=out, device="cuda")
        L.call("gptq_matmul_nt", _ops._p(a), aplanes * N, _ops._p(b), 3 * N, L.BF16, M, K, N, aplanes, 3,
               _ops._p(flags), _ops._p(None), 0, _ops._p(y), K, _ops.dtype_code(out), _ops._stream(a.device))
        ref = A.double().sum(0) @ B[:2 + flag].double().sum(0).t()
        assert torch.equal(y, ref.to(out))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gradient_of_weights_that_cancel(dtype):
    """Pairs of rows whose fp32 weights differ past 16 bits: their gradients
    cancel down to what the third plane holds."""
    from distributed_gptq_amd import _ops
    N, K, gs = 256, 384, 64
    codes, s, z, g = params(N, K, 4, gs, torch.float32, 3)
    codes[1::2], z[1::2] = codes[::2], z[::2]
    s[1::2] = s[::2] * (1 + 2.0 ** -19)
    sign = torch.where(torch.arange(N, device="cuda") % 2 == 0, 1.0, -1.0)
    go = ((torch.randint(0, 2, (33, N // 2), generator=g, device="cuda") * 2 - 1).repeat_interleave(2, 1) * sign).to(dtype)
    q = _ops.pack(codes, 4)
    W = _ops.dequant(q, 4, s, z, K, group_size=gs)
    up = 2.0 ** 10  # (keeps the differences in fp16's normal range)
    gx = _ops.linear_grad_input(go * up, q, 4, s, z, K, gs).double() / up
    ref = go.double() @ W.double()
    # 256 terms of at most 2^-3 in fp32, cancelling pair by pair within an MFMA: far below the third plane's part
    two = (W.double() - (W.bfloat16().double() + (W - W.bfloat16().float()).bfloat16().double()))
    lost = (go.double() @ two).norm()
    assert (gx - ref).norm() < 0.25 * lost, ((gx - ref).norm(), lost)
