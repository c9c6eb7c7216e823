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
