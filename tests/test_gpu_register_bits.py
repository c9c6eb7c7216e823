"""The register dequant-GEMM's staged scales and zeros against the fp64 oracle."""
import numpy as np
import pytest
import torch

from linear_check import check_linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sdt", [torch.float16, torch.float32])
@pytest.mark.parametrize("bits", [4, 3])
def test_last_scale_of_odd_rows(bits, sdt):
    """One group a row and an odd number of rows: the 16-bit records of the
    last workgroup end in half a word; 32-bit records take each value of a
    load."""
    from distributed_gptq_amd import _ops
    rng = np.random.default_rng(bits)
    K = 1024
    for N in (37, 4101):
        codes = rng.integers(0, 2 ** bits, (N, K)).astype(np.uint8)
        s = torch.from_numpy(rng.uniform(1e-3, 1e-2, (N, 1))).half()
        z = torch.from_numpy(rng.integers(0, 2 ** bits, (N, 1)).astype(np.float64)).half()
        packed = _ops.pack(torch.from_numpy(codes).cuda(), bits)
        s, z = s.to(sdt), z.to(sdt)
        for M in (2, 16):
            x = torch.from_numpy(rng.standard_normal((M, K))).half()
            y = _ops.linear(x.cuda(), packed, bits, s.cuda(), z.cuda(), K, group_size=K)
            check_linear(y, x, codes, s, z, np.zeros(K, np.int32), None, bits=bits)
