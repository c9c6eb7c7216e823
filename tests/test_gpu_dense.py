"""The row-wise dequantisation at the edges of its workgroups, against the
formula."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


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
