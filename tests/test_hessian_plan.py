"""The Hessian launch's plan (whole tiles and finer-cut tail): its properties
on the CPU under the sanitizers, its results against fp64 on the GPU."""
import os
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "distributed_gptq_amd", "csrc")


def test_plan_properties(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "hessian_plan_check")
    subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host", "hessian_plan_check.cpp"),
                    os.path.join(CSRC, "plan.cpp"), os.path.join(CSRC, "status.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "0 check(s) failed" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,K", [
    (40, 8),          # one tile, added to H by the tile kernel
    (700, 776),       # partial last tiles, one split
    (1700, 5128),     # 231 tiles of one split, the last rows and columns 8 past a tile
    (3000, 6152),     # 325 tiles: 256 in one split, the tail in finer ones
    (9000, 4104),     # four splits and a finer tail, both through partial tiles
    (2100, 11272),    # 1035 tiles: four whole rounds and a tail
])
def test_against_fp64(n, K, dtype):
    """H += X^T X from a symmetric H: within an fp32 sum's bound of the fp64
    sum, and still exactly symmetric."""
    from distributed_gptq_amd import _ops
    g = torch.Generator(device="cuda").manual_seed(n)
    X = torch.randn(n, K, generator=g, device="cuda").to(dtype)
    H0 = torch.randn(K, K, generator=g, device="cuda")
    H0 = torch.tril(H0) + torch.tril(H0, -1).t()
    H = H0.clone()
    _ops.hessian_accumulate(H, X)
    assert torch.equal(H, H.t())
    for part in range(0, K, 2048):
        rows = slice(part, min(K, part + 2048))
        Xp = X[:, rows].double().t().contiguous()
        ref = H0[rows].double() + Xp @ X.double()
        mag = H0[rows].double().abs() + Xp.abs() @ X.double().abs()
        # MFMA steps of 16 products into one accumulator, then the splits and H
        bound = (n / 16 + 16 + 64) * 2.0 ** -24 * mag
        assert ((H[rows].double() - ref).abs() <= bound).all()
