"""The kernels whose MFMAs are inline asm: the compiler does not know that
their accumulators are MFMA results, so nothing but the source's own wait
(mfma_settle) separates the last MFMA from a read of them.  In the generated
code no accumulator may be read or moved between the two."""
import os
import re
import shutil
import subprocess

import pytest

from distributed_gptq_amd import build

HIPCC = build.HIPCC if os.path.exists(build.HIPCC) else shutil.which("hipcc")
WAIT = ["s_nop 7"] * 3


@pytest.mark.skipif(HIPCC is None, reason="hipcc not available")
@pytest.mark.parametrize("name", ["dense", "hessian"])
def test_accumulators_are_read_after_the_wait(name, tmp_path):
    out = tmp_path / f"{name}.s"
    subprocess.run([HIPCC, *build.COMMON_FLAGS, "-S", "--cuda-device-only", os.path.join(build.CSRC, f"{name}.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    code = [t for t in (line.split(";")[0].strip() for line in out.read_text().split("\n")) if t]
    waits = [i for i in range(len(code)) if code[i:i + 3] == WAIT]
    assert waits
    for i in waits:
        last = max(j for j in range(i) if code[j].startswith("v_mfma"))
        between = [t for t in code[last + 1:i] if re.search(r"\ba(\d|\[)", t)]
        # (zeros written on the path without a stage)
        assert all(re.fullmatch(r"v_accvgpr_write_b32 a\d+, 0", t) for t in between), between
