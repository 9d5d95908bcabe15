"""Registers of the multi-row decode partials on the bf16 cache (CPU: hipcc cross-compiles gfx950 and
reports each kernel's resources).

The addresses of a tile's LDS-DMA loads must stay in registers or be made anew: where the compiler
spills them, each load of a round is preceded by the reload of its address, which waits for every load
before it, and the look-ahead becomes a chain of memory latencies (8 rows at 16 / 2 heads on 64,000
positions: 64.2 us with 41 spilled registers against 51.8 us for the loop without look-ahead)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from test_decode_issue_order import _build_module


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(),
                    reason="hipcc not installed")
def test_bf16_cols_kernels_do_not_spill():
    b = _build_module()
    src = b.CSRC / "attn_decode.hip"
    cmd = [b.HIPCC, *b.HIP_FLAGS, *b.SOURCE_FLAGS.get(src.name, []), "--offload-device-only", "-c",
           "-Rpass-analysis=kernel-resource-usage", str(src), "-o", "/dev/null"]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    usage = {}
    for line in r.stdout.splitlines():
        if m := re.search(r"Function Name: (\S+)", line):
            usage[m.group(1)] = cur = {}
        elif m := re.search(r"remark: .*?(VGPRs Spill|ScratchSize \[bytes/lane\]): (\d+)", line):
            cur[m.group(1)] = int(m.group(2))
    cols = {k: v for k, v in usage.items() if re.search(r"attn_partials_cols_kernelILi\dELi\dELb0E", k)}
    assert len(cols) >= 3, sorted(usage)  # 2, 3 and 4 column tiles
    assert all(v == {"VGPRs Spill": 0, "ScratchSize [bytes/lane]": 0} for v in cols.values()), cols
