"""Every barrier of the split-operand attention kernels waits for the wave's LDS
accesses by itself (CPU only: hipcc cross-compiles).

The kernels' two barriers a key block separate its LDS reads from the refill of
the same buffer.  A read still in flight at the barrier could return the next
block's values, so the wait has to stand before the barrier; that an MFMA which
uses the read's result happens to be scheduled earlier is no guarantee.
"""

import os
import re
import shutil
import subprocess

import pytest

from cutilegpt_amd import build as B


def _barriers(lines):
    """(kernel, line, has a wait for LDS) of every s_barrier: the wait is an
    s_waitcnt lgkmcnt(0) in the barrier's own basic block with no LDS access
    after it."""
    kernel, waits = None, False
    for i, line in enumerate(l.strip() for l in lines):
        m = re.match(r"(_ZN4cgpt\w+):", line)
        if m:
            kernel = m.group(1)
        if re.match(r"[.\w]+:", line):       # a label: another block
            waits = False
        elif line.startswith("ds_"):
            waits = False
        elif line.startswith("s_waitcnt") and "lgkmcnt(0)" in line:
            waits = True
        elif line.startswith("s_barrier"):
            yield kernel, i + 1, waits


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"),
                    reason="needs hipcc")
@pytest.mark.parametrize("src", ["attention_split.hip"])
def test_barriers_wait_for_lds(tmp_path, src):
    out = tmp_path / "k.s"
    cmd = [B.hipcc(), *B.HIPCC_FLAGS, *B.FILE_FLAGS.get(src, []), "--cuda-device-only", "-S",
           os.path.join(B.CSRC, src), "-o", str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    found = [b for b in _barriers(out.read_text().splitlines()) if b[0] and "attn_fwd_split_kernel" in b[0]]
    assert len(found) >= 4  # two kernels, two barriers a key block each
    assert all(ok for _, _, ok in found), [b for b in found if not b[2]]
