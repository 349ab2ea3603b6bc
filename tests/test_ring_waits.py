"""The FP64 products' LDS rings as compiled for gfx950: before each barrier that hands a slot over,
a wave has waited for its loads into the next slot and for its own reads of the last one.

A read still in flight there could return what another wave's LDS-DMA has already overwritten, once
in a while and only with another schedule, so this looks at the assembly of the sources instead of
at results."""
import os
import shutil
import subprocess

import pytest

from rspacedist_amd import build


@pytest.mark.skipif(shutil.which(build.HIPCC) is None, reason="no hipcc here")
def test_barriers_wait_for_reads_and_loads(tmp_path):
    out = tmp_path / "gemm_f64.s"
    subprocess.run([build.HIPCC, *build.CFLAGS, "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, "gemm_f64.hip"), "-o", str(out)], check=True, capture_output=True)
    rings, kernel, waits = {}, None, ""
    for line in out.read_text().splitlines():
        s = line.strip()
        if line.startswith("_Z") and ":" in line:
            kernel = line.split(":")[0]
        elif s.startswith("s_waitcnt"):
            waits = s
        elif s.startswith(("ds_", "buffer_load")):
            waits = ""  # issued after the last wait
        elif s.startswith("s_barrier") and ("k_tn_f64_lds" in kernel or "k_nn_f64E" in kernel):
            rings.setdefault(kernel, []).append(waits)
    assert len(rings) == 2, sorted(rings)
    for kernel, found in rings.items():
        assert len(found) == 1 and "vmcnt(0)" in found[0] and "lgkmcnt(0)" in found[0], (kernel, found)
