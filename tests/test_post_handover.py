"""The NaN fill's tiles pass from one workgroup to another through a flag that one
wave releases.  Its release waits for that wave's own stores only, so every wave has
to wait for its own before the barrier in front of it.  Read from the assembly that
the compiler makes of the kernel; no GPU runs."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
def test_every_wave_waits_for_its_stores_before_the_release(tmp_path):
    asm = tmp_path / "post.s"
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + os.path.join(ROOT, "include"), "-S",
                    os.path.join(ROOT, "pseudoctimaging_amd", "csrc", "pct_post.hip"),
                    "-o", str(asm)], check=True, capture_output=True)
    text = asm.read_text()
    start = re.search(r"^\S*fill_tiles_kernel\S*:", text, re.M)
    lines = [s.split(";")[0].strip() for s in text[start.start():].split("s_endpgm")[0].split("\n")]
    release = [i for i, s in enumerate(lines) if s.startswith("buffer_wbl2")]
    assert len(release) == 1
    barrier = max(i for i in range(release[0]) if lines[i] == "s_barrier")
    run = []   # the straight line that ends in the barrier
    for s in reversed(lines[:barrier]):
        if s.startswith((".L", "s_cbranch", "s_branch", "global_store", "s_barrier")):
            break
        run.append(s)
    assert any(s.startswith("s_waitcnt") and "vmcnt(0)" in s for s in run), run
