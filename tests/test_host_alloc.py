"""Host code after a failed device allocation or fill, on the CPU: the source under test is
compiled into a small program (host_alloc.cpp) whose HIP calls work on host memory and fail on
request."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to compile the library's host code")
@pytest.mark.parametrize("part", ["CFM", "RUNTIME"])
def test_failed_allocation_leaves_nothing_stale(tmp_path, part):
    src = os.path.join(ROOT, "index-tts-rs_amd", "csrc", {"CFM": "cfm.cpp", "RUNTIME": "runtime.cpp"}[part])
    exe = str(tmp_path / part)
    # (the kernels' launchers stay undefined: nothing here reaches them)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", f'-DSOURCE="{src}"',
                    f"-D{part}", os.path.join(ROOT, "tests", "host_alloc.cpp"), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all", "-lpthread"], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
