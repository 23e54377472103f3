"""The order of a context's calls over several streams, on the host: the
library's bh_api.cpp built on a model of the HIP runtime (tests/host/
streams_host.cpp) that says which launches the streams and events order.
Launches that share a context's memory must be ordered."""
import shutil
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent / "host"
ROOT = HOST.parent.parent
CSRC = ROOT / "blackhole_8_amd" / "csrc"
HIP = Path("/opt/rocm/include")


def test_calls_keep_their_order_across_streams(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None or not (HIP / "hip" / "hip_runtime.h").exists():
        pytest.skip("no host C++ compiler or no HIP headers")
    exe = tmp_path / "streams_host"
    subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", str(HIP),
                    f"-I{ROOT / 'include'}", f"-I{CSRC}", str(HOST / "streams_host.cpp"),
                    str(CSRC / "bh_api.cpp"), str(CSRC / "bh_host_util.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count(" ok\n") >= 4
