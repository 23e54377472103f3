"""The FP64 march's chord choice on the host: the device code of
bh_trace64.h, built with the host compiler (tests/host), must give the same
outcome to the bit whether it tests every chord or only those that can meet
an object, over every form of scene the FP64 precision accepts."""
import shutil
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent / "host"
ROOT = HOST.parent.parent


def test_chosen_chords_give_every_chords_outcome(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "trace64_host"
    subprocess.run([cxx, "-std=c++17", "-O2", "-ffp-contract=off", f"-I{HOST}",
                    f"-I{ROOT / 'blackhole_8_amd' / 'csrc'}", f"-I{ROOT / 'include'}",
                    str(HOST / "trace64_host.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), "60"], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    lines = [ln.split() for ln in r.stdout.splitlines() if " rays " in ln]
    assert len(lines) == 10
    for name, _, rays, _, hits, _, differ in lines:
        assert int(rays) == 24000 and int(differ) == 0, name
        assert int(hits) > 500, name
