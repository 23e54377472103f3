"""The FP64 replay of a known outcome on the host: replay64 of bh_trace64.h,
built with the host compiler (tests/host), must replay every disc hit and every
uncaptured miss of the march, with the march's bits."""
import shutil
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent / "host"
ROOT = HOST.parent.parent


def test_every_hit_and_miss_replays(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "replay64_host"
    subprocess.run([cxx, "-std=c++17", "-O2", "-ffp-contract=off", f"-I{HOST}",
                    f"-I{ROOT / 'blackhole_8_amd' / 'csrc'}", f"-I{ROOT / 'include'}",
                    str(HOST / "replay64_host.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), "60"], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    rows = {c: (int(d), int(m), int(n)) for c, _, d, _, m, _, n in
            (ln.split() for ln in r.stdout.splitlines() if " disc " in ln)}
    assert len(rows) == 10
    assert all(n == 0 for _, _, n in rows.values())
    assert all(rows[c][0] > 1000 for c in rows if c not in ("hole", "away", "inside"))
    assert all(rows[c][1] > 5000 for c in rows if c != "inside")
