"""The transfers' ring, threads and pinned memory on the CPU (host_transfer.cpp)."""
from __future__ import annotations

import subprocess

from _fake_hip import program


def test_transfers_on_the_host(tmp_path):
    exe = program("host_transfer.cpp", tmp_path, without=("transfer.hip",))
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, f"status {r.returncode}\n{r.stdout[-3000:]}{r.stderr}"
