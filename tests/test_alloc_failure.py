"""Every device allocation of an upload, of the search's slabs and of the
recorded sets fails once, on the CPU: the call reports it, and no later call
works with buffers that are missing or of another size (host_alloc_failure.cpp)."""
from __future__ import annotations

import subprocess

from _fake_hip import program


def test_failed_allocations_leave_no_capacity(tmp_path):
    exe = program("host_alloc_failure.cpp", tmp_path)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, f"status {r.returncode}\n{r.stdout[-3000:]}{r.stderr}"
