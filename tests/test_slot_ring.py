"""CPU: bookkeeping of the parameter ring (runs of slots, held and queued
ones, waits), built and run under the address and undefined-behaviour
sanitizers."""
from __future__ import annotations

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_slot_ring(tmp_path):
    exe = tmp_path / "slot_ring_main"
    cmd = ["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Werror", "-fsanitize=address,undefined",
           "-fno-sanitize-recover=all", f"-I{ROOT / 'genesis4_cuda_port_amd' / 'csrc'}",
           str(ROOT / "tests" / "slot_ring_main.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    assert "done" in res.stdout
