"""CPU: the order of the persistent grid's work (fa_plan.cpp) against a list written out by plain loops."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

from flash_attn_npu_amd import build as B


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_unit_once_in_the_stated_order(tmp_path):
    exe = tmp_path / "tile_order_check"
    src = Path(__file__).resolve().parent / "tile_order_check.cpp"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{B.INCLUDE_DIR}", f"-I{B.PLAN_SRC.parent}",
                    str(src), "-o", str(exe)], check=True, capture_output=True, text=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0 and "tile order ok" in proc.stdout, proc.stdout + proc.stderr
