"""The numbering of the one-launch passes' hand-over words on the host, where the numbers turn
(tests/native/fuse_words_check.cpp)."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "native" / "fuse_words_check.cpp"


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_no_word_outlives_its_number(tmp_path):
    exe = tmp_path / "fuse_words_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-fsanitize=address,undefined", str(SRC), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
