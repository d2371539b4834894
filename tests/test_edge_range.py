"""Positions in the edge arrays (medusa_amd/csrc/edge_range.h, compiled here with g++): walks and parts of
ranges that end up to the last position below 2^32 take every edge once and end."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_ranges_up_to_the_last_position(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = tmp_path / "edge_range_check"
    subprocess.run([gxx, "-O2", "-std=c++17", "-iquote", str(ROOT / "medusa_amd" / "csrc"), "-o", str(exe),
                    str(ROOT / "tests" / "edge_range_check.cpp")], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.stdout.strip() == "ok", r.stdout
