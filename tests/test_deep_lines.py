"""The deep-ring kernel's load addresses on the CPU: tests/host/deep_lines.cpp walks over them."""
import subprocess
from pathlib import Path

HOST = Path(__file__).resolve().parent / "host"


def test_every_chunk_is_loaded_once_and_no_load_leaves_its_row(tmp_path):
    exe = tmp_path / "deep_lines"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", str(HOST / "deep_lines.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
