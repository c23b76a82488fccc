"""Host check of the staged device-to-host copy (csrc/download.hpp) with the
device played by memory (no GPU): sizes, missing threads, no ring, failures."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_download(tmp_path):
    exe = tmp_path / "download_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-pthread", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "download_check.cpp")], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "download check passed" in r.stdout
