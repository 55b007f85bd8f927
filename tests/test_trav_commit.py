"""The rule by which a traversal replaces a {value, parent} word, against interleaved
writers on the host: SSWP never takes a parent on equal widths (no parent cycles), SSSP
and BFS end with the smallest word."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_commit_under_interleaved_writers(tmp_path):
    exe = tmp_path / "trav_commit"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", str(ROOT / "tests" / "c" / "trav_commit.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "PASS", out.stdout + out.stderr
