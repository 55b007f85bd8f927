"""Headers of the library that hold no device code, tested on the host: the rule by which
a traversal replaces a {value, parent} word, against interleaved writers (SSWP never takes
a parent on equal widths, so no parent cycles; SSSP and BFS end with the smallest word),
the cuts of the binned layout's ordering up to 2^32 - 2 edges, and the read-back's copying
threads when an allocation fails."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.parametrize("name", ["trav_commit", "sort_tiles", "copiers"])
def test_host_header(tmp_path, name):
    exe = tmp_path / name
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread",
                    str(ROOT / "tests" / "c" / f"{name}.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "PASS", out.stdout + out.stderr
