"""Where the decode kernels keep a K split's partials, built for the host: the
index of a split past the first passes 32 bits at sizes whose tokens * hidden
does not (64 tokens, hidden 2^24, 7 splits)."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_split_index_past_32_bits(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc is not installed")
    exe = tmp_path / "split_index"
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-I", str(ROOT / "complexity-framework_amd/csrc"),
                    str(ROOT / "tests/split_index_check.cpp"), "-o", str(exe)], check=True)
    cases = [(s, m, n, r, c) for s in (0, 1, 2, 6, 7) for m, n in ((1, 1), (16, 896), (64, 65536), (64, 1 << 24))
             for r, c in ((0, 0), (m - 1, n - 1))]
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True, text=True,
                         check=True).stdout.split()
    want = [s * m * n + r * n + c for s, m, n, r, c in cases]
    assert max(want) >= 1 << 32 and [int(v) for v in out] == want
    # the store and both sums go through it, their steps from split to split included
    src = (ROOT / "complexity-framework_amd/csrc/trmoe_skinny.hip").read_text()
    steps = src.count("const int64_t plane = split_index(1, a.M, a.N, 0, 0);")
    assert steps == 2 and src.count("split_index(") == 1 + steps and "int plane" not in src
