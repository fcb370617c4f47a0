"""The fixed-point comparisons of the fused kernel, evaluated by the host
compiler in constant expressions, where undefined arithmetic does not compile."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "curvelet_construction_on_gpu_amd" / "csrc"


@pytest.mark.parametrize("t,is_open", [("0", True), ("kFixTol", True), ("-kFixTol", True), ("kFixTol + 1", False),
                                       ("-kFixTol - 1", False), ("INT_MAX", False), ("INT_MAX - kFixTol", False),
                                       ("INT_MIN", False), ("INT_MIN + kFixTol", False)])
def test_open_key(tmp_path, t, is_open):
    src = tmp_path / "t.cpp"
    src.write_text(f"""#include <climits>
#include "{CSRC / 'cvg_fixed.hpp'}"
using namespace cvg;
static_assert((open_key({t}) <= 2u * kFixTol) == {str(is_open).lower()}, "");
""")
    cxx = shutil.which("g++") or "g++"
    r = subprocess.run([cxx, "-std=c++17", "-fsyntax-only", str(src)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
