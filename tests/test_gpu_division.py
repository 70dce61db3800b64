"""The divisions that take the compiler's place in the exponential, the
logarithm and the Poisson sums, against the compiler's own, bit for bit
(tests/cpp/test_division.hip, built by `python g4hepem_amd/build.py cpp`)."""
import subprocess
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu


def test_divisions_round_as_divisions():
    binary = Path(__file__).resolve().parent / "cpp" / "test_division"
    assert binary.exists(), f"{binary} is not built (python g4hepem_amd/build.py cpp)"
    p = subprocess.run([str(binary)], capture_output=True, text=True, timeout=100)
    print(p.stdout, flush=True)
    assert p.returncode == 0, p.stdout + p.stderr
    assert "ALL OK" in p.stdout
