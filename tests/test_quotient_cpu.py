"""mh::quotient (meshhashing_amd/csrc/mh_div.h), the division by the voxel size
of the raycast's and the mesher's samples, equals the IEEE division bit for bit:
every mantissa at one exponent (scaling by powers of two changes nothing while
nothing under- or overflows), and a stride of them over the whole range that its
comment states, for the voxel sizes of the configurations and awkward ones."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    out = tmp_path_factory.mktemp("quotient") / "quotient"
    subprocess.run([gxx, "-std=c++17", "-O2", "-ffp-contract=off",
                    f"-I{ROOT / 'meshhashing_amd' / 'csrc'}", str(ROOT / "tests" / "quotient_main.cpp"), "-o", str(out)],
                   check=True)
    return out


SIZES = ["0.005", "0.01", "0.02", "0.03", "0.04", "0.001", "0.0125", "0.0625", "1.0", "0x1.fffffep-1",
         "0x1.000002p-7", "0x1.fffffep-8", "0x1.5555p-6", "0x1p-20", "0x1p20", "0x1.a3c5e7p3"]


@pytest.mark.parametrize("d", SIZES)
def test_quotient_is_the_ieee_division(exe, d):
    for lo, hi, step in ((0, 0, 1), (-100, 100, 40013)):
        bad, n, zero = map(int, subprocess.run([str(exe), d, str(lo), str(hi), str(step)], capture_output=True,
                                               text=True, check=True).stdout.split())
        assert n > 40000 and bad == 0 and zero == 1
