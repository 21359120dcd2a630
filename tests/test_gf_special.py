"""The library's own exp, erfcx and whole powers (goofit_amd/csrc/gf_math.h), built for the
host with the same operations as on the device (tests/cpp/special_check.cpp) and compared
with long double.

Bars, in units of 2^-53 of the value: exp below 2 (one unit in the last place is 1 to 2 of
them); erfcx below 5.5 (its polynomial is cut at 0.3; two factors of the scale and the
reciprocal round by 0.5 to 1.5 each, Horner's last steps by 1); powers below 1.01 (h + l
holds the power to 2^-100, one rounding; the long double reference's 20 factors are good to
0.01), negative ones below 1.01 + the reciprocal's correction; powers in the subnormal range
below 1.01 of its spacing 2^-1074, whichever sign the exponent has."""
import math
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("gfspecial") / "special_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "goofit_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "special_check.cpp"), "-o", exe], check=True)
    return subprocess.run([exe, "400000", "5"], check=True, capture_output=True, text=True).stdout


@pytest.mark.parametrize("name,bar", [("exp_range", 2.0), ("exp_small", 2.0), ("erfcx_low", 5.5), ("erfcx_mid", 5.5),
                                      ("erfcx_high", 5.5), ("powi", 1.01), ("powi_negative", 1.02),
                                      ("powi_large", 1.01), ("powi_tiny", 1.01), ("powi_negative_tiny", 1.01)])
def test_accuracy(report, name, bar):
    m = re.search(name + r" n=(\d+) err=([\d.]+|nan|inf) at=(\S+)", report)
    assert int(m.group(1)) >= 330_000 and float(m.group(2)) < bar, m.group(0)


def test_special_values(report):
    rows = re.findall(r"special (exp|powi) (x=\S+(?: n=\S+)?) y=(\S+) library=(\S+)", report)
    assert len(rows) == 11 + 7 * 6
    for f, x, y, lib in rows:
        y, lib = float(y), float(lib)
        assert (math.isnan(y) and math.isnan(lib)) or y == lib, (f, x, y, lib)
    e = dict(re.findall(r"special erfcx x=(\S+) y=(\S+)", report))
    assert abs(float(e["0"]) - 1) < 3e-16 and math.isnan(float(e["nan"]))
    assert 0 <= float(e["inf"]) == float(e["9.9999999999999997e+199"]) < 1e-150
