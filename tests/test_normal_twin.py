"""The normal and log-normal transforms' functions (include/rocrand/rocrand_amd_math.h)
compiled for the host from the same source as the device (tests/normal_twin.cpp): the float
log, sin, cos and exp are the correctly rounded ones (but next to a rounding boundary: at
most one of a row's million or more), the float pair is within 0.508 ulp and the double pair
within 0.52 ulp of exact, both within 2 ulp of the reference's steps over this libm."""
import os
import subprocess

import pytest

from test_dmath_twin import GCC_LIB, HERE, HIPCC, ROOT


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    if not os.path.exists(HIPCC) or not os.path.exists(os.path.join(GCC_LIB, "include", "quadmath.h")):
        pytest.skip("hipcc or libquadmath not available")
    exe = tmp_path_factory.mktemp("ntwin") / "normal_twin"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-ffp-contract=off", f"-I{os.path.join(ROOT, 'include')}",
                    "-isystem", os.path.join(GCC_LIB, "include"), "-x", "hip", "--offload-arch=gfx950",
                    os.path.join(HERE, "normal_twin.cpp"), "-o", str(exe), f"-L{GCC_LIB}", "-lquadmath"],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe), "400000"], check=True, capture_output=True, text=True).stdout
    return {ln.split()[0]: [int(v) for v in ln.split()[1:]] for ln in out.strip().splitlines()}


@pytest.mark.parametrize("name", ["log", "sincos", "exp"])
def test_float_functions_correctly_rounded(rows, name):
    bad, total = rows[name]
    assert total > 1_000_000
    assert bad <= 1
    assert rows["special"] == [1, 1, 1, 1]


@pytest.mark.parametrize("name,values,most,steps", [
    ("pair_f32", 4000000, 508000, 1_000_000), ("pair_f32_mrg32", 4000000, 508000, 1_000_000),
    ("pair_f32_mrg31", 4000000, 508000, 1_000_000), ("pair_f64", 800000, 520000, 1_500_000)])
def test_pairs(rows, name, values, most, steps):
    """Before its one rounding the float pair is within 2^-31 of exact (2^-7 of the narrowest ulp),
    the double pair within 2^-58."""
    n, worst, beyond, host = rows[name]
    assert n == values
    assert worst <= most
    assert beyond == 0
    assert host >= steps  # the steps rounded one by one are further off: the comparison is not vacuous


@pytest.mark.parametrize("name", ["quarter_words", "quarter_mrg32", "quarter_mrg31"])
def test_double_pair_next_to_quarter_turns(rows, name):
    """There the small sine or cosine is a table entry rounded to a double (half an ulp), and
    the result is rounded once (another half)."""
    n, worst, beyond, steps = rows[name]
    assert n > 400000
    assert worst <= 1_000_000
    assert beyond == 0
    assert steps >= 1_500_000  # the steps rounded one by one are further off


def test_doubles_before_their_rounding_to_float(rows):
    """The worst relative errors (100 log2) of the doubles that sincosf_unit and expf_acc round:
    sin and cos a few roundings of 2^-53 (next to their zeros too), exp the r^6/720 that its
    series leaves out at |r| = 0.0109 (2^-48.6) and a few roundings."""
    sincos, exp = rows["steps"]
    assert sincos <= -5100
    assert exp <= -4840
