"""The controllers' pow (csrc/de_pow_libm.h, libm_pow_const), built for the host and
in the device library: the bits of libm_pow for every exponent in use, over all regimes of x -- random bit
patterns (negative, subnormal, NaN), error norms, arguments near 1 (where y log x
falls below 2^-54), the table's interval ends and the special values.  Exponents
outside the range whose special cases it leaves out do not compile."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EXE = os.path.join(HERE, "cpp", "_build", "pow_check")


def arguments():
    rng = np.random.default_rng(7)
    bits = rng.integers(0, 2 ** 64, 200000, dtype=np.uint64).view(np.float64)
    norms = 10.0 ** rng.uniform(-300, 300, 200000)
    usual = 10.0 ** rng.uniform(-12, 4, 200000)
    k = rng.integers(-(1 << 14), 1 << 14, 100000)
    near = np.concatenate([1.0 + k * 2.0 ** -52, 1.0 + k * 2.0 ** -53])
    sub = rng.integers(1, 1 << 52, 50000, dtype=np.uint64).view(np.float64)
    edges = (np.uint64(0x3fe6955500000000) + (np.arange(0, 129, dtype=np.uint64) << np.uint64(45)))
    ends = np.concatenate([(edges + np.uint64(d)).view(np.float64) for d in (0, 1)] +
                          [(edges - np.uint64(1)).view(np.float64)])
    scaled = np.concatenate([ends * 2.0 ** e for e in (-1021, -900, -60, -1, 1, 52, 700, 1022)])
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -np.nan, 1.0, -1.0, 5e-324, -5e-324,
                        2.2250738585072014e-308, 2.225073858507201e-308, 1.7976931348623157e308])
    with np.errstate(all="ignore"):
        return np.concatenate([bits, norms, usual, near, sub, ends, scaled, special])


def test_pow_const_has_libm_pow_bits():
    subprocess.check_call(["make", "-s", "-C", os.path.join(HERE, "cpp"), "_build/pow_check"])
    out = subprocess.run([EXE], input=arguments().tobytes(), capture_output=True, timeout=300)
    assert out.returncode == 0, out.stdout.decode()[-2000:]
    assert b", 0 differ" in out.stdout


@pytest.mark.parametrize("exponent,takes", [
    ("-0.2", True), ("1.0 / 9.0", True), ("-(1.0 / 3.0)", True), ("0x1p-10", True),
    ("0.5", False), ("-0.5", False), ("1.0 / 1.0", False), ("0.0", False), ("0x1p-11", False),
    ("x", False)])  # x: known at run time only
def test_exponents_outside_its_range_do_not_compile(exponent, takes):
    src = ('#include "de_lane.h"\ndouble f(double x) { return DE_CTRL_POW(x, %s); }\n' % exponent)
    out = subprocess.run(
        ["g++", "-std=c++17", "-fsyntax-only", "-Wno-unknown-pragmas", "-x", "c++", "-I",
         os.path.join(HERE, "..", "differential-equations_amd", "csrc"), "-"],
        input=src, capture_output=True, text=True, timeout=120)
    assert (out.returncode == 0) == takes, out.stderr[-2000:]
    if not takes:
        assert "constant" in out.stderr


@pytest.mark.gpu
def test_device_build_has_the_host_bits(orc):
    import deamd
    x = arguments()
    for y in [-0.2, 0.2, -0.125, 0.125] + [s / k for k in (4, 6, 7, 9) for s in (-1.0, 1.0)] + \
            [2.0 ** -10, -0.499]:
        ys, out = np.full_like(x, y), np.empty_like(x)
        deamd._abi.check(deamd.lib().de_diag_pow(deamd._ptr(x), deamd._ptr(ys),
                                                 deamd._ptr(out), len(x)))
        want = orc.pow_many(x, ys)
        assert ((out.view(np.uint64) == want.view(np.uint64)) |
                (np.isnan(out) & np.isnan(want))).all(), y
