"""The face arithmetic of compas_amd/csrc/cmp_device.hpp on the host (tests/device_math_host.cpp): the short
quotient and root against IEEE, WENO5 face states against the oracle's ratio form over the exponent range."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle

HERE = os.path.dirname(os.path.abspath(__file__))
EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def dev(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("device_math") / "device_math.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-w", "-shared", "-fPIC",
                           "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(rocm, "include"),
                           os.path.join(HERE, "device_math_host.cpp"), "-o", so])
    lib = ctypes.CDLL(so)
    lib.host_errors.argtypes = [ctypes.c_double, ctypes.c_double]

    def call(name, *arrays, out=1):
        a = [np.ascontiguousarray(x, dtype=np.float64) for x in arrays]
        res = [np.empty(len(a[0])) for _ in range(out)]
        getattr(lib, name)(ctypes.c_long(len(a[0])), *[ctypes.c_void_p(x.ctypes.data) for x in a + res])
        return res if out > 1 else res[0]

    call.errors, call.lib = lib.host_errors, lib
    yield call


# the hardware's v_rcp_f64 and v_rsq_f64 were measured within 2^-24.4 and 2^-24.2 of the exact values
@pytest.mark.parametrize("err", [-2.0 ** -24, -2.0 ** -27, 0.0, 2.0 ** -26, 2.0 ** -24])
def test_short_quotient_and_root_are_ieee(dev, err):
    """After a Newton step the reciprocal is within 2^-48, the quotient's correction within 2^-95 of it: the
    rounded result differs from IEEE only where the exact one lies that close to a rounding boundary, 2^-41 of
    all operands."""
    dev.errors(err, err)
    rng = np.random.default_rng(7)
    n = 200000
    mant = lambda: rng.uniform(1.0, 2.0, n) * rng.choice([-1.0, 1.0], n)  # noqa: E731
    d = mant() * 10.0 ** rng.uniform(-289, 289, n)
    q = mant() * 10.0 ** rng.uniform(-100, 100, n)
    a = np.where(np.abs(np.log10(np.abs(d)) + np.log10(np.abs(q))) < 290, q, 1.0 / q) * d
    a = np.where(np.isfinite(a) & (np.abs(a) > 1e-290) & (np.abs(a) < 1e290), a, d)
    assert (dev("host_quot", a, d) == a / d).all()
    x = np.abs(d)
    assert (dev("host_sqrt", x) == np.sqrt(x)).all()
    # denominators outside the range, and what IEEE division gives for them
    with np.errstate(all="ignore"):
        a = np.array([1.0, -1.0, 0.0, 1.0, 1.0, 1e-300, 3.0, np.nan, 1.0])
        d = np.array([0.0, 0.0, 0.0, np.inf, -np.inf, 1e-300, 5e-324, 1.0, np.nan])
        np.testing.assert_array_equal(dev("host_quot", a, d), a / d)
        x = np.array([0.0, np.inf, 5e-324, 1e-300, 1e300, -1.0, np.nan])
        np.testing.assert_array_equal(dev("host_sqrt", x), np.sqrt(x))


def _stencils(rng, n):
    """Six-cell stencils of unit size: random, plateaus of 2 to 5 cells between jumps of any relative size,
    single jumps, ramps that end, smooth data, rounding-level differences."""
    out = [rng.uniform(-1.0, 1.0, (n, 6))]
    for width in (2, 3, 4, 5):
        for first in range(0, 7 - width):
            v = rng.uniform(-1.0, 1.0, (n, 6)) * 2.0 ** rng.integers(-120, 1, (n, 6))
            v[:, first:first + width] = rng.uniform(-1.0, 1.0, (n, 1)) * 2.0 ** rng.integers(-120, 1, (n, 1))
            out.append(v)
    for k in range(1, 6):
        v = np.ones((n, 6)) * rng.uniform(0.5, 1.0, (n, 1))
        v[:, k:] = rng.uniform(-1.0, 0.4, (n, 1))
        out.append(v)
    i = np.arange(6.0)
    out.append(np.maximum(0.0, i - rng.integers(0, 6, (n, 1))) * 0.1)
    out.append(np.sin(0.2 * i + rng.uniform(0, 6, (n, 1))))
    out.append(1.0 + 2.0 ** -52 * rng.integers(0, 3, (n, 6)))
    return np.concatenate(out)


# 2^133 is 1e40, where the products of four indicators leave the double range from above
@pytest.mark.parametrize("power", [-400, -140, -60, 0, 60, 110, 127, 133, 150, 200, 400, 500])
@pytest.mark.parametrize("form", ["host_weno5_faces", "host_weno5"])
def test_weno5_over_the_exponents(dev, form, power):
    """WENO5 has no scale of its own: the face states of 2^p v are 2^p times those of v. Reference: the ratio
    form at unit size. The bound: about 40 roundings of numbers up to 8 max |v| in the indicators, the weights and
    the sum, each indicator's relative error amplified up to 8 times by its cancellation and doubled by its square."""
    if form == "host_weno5" and abs(power) > 450:
        pytest.skip("its indicators are not scaled: they leave the double range, as the ratio form's do")
    dev.errors(2.0 ** -25, 2.0 ** -25)
    v = _stencils(np.random.default_rng(11), 200)
    L, R = dev(form, v * 2.0 ** power, out=2)
    lib = oracle.load()
    with np.errstate(all="ignore"):
        rl = np.array([lib.ref_weno5(*s[:5], 1) for s in v])
        rr = np.array([lib.ref_weno5(*s[1:], -1) for s in v])
    assert np.isfinite(L).all() and np.isfinite(R).all()
    bound = 40 * 8 * 2 * EPS * np.abs(v).max(axis=1)
    assert (np.abs(np.ldexp(L, -power) - rl) <= bound).all()
    assert (np.abs(np.ldexp(R, -power) - rr) <= bound).all()


@pytest.mark.parametrize("sj,sk", [(38, 38 * 38), (2 ** 27, 0), (2 ** 28 + 7, 0), (20006, 430000000), (2, 2 ** 30)])
def test_cells_of_a_tile_of_a_very_large_box(dev, sj, sk):
    """The staged cells' offsets from their tile's first cell, also where a tile's few rows or planes are more than
    2^31 cells apart (a 2D box of 2^27 by 15 is 128 GB)."""
    for d in [(0, 0, 0), (-3, 0, 0), (18, 0, 0), (0, -3, 0), (0, 17, 0), (0, 0, -3), (0, 0, 5), (18, 17, 5)]:
        if sk == 0 and d[2]:
            continue
        step, index = ctypes.c_longlong(), ctypes.c_longlong()
        dev.lib.host_fab_step(ctypes.c_longlong(sj), ctypes.c_longlong(sk), (ctypes.c_int * 3)(32, 15, 3),
                              (ctypes.c_int * 3)(*d), ctypes.byref(step), ctypes.byref(index))
        assert step.value == index.value
