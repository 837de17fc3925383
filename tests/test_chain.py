"""The kernels' addition chains (square-wheel_amd/csrc/sw_chain.h: the depth rasteriser's stepped 1 / z,
rasterizer.rs:1414-1474) against the walked chain, bit for bit: steps much smaller and larger than the start,
exact half-way steps (the rounding's ties) from even and odd mantissas, crossings of powers of two in both
directions and of zero, denormals, infinities and NaN, chains as long as a row."""
import ctypes as C
import os
import subprocess
import time

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "chain_check.cpp")
HDR = os.path.join(os.path.dirname(HERE), "square-wheel_amd", "csrc", "sw_chain.h")
LIB = os.path.join(HERE, "native", "libchain_check.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < max(os.path.getmtime(SRC), os.path.getmtime(HDR)):
        # -mfma: __builtin_fmaf as one rounding, like the GPU's
        subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-fPIC", "-shared", "-ffp-contract=off", "-o", LIB, SRC], check=True)
    lib = C.CDLL(LIB)
    for name in ("check_chains", "check_chain_ends"):
        getattr(lib, name).restype = C.c_uint64
    return lib


def _check(lib, start, step, n):
    start, step = np.ascontiguousarray(start, np.float32), np.ascontiguousarray(step, np.float32)
    first = (C.c_uint32 * 2)()
    bad = lib.check_chains(C.c_void_p(start.ctypes.data), C.c_void_p(step.ctypes.data), len(start), n, first)
    assert bad == 0, f"{bad} values, first: start {start[first[0]]!r} step {step[first[0]]!r} length {first[1]}"


def test_random_chains(lib):
    rng = np.random.default_rng(5)
    n = 60000
    start = rng.uniform(0.5, 1.0, n) * np.exp2(rng.integers(-40, 40, n)) * rng.choice([-1, 1], n)
    step = start * rng.uniform(-1, 1, n) * np.exp2(-rng.integers(0, 30, n).astype(np.float64))
    _check(lib, start, step, 300)


def test_half_way_steps(lib):
    """Steps of (m + 1/2) units in the last place, from even and odd mantissas, near both ends of a binade."""
    rng = np.random.default_rng(6)
    n = 40000
    e = rng.integers(-20, 20, n)
    ulp = np.exp2(e - 23.0)
    mant = rng.choice([2 ** 23 + 1, 2 ** 23 + 2, 2 ** 24 - 2, 2 ** 24 - 3], n) + rng.integers(-400, 400, n)
    start = np.clip(mant, 2 ** 23, 2 ** 24 - 1) * ulp * rng.choice([-1, 1], n)
    step = (rng.integers(-60, 60, n) + 0.5) * ulp
    _check(lib, start, step, 200)


def test_special_values(lib):
    tiny, big = np.float32(1e-45), np.float32(3e38)
    values = np.array([0.0, -0.0, tiny, -tiny, 1.17549435e-38, 1.1754942e-38, 1.0, -1.0, 2.0 - 2 ** -23, 0.5, big, -big, np.inf,
                       -np.inf, np.nan, 1e-30, 3e-39], np.float32)
    a, b = np.meshgrid(values, np.concatenate([values, values * np.float32(2 ** -10), values * np.float32(2 ** -24)]))
    with np.errstate(all="ignore"):
        _check(lib, a.ravel(), b.ravel(), 400)


def test_long_chains(lib):
    rng = np.random.default_rng(7)
    n = 3000
    start = (rng.uniform(1e-4, 4.0, n)).astype(np.float32)
    step = (start * rng.uniform(-1, 1, n) * np.exp2(-rng.integers(8, 26, n).astype(np.float64))).astype(np.float32)
    for length in (1000, 16384, 65535):
        assert lib.check_chain_ends(C.c_void_p(start.ctypes.data), C.c_void_p(step.ctypes.data), n, length) == 0


def test_chains_that_are_or_become_infinite_or_nan_end_at_once(lib):
    """A chain that reaches infinity or NaN stays there: its end is found in a few steps and not walked (walked three
    additions at a time these chains take seconds)."""
    f = np.float32
    values = np.array([0.0, 1.0, -2.5, 3e38, -3e38, np.inf, -np.inf, np.nan], f)
    steps = np.array([1.0, -1.0, 2e37, -3e38, 3.4e38, np.inf, -np.inf, np.nan], f)
    start, step = (np.ascontiguousarray(a.ravel()) for a in np.meshgrid(values, steps))
    with np.errstate(all="ignore"):
        walked = start.copy()
        for _ in range(200):
            walked = (walked + step).astype(f)
    lost = ~np.isfinite(walked)
    start, step, walked = (np.ascontiguousarray(a[lost]) for a in (start, step, walked))
    assert len(start) > 40
    out = np.empty_like(start)
    t = time.perf_counter()
    lib.chain_ends(C.c_void_p(start.ctypes.data), C.c_void_p(step.ctypes.data), len(start), 2 ** 24 - 1, C.c_void_p(out.ctypes.data))
    took = time.perf_counter() - t
    assert np.array_equal(np.isnan(out), np.isnan(walked)) and np.array_equal(out[~np.isnan(out)], walked[~np.isnan(walked)])
    assert took < 0.05, f"{took:.3f} s"
