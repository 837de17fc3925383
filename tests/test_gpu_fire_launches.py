"""The fire step's launch forms (sw_fire_step) against the oracle, bit for bit: the points in the kernel's
arguments (both argument sizes, their limits) and beyond them through device memory, maps of less than a
block, rows of several chunks of the slow variant, and buffers that are not 4-byte aligned."""
import ctypes as C

import numpy as np
import pytest

import oracle
import sw_abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slow", [0, 1])
@pytest.mark.parametrize("log2", [(4, 4), (9, 5), (5, 9)])
@pytest.mark.parametrize("points", [0, 1, 64, 65, 512, 513])
def test_fire_step_points(gpu_ctx, slow, log2, points):
    lw, lh = log2
    n = 1 << (lw + lh)
    rng = np.random.default_rng([lw, lh, points, slow])
    heat = rng.integers(0, 256, n).astype(np.uint8)
    p = np.zeros(points, A.HEAT_POINT_DTYPE)
    # crowded into an eighth of the rows, so that addresses repeat; coordinates wrap, heat keeps its low byte
    p["x"], p["y"] = rng.integers(0, 5 << lw, points), (1 << lh) - 1 - rng.integers(0, max((1 << lh) // 8, 2), points)
    p["heat"] = rng.integers(0, 1 << 12, points)
    print(f"fire step {lw}x{lh} slow={slow} points={points}", flush=True)
    got = gpu_ctx.fire_steps(heat, lw, lh, 1.0, slow, [p, p[: points // 2]])
    ref = oracle.fire_step(oracle.fire_step(heat, lw, lh, 1.0, slow, p), lw, lh, 1.0, slow, p[: points // 2])
    assert np.array_equal(got, ref), np.count_nonzero(got != ref)


@pytest.mark.parametrize("shift", [(0, 1), (3, 0), (2, 2)])
def test_fire_step_unaligned_buffers(gpu_ctx, shift):
    lw, lh = 6, 5
    n = 1 << (lw + lh)
    rng = np.random.default_rng(shift)
    heat = rng.integers(0, 256, n).astype(np.uint8)
    p = np.zeros(9, A.HEAT_POINT_DTYPE)
    p["x"], p["y"], p["heat"] = rng.integers(0, 64, 9), rng.integers(0, 32, 9), 255
    src = gpu_ctx.to_device(np.concatenate([np.zeros(shift[0], np.uint8), heat]))
    dst = gpu_ctx.to_device(np.full(n + 8, 7, np.uint8))
    try:
        print(f"fire step at byte offsets {shift}", flush=True)
        gpu_ctx.check(gpu_ctx.lib.sw_fire_step(gpu_ctx.h, C.c_void_p(src.ptr.value + shift[0]), C.c_void_p(dst.ptr.value + shift[1]),
                                               lw, lh, 0.97, 0, C.c_void_p(p.ctypes.data), len(p)), "sw_fire_step")
        gpu_ctx.check(gpu_ctx.lib.sw_sync(gpu_ctx.h), "sw_sync")
        out = dst.read(np.uint8, n + 8)
    finally:
        src.free()
        dst.free()
    assert np.array_equal(out[shift[1]:shift[1] + n], oracle.fire_step(heat, lw, lh, 0.97, False, p))
    assert np.all(out[:shift[1]] == 7) and np.all(out[shift[1] + n:] == 7)


@pytest.mark.parametrize("slow", [False, True])
@pytest.mark.parametrize("log2", [(4, 4), (5, 6), (9, 5)])
@pytest.mark.parametrize("shift", [(0, 0), (0, 1), (3, 0)])
def test_fire_update_alone(gpu_ctx, slow, log2, shift):
    """A step without points, both alignments: maps of less than a block and of several, rows of one and of two passes."""
    lw, lh = log2
    n = 1 << (lw + lh)
    heat = np.random.default_rng([lw, lh, slow, *shift]).integers(0, 256, n).astype(np.uint8)
    src = gpu_ctx.to_device(np.concatenate([np.zeros(shift[0], np.uint8), heat]))
    dst = gpu_ctx.to_device(np.full(n + 8, 7, np.uint8))
    try:
        print(f"fire step of {1 << lw} x {1 << lh} without points slow={slow} at byte offsets {shift}", flush=True)
        gpu_ctx.check(gpu_ctx.lib.sw_fire_step(gpu_ctx.h, C.c_void_p(src.ptr.value + shift[0]), C.c_void_p(dst.ptr.value + shift[1]),
                                               lw, lh, 0.97, int(slow), None, 0), "sw_fire_step")
        gpu_ctx.check(gpu_ctx.lib.sw_sync(gpu_ctx.h), "sw_sync")
        out = dst.read(np.uint8, n + 8)
    finally:
        src.free()
        dst.free()
    ref = oracle.fire_step(heat, lw, lh, 0.97, slow, np.zeros(0, A.HEAT_POINT_DTYPE))
    assert np.array_equal(out[shift[1]:shift[1] + n], ref)
    assert np.all(out[:shift[1]] == 7) and np.all(out[shift[1] + n:] == 7)
