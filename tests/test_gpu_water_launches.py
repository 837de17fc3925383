"""The water step's and texture's launch forms (sw_water_step, sw_water_make_texture) against the oracle, bit
for bit: points in the kernel's arguments (both argument sizes, their limits) and beyond them, repeated and
on the edges of blocks and of the torus, fields of less than a block, and fields that are not 16-byte (or, for
the texture, 8-byte) aligned."""
import ctypes as C

import numpy as np
import pytest

import oracle
import sw_abi as A
import sw_host

pytestmark = pytest.mark.gpu


def _points(rng, lw, lh, n):
    p = np.zeros(n, A.WAVE_POINT_DTYPE)
    p["x"], p["y"] = rng.integers(0, 3 << lw, n), rng.integers(0, 3 << lh, n)
    # edges: columns 0 and w - 1, the rows on both sides of a 1024-element block's edge, corners
    edge_rows = [0, (1 << lh) - 1, (1024 >> lw) or 1, ((1024 >> lw) or 1) - 1]
    for k in range(0, n, 3):
        p[k]["x"], p[k]["y"] = [0, (1 << lw) - 1, 5][k % 2 if k % 4 else 2], edge_rows[k % 4]
    p["value"] = rng.normal(size=n) * 2
    if n > 5:
        p[4]["x"], p[4]["y"] = p[1]["x"], p[1]["y"]
        p[n - 1]["x"], p[n - 1]["y"] = p[1]["x"], p[1]["y"]
        p[1]["value"], p[4]["value"] = 1e8, -1e8  # the order of an address's additions shows
    return p


@pytest.mark.parametrize("log2", [(4, 4), (7, 6), (11, 5), (5, 11)])
@pytest.mark.parametrize("points", [1, 16, 64, 65, 256, 257])
def test_water_step_points(gpu_ctx, log2, points):
    lw, lh = log2
    n = 1 << (lw + lh)
    rng = np.random.default_rng([lw, lh, points])
    f, fo = rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    steps = [_points(rng, lw, lh, points), _points(rng, lw, lh, points // 2), _points(rng, lw, lh, points)]
    att = np.float32(0.99)
    print(f"water step {lw}x{lh} points={points}", flush=True)
    a, b = gpu_ctx.water_steps(f, fo, lw, lh, att, steps)
    for p in steps:
        f, fo = oracle.water_step(f, fo, lw, lh, att, p)
    assert np.array_equal(a.view(np.uint32), f.view(np.uint32))
    assert np.array_equal(b.view(np.uint32), fo.view(np.uint32))


@pytest.mark.parametrize("log2", [(4, 4), (5, 4), (9, 5), (10, 5), (11, 4), (12, 6)])
@pytest.mark.parametrize("points", [9, 64, 250])
def test_water_step_crowded_points(gpu_ctx, log2, points):
    """Points side by side in one corner, over the torus's seams, and many of them at one address: rows shorter than a
    block, exactly one, and several blocks long (a row's ends then lie in other blocks)."""
    lw, lh = log2
    n, w, h = 1 << (lw + lh), 1 << lw, 1 << lh
    rng = np.random.default_rng([lw, lh, points])
    f, fo = rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    p = np.zeros(points, A.WAVE_POINT_DTYPE)
    p["x"], p["y"] = (w + rng.integers(-4, 4, points)) % w, (h + rng.integers(-3, 3, points)) % h
    p["x"][1::4] = (1024 + rng.integers(-2, 2, len(p[1::4]))) % w  # both sides of a block's end inside a row
    p["x"][2::4], p["y"][2::4] = 0, 0
    p["value"] = rng.normal(size=points) * np.exp2(rng.integers(-20, 20, points))
    att = np.float32(0.99)
    print(f"water crowded points {lw}x{lh} points={points}", flush=True)
    a, b = gpu_ctx.water_steps(f, fo, lw, lh, att, [p, p[::-1].copy()])
    for q in (p, p[::-1].copy()):
        f, fo = oracle.water_step(f, fo, lw, lh, att, q)
    assert np.array_equal(a.view(np.uint32), f.view(np.uint32))
    assert np.array_equal(b.view(np.uint32), fo.view(np.uint32))


@pytest.mark.parametrize("log2", [(4, 4), (5, 5), (10, 4), (4, 11), (9, 9), (10, 11)])
@pytest.mark.parametrize("shift", [(0, 0), (1, 2)])
def test_water_step_without_points(gpu_ctx, log2, shift):
    """The kernel without points, between steps with one (whose ticket it leaves alone), on fields of less than a
    block to the largest, 16-byte aligned and not."""
    lw, lh = log2
    n = 1 << (lw + lh)
    rng = np.random.default_rng([lw, lh])
    f, fo = rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    steps = [_points(rng, lw, lh, k) for k in (0, 0, 1, 0, 257, 1)]
    att = np.float32(0.97)
    print(f"water steps without points {lw}x{lh} shift={shift}", flush=True)
    bufs = [gpu_ctx.to_device(np.concatenate([np.full(s, 9, np.float32), v, np.full(4, 9, np.float32)])) for s, v in zip(shift, (f, fo))]
    ptr = [C.c_void_p(b.ptr.value + 4 * s) for s, b in zip(shift, bufs)]
    try:
        for k, p in enumerate(steps):
            gpu_ctx.check(gpu_ctx.lib.sw_water_step(gpu_ctx.h, ptr[k % 2], ptr[1 - k % 2], lw, lh, C.c_float(att),
                                                    C.c_void_p(p.ctypes.data) if len(p) else None, len(p)), "sw_water_step")
        got = [b.read(np.float32, n + s + 4) for s, b in zip(shift, bufs)]
    finally:
        for b in bufs:
            b.free()
    for p in steps:
        f, fo = oracle.water_step(f, fo, lw, lh, att, p)
    for g, s, ref in zip(got, shift, (f, fo)):
        assert np.array_equal(g[s:s + n].view(np.uint32), ref.view(np.uint32))
        assert np.all(g[:s] == 9) and np.all(g[s + n:] == 9)


@pytest.mark.parametrize("shift", [(1, 0), (0, 3), (2, 2)])
def test_water_unaligned_fields(gpu_ctx, shift):
    lw, lh = 6, 6
    n = 1 << (lw + lh)
    rng = np.random.default_rng(shift)
    f, fo = rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    p = _points(rng, lw, lh, 12)
    att = np.float32(0.98)
    m = sw_host.Map(seed=3, grid=(10, 10, 4), texture_size=64, num_materials=3, num_decal_textures=1, num_model_textures=1)
    m.data.levels["flags"][0:5] |= 1
    params = A.WaterTextureParams(0, 5, A.WATER_COLOR_DEFORMED, 0, 0.3, 0)
    bufs = [gpu_ctx.to_device(np.concatenate([np.full(s, 9, np.float32), v, np.full(4, 9, np.float32)])) for s, v in zip(shift, (f, fo))]
    ptr = [C.c_void_p(b.ptr.value + 4 * s) for s, b in zip(shift, bufs)]
    mh = gpu_ctx.upload_map(m.data)
    try:
        print(f"water step and texture at float offsets {shift}", flush=True)
        gpu_ctx.check(gpu_ctx.lib.sw_water_step(gpu_ctx.h, ptr[0], ptr[1], lw, lh, C.c_float(att), C.c_void_p(p.ctypes.data), len(p)),
                      "sw_water_step")
        gpu_ctx.check(gpu_ctx.lib.sw_water_make_texture(gpu_ctx.h, mh, ptr[0], lw, lh, C.byref(params)), "sw_water_make_texture")
        got = [b.read(np.float32, n + s + 4) for s, b in zip(shift, bufs)]
        texels = gpu_ctx.map_read(mh, 0, 0, len(m.data.texels))
    finally:
        gpu_ctx.release_map(mh)
        for b in bufs:
            b.free()
    # the step writes the new field over the old one; the field keeps its own values with the points added
    ra, rb = oracle.water_step(f, fo, lw, lh, att, p)
    for g, s, ref in zip(got, shift, (rb, ra)):
        assert np.array_equal(g[s:s + n].view(np.uint32), ref.view(np.uint32))
        assert np.all(g[:s] == 9) and np.all(g[s + n:] == 9)
    ref = oracle.water_make_texture(m.data, rb, lw, lh, params)
    assert np.array_equal(texels.view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("log2", [(4, 4), (5, 6), (6, 7), (9, 5)])
@pytest.mark.parametrize("shift", [(0, 0), (1, 0), (0, 3)])
def test_water_step_alone(gpu_ctx, log2, shift):
    """A step without points: fields of less than a block, of a block for some XCDs and of several for each, both alignments."""
    lw, lh = log2
    n = 1 << (lw + lh)
    rng = np.random.default_rng([lw, lh, *shift])
    f, fo = rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    bufs = [gpu_ctx.to_device(np.concatenate([np.full(s, 9, np.float32), v, np.full(4, 9, np.float32)])) for s, v in zip(shift, (f, fo))]
    ptr = [C.c_void_p(b.ptr.value + 4 * s) for s, b in zip(shift, bufs)]
    try:
        print(f"water step of {1 << lw} x {1 << lh} without points at float offsets {shift}", flush=True)
        gpu_ctx.check(gpu_ctx.lib.sw_water_step(gpu_ctx.h, ptr[0], ptr[1], lw, lh, C.c_float(0.98), None, 0), "sw_water_step")
        gpu_ctx.check(gpu_ctx.lib.sw_sync(gpu_ctx.h), "sw_sync")
        got = [b.read(np.float32, n + s + 4) for s, b in zip(shift, bufs)]
    finally:
        for b in bufs:
            b.free()
    new, old = oracle.water_step(f, fo, lw, lh, np.float32(0.98), np.zeros(0, A.WAVE_POINT_DTYPE))
    for g, s, ref in zip(got, shift, (old, new)):
        assert np.array_equal(g[s:s + n].view(np.uint32), ref.view(np.uint32))
        assert np.all(g[:s] == 9) and np.all(g[s + n:] == 9)


def test_water_texture_level_not_on_16_bytes(gpu_ctx):
    """A level that starts on an odd texel (8 bytes past a multiple of 16)."""
    lw, lh = 5, 4
    rng = np.random.default_rng(4)
    sizes = [(max(32 >> k, 1), max(16 >> k, 1)) for k in range(5)]
    levels = []
    off = 1
    for w, h in sizes:
        levels.append((off, w, h, A.TEX_HAS_NORMAL_MAP, 0))
        off += w * h
    texels = np.zeros(off, A.TEXEL_DTYPE)
    texels["diffuse"] = rng.integers(0, 1 << 32, off, dtype=np.uint32)
    d = A.MapData(texels, np.zeros(1, np.uint32), np.zeros((1, 3), np.float32), np.zeros(1, A.DIRLM_DTYPE),
                  np.array(levels, dtype=A.LEVEL_DTYPE))
    field = rng.normal(size=32 * 16).astype(np.float32)
    params = A.WaterTextureParams(0, 0, A.WATER_COLOR_KEEP, 0, 0.5, 0)
    mh = gpu_ctx.upload_map(d)
    try:
        gpu_ctx.water_make_texture(mh, field, lw, lh, params)
        got = gpu_ctx.map_read(mh, 0, 0, off)
    finally:
        gpu_ctx.release_map(mh)
    ref = oracle.water_make_texture(d, field, lw, lh, params)
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))
