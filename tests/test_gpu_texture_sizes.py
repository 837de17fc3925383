"""Texture operations over sizes and shifts at the edges of their index arithmetic, against the oracle: widths
that are and are not powers of two, levels of less than a block and of several, sources of other sizes, shifts
of any sign up to the limits of 32 bits, destinations that the first operation overwrites or blends into, calls
of more destinations than a wave probes at once and of arguments around the size from which a kernel copies them."""
import numpy as np
import pytest

import oracle
import sw_abi as A

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (37, 5), (300, 7), (1024, 3), (64, 64), (33, 65), (1, 1025), (513, 2), (96, 48), (7, 1)]
I32 = 2**31 - 1


@pytest.mark.parametrize("lite", [False, True])
@pytest.mark.parametrize("first_blend", [A.BLEND_NONE, A.BLEND_AVERAGE])
def test_layer_sizes_and_shifts(gpu_ctx, lite, first_blend):
    rng = np.random.default_rng([7, int(lite), first_blend])
    n = len(SIZES)
    levels = np.zeros(3 * n, dtype=A.LEVEL_DTYPE)  # n destinations, then 2 n sources
    offset = 0
    for i, (w, h) in enumerate(SIZES * 3):
        levels[i]["offset"], levels[i]["width"], levels[i]["height"] = offset, w, h
        levels[i]["flags"] = A.TEX_LITE_LEVEL if lite else 0
        offset += w * h
    raw = rng.integers(0, 1 << 32, size=(offset, 2), dtype=np.uint32)
    tex = np.zeros(1 if lite else offset, dtype=A.TEXEL_DTYPE)
    if not lite:
        tex = np.ascontiguousarray(raw).view(A.TEXEL_DTYPE).reshape(-1)
    data = A.MapData(tex, raw[:, 0].copy() if lite else np.zeros(1, np.uint32), np.zeros((1, 3), np.float32),
                     np.zeros(1, A.DIRLM_DTYPE), levels)
    shifts = [0, 1, -1, 37, -1000003, I32, I32 - 1, I32 - 40, -I32 - 1, 65536]
    ops = np.zeros(3 * n, dtype=A.TEXTURE_OP_DTYPE)
    for i in range(3 * n):
        d = i // 3
        ops[i]["kind"] = A.TEXOP_LAYER_LITE if lite else A.TEXOP_LAYER
        ops[i]["dst_level"], ops[i]["src_level"] = d, n + int(rng.integers(0, 2 * n))
        ops[i]["blend"] = first_blend if i % 3 == 0 else int(rng.integers(0, 5))
        ops[i]["shift"] = (shifts[(i * 7 + d) % len(shifts)], shifts[(i * 3 + 1) % len(shifts)])
        ops[i]["light"] = [(1.0, 1.0, 1.0), (0.5, 1.5, 0.25)][int(rng.integers(0, 2))]
    print(f"case texture sizes lite={lite} first blend={first_blend}", flush=True)
    mh = gpu_ctx.upload_map(data)
    try:
        gpu_ctx.apply_texture_ops(mh, ops, np.zeros(0, np.int32))
        rtex, rlite = oracle.apply_texture_ops(data, ops, np.zeros(0, np.int32))
        if lite:
            assert np.array_equal(gpu_ctx.map_read(mh, 1, 0, len(rlite)), rlite)
        else:
            assert np.array_equal(gpu_ctx.map_read(mh, 0, 0, len(rtex)).view(np.uint64), rtex.view(np.uint64))
    finally:
        gpu_ctx.release_map(mh)


@pytest.mark.parametrize("destinations", [64, 65, 200, 5000])
@pytest.mark.parametrize("extra", [-4, 0, 4, 40000])
def test_many_destinations_and_argument_sizes(gpu_ctx, destinations, extra):
    """Small levels of both kinds in turn, some of several blocks: the block's run is searched in two levels above 64
    runs, in three above 4096. The shift table ends `extra` bytes past 16 KiB of arguments (records of 32 bytes per
    destination and 48 per operation, each part on 256 bytes) where they leave room for it, and its last entries are
    used."""
    rng = np.random.default_rng([destinations, extra + 4])
    n = destinations
    levels = np.zeros(2 * n + 2, dtype=A.LEVEL_DTYPE)  # destinations, sources, a source for each kind of other size
    offset = [0, 0]
    for i in range(2 * n + 2):
        lite = i % 2
        w, h = (16, 16) if i >= 2 * n else ([(8, 8), (8, 8), (40, 60), (5, 3)] if n < 1000 else [(8, 8)])[i % n // 2 % (4 if n < 1000 else 1)]
        if n % 2 and n <= i < 2 * n:
            lite = (i - n) % 2
        levels[i]["offset"], levels[i]["width"], levels[i]["height"] = offset[lite], w, h
        levels[i]["flags"] = A.TEX_LITE_LEVEL if lite else 0
        offset[lite] += w * h
    raw = rng.integers(0, 1 << 32, size=(offset[0], 2), dtype=np.uint32)
    data = A.MapData(np.ascontiguousarray(raw).view(A.TEXEL_DTYPE).reshape(-1), rng.integers(0, 1 << 32, offset[1], dtype=np.uint32),
                     np.zeros((1, 3), np.float32), np.zeros(1, A.DIRLM_DTYPE), levels)
    per = 2 if n <= 200 else 1
    ops = np.zeros(per * n, dtype=A.TEXTURE_OP_DTYPE)
    up = lambda x: (x + 255) // 256 * 256
    used = up(up(32 * n) + 48 * len(ops))
    shifts = rng.integers(-100, 100, max((16384 + extra - used) // 4, 64)).astype(np.int32)
    for i in range(len(ops)):
        d = i // per
        turb = i % per == 0 and int(levels[d]["width"]) == 8
        lite = bool(levels[d]["flags"])
        ops[i]["kind"] = A.TEXOP_TURB if turb else A.TEXOP_LAYER_LITE if lite else A.TEXOP_LAYER
        ops[i]["dst_level"], ops[i]["src_level"] = d, n + d if turb or d % 3 else 2 * n + int(lite)
        ops[i]["blend"], ops[i]["shift"] = int(rng.integers(0, 5)), rng.integers(-50, 50, 2)
        ops[i]["light"], ops[i]["turb_shifts"] = rng.uniform(0.2, 1.5, 3), len(shifts) - 8 - int(rng.integers(0, 40))
    print(f"case texture destinations={n} extra={extra}", flush=True)
    mh = gpu_ctx.upload_map(data)
    try:
        gpu_ctx.apply_texture_ops(mh, ops, shifts)
        rtex, rlite = oracle.apply_texture_ops(data, ops, shifts)
        assert np.array_equal(gpu_ctx.map_read(mh, 1, 0, len(rlite)), rlite)
        assert np.array_equal(gpu_ctx.map_read(mh, 0, 0, len(rtex)).view(np.uint64), rtex.view(np.uint64))
    finally:
        gpu_ctx.release_map(mh)
