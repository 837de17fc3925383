"""Texture operations over sizes and shifts at the edges of their index arithmetic, against the oracle: widths
that are and are not powers of two, levels of less than a block and of several, sources of other sizes, shifts
of any sign up to the limits of 32 bits, destinations that the first operation overwrites or blends into."""
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
