"""Every raster tile size (16, 32 and 64 x 4, 8 and 16 pixels, chosen from the views' sizes and the tile rows)
against the oracle: views whose last column and last rows are cut at every unit of 16 x 4 pixels, a view that
draws over what is there, both colour sizes, a re-run after the tile rows were set anew."""
import ctypes as C

import numpy as np
import pytest

import oracle
import scenes
import sw_abi as A

pytestmark = pytest.mark.gpu

# tile widths by rows: 4 -> 16, 32, 64; 8 -> 16, 32, 32; 16 -> 16
SMALL = (((1, 1), (17, 5), (50, 31)), ((1003, 603), (33, 2)), ((1405, 803), (79, 9)))


def _check(ctx, rows, bits, sizes, seed):
    m, b = scenes.make_batch(seed, color_bits=bits, view_sizes=sizes)
    b.views["clear_background"][-1] = 0  # the last view draws over the buffer (zeros)
    prev = ctx.tile_rows()
    mh = ctx.upload_map(m)
    out = ctx.to_device(np.zeros(b.fb_texels, dtype=b.color_dtype))
    try:
        ctx.set_tile_rows(rows)
        fb = ctx.render_batch(mh, b, out=out)
    finally:
        out.free()
        ctx.set_tile_rows(prev)
        ctx.release_map(mh)
    ofb = oracle.render(m, b, mode=oracle.MODE_EXACT)[0]
    assert np.array_equal(fb, ofb), f"{np.count_nonzero(fb != ofb)} pixels differ"


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("rows", [4, 8, 16])
@pytest.mark.parametrize("sizes", SMALL)
def test_tile_sizes(gpu_ctx, rows, bits, sizes):
    print(f"case raster tiles rows={rows} bits={bits} sizes={sizes}", flush=True)
    _check(gpu_ctx, rows, bits, sizes, 700 + rows)


@pytest.mark.parametrize("rows,bits", [(8, 64), (16, 32), (16, 64)])
def test_largest_tiles(gpu_ctx, rows, bits):
    """512 pixels to a tile, from 131,072 tiles of 256 on."""
    print(f"case raster largest tiles rows={rows} bits={bits}", flush=True)
    _check(gpu_ctx, rows, bits, ((16381, 2083), (61, 13)), 720 + rows)


@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("rows", [4, 16])
def test_rerun_keeps_its_tiling(plain, rows):
    """More span records than a fresh context holds: the raster is run again, with the tiling its views were given
    even if the tile rows were set in between. (More than 2^25 rows of views over all draws, so that records are
    counted and not laid out per draw; more than 2^20 records in them.)"""
    print(f"case rerun plain={plain} rows={rows}", flush=True)
    m, b = scenes.make_batch(77, view_sizes=((24, 16384),), surfaces_per_view=8, draws_per_view=2100, triangles=False)
    ref = oracle.render(m, b, mode=oracle.MODE_EXACT)[0]
    ctx = A.Context(0)
    try:
        mh, v = ctx.upload_map(m), b.views[0]
        fb = np.zeros(b.fb_texels, dtype=b.color_dtype)
        if plain:
            cam = (C.c_float * 3)(*[float(x) for x in v["cam_pos"]])
            ctx.check(ctx.lib.sw_frame_begin(ctx.h, mh, 32, 24, 16384, cam, 1, int(v["background_color"])), "begin")
            ctx.check(ctx.lib.sw_build_surfaces(ctx.h, b.surfaces.ctypes.data, len(b.surfaces), b.lights.ctypes.data, len(b.lights),
                                                b.light_indices.ctypes.data, len(b.light_indices)), "surfaces")
            ctx.check(ctx.lib.sw_raster_draws(ctx.h, b.draws.ctypes.data, len(b.draws), b.vertex_data.ctypes.data,
                                              len(b.vertex_data)), "draws")
            ctx.set_tile_rows(rows)
            ctx.check(ctx.lib.sw_frame_end(ctx.h, fb.ctypes.data, 24 * 4, 0), "end")
        else:
            out = ctx.alloc(b.fb_texels * 4)
            cb = b.ctypes_batch()
            ctx.check(ctx.lib.sw_render_batch_async(ctx.h, mh, C.byref(cb), out.ptr), "render")
            ctx.set_tile_rows(rows)
            ctx.check(ctx.lib.sw_batch_wait(ctx.h), "wait")
            fb = out.read(b.color_dtype, b.fb_texels)
            out.free()
        assert ctx.lib.sw_last_reruns(ctx.h) > 0
        ctx.release_map(mh)
    finally:
        ctx.close()
    assert np.array_equal(fb, ref), f"{np.count_nonzero(fb != ref)} pixels differ"
