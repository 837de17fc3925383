"""Every raster tile size (16, 32 and 64 x 4, 8 and 16 pixels, chosen from the views' sizes and the tile rows)
against the oracle: views whose last column and last rows are cut at every unit of 16 x 4 pixels, a view that
draws over what is there, both colour sizes."""
import numpy as np
import pytest

import oracle
import scenes

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
