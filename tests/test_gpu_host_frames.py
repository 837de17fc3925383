"""Frames and batches of host-resident command buffers: the queued uploads (several calls before the raster, buffers
that grow, arrays past the size that is queued) and the copy of the frame back (pinned and pageable destinations,
offsets, padded rows; left alone after an error), against the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
import scenes
import sw_abi as A

pytestmark = pytest.mark.gpu


def _p(a, offset=0):
    return C.c_void_p((a.data_ptr() if isinstance(a, torch.Tensor) else a.ctypes.data) + offset)


def _draw(ctx, mh, b, before=None):
    v = b.views[0]
    cam = (C.c_float * 3)(*[float(x) for x in v["cam_pos"]])
    ctx.check(ctx.lib.sw_frame_begin(ctx.h, mh, b.color_bits, int(v["width"]), int(v["height"]), cam, 1, int(v["background_color"])), "begin")
    for s in (before, b) if before else (b,):
        ctx.check(ctx.lib.sw_build_surfaces(ctx.h, _p(s.surfaces), len(s.surfaces), _p(s.lights), len(s.lights), _p(s.light_indices),
                                            len(s.light_indices)), "surfaces")
    ctx.check(ctx.lib.sw_raster_draws(ctx.h, _p(b.draws), len(b.draws), _p(b.vertex_data), len(b.vertex_data)), "draws")


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("size", [(160, 100), (97, 61), (1, 1), (3, 200), (640, 401)])
def test_frame_destinations(gpu_ctx, bits, size):
    print(f"case host frame {size} bits={bits}", flush=True)
    w, h = size
    m, b = scenes.make_batch(w + h, color_bits=bits, view_sizes=(size,))
    ref = oracle.render(m, b, mode=oracle.MODE_EXACT)[0].reshape(h, w)
    px, row = bits // 8, w * bits // 8
    mh = gpu_ctx.upload_map(m)
    try:
        for pinned in (True, False):
            for offset, pitch in ((0, row), (16, row), (8, row), (0, row + 24)):
                buf = torch.full((offset + pitch * h + 64,), 0x5A, dtype=torch.uint8, pin_memory=pinned)
                _draw(gpu_ctx, mh, b)
                gpu_ctx.check(gpu_ctx.lib.sw_frame_end(gpu_ctx.h, _p(buf, offset), pitch, 0), "end")
                raw = buf.numpy()
                rows = raw[offset:offset + pitch * h].reshape(h, pitch)
                out = np.ascontiguousarray(rows[:, :row]).view(np.uint64 if px == 8 else np.uint32).reshape(h, w)
                assert np.array_equal(out, ref), (pinned, offset, pitch)
                assert np.all(rows[:-1, row:] == 0x5A) and np.all(raw[:offset] == 0x5A) and np.all(raw[offset + pitch * h:] == 0x5A)
    finally:
        gpu_ctx.release_map(mh)


def test_uploads_of_growing_and_repeated_calls(gpu_ctx):
    """Surfaces set twice before the draws (the second replaces the first), frames of growing command buffers."""
    m, small = scenes.make_batch(41, view_sizes=((160, 120),), draws_per_view=3)
    mh = gpu_ctx.upload_map(m)
    try:
        for draws in (5, 400, 30, 3000):
            print(f"case uploads draws={draws}", flush=True)
            b = scenes.make_batch(41, view_sizes=((160, 120),), surfaces_per_view=24 + draws // 20, draws_per_view=draws)[1]
            ref = oracle.render(m, b, mode=oracle.MODE_EXACT)[0]
            out = torch.zeros(160 * 120, dtype=torch.int32, pin_memory=True)
            _draw(gpu_ctx, mh, b, before=small)
            gpu_ctx.check(gpu_ctx.lib.sw_frame_end(gpu_ctx.h, _p(out), 160 * 4, 0), "end")
            assert np.array_equal(out.numpy().view(np.uint32), ref), draws
    finally:
        gpu_ctx.release_map(mh)


def test_batch_arrays_past_the_queued_size(gpu_ctx):
    print("case batch of large host arrays", flush=True)
    m, b = scenes.make_batch(43, view_sizes=((64, 48),) * 60, surfaces_per_view=40, draws_per_view=200)
    assert b.draws.nbytes > 1 << 20 > b.surfaces.nbytes
    ref = oracle.render(m, b, mode=oracle.MODE_EXACT)[0]
    mh = gpu_ctx.upload_map(m)
    try:
        for _ in range(3):
            assert np.array_equal(gpu_ctx.render_batch(mh, b), ref)
    finally:
        gpu_ctx.release_map(mh)


@pytest.mark.parametrize("views", [1, 2])
@pytest.mark.parametrize("missing", ["surfaces", "draws", "vertex_data"])
def test_missing_host_array_is_an_error(gpu_ctx, missing, views):
    """A null array with a count is refused before any of the batch is read or queued, synchronously and not, and the
    next batch of the context is drawn as usual."""
    print(f"case missing {missing} views={views}", flush=True)
    m, b = scenes.make_batch(44, view_sizes=((64, 48),) * views)
    ref = oracle.render(m, b, mode=oracle.MODE_EXACT)[0]
    out = torch.zeros(b.fb_texels, dtype=torch.int32, device="cuda")
    mh = gpu_ctx.upload_map(m)
    try:
        cb = b.ctypes_batch()
        setattr(cb, missing, None)
        for render in (gpu_ctx.lib.sw_render_batch, gpu_ctx.lib.sw_render_batch_async):
            with pytest.raises(A.SwError, match="null surfaces, draws or vertex data"):
                gpu_ctx.check(render(gpu_ctx.h, mh, C.byref(cb), _p(out)), "render")
        assert np.array_equal(gpu_ctx.render_batch(mh, b), ref)
    finally:
        gpu_ctx.release_map(mh)


@pytest.mark.parametrize("bits", [32, 64])
def test_pinned_destination_after_an_error(gpu_ctx, bits):
    """The copy into pinned memory is queued before the frame's errors are known: an invalid surface (a texture level out
    of range) is reported and leaves the destination as it was; the next frame into it is the oracle's."""
    print(f"case pinned destination after an error bits={bits}", flush=True)
    m, b = scenes.make_batch(45, color_bits=bits, view_sizes=((160, 120),))
    bad = scenes.make_batch(45, color_bits=bits, view_sizes=((160, 120),))[1]
    bad.surfaces["flags"][3] |= A.SURF_DIFFUSE_LAYER
    bad.surfaces["texture_level"][3] = 0xFFFFFF
    ref = oracle.render(m, b, mode=oracle.MODE_EXACT)[0]
    row = 160 * bits // 8
    out = torch.full((row * 120,), 0x5A, dtype=torch.uint8, pin_memory=True)
    mh = gpu_ctx.upload_map(m)
    try:
        for _ in range(2):
            _draw(gpu_ctx, mh, bad)
            with pytest.raises(A.SwError, match="invalid surface descriptor"):
                gpu_ctx.check(gpu_ctx.lib.sw_frame_end(gpu_ctx.h, _p(out), row, 0), "end")
            assert np.all(out.numpy() == 0x5A)
            _draw(gpu_ctx, mh, b)
            gpu_ctx.check(gpu_ctx.lib.sw_frame_end(gpu_ctx.h, _p(out), row, 0), "end")
            assert np.array_equal(out.numpy().view(ref.dtype), ref)
            out.fill_(0x5A)
    finally:
        gpu_ctx.release_map(mh)
