"""The blur's tiles, reaches and taps, the downscale's row parts and the tonemap's 2 x 2 groups at their edges,
against the oracle: bloom buffers around multiples of 32 texels, frames of one bloom texel, radii at both ends
of each reach (2, 4, 8, 12, 16), full-range lanes."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("linear", [False, True])
@pytest.mark.parametrize("scale_log2,sigma", [(1, 0.4), (1, 1.0), (1, 1.3), (1, 2.0), (1, 2.6), (1, 4.0), (1, 5.5), (1, 5.9), (1, 8.0), (1, 9.0), (2, 8.0),
                                              (2, 30.0), (3, 12.0)])
@pytest.mark.parametrize("bw,bh,extra", [(1, 1, 0), (1, 70, 1), (31, 33, 1), (32, 32, 0), (65, 3, 1), (258, 64, 1)])
def test_bloom_edges(gpu_ctx, scale_log2, sigma, linear, bw, bh, extra):
    w, h = (bw << scale_log2) + extra, (bh << scale_log2) + extra
    print(f"case bloom {w}x{h} scale_log2 {scale_log2} sigma {sigma} linear {linear}", flush=True)
    rng = np.random.default_rng([w, h, int(sigma * 10)])
    hdr = rng.integers(0, 1 << 63, size=(h, w), dtype=np.uint64) * np.uint64(2)
    hdr[rng.random((h, w)) < 0.3] = 0
    hdr[rng.random((h, w)) < 0.1] = np.uint64(0xFFFFFFFFFFFFFFFF)
    out, avg = gpu_ctx.postprocess(hdr, 0.004, (1.0, 0.8, 1.2), bloom=(sigma, scale_log2, 0.5, linear))
    ref, ravg, radius, _ = oracle.bloom(hdr, 0.004, (1.0, 0.8, 1.2), sigma, scale_log2, 0.5, linear)
    assert np.array_equal(out, ref), f"{np.count_nonzero(out != ref)} pixels differ (radius {radius})"
    assert np.array_equal(avg, ravg)
