"""The depth rasteriser's row passes (sw_render_depth) against the oracle, bit for bit: rows wider than one
pass of 256 columns and ragged ones, rows of which only some passes hold a span, more than 64 draws over a target (several chunks, overwriting only,
mixed and depth-tested only), more than 64 targets, pixels that no draw covers, and equations whose chains of
additions cross powers of two and zero."""
import numpy as np
import pytest

import oracle
import scenes
import sw_abi as A

pytestmark = pytest.mark.gpu


def _scene(rng, sizes, draws_per_target, test_of, steep=False):
    targets = np.zeros(len(sizes), dtype=A.DEPTH_TARGET_DTYPE)
    draws, vdata, ints, off = [], [], 0, 0
    for t, (w, h) in enumerate(sizes):
        n = draws_per_target(t)
        targets[t]["offset"], targets[t]["width"], targets[t]["height"] = off, w, h
        targets[t]["first_draw"], targets[t]["num_draws"] = len(draws), n
        targets[t]["flags"] = A.DEPTH_CIRCLE if w == h and t % 2 else 0
        off += w * h
        for i in range(n):
            fx, de, _ = scenes.make_polygon(rng, w, h, 16, 16, A.TC_PERSPECTIVE, thin=i % 5 == 1)
            d = np.zeros(1, dtype=A.DEPTH_DRAW_DTYPE)[0]
            d["first_vertex_int"], d["num_vertices"], d["depth_test"] = ints, len(fx) // 2, test_of(i)
            # steep: 1 / z from far below a power of two to far above it, or through zero, along a row
            d["depth_equation"] = rng.normal(size=3) * [3e-3, 2e-3, 0.5] if steep else de
            draws.append(d)
            vdata.append(fx)
            ints += len(fx)
    return targets, np.array(draws, dtype=A.DEPTH_DRAW_DTYPE), np.concatenate(vdata).astype(np.int32), off


CASES = {
    "wide": ([(1500, 5), (4099, 3), (257, 64), (255, 9), (1, 40)], lambda t: 20, lambda i: int(i % 4 == 3), False),
    "many_draws": ([(300, 40), (64, 64)], lambda t: 200, lambda i: 0, False),
    "many_mixed": ([(300, 40), (64, 64)], lambda t: 150, lambda i: int(i % 3 == 0), False),
    "tests_only": ([(130, 50)], lambda t: 70, lambda i: 1, False),
    "many_targets": ([(9 + t % 5, 3 + t % 7) for t in range(150)], lambda t: t % 4, lambda i: int(i == 2), False),
    "steep": ([(700, 60), (256, 256)], lambda t: 90, lambda i: int(i % 6 == 5), True),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_depth_rows_bit_exact(gpu_ctx, name):
    sizes, draws_per_target, test_of, steep = CASES[name]
    rng = np.random.default_rng(len(name))
    targets, draws, vdata, n = _scene(rng, sizes, draws_per_target, test_of, steep)
    init = rng.uniform(-0.01, 0.01, size=n).astype(np.float32)
    print(f"depth rows {name}: {len(draws)} draws, {n} texels", flush=True)
    out = gpu_ctx.render_depth(targets, draws, vdata, init)
    ref = oracle.render_depth(targets, draws, vdata, init)
    bad = np.flatnonzero(out.view(np.uint32) != ref.view(np.uint32))
    assert bad.size == 0, f"{bad.size} texels differ, first {bad[:5].tolist()}"
    assert np.any(out != init)


@pytest.mark.parametrize("test", ["overwrite", "mixed", "tests"])
def test_wide_rows_of_narrow_polygons(gpu_ctx, test):
    """Rows wide enough that the passes which a span meets are found first: polygons a few dozen columns wide on and
    around the ends of passes (256 columns) and of groups of 64 passes, circles whose outside lies in other passes."""
    rng = np.random.default_rng(31)
    sizes = [(1024, 9), (1025, 30), (1100, 1100), (2049, 2049), (5000, 7), (16384, 5), (16385, 6), (33000, 3), (65535, 2)]
    targets = np.zeros(len(sizes), dtype=A.DEPTH_TARGET_DTYPE)
    draws, vdata, ints, off = [], [], 0, 0
    for t, (w, h) in enumerate(sizes):
        targets[t]["offset"], targets[t]["width"], targets[t]["height"] = off, w, h
        targets[t]["first_draw"], targets[t]["num_draws"] = len(draws), 70
        targets[t]["flags"] = A.DEPTH_CIRCLE if w == h else 0
        off += w * h
        for i in range(70):
            fx, de, _ = scenes.make_polygon(rng, 48, h, 16, 16, A.TC_PERSPECTIVE)
            x = [int(rng.integers(0, w)), 256 * int(rng.integers(0, w // 256)) - 24, 16384 - 24, w - 30][i % 4 if i % 8 < 4 else 0]
            v = fx.astype(np.int64)
            v[0::2] += min(x, 32600) << 16  # fixed16 coordinates end at 32767
            d = np.zeros(1, dtype=A.DEPTH_DRAW_DTYPE)[0]
            d["first_vertex_int"], d["num_vertices"] = ints, len(v) // 2
            d["depth_equation"], d["depth_test"] = de, {"overwrite": 0, "mixed": i % 3 == 0, "tests": 1}[test]
            draws.append(d)
            vdata.append(np.clip(v, -2**31, 2**31 - 1).astype(np.int32))
            ints += len(v)
    draws, vdata = np.array(draws, dtype=A.DEPTH_DRAW_DTYPE), np.concatenate(vdata)
    init = rng.uniform(-0.01, 0.01, size=off).astype(np.float32)
    print(f"depth wide rows {test}: {len(draws)} draws, {off} texels", flush=True)
    out = gpu_ctx.render_depth(targets, draws, vdata, init)
    ref = oracle.render_depth(targets, draws, vdata, init)
    bad = np.flatnonzero(out.view(np.uint32) != ref.view(np.uint32))
    assert bad.size == 0, f"{bad.size} texels differ, first {bad[:5].tolist()}"
    assert np.any(out != init)


def test_infinite_and_nan_equations(gpu_ctx):
    """Equations that are infinite or NaN from the start, or overflow along a row or down a part, beside ordinary ones."""
    rng = np.random.default_rng(33)
    targets, draws, vdata, n = _scene(rng, [(1500, 40), (300, 64), (64, 64)], lambda t: 40, lambda i: int(i % 4 == 1))
    bad = np.array([[0, 0, np.inf], [0, 0, -np.inf], [1e36, 0, 3e38], [0, -2e37, -3e38], [np.inf, 0, 1], [-3e38, 3e38, 0], [np.nan, 0, 0],
                    [0, np.nan, 1]], np.float32)
    draws["depth_equation"][::5] = bad[np.arange(len(draws[::5])) % len(bad)]
    init = rng.uniform(-0.01, 0.01, size=n).astype(np.float32)
    print(f"depth of infinite equations: {len(draws)} draws, {n} texels", flush=True)
    out = gpu_ctx.render_depth(targets, draws, vdata, init)
    ref = oracle.render_depth(targets, draws, vdata, init)
    assert np.count_nonzero(~np.isfinite(ref)) > n // 20
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(out), nan) and np.array_equal(out.view(np.uint32)[~nan], ref.view(np.uint32)[~nan])
