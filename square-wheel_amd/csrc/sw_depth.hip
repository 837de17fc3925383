// The depth rasteriser of shadow maps (DepthRasterizer, rasterizer.rs:1295-1474): convex polygons
// with a 1 / z equation drawn into f32 depth buffers, overwriting (back-to-front order) or keeping
// the larger value (depth test).
//
// The reference steps 1 / z by additions along a span (inv_z += d_inv_z_dx) and along the rows of a
// polygon part (line_inv_z += d_inv_z_dy); float addition rounds at every step, so each value is the
// end of a chain of additions, which sw_chain.h gives without walking it: every row's and every
// pixel's value on its own.
//
//   k_depth_setup   one wave per draw: the edge walk into parts (identical on all lanes, comparisons
//                   only), the parts' slopes one part per lane, then one row per lane: the span's x
//                   range and its first pixel's 1 / z. Reads the packed draws, their targets and vertices
//                   straight from pinned host memory (each draw and vertex once, a target's 40 bytes once
//                   per draw: no copy goes ahead of the launch) and leaves in device memory what the
//                   raster reads many times.
//   k_depth_raster  one wave per depth-buffer row: the row's spans of the target's draws from the last
//                   to the first, each taking the pixels no later overwriting draw has taken (64-pixel
//                   masks, scalar arithmetic), until all are taken; then each pixel's 1 / z once.
#include <cstring>
#include <string>
#include <vector>

#include "sw_internal.h"
#include "sw_device.h"
#include "sw_chain.h"

using namespace swd;

namespace
{

SW_DEV int32_t imax32(int32_t a, int32_t b) { return a > b ? a : b; }
SW_DEV int32_t imin32(int32_t a, int32_t b) { return a < b ? a : b; }

struct alignas(8) DepthRow
{
	uint16_t x0, x1; // [x0, x1): the span's pixels (empty when x0 >= x1)
	float inv_z; // 1 / z at x0
};

struct DepthDrawDev
{
	uint32_t first_vertex_int, num_vertices;
	float dx, dy, k; // DepthEquation
	uint32_t depth_test;
	uint32_t target;
	uint32_t pad;
};

struct DepthTargetDev
{
	uint64_t offset; // of the depth buffer in the texels
	uint64_t rec_base; // row records: rec_base + y * num_draws + (draw - first_draw)
	uint32_t w, h;
	uint32_t first_draw, num_draws;
	uint32_t first_row; // raster rows: first_row + y
	uint32_t flags; // SW_DEPTH_*
};

// What the raster reads of a draw, beside its row records.
struct alignas(16) DepthDrawInfo
{
	int32_t first, end; // rows [first, end) have records
	float dx;
	uint32_t depth_test;
};

// make_shadow_map_circle (light.rs:130-154): texels [0, dx) and [size - dx, size) of row y are
// outside the inscribed circle
SW_DEV uint32_t circle_margin(int32_t size, int32_t y)
{
	const int32_t radius = size / 2, dy = y - radius;
	const int32_t r2 = radius * radius - dy * dy;
	const int32_t half = int32_t(__builtin_ceilf(__builtin_sqrtf(float(r2 > 0 ? r2 : 0))));
	return uint32_t(radius - (half < radius ? half : radius));
}

struct DepthLaunch
{
	const DepthDrawDev* draws; // pinned host memory: draws, targets and vertices
	const DepthTargetDev* host_targets;
	const int32_t* vdata;
	DepthTargetDev* targets; // device memory, written by the setup
	DepthDrawInfo* infos;
	DepthRow* rows;
	float* texels;
	uint32_t num_draws, num_targets, num_rows;
};

#define MAX_DEPTH_PARTS SW_MAX_POLYGON_VERTICES

SW_DEV int32_t lane_pull(int32_t v, uint32_t src) { return __builtin_amdgcn_ds_bpermute(int32_t(src << 2), v); }
SW_DEV float lane_pull_f(float v, uint32_t src) { return __builtin_bit_cast(float, lane_pull(__builtin_bit_cast(int, v), src)); }
SW_DEV int32_t rl(int32_t v, uint32_t lane) { return __builtin_amdgcn_readlane(v, lane); }

// Four draws per block, a wave each; blocks past the draws copy the targets to device memory.
__global__ __launch_bounds__(256) void k_depth_setup(DepthLaunch L, uint32_t draw_blocks)
{
	const uint32_t lane = threadIdx.x & 63u;
	if(blockIdx.x >= draw_blocks)
	{
		const uint32_t words = L.num_targets * uint32_t(sizeof(DepthTargetDev) / 4u);
		const uint32_t i = (blockIdx.x - draw_blocks) * 256u + threadIdx.x;
		if(i < words)
			reinterpret_cast<uint32_t*>(L.targets)[i] = reinterpret_cast<const uint32_t*>(L.host_targets)[i];
		return;
	}
	const uint32_t di = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
	if(di >= L.num_draws)
		return; // uniform over the wave; no barriers below
	const DepthDrawDev d = L.draws[di];
	const DepthTargetDev t = L.host_targets[d.target];
	const uint32_t n = d.num_vertices;
	int32_t vx = 0, vy = 0; // lane i: vertex i
	if(lane < n)
	{
		vx = L.vdata[d.first_vertex_int + lane * 2u];
		vy = L.vdata[d.first_vertex_int + lane * 2u + 1u];
	}
	// fill_polygon (rasterizer.rs:1315-1412): from the lowest vertex up both chains; lane p keeps part p
	uint32_t lower = 0, np = 0;
	int32_t min_y = rl(vy, 0);
	for(uint32_t i = 0; i < n; ++i)
		if(rl(vy, i) < min_y)
		{
			min_y = rl(vy, i);
			lower = i;
		}
	uint32_t left = lower, right = lower;
	int32_t cur_y = min_y;
	const int32_t H = int32_t(t.h);
	uint32_t pl = 0, pnl = 0, pr = 0, pnr = 0;
	int32_t p_cur = 0, p_y0 = 0, p_y1 = 0;
	bool p_wide = false;
	for(uint32_t guard = 0; guard < 2 * n + 2; ++guard)
	{
		const uint32_t next_left = left + n - 1 >= n ? left + n - 1 - n : left + n - 1;
		const uint32_t next_right = right + 1 >= n ? right + 1 - n : right + 1;
		const int32_t ly = rl(vy, left), nly = rl(vy, next_left), ry = rl(vy, right), nry = rl(vy, next_right);
		const int32_t dy_left = nly - ly, dy_right = nry - ry;
		const int32_t next_y = nly < nry ? nly : nry;
		const bool wide = dy_left > FIXED16_HALF && dy_right > FIXED16_HALF;
		const bool thin = !wide && dy_left > 0 && dy_right > 0 && fixed16_round_to_int(cur_y) < fixed16_round_to_int(next_y);
		if((wide || thin) && np < MAX_DEPTH_PARTS)
		{
			if(lane == np)
			{
				pl = left;
				pnl = next_left;
				pr = right;
				pnr = next_right;
				p_cur = cur_y;
				p_wide = wide;
				p_y0 = imax32(fixed16_round_to_int(cur_y), 0);
				p_y1 = imin32(fixed16_round_to_int(next_y), H);
			}
			np++;
		}
		if(next_left == next_right)
			break;
		if(nry < nly)
			right = next_right;
		else
			left = next_left;
		cur_y = next_y;
	}
	// the parts' sides and first rows (fill_polygon, fill_polygon_part :1414-1465), lane p for part p;
	// every lane takes part in the exchanges
	const int32_t lx = lane_pull(vx, pl), ly = lane_pull(vy, pl), nlx = lane_pull(vx, pnl), nly = lane_pull(vy, pnl);
	const int32_t rx = lane_pull(vx, pr), ry = lane_pull(vy, pr), nrx = lane_pull(vx, pnr), nry = lane_pull(vy, pnr);
	int32_t xl = 0, xr = 0, dl = 0, dr = 0;
	float line_inv_z = 0.0f;
	if(lane < np)
	{
		int32_t xs_l, xs_r;
		if(p_wide)
		{
			dl = fixed16_div(nlx - lx, nly - ly);
			dr = fixed16_div(nrx - rx, nry - ry);
			xs_l = lx + fixed16_mul(dl, p_cur - ly);
			xs_r = rx + fixed16_mul(dr, p_cur - ry);
		}
		else
		{
			const int32_t thin_line_y = int_to_fixed16(fixed16_round_to_int(p_cur)) + FIXED16_HALF;
			xs_l = lx + fixed16_mul_div(thin_line_y - ly, nlx - lx, nly - ly);
			xs_r = rx + fixed16_mul_div(thin_line_y - ry, nrx - rx, nry - ry);
		}
		const int32_t y_start_delta = int_to_fixed16(p_y0) + FIXED16_HALF - p_cur;
		xl = xs_l + fixed16_mul(y_start_delta, dl) + FIXED16_HALF;
		xr = xs_r + fixed16_mul(y_start_delta, dr) + FIXED16_HALF;
		line_inv_z = float(p_y0) * d.dy + 0.5f * (d.dx + d.dy) + d.k;
	}
	int32_t first = H, end = 0;
	for(uint32_t q = 0; q < np; ++q)
	{
		const int32_t y0 = rl(p_y0, q), y1 = rl(p_y1, q);
		if(y0 < y1)
		{
			first = imin32(first, y0);
			end = imax32(end, y1);
		}
	}
	// a row per lane: its part is the last one that holds it
	for(int32_t yb = first; yb < end; yb += 64)
	{
		const int32_t y = yb + int32_t(lane);
		uint32_t part = MAX_DEPTH_PARTS;
		for(uint32_t q = 0; q < np; ++q)
		{
			const int32_t y0 = rl(p_y0, q), y1 = rl(p_y1, q);
			part = y >= y0 && y < y1 ? q : part;
		}
		const uint32_t src = part < MAX_DEPTH_PARTS ? part : 0u;
		const int32_t y0 = lane_pull(p_y0, src);
		const int32_t r_xl = lane_pull(xl, src), r_xr = lane_pull(xr, src), r_dl = lane_pull(dl, src), r_dr = lane_pull(dr, src);
		const float r_z = lane_pull_f(line_inv_z, src);
		if(y < end)
		{
			DepthRow row{0, 0, 0.0f};
			if(part < MAX_DEPTH_PARTS)
			{
				const uint32_t r = uint32_t(y - y0);
				const int32_t x_left = wadd(r_xl, wmul(int32_t(r), r_dl)), x_right = wadd(r_xr, wmul(int32_t(r), r_dr));
				const int32_t x0 = imax32(fixed16_floor_to_int(x_left), 0), x1 = imin32(fixed16_floor_to_int(x_right), int32_t(t.w));
				if(x0 < x1)
					row = DepthRow{uint16_t(x0), uint16_t(x1), swchain::chain_add(r_z, d.dy, r) + float(x0) * d.dx};
			}
			L.rows[t.rec_base + uint64_t(uint32_t(y)) * t.num_draws + (di - t.first_draw)] = row;
		}
	}
	if(lane == 0)
		L.infos[di] = DepthDrawInfo{first < end ? first : 0, first < end ? end : 0, d.dx, d.depth_test};
}

// bits [0, n) of 64, n clamped to [0, 64]
SW_DEV uint64_t low_bits(int32_t n) { return n <= 0 ? 0ull : n >= 64 ? ~0ull : (1ull << n) - 1ull; }
// the bits of [x0, x1) that lie in the 32 columns from base on
SW_DEV uint32_t span_bits(int32_t x0, int32_t x1, int32_t base)
{
	const int32_t a = imax32(x0 - base, 0), b = imin32(x1 - base, 32);
	return a < b ? (~0u << a) & (~0u >> (32 - b)) : 0u;
}

#define DEPTH_SEGMENTS 4u // 64-pixel segments a wave holds at once
#define DEPTH_PASS (64u * DEPTH_SEGMENTS) // columns of a pass
#define DEPTH_GROUP (64u * DEPTH_PASS) // columns of 64 passes
#define DEPTH_NARROW (4u * DEPTH_PASS) // wider rows look at all their draws' spans first
#define DEPTH_FOUND 128u // and keep that many in LDS

// A draw's span of a row, packed x0 | x1 << 16 (0: none).
struct alignas(16) RowSpan
{
	uint32_t span;
	float inv_z; // 1 / z at x0
	float dx;
	uint32_t depth_test;
};

// the passes, a bit each, of the group of columns from base on that [x0, x1) meets
SW_DEV uint64_t pass_bits(uint32_t x0, uint32_t x1, uint32_t base)
{
	if(x0 >= x1 || x1 <= base || x0 >= base + DEPTH_GROUP)
		return 0ull;
	const uint32_t a = x0 > base ? (x0 - base) / DEPTH_PASS : 0u;
	return low_bits(int32_t((x1 - base + DEPTH_PASS - 1u) / DEPTH_PASS)) & ~low_bits(int32_t(a));
}

// The rows of a 256 x 256 cube side take one pass of 256 columns each. A back-to-front list overwrites
// most pixels several times: walked backwards, a row is finished after its nearest spans, and each pixel's
// chain is evaluated once instead of once per draw that covers it. Eight lights' 256 x 256 cube maps (3.1
// Mtexels, 1,633 draws): 33.6 us with every span filled in draw order by 16-lane chains, now 19.
// WIDE (a target wider than DEPTH_NARROW): a row's draws are looked at once, which gives the passes that a span meets
// and a list of the spans for them. Without it every pass loads every draw's record, also where none has a span:
// 300 polygons of up to 32 x 32 pixels in a 4096 x 4096 target 76.0 us a call, 38.1 so (54.9 with every span filled in
// draw order), in 16384 x 512 156.9, 49.7 (57.9). Rows of up to four passes go without (twelve targets of 640 x 640
// with 40 such polygons 38.9 us a call, 40.1 with the list).
template <bool WIDE>
__global__ __launch_bounds__(256) void k_depth_raster(DepthLaunch L)
{
	__shared__ RowSpan found[WIDE ? 4 : 1][WIDE ? DEPTH_FOUND : 1]; // a wave's: the spans of a wide row
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
	if(wave >= L.num_rows)
		return; // uniform over the wave; no barriers below
	// the row's target: the last one whose rows start at or before this one, 64 targets a step
	uint32_t ti = 0;
	for(uint32_t base = 0; base < L.num_targets; base += 64u)
	{
		const bool le = base + lane < L.num_targets && L.targets[base + lane].first_row <= wave;
		const uint32_t count = uint32_t(__popcll(__ballot(le)));
		if(count)
			ti = base + count - 1u;
		if(count < 64u)
			break;
	}
	const DepthTargetDev t = L.targets[ti];
	const int32_t y = int32_t(wave - t.first_row);
	const DepthRow* rows = L.rows + t.rec_base + uint64_t(uint32_t(y)) * t.num_draws;
	float* out = L.texels + t.offset + uint64_t(uint32_t(y)) * t.w;
	// the row's spans in draw order: those of all draws, or (listed) the ones found
	uint32_t n = t.num_draws;
	bool listed = false;
	auto load_span = [&](bool ok, uint32_t i) -> RowSpan {
		if(!ok)
			return RowSpan{0u, 0.0f, 0.0f, 0u};
		if(WIDE && listed)
			return found[threadIdx.x >> 6][i];
		// both records whole, and no condition between them: a second trip to memory otherwise
		const uint2 r = *reinterpret_cast<const uint2*>(rows + i); // not written outside the draw's rows: dropped here
		const uint4 info = *reinterpret_cast<const uint4*>(L.infos + t.first_draw + i);
		const bool has = (y >= int32_t(info.x)) & (y < int32_t(info.y)) & ((r.x & 0xFFFFu) < r.x >> 16);
		return RowSpan{has ? r.x : 0u, __builtin_bit_cast(float, r.y), __builtin_bit_cast(float, info.z), info.w};
	};
	const uint32_t margin = t.flags & SW_DEPTH_CIRCLE ? circle_margin(int32_t(t.w), y) : 0u;
	for(uint32_t base_x = 0; base_x < t.w; base_x += DEPTH_GROUP)
	{
		uint64_t passes = pass_bits(0u, t.w, base_x);
		if(WIDE && t.w > DEPTH_NARROW)
		{
			// only the passes that a span, or what lies outside the circle, meets; the spans are listed for them
			uint64_t met = pass_bits(0u, margin, base_x) | pass_bits(t.w - margin, t.w, base_x);
			uint32_t count = 0;
			for(uint32_t base = 0; base < n; base += 64u)
			{
				const RowSpan r = load_span(base + lane < n, base + lane);
				met |= pass_bits(r.span & 0xFFFFu, r.span >> 16, base_x);
				const uint64_t has = __ballot(r.span != 0u);
				const uint32_t at = count + uint32_t(__popcll(has & ((1ull << lane) - 1ull)));
				if(!listed && r.span != 0u && at < DEPTH_FOUND)
					found[threadIdx.x >> 6][at] = r;
				count += uint32_t(__popcll(has));
			}
			if(count <= DEPTH_FOUND)
			{
				__builtin_amdgcn_wave_barrier(); // the wave's own LDS operations take effect in order
				listed = true;
				n = count;
			}
#pragma unroll
			for(int off = 32; off > 0; off >>= 1)
				met |= __shfl_xor(met, off);
			passes &= uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int32_t(met)))) |
				(uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int32_t(met >> 32)))) << 32);
		}
		for(; passes; passes &= passes - 1u)
		{
			const uint32_t cx = base_x + uint32_t(__builtin_ctzll(passes)) * DEPTH_PASS;
			uint64_t open[DEPTH_SEGMENTS]; // pixels no overwriting draw has taken yet
			float z[DEPTH_SEGMENTS];
			uint32_t from[DEPTH_SEGMENTS]; // the place in draw order of the span that took the pixel, + 1
			uint64_t any_open = 0;
			bool tests = false;
#pragma unroll
			for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
			{
				open[s] = low_bits(int32_t(t.w) - int32_t(cx + 64u * s));
				any_open |= open[s];
				z[s] = 0.0f;
				from[s] = 0;
			}
			// backwards, 64 spans at a time: lane k holds span end - 1 - k
			for(uint32_t end = n; end > 0u && any_open; end = end > 64u ? end - 64u : 0u)
			{
				const RowSpan r = load_span(lane < end, end - 1u - lane);
				const bool meets = (r.span >> 16) > cx && (r.span & 0xFFFFu) < cx + DEPTH_PASS && r.span != 0u;
				tests = tests || __ballot(meets && r.depth_test != 0u) != 0;
				uint64_t hits = __ballot(meets && r.depth_test == 0u);
				// every lane's span as bits of the segments, so that a hit costs two readlanes, three scalar
				// operations and a select per segment
				uint32_t src[DEPTH_SEGMENTS], bits[DEPTH_SEGMENTS][2];
#pragma unroll
				for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
				{
					src[s] = 64u;
#pragma unroll
					for(uint32_t h = 0; h < 2; ++h)
						bits[s][h] = span_bits(int32_t(r.span & 0xFFFFu), int32_t(r.span >> 16), int32_t(cx + 64u * s + 32u * h));
				}
				while(hits && any_open)
				{
					const uint32_t k = uint32_t(__builtin_ctzll(hits));
					hits &= hits - 1u;
					any_open = 0;
#pragma unroll
					for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
					{
						const uint64_t take = open[s] & (uint64_t(uint32_t(rl(int32_t(bits[s][0]), k))) | (uint64_t(uint32_t(rl(int32_t(bits[s][1]), k))) << 32));
						open[s] ^= take;
						any_open |= open[s];
						src[s] = __builtin_amdgcn_inverse_ballot_w64(take) ? k : src[s];
					}
				}
				// the pixels taken in this chunk: their chain's end
#pragma unroll
				for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
				{
					if(__ballot(src[s] < 64u) == 0)
						continue;
					const uint32_t k = src[s] & 63u;
					const float start = lane_pull_f(r.inv_z, k), step = lane_pull_f(r.dx, k);
					const uint32_t x0 = uint32_t(lane_pull(int32_t(r.span), k)) & 0xFFFFu;
					if(src[s] < 64u)
					{
						z[s] = swchain::chain_add(start, step, cx + 64u * s + lane - x0);
						from[s] = end - k;
					}
				}
			}
			if(tests)
			{
				// depth-tested draws over the pixels' overwriting draw (or the buffer's value), in order
#pragma unroll
				for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
				{
					const uint32_t x = cx + 64u * s + lane;
					if(from[s] == 0 && x < t.w)
						z[s] = out[x];
				}
				for(uint32_t base = 0; base < n; base += 64u)
				{
					const RowSpan r = load_span(base + lane < n, base + lane);
					uint64_t hits = __ballot((r.span >> 16) > cx && (r.span & 0xFFFFu) < cx + DEPTH_PASS && r.span != 0u && r.depth_test != 0u);
					while(hits)
					{
						const uint32_t k = uint32_t(__builtin_ctzll(hits));
						hits &= hits - 1u;
						const uint32_t sp = uint32_t(rl(int32_t(r.span), k)), x0 = sp & 0xFFFFu, x1 = sp >> 16;
						const float start = __builtin_bit_cast(float, rl(__builtin_bit_cast(int, r.inv_z), k));
						const float step = __builtin_bit_cast(float, rl(__builtin_bit_cast(int, r.dx), k));
#pragma unroll
						for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
						{
							const uint32_t x = cx + 64u * s + lane;
							if(x >= x0 && x < x1 && base + k + 1u > from[s])
								z[s] = fmax_r(swchain::chain_add(start, step, x - x0), z[s]);
						}
					}
				}
			}
#pragma unroll
			for(uint32_t s = 0; s < DEPTH_SEGMENTS; ++s)
			{
				const uint32_t x = cx + 64u * s + lane;
				const bool outside = (t.flags & SW_DEPTH_CIRCLE) && (x < margin || x >= t.w - margin);
				// with depth tests every pixel is stored (one that no draw touched as it was)
				if(x < t.w && (outside || tests || !__builtin_amdgcn_inverse_ballot_w64(open[s])))
					out[x] = outside ? 1.0e24f : z[s];
			}
		}
	}
}

} // namespace

namespace swk
{
int depth_plan(const sw_depth_target* targets, uint32_t num_targets, const sw_depth_draw* draws, uint32_t num_draws,
	uint64_t num_vertex_ints, uint64_t num_texels, std::vector<char>& packed, DepthPlan& plan, std::string& error)
{
	std::vector<DepthTargetDev> tg(num_targets);
	std::vector<DepthDrawDev> dd(num_draws);
	uint64_t rec = 0;
	uint32_t rows = 0, next_draw = 0, max_width = 0;
	for(uint32_t i = 0; i < num_targets; ++i)
	{
		const sw_depth_target& t = targets[i];
		const std::string which = "depth target " + std::to_string(i) + ": ";
		if(t.width == 0 || t.height == 0 || t.width > 65535 || t.height > 65535)
			return (error = which + "size out of range"), -1;
		if(t.offset > num_texels || uint64_t(t.width) * t.height > num_texels - t.offset)
			return (error = which + "buffer outside the depth texels"), -1;
		if(t.first_draw != next_draw || uint64_t(t.first_draw) + t.num_draws > num_draws)
			return (error = which + "draw range not following the previous target's"), -1;
		next_draw = t.first_draw + t.num_draws;
		if(t.flags & ~SW_DEPTH_CIRCLE)
			return (error = which + "unknown flags"), -1;
		if((t.flags & SW_DEPTH_CIRCLE) && t.width != t.height)
			return (error = which + "the circle needs a square target"), -1;
		if(uint64_t(rows) + t.height > 0x7FFFFFFFu)
			return (error = "depth targets: too many rows"), -1;
		tg[i] = DepthTargetDev{t.offset, rec, t.width, t.height, t.first_draw, t.num_draws, rows, t.flags};
		rows += t.height;
		max_width = max_width > t.width ? max_width : t.width;
		rec += uint64_t(t.height) * t.num_draws;
		for(uint32_t k = t.first_draw; k < t.first_draw + t.num_draws; ++k)
		{
			const sw_depth_draw& s = draws[k];
			if(s.num_vertices < 3 || s.num_vertices > SW_MAX_POLYGON_VERTICES ||
				uint64_t(s.first_vertex_int) + 2ull * s.num_vertices > num_vertex_ints)
				return (error = "depth draw " + std::to_string(k) + ": vertices out of range"), -1;
			dd[k] = DepthDrawDev{s.first_vertex_int, s.num_vertices, s.depth_equation[0], s.depth_equation[1], s.depth_equation[2],
				s.depth_test ? 1u : 0u, i, 0};
		}
	}
	if(next_draw != num_draws)
		return (error = "depth draws not covered by the targets"), -1;
	plan.targets_at = (sizeof(DepthDrawDev) * dd.size() + 255) & ~size_t(255);
	plan.bytes = plan.targets_at + sizeof(DepthTargetDev) * tg.size();
	plan.row_records = rec;
	plan.rows = rows;
	plan.max_width = max_width;
	plan.num_draws = num_draws;
	plan.num_targets = num_targets;
	packed.assign(plan.bytes, 0);
	std::memcpy(packed.data(), dd.data(), sizeof(DepthDrawDev) * dd.size());
	std::memcpy(packed.data() + plan.targets_at, tg.data(), sizeof(DepthTargetDev) * tg.size());
	return 0;
}

size_t depth_row_record_bytes() { return sizeof(DepthRow); }
size_t depth_work_bytes(const DepthPlan& plan)
{
	return ((sizeof(DepthTargetDev) * plan.num_targets + 255) & ~size_t(255)) + sizeof(DepthDrawInfo) * plan.num_draws;
}

void launch_depth(hipStream_t st, const char* args, const int32_t* vdata, const DepthPlan& plan, char* work, void* rows, float* texels,
	bool raster)
{
	DepthLaunch L{reinterpret_cast<const DepthDrawDev*>(args), reinterpret_cast<const DepthTargetDev*>(args + plan.targets_at), vdata,
		reinterpret_cast<DepthTargetDev*>(work),
		reinterpret_cast<DepthDrawInfo*>(work + ((sizeof(DepthTargetDev) * plan.num_targets + 255) & ~size_t(255))),
		static_cast<DepthRow*>(rows), texels, plan.num_draws, plan.num_targets, plan.rows};
	if(plan.num_draws == 0 || plan.rows == 0)
		return;
	const uint32_t draw_blocks = (plan.num_draws + 3u) / 4u;
	const uint32_t copy_blocks = (plan.num_targets * uint32_t(sizeof(DepthTargetDev) / 4u) + 255u) / 256u;
	if(!raster)
		hipLaunchKernelGGL(k_depth_setup, dim3(draw_blocks + copy_blocks), dim3(256), 0, st, L, draw_blocks);
	else if(plan.max_width > DEPTH_NARROW)
		hipLaunchKernelGGL(k_depth_raster<true>, dim3((plan.rows + 3u) / 4u), dim3(256), 0, st, L);
	else
		hipLaunchKernelGGL(k_depth_raster<false>, dim3((plan.rows + 3u) / 4u), dim3(256), 0, st, L);
}
} // namespace swk
