// Per-frame texture animation on the map's resident textures (the map materials processor's
// generative effects): turbulence distortion (generative_texture_effect_turb.rs:89-138), texture
// layers (generative_texture_effect_layered.rs:162-381) and emissive layers (the layered effect's
// use of mix_surface_with_texture, surfaces.rs:854-971).
//
// One launch applies a list of operations. Consecutive operations with the same destination level
// form a run; every thread takes destination texels of one run and applies the run's operations to
// them in order (each operation reads only its source and the same destination texel, so doing
// them texel by texel gives the reference's level-by-level result).
#include <algorithm>
#include <bitset>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "sw_internal.h"
#include "sw_device.h"
#include "sw_divide.h"

using namespace swd;

namespace
{

#define TEXOP_BLOCK 256u
#define TEXOP_PER_THREAD 4u

struct TexLevel
{
	uint64_t offset;
	uint32_t w, h;
};

SW_DEV uint32_t wrap(int32_t v, uint32_t n)
{
	// rem_euclid for a positive divisor
	const int32_t r = v % int32_t(n);
	return uint32_t(r < 0 ? r + int32_t(n) : r);
}

// ColorVecI::from_color32(src) * light_vec >> 8 (light_vec = cvtps2dq(light * 256), alpha lane 0)
SW_DEV CI modulate(uint32_t c, const int32_t* lv)
{
	const CI t = Color32T::to_ci(c);
	return CI{wmul(t.b, lv[0]) >> 8, wmul(t.g, lv[1]) >> 8, wmul(t.r, lv[2]) >> 8, wmul(t.a, 0) >> 8};
}
SW_DEV CI ci_add2(CI a, CI b) { return CI{wadd(a.b, b.b), wadd(a.g, b.g), wadd(a.r, b.r), wadd(a.a, b.a)}; }
SW_DEV CI ci_shr2(CI a, int k) { return CI{a.b >> k, a.g >> k, a.r >> k, a.a >> k}; }
SW_DEV CI ci_blend(CI src, CI dst, int32_t alpha)
{
	const int32_t ia = 255 - alpha;
	return CI{wadd(wmul(src.b, alpha), wmul(dst.b, ia)) >> 8, wadd(wmul(src.g, alpha), wmul(dst.g, ia)) >> 8,
		wadd(wmul(src.r, alpha), wmul(dst.r, ia)) >> 8, wadd(wmul(src.a, alpha), wmul(dst.a, ia)) >> 8};
}

enum : uint32_t
{
	RUN_LITE = 1, // destination (and sources) are TextureLite levels
	RUN_OVERWRITES = 2, // the first operation leaves nothing of what the destination holds
};

struct TexOpRun
{
	uint32_t first_op, num_ops;
	uint32_t first_block;
	uint32_t flags;
	TexLevel dst;
};

enum : uint32_t
{
	OP_TURB = 1,
	OP_MODULATE = 2, // layers: a light component outside [0.98, 1.02] (impl_1, :231-242)
	OP_OVERFLOWS = 4, // layers: shift + row can overflow (and the height is no power of two), which the rem_euclid sees
	OP_BLEND_SHIFT = 8,
};

struct DevTexOp
{
	uint32_t flags;
	uint32_t turb_shifts; // TURB: first shift of the level
	uint32_t add[2]; // layers: the source texel is (destination + add) mod size
	int32_t shift_v;
	int32_t light_vec[3]; // lanes B, G, R
	TexLevel src;
};

struct TexOpLaunch
{
	const TexOpRun* runs;
	uint32_t num_runs;
	const DevTexOp* ops;
	const int32_t* turb_shifts;
	sw_texel* texels;
	uint32_t* lite;
};

// apply_texture_layer_impl_2 (generative_texture_effect_layered.rs:255-381), one texel
SW_DEV sw_texel layer_texel(const DevTexOp& op, sw_texel dst, sw_texel src)
{
	if(op.flags & OP_MODULATE)
	{
		const CI m = modulate(src.diffuse, op.light_vec);
		switch(op.flags >> OP_BLEND_SHIFT)
		{
		case SW_BLEND_NONE: return sw_texel{Color32T::from_ci(m), src.packed_normal_roughness};
		case SW_BLEND_AVERAGE:
			dst.diffuse = Color32T::from_ci(ci_shr2(ci_add2(m, Color32T::to_ci(dst.diffuse)), 1));
			return dst;
		case SW_BLEND_ADDITIVE: dst.diffuse = Color32T::from_ci(ci_add2(m, Color32T::to_ci(dst.diffuse))); return dst;
		case SW_BLEND_ALPHA_TEST: return Color32T::test_alpha(src.diffuse) ? sw_texel{Color32T::from_ci(m), src.packed_normal_roughness} : dst;
		case SW_BLEND_ALPHA_BLEND:
			dst.diffuse = Color32T::from_ci(ci_blend(m, Color32T::to_ci(dst.diffuse), Color32T::get_alpha(src.diffuse)));
			return dst;
		default: return dst;
		}
	}
	switch(op.flags >> OP_BLEND_SHIFT)
	{
	case SW_BLEND_NONE: return src;
	case SW_BLEND_AVERAGE: dst.diffuse = Color32T::average(dst.diffuse, src.diffuse); return dst;
	case SW_BLEND_ADDITIVE:
		dst.diffuse = Color32T::from_ci(ci_add2(Color32T::to_ci(src.diffuse), Color32T::to_ci(dst.diffuse)));
		return dst;
	case SW_BLEND_ALPHA_TEST: return Color32T::test_alpha(src.diffuse) ? src : dst;
	case SW_BLEND_ALPHA_BLEND:
		dst.diffuse =
			Color32T::from_ci(ci_blend(Color32T::to_ci(src.diffuse), Color32T::to_ci(dst.diffuse), Color32T::get_alpha(src.diffuse)));
		return dst;
	default: return dst;
	}
}

// mix_surface_with_texture_impl (surfaces.rs:903-971) on a Color32 destination, one texel
SW_DEV uint32_t lite_layer_texel(const DevTexOp& op, uint32_t dst, uint32_t src)
{
	const CI m = modulate(src, op.light_vec);
	switch(op.flags >> OP_BLEND_SHIFT)
	{
	case SW_BLEND_NONE: return Color32T::from_ci(m);
	case SW_BLEND_AVERAGE: return Color32T::from_ci(ci_shr2(ci_add2(m, Color32T::to_ci(dst)), 1));
	case SW_BLEND_ADDITIVE: return Color32T::from_ci(ci_add2(m, Color32T::to_ci(dst)));
	case SW_BLEND_ALPHA_TEST: return Color32T::test_alpha(src) ? Color32T::from_ci(m) : dst;
	case SW_BLEND_ALPHA_BLEND: return Color32T::from_ci(ci_blend(m, Color32T::to_ci(dst), Color32T::get_alpha(src)));
	default: return dst;
	}
}

SW_DEV sw_texel blend_layer(const DevTexOp& op, sw_texel dst, sw_texel src) { return layer_texel(op, dst, src); }
SW_DEV uint32_t blend_layer(const DevTexOp& op, uint32_t dst, uint32_t src) { return lite_layer_texel(op, dst, src); }

// (destination + add) mod size for the texels of a thread; one division for all where size is no power of two.
template <uint32_t N>
SW_DEV void wrap_all(const uint32_t (&at)[N], uint32_t add, uint32_t size, uint32_t (&out)[N])
{
	if((size & (size - 1)) == 0)
	{
#pragma unroll
		for(uint32_t k = 0; k < N; ++k)
			out[k] = (at[k] + add) & (size - 1);
	}
	else
	{
		const double inv = 1.0 / double(size);
#pragma unroll
		for(uint32_t k = 0; k < N; ++k)
			out[k] = swdiv::mod_rcp(at[k] + add, size, swdiv::NO_MASK, inv);
	}
}

// The operation's source texels of a thread's destination texels.
template <class T, uint32_t N>
SW_DEV void load_sources(const TexOpLaunch& L, const TexOpRun& run, const DevTexOp& op, const T* texels, const uint32_t (&x)[N],
	const uint32_t (&y)[N], T (&out)[N])
{
	uint32_t su[N], sv[N];
	if(op.flags & OP_TURB)
	{
		// make_turb_distortion (generative_texture_effect_turb.rs:89-138): the source texel at
		// (x + shift[y], y + shift[x]), wrapped by the power-of-two masks
		const int32_t* shifts = L.turb_shifts + op.turb_shifts;
#pragma unroll
		for(uint32_t k = 0; k < N; ++k)
		{
			su[k] = (x[k] + uint32_t(shifts[y[k]])) & (op.src.w - 1);
			sv[k] = (y[k] + uint32_t(shifts[x[k]])) & (op.src.h - 1);
		}
	}
	else
	{
		// u steps from rem_euclid(shift) with a wrap at the width, v is the rem_euclid of each row's sum
		wrap_all(x, op.add[0], op.src.w, su);
		if(op.flags & OP_OVERFLOWS)
#pragma unroll
			for(uint32_t k = 0; k < N; ++k)
				sv[k] = wrap(op.shift_v + int32_t(y[k]), op.src.h);
		else
			wrap_all(y, op.add[1], op.src.h, sv);
	}
	const T* src = texels + op.src.offset;
#pragma unroll
	for(uint32_t k = 0; k < N; ++k)
		out[k] = src[uint64_t(sv[k]) * op.src.w + su[k]];
}

// A block's texels of a run: all operations in turn on TEXOP_PER_THREAD texels of a thread together; an
// operation's sources are requested before the previous one is blended.
template <class T>
SW_DEV void texture_run(const TexOpLaunch& L, const TexOpRun& run, T* texels)
{
	constexpr uint32_t N = TEXOP_PER_THREAD;
	const uint32_t w = run.dst.w, h = run.dst.h;
	const uint64_t n = uint64_t(w) * h;
	const uint64_t base = uint64_t(blockIdx.x - run.first_block) * (TEXOP_BLOCK * N) + threadIdx.x;
	T* dst = texels + run.dst.offset;
	uint32_t at[N], x[N], y[N]; // threads past the end work on the last texel and store nothing
	const bool pow2 = (w & (w - 1)) == 0;
	const double inv_w = pow2 ? 0.0 : 1.0 / double(w);
#pragma unroll
	for(uint32_t k = 0; k < N; ++k)
	{
		at[k] = uint32_t(std::min<uint64_t>(base + k * TEXOP_BLOCK, n - 1)); // n <= 2^32
		if(pow2)
		{
			x[k] = at[k] & (w - 1);
			y[k] = at[k] >> __builtin_ctz(w);
		}
		else
			y[k] = swdiv::div_rcp(at[k], w, inv_w, x[k]);
	}
	T v[N], s[N];
	const DevTexOp* ops = L.ops + run.first_op;
	DevTexOp op = ops[0];
	load_sources(L, run, op, texels, x, y, s);
	if(!(run.flags & RUN_OVERWRITES))
#pragma unroll
		for(uint32_t k = 0; k < N; ++k)
			v[k] = dst[at[k]];
#pragma unroll 1
	for(uint32_t o = 0; o < run.num_ops; ++o)
	{
		const DevTexOp next = ops[std::min(o + 1, run.num_ops - 1)];
		T next_s[N];
		if(o + 1 < run.num_ops)
			load_sources(L, run, next, texels, x, y, next_s);
#pragma unroll
		for(uint32_t k = 0; k < N; ++k)
		{
			v[k] = op.flags & OP_TURB ? s[k] : blend_layer(op, v[k], s[k]);
			s[k] = next_s[k];
		}
		op = next;
	}
#pragma unroll
	for(uint32_t k = 0; k < N; ++k)
		if(base + k * TEXOP_BLOCK < n)
			dst[at[k]] = v[k];
}

// Bound by latency: a few hundred blocks, each a chain of run, operation and texel loads. 8 textures of
// 256 x 256 texels and their mips, 80 operations: 15.3 us with a binary search for the run and a texel after
// another, its row and wrapped coordinates by integer division; now 8.4 (an
// argument record of 40 bytes rather than 96: the arguments of a call then stay below the 16 KiB from which a copy
// costs 10 us more).
__global__ __launch_bounds__(TEXOP_BLOCK) void k_texture_ops(TexOpLaunch L)
{
	// the block's run: the last run starting at or before this block, a probe per lane and level
	const uint32_t lane = threadIdx.x & 63;
	uint32_t lo = 0;
	for(uint32_t n = L.num_runs; n > 1;)
	{
		const uint32_t step = (n + 63u) / 64u, probe = lo + lane * step;
		const uint64_t le = __ballot(lane * step < n && L.runs[probe].first_block <= blockIdx.x);
		const uint32_t last = 63u - uint32_t(__builtin_clzll(le)); // lane 0's run starts at or before the block
		lo += last * step;
		n = std::min(step, n - last * step);
	}
	const TexOpRun& run = L.runs[lo];
	if(run.flags & RUN_LITE)
		texture_run(L, run, L.lite);
	else
		texture_run(L, run, L.texels);
}

// make_skybox_side_texture / make_skybox_side_texture64 (textures.rs:183-229): the top-left
// size x size pixels of the image, (c * trunc(brightness * 256)) >> 8 per lane with the alpha lane
// multiplied by 0, packed with unsigned saturation.
template <class CT>
__global__ __launch_bounds__(256) void k_skybox_mip0(
	const typename CT::T* __restrict__ image, uint32_t image_w, uint32_t size, int32_t brightness, typename CT::T* __restrict__ dst)
{
	const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
	if(x >= size)
		return;
	const CI c = CT::to_ci(image[uint64_t(y) * image_w + x]);
	dst[uint64_t(y) * size + x] =
		CT::from_ci(CI{wmul(c.b, brightness) >> 8, wmul(c.g, brightness) >> 8, wmul(c.r, brightness) >> 8, wmul(c.a, 0) >> 8});
}

// make_skybox_side_texture_mips (textures.rs:231-286): (p00 + p01 + p10 + p11) >> 2 per lane
template <class CT>
__global__ __launch_bounds__(256) void k_skybox_mip(
	const typename CT::T* __restrict__ prev, uint32_t ps, uint32_t size, typename CT::T* __restrict__ dst)
{
	// prev: the previous level, ps x ps (ps = 2 size or 2 size + 1)
	const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
	if(x >= size)
		return;
	const CI p00 = CT::to_ci(prev[uint64_t(2 * y) * ps + 2 * x]), p01 = CT::to_ci(prev[uint64_t(2 * y + 1) * ps + 2 * x]);
	const CI p10 = CT::to_ci(prev[uint64_t(2 * y) * ps + 2 * x + 1]), p11 = CT::to_ci(prev[uint64_t(2 * y + 1) * ps + 2 * x + 1]);
	dst[uint64_t(y) * size + x] = CT::from_ci(ci_shr2(ci_add2(ci_add2(p00, p01), ci_add2(p10, p11)), 2));
}

} // namespace

namespace swk
{
// A skybox side and its mips (size, size/2, ... down to 1, at most five levels) back to back at dst.
void launch_skybox_side(hipStream_t st, uint32_t color_bits, const void* image, uint32_t image_w, uint32_t size, int32_t brightness,
	void* dst)
{
	if(color_bits == 64)
	{
		uint64_t* d = static_cast<uint64_t*>(dst);
		hipLaunchKernelGGL(k_skybox_mip0<Color64T>, dim3((size + 255) / 256, size), dim3(256), 0, st, static_cast<const uint64_t*>(image),
			image_w, size, brightness, d);
		for(uint32_t mip = 1, s = size; mip < 5 && (s >> 1); ++mip, d += uint64_t(s) * s, s >>= 1)
			hipLaunchKernelGGL(k_skybox_mip<Color64T>, dim3(((s >> 1) + 255) / 256, s >> 1), dim3(256), 0, st, d, s, s >> 1, d + uint64_t(s) * s);
	}
	else
	{
		uint32_t* d = static_cast<uint32_t*>(dst);
		hipLaunchKernelGGL(k_skybox_mip0<Color32T>, dim3((size + 255) / 256, size), dim3(256), 0, st, static_cast<const uint32_t*>(image),
			image_w, size, brightness, d);
		for(uint32_t mip = 1, s = size; mip < 5 && (s >> 1); ++mip, d += uint64_t(s) * s, s >>= 1)
			hipLaunchKernelGGL(k_skybox_mip<Color32T>, dim3(((s >> 1) + 255) / 256, s >> 1), dim3(256), 0, st, d, s, s >> 1, d + uint64_t(s) * s);
	}
}

// Validates the operations against the map's level table and packs the launch arguments (runs,
// then operations at `ops_at`) into `packed`.
int pack_texture_ops(const sw_texture_op* ops, uint32_t num_ops, const sw_texture_level* levels, uint32_t num_levels,
	uint32_t num_turb_shifts, std::vector<char>& packed, TexOpPlan& plan, std::string& error)
{
	std::vector<TexOpRun> runs;
	std::vector<DevTexOp> dops(num_ops);
	std::vector<uint8_t> is_dst(num_levels, 0); // levels that a run writes
	uint32_t blocks = 0;
	for(uint32_t i = 0; i < num_ops; ++i)
	{
		const sw_texture_op& op = ops[i];
		auto fail = [&](const char* what) { return (error = "texture op " + std::to_string(i) + ": " + what), -1; };
		if(op.kind > SW_TEXOP_LAYER_LITE)
			return fail("unknown kind");
		if(op.dst_level >= num_levels || op.src_level >= num_levels)
			return fail("level out of range");
		const sw_texture_level& dl = levels[op.dst_level];
		const sw_texture_level& sl = levels[op.src_level];
		const bool dlite = (dl.flags & SW_TEX_LITE_LEVEL) != 0, slite = (sl.flags & SW_TEX_LITE_LEVEL) != 0;
		if(dlite != slite || (op.kind == SW_TEXOP_LAYER && dlite) || (op.kind == SW_TEXOP_LAYER_LITE && !dlite))
			return fail("level kinds do not fit the operation");
		if(op.dst_level == op.src_level)
			return fail("source and destination are the same level");
		if(op.kind == SW_TEXOP_TURB)
		{
			if(sl.width != dl.width || sl.height != dl.height || (dl.width & (dl.width - 1)) || (dl.height & (dl.height - 1)))
				return fail("turbulence needs equal power-of-two sizes");
			if(uint64_t(op.turb_shifts) + std::max(dl.width, dl.height) > num_turb_shifts)
				return fail("turbulence shifts out of range");
		}
		else if(op.blend > SW_BLEND_ALPHA_BLEND)
			return fail("unknown blending mode");
		DevTexOp& d = dops[i];
		d.flags = op.kind == SW_TEXOP_TURB ? OP_TURB : op.blend << OP_BLEND_SHIFT;
		for(int c = 0; c < 3; ++c)
			d.flags |= (op.light[c] < 0.98f || op.light[c] > 1.02f) ? OP_MODULATE : 0u;
		d.turb_shifts = op.turb_shifts;
		d.shift_v = op.shift[1];
		// ColorVecI::from_color_f32x3(light * 256): cvtps2dq (round half even, "integer indefinite"
		// out of range), lanes B, G, R
		for(int c = 0; c < 3; ++c)
		{
			const float v = op.light[2 - c] * 256.0f;
			d.light_vec[c] = (v >= -2147483648.0f && v < 2147483648.0f) ? int32_t(std::nearbyint(v)) : INT32_MIN;
		}
		d.src = TexLevel{sl.offset, sl.width, sl.height};
		const uint32_t src_size[2] = {sl.width, sl.height};
		for(int c = 0; c < 2; ++c)
		{
			const int64_t size = src_size[c];
			const bool pow2 = (size & (size - 1)) == 0;
			d.add[c] = pow2 ? uint32_t(op.shift[c]) : uint32_t((op.shift[c] % size + size) % size);
			if(c == 1 && !pow2 && int64_t(op.shift[1]) + dl.height > INT32_MAX)
				d.flags |= OP_OVERFLOWS;
		}
		if(runs.empty() || ops[runs.back().first_op].dst_level != op.dst_level)
		{
			if(is_dst[op.dst_level])
				return fail("a destination's operations must be consecutive");
			is_dst[op.dst_level] = 1;
			TexOpRun r{};
			r.first_op = i;
			r.num_ops = 0;
			r.first_block = blocks;
			r.dst = TexLevel{dl.offset, dl.width, dl.height};
			// SW_BLEND_NONE: as layer_texel and lite_layer_texel do
			r.flags = (dlite ? RUN_LITE : 0u) | (op.kind == SW_TEXOP_TURB || op.blend == SW_BLEND_NONE ? RUN_OVERWRITES : 0u);
			const uint64_t nb = (uint64_t(dl.width) * dl.height + TEXOP_BLOCK * TEXOP_PER_THREAD - 1) / (TEXOP_BLOCK * TEXOP_PER_THREAD);
			if(blocks + nb > 0x7FFFFFFFull)
				return (error = "texture ops: too many texels"), -1;
			blocks += uint32_t(nb);
			runs.push_back(r);
		}
		runs.back().num_ops++;
	}
	for(uint32_t i = 0; i < num_ops; ++i)
		if(is_dst[ops[i].src_level])
			return (error = "texture op " + std::to_string(i) + ": its source is the destination of another operation"), -1;
	const size_t runs_bytes = sizeof(TexOpRun) * runs.size();
	plan.ops_at = (runs_bytes + 255) & ~size_t(255);
	plan.bytes = plan.ops_at + sizeof(DevTexOp) * dops.size();
	plan.blocks = blocks;
	plan.num_runs = uint32_t(runs.size());
	packed.assign(plan.bytes, 0);
	std::memcpy(packed.data(), runs.data(), runs_bytes);
	std::memcpy(packed.data() + plan.ops_at, dops.data(), sizeof(DevTexOp) * dops.size());
	return 0;
}

void launch_texture_ops(hipStream_t st, const char* args_dev, const TexOpPlan& plan, const int32_t* turb_shifts_dev, sw_texel* texels,
	uint32_t* lite)
{
	if(plan.blocks == 0)
		return;
	TexOpLaunch L{reinterpret_cast<const TexOpRun*>(args_dev), plan.num_runs, reinterpret_cast<const DevTexOp*>(args_dev + plan.ops_at),
		turb_shifts_dev, texels, lite};
	hipLaunchKernelGGL(k_texture_ops, dim3(plan.blocks), dim3(TEXOP_BLOCK), 0, st, L);
}
} // namespace swk

namespace
{

// ---------------------------------------------------------------------------------------------
// Water (generative_texture_effect_water.rs)
// ---------------------------------------------------------------------------------------------
// add_point_value (:68-76) for more points than a step's kernel arguments hold, 64 at a time: the first
// point of each address in a batch adds the batch's values for that address in order (points at one address add up in the
// reference's order; distinct addresses go in parallel); batches follow each other.
__global__ __launch_bounds__(64) void k_water_points(float* field, float* field_old, const sw_wave_point* pts, uint32_t n,
	uint32_t log2w, uint32_t log2h)
{
	__shared__ uint32_t sa[64];
	__shared__ float sv[64];
	const uint32_t lane = threadIdx.x;
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	for(uint32_t base = 0; base < n; base += 64)
	{
		const uint32_t cnt = n - base < 64u ? n - base : 64u;
		uint32_t a = 0;
		if(lane < cnt)
		{
			const sw_wave_point p = pts[base + lane];
			a = (p.x & mx) + ((p.y & my) << log2w);
			sa[lane] = a;
			sv[lane] = p.value;
		}
		__syncthreads();
		if(lane < cnt)
		{
			bool first = true;
			for(uint32_t k = 0; k < lane; ++k)
				first = first && sa[k] != a;
			if(first)
			{
				float f = field[a], fo = field_old[a];
				for(uint32_t k = lane; k < cnt; ++k)
					if(sa[k] == a)
					{
						f += sv[k];
						fo -= sv[k];
					}
				field[a] = f;
				field_old[a] = fo;
			}
		}
		__syncthreads();
	}
}

// The end of the run of equal addresses that starts at k, of n ascending ones: known ahead, so that the loads of the
// run's values do not wait for each comparison (two queued steps of 256 points at one address 87.6 us, now 17.9).
SW_DEV uint32_t same_address_end(const uint32_t* address, uint32_t k, uint32_t n)
{
	const uint32_t a = address[k];
	uint32_t lo = k + 1u, hi = lo < n && address[lo] == a ? n : lo; // mostly a point alone
	while(lo < hi)
	{
		const uint32_t mid = (lo + hi) / 2u;
		if(address[mid] == a)
			lo = mid + 1u;
		else
			hi = mid;
	}
	return lo;
}

// Four consecutive elements of a thread and what the stencil reads for them.
struct WaterQuad
{
	uint32_t block, i, il, ir; // the block's place in the field; the first element, the neighbours left and right of the four
	bool in;
	float c[6], u[4], d[4], o[4]; // the row from il to ir, the elements above and below, the old field
};

// The thread's four elements, read. VEC: both buffers are 16-byte aligned.
// Blocks are dealt to the eight XCDs in turn: each takes a contiguous eighth of the field, so that a row's
// neighbours above and below come from the same L2 (four queued steps of 1024 x 1024 without points: 23.8 us
// with consecutive blocks on different XCDs, 16.9 so). The number of blocks comes from the size: read as gridDim it
// would have the runtime fill in the kernel's hidden arguments for every launch.
template <bool VEC>
SW_DEV WaterQuad water_load(const float* src, const float* old, uint32_t log2w, uint32_t log2h)
{
	WaterQuad q;
	const uint32_t each = (1u << (log2w + log2h)) / (8u * swk::WATER_BLOCK); // blocks of an XCD
	q.block = each ? blockIdx.x % 8u * each + blockIdx.x / 8u : blockIdx.x;
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	q.i = q.block * swk::WATER_BLOCK + threadIdx.x * 4u;
	q.in = (q.i >> (log2w + log2h)) == 0;
	const uint32_t x = q.i & mx, y = q.i >> log2w;
	const uint32_t row = y << log2w, up = (((y - 1u) & my) << log2w) + x, down = (((y + 1u) & my) << log2w) + x;
	q.il = row + ((x - 1u) & mx);
	q.ir = row + ((x + 4u) & mx);
	if(q.in)
	{
		q.c[0] = src[q.il];
		q.c[5] = src[q.ir];
		if(VEC)
		{
			const float4 c4 = *reinterpret_cast<const float4*>(src + q.i), u4 = *reinterpret_cast<const float4*>(src + up),
						 d4 = *reinterpret_cast<const float4*>(src + down), o4 = *reinterpret_cast<const float4*>(old + q.i);
			q.c[1] = c4.x, q.c[2] = c4.y, q.c[3] = c4.z, q.c[4] = c4.w;
			q.u[0] = u4.x, q.u[1] = u4.y, q.u[2] = u4.z, q.u[3] = u4.w;
			q.d[0] = d4.x, q.d[1] = d4.y, q.d[2] = d4.z, q.d[3] = d4.w;
			q.o[0] = o4.x, q.o[1] = o4.y, q.o[2] = o4.z, q.o[3] = o4.w;
		}
		else
#pragma unroll
			for(uint32_t k = 0; k < 4; ++k)
			{
				q.c[k + 1] = src[q.i + k];
				q.u[k] = src[up + k];
				q.d[k] = src[down + k];
				q.o[k] = old[q.i + k];
			}
	}
	return q;
}

// update_wave_field (:307-418) of the thread's elements
template <bool VEC>
SW_DEV void water_store(const WaterQuad& q, float* dst, float attenuation)
{
	if(!q.in)
		return;
	float r[4];
#pragma unroll
	for(uint32_t k = 0; k < 4; ++k)
	{
		const float sum = ((q.c[k] + q.c[k + 2]) + q.u[k]) + q.d[k];
		r[k] = (sum * 0.5f - q.o[k]) * attenuation;
	}
	if(VEC)
		*reinterpret_cast<float4*>(dst + q.i) = make_float4(r[0], r[1], r[2], r[3]);
	else
#pragma unroll
		for(uint32_t k = 0; k < 4; ++k)
			dst[q.i + k] = r[k];
}

// A step without points: the field is a torus (rows and columns wrap). Its own kernel, with no more arguments than it
// needs: queued steps of a field up to 256 x 256 are bound by the host's launches, and those by the bytes of arguments
// (4.2 us a step with the points' arguments or, without them, with gridDim's, 3.7 so).
template <bool VEC>
__global__ __launch_bounds__(256) void k_water_step(float* __restrict__ dst, const float* __restrict__ src, uint32_t log2w, uint32_t log2h,
	float attenuation)
{
	const WaterQuad q = water_load<VEC>(src, dst, log2w, log2h);
	water_store<VEC>(q, dst, attenuation);
}

// A step with its points (add_point_value, :68-76), which travel in the kernel's arguments. The stencil reads the
// field with the points added: a block that points touch passes its values through LDS, where a thread per address adds that address's points in their order (the
// reference's) wherever the value is held and subtracts them from the old field (every thread comparing each
// point's address with those of the 18 values it held took 0.2 us a point: two queued steps of 32 x 32 with 200
// points 82.8 us, 67 with the points in a kernel ahead of the step, now 12.9). The field itself is updated
// by the last of the blocks that read any point's element (they take tickets; nobody waits), when all of
// them have read it. One launch per step, no copy ahead of it. A 1024 x 1024 step with 16 points takes 5.7 us
// (2.9 us of copy, 4.3 us of points and 5.3 us of stencil as three operations); its 12.6 MB take 2.6 us at
// the rate of a large copy.
template <uint32_t N, bool VEC>
__global__ __launch_bounds__(256) void k_water_step_points(float* __restrict__ dst, float* __restrict__ src, uint32_t log2w, uint32_t log2h,
	float attenuation, swk::WavePoints<N> pts, uint32_t readers, uint32_t* __restrict__ ticket)
{
	// the block's values by element (its own, their neighbours above and below, the old field, the
	// neighbours left and right of its ends), and whether points touch them
	__shared__ __align__(16) float l_own[swk::WATER_BLOCK], l_up[swk::WATER_BLOCK], l_down[swk::WATER_BLOCK], l_old[swk::WATER_BLOCK],
		l_ends[2], l_value[N];
	__shared__ uint32_t l_address[N], touched, reads, last;
	WaterQuad q = water_load<VEC>(src, dst, log2w, log2h);
	if(threadIdx.x == 0)
		touched = reads = 0;
	__syncthreads();
	// thread k's point: its address, whether it is the first of its address, and the elements that it is read by
	static_assert(N <= 256u);
	const uint32_t k = threadIdx.x, b0 = q.block * swk::WATER_BLOCK;
	const bool has = k < pts.n;
	const uint32_t a = pts.address[has ? k : 0u], before = pts.address[has && k > 0u ? k - 1u : 0u];
	const float v0 = pts.value[has ? k : 0u];
	const bool first = has && (k == 0u || before != a);
	if(has)
	{
		l_address[k] = a;
		l_value[k] = v0;
	}
	uint32_t at[4]; // of the block: its right, left, lower and upper neighbour, whose left, ... neighbour it is
	bool read = false;
#pragma unroll
	for(uint32_t n = 0; n < 4; ++n)
	{
		at[n] = swk::water_neighbour(a, n ^ 1u, log2w, log2h) - b0;
		read = read || at[n] < swk::WATER_BLOCK;
	}
	const uint32_t own = a - b0;
	if(has && read)
		reads = 1; // every writer writes 1
	if(has && (read || own < swk::WATER_BLOCK))
		touched = 1;
	__syncthreads();
	if(touched)
	{
		// uniform over the block: the values go through LDS, where a thread per address adds its points in turn
		const uint32_t t4 = threadIdx.x * 4u;
		*reinterpret_cast<float4*>(l_own + t4) = make_float4(q.c[1], q.c[2], q.c[3], q.c[4]);
		*reinterpret_cast<float4*>(l_up + t4) = make_float4(q.u[0], q.u[1], q.u[2], q.u[3]);
		*reinterpret_cast<float4*>(l_down + t4) = make_float4(q.d[0], q.d[1], q.d[2], q.d[3]);
		*reinterpret_cast<float4*>(l_old + t4) = make_float4(q.o[0], q.o[1], q.o[2], q.o[3]);
		// the neighbour left of an element of the block is its predecessor, or lies at its row's other end: in the
		// block if it holds whole rows, else only the first thread's is outside (right alike)
		const bool left_in = q.il - b0 < swk::WATER_BLOCK, right_in = q.ir - b0 < swk::WATER_BLOCK;
		if(!left_in)
			l_ends[0] = q.c[0];
		if(!right_in)
			l_ends[1] = q.c[5];
		__syncthreads();
		if(first && (read || own < swk::WATER_BLOCK))
		{
			// whatever place holds the element's value, all of them hold the same
			const bool is_own = own < swk::WATER_BLOCK, is_left = !is_own && at[0] < swk::WATER_BLOCK,
					   is_right = !is_own && at[1] < swk::WATER_BLOCK, is_up = at[2] < swk::WATER_BLOCK, is_down = at[3] < swk::WATER_BLOCK;
			float f = is_own ? l_own[own] : is_left ? l_ends[0] : is_right ? l_ends[1] : is_up ? l_up[at[2]] : l_down[at[3]];
			float old = is_own ? l_old[own] : 0.0f;
			const uint32_t end = same_address_end(l_address, k, pts.n);
#pragma unroll 8
			for(uint32_t j = k; j < end; ++j)
			{
				f += l_value[j];
				old -= l_value[j];
			}
			if(is_own)
			{
				l_own[own] = f;
				l_old[own] = old;
			}
			if(is_left)
				l_ends[0] = f;
			if(is_right)
				l_ends[1] = f;
			if(is_up)
				l_up[at[2]] = f;
			if(is_down)
				l_down[at[3]] = f;
		}
		__syncthreads();
		const float4 c4 = *reinterpret_cast<const float4*>(l_own + t4), u4 = *reinterpret_cast<const float4*>(l_up + t4),
					 d4 = *reinterpret_cast<const float4*>(l_down + t4), o4 = *reinterpret_cast<const float4*>(l_old + t4);
		q.c[0] = left_in ? l_own[q.il - b0] : l_ends[0];
		q.c[1] = c4.x, q.c[2] = c4.y, q.c[3] = c4.z, q.c[4] = c4.w;
		q.c[5] = right_in ? l_own[q.ir - b0] : l_ends[1];
		q.u[0] = u4.x, q.u[1] = u4.y, q.u[2] = u4.z, q.u[3] = u4.w;
		q.d[0] = d4.x, q.d[1] = d4.y, q.d[2] = d4.z, q.d[3] = d4.w;
		q.o[0] = o4.x, q.o[1] = o4.y, q.o[2] = o4.z, q.o[3] = o4.w;
	}
	water_store<VEC>(q, dst, attenuation);
	if(!reads)
		return; // uniform over the block
	// Every element of the field that this block reads has been read: the sums made of them were stored
	// before the barrier. That is the condition the ticket stands on, and it is the hardware's order, not the
	// memory model's: a block must read nothing of the field after its barrier (no prefetch, no load that a
	// later change moves behind it), for the last reader may be writing it then. Nothing else has to be ordered
	// (the field is only read until the last reader writes it), so the ticket is relaxed: a fence here would
	// write back the L2's dirty lines, most of the new field, once per reading block (the step took 10.7 us
	// with fences).
	__syncthreads();
	if(threadIdx.x == 0)
		last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == readers - 1u ? 1u : 0u;
	__syncthreads();
	if(!last)
		return;
	// the last reader: an address's points lie together, its first point's thread adds them up in order
	if(k < pts.n && (k == 0u || l_address[k - 1u] != l_address[k]))
	{
		const uint32_t a = l_address[k];
		const uint32_t end = same_address_end(l_address, k, pts.n);
		float f = src[a];
#pragma unroll 8
		for(uint32_t j = k; j < end; ++j)
			f += l_value[j];
		src[a] = f;
	}
	if(threadIdx.x == 0)
		*ticket = 0;
}

// PackedNormalRoughness::pack (textures.rs:33-39, fast_math.rs:64-78): x 127 per lane, cvtps2dq,
// signed saturation to bytes. A value here is at most 127 in magnitude up to rounding, or NaN (a normal's
// lane, a roughness), never above 2^31, so the saturation can go first: NaN becomes -128, as cvtps2dq's
// "integer indefinite" does, and adding 1.5 * 2^23 rounds to the nearest even integer in the low bits.
SW_DEV uint32_t pack_lane(float v)
{
	return __float_as_uint(__builtin_fminf(__builtin_fmaxf(v * 127.0f, -128.0f), 127.0f) + 12582912.0f) & 0xFFu;
}
SW_DEV int32_t pack_normal_roughness_dev(float x, float y, float z, float r)
{
	return int32_t(pack_lane(x) | (pack_lane(y) << 8) | (pack_lane(z) << 16) | (pack_lane(r) << 24));
}

// make_wavy_texture_impl (:497-682) per texel: the normal from the field's central differences dx, dy,
// normalised as cgmath's normalize (v * (1 / |v|)), colours by mode
SW_DEV sw_texel water_texel(float dx, float dy, uint32_t log2w, uint32_t log2h, const swk::WaterTexLaunch& w, const sw_texel* texels,
	uint32_t x, uint32_t y)
{
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	const uint32_t row = y << log2w, i = x + row;
	const float m2 = (dx * dx + dy * dy) + 1.0f;
	const float s = 1.0f / __builtin_sqrtf(m2);
	const float nx = dx * s, ny = dy * s, nz = s;
	const sw_texel* color = texels + w.color_offset;
	uint32_t diffuse;
	if(w.color_mode == SW_WATER_COLOR_KEEP)
		diffuse = w.init == SW_WATER_INIT_BASE_COLOR ? w.base_color
			: w.init == SW_WATER_INIT_SOURCE      ? color[i].diffuse
												  : texels[w.dst_offset[0] + i].diffuse;
	else
	{
		const int32_t du = int32_t(nx * 16.0f);
		const uint32_t u = (x + uint32_t(du)) & mx;
		if(w.color_mode == SW_WATER_COLOR_DEFORMED)
		{
			const int32_t dv = int32_t(ny * 16.0f);
			const uint32_t v = (y + uint32_t(dv)) & my;
			diffuse = color[u + (v << log2w)].diffuse;
		}
		else
			diffuse = color[u + row].diffuse;
	}
	sw_texel t;
	t.diffuse = diffuse;
	t.packed_normal_roughness = pack_normal_roughness_dev(nx, ny, nz, w.roughness);
	return t;
}

// Color32::get_average_4 (color.rs:51-71)
SW_DEV uint32_t average_4(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3)
{
	uint32_t s0 = 0, s1 = 0, s2 = 0, s3 = 0;
	const uint32_t c[4] = {c0, c1, c2, c3};
	for(int k = 0; k < 4; ++k)
	{
		s0 += c[k] & 0x000000FFu;
		s1 += c[k] & 0x0000FF00u;
		s2 += c[k] & 0x00FF0000u;
		s3 += (c[k] & 0xFF000000u) >> 2;
	}
	return (s0 >> 2) | ((s1 >> 2) & 0x0000FF00u) | ((s2 >> 2) & 0x00FF0000u) | (s3 & 0xFF000000u);
}

SW_DEV void unpack_normal_roughness_dev(int32_t p, float& x, float& y, float& z, float& r)
{
	const float k = 1.0f / 127.0f;
	x = float(int8_t(p & 0xFF)) * k;
	y = float(int8_t((p >> 8) & 0xFF)) * k;
	z = float(int8_t((p >> 16) & 0xFF)) * k;
	r = float(int8_t((p >> 24) & 0xFF)) * k;
}

// build_texture_mip (textures.rs:309-362) for one texel
SW_DEV sw_texel texel_mip(sw_texel p00, sw_texel p01, sw_texel p10, sw_texel p11)
{
	float n[4][3], r[4];
	unpack_normal_roughness_dev(p00.packed_normal_roughness, n[0][0], n[0][1], n[0][2], r[0]);
	unpack_normal_roughness_dev(p01.packed_normal_roughness, n[1][0], n[1][1], n[1][2], r[1]);
	unpack_normal_roughness_dev(p10.packed_normal_roughness, n[2][0], n[2][1], n[2][2], r[2]);
	unpack_normal_roughness_dev(p11.packed_normal_roughness, n[3][0], n[3][1], n[3][2], r[3]);
	const float sx = ((n[0][0] + n[1][0]) + n[2][0]) + n[3][0];
	const float sy = ((n[0][1] + n[1][1]) + n[2][1]) + n[3][1];
	const float sz = ((n[0][2] + n[1][2]) + n[2][2]) + n[3][2];
	const float len = __builtin_fmaxf(__builtin_sqrtf((sx * sx + sy * sy) + sz * sz), 0.000001f);
	const float deviation = (1.0f - len * 0.25f) / 0.5f;
	const float rs = ((r[0] + r[1]) + r[2]) + r[3];
	const float dr = __builtin_fminf(__builtin_fmaxf(__builtin_fmaf(rs, 0.25f, deviation), 1.0f / 126.0f), 1.0f);
	sw_texel t;
	t.diffuse = average_4(p00.diffuse, p01.diffuse, p10.diffuse, p11.diffuse);
	t.packed_normal_roughness = pack_normal_roughness_dev(sx / len, sy / len, sz / len, dr);
	return t;
}

// The lane's 2 x 2 square of texels at Morton distance step (the square's first lane, then x + 1 at step,
// y + 1 at 2 * step) as one texel of the next mip.
SW_DEV sw_texel quad_mip(sw_texel t, uint32_t lane, uint32_t step)
{
	const uint32_t first = lane & ~(4u * step - 1u);
	auto from = [&](uint32_t l) {
		sw_texel r;
		r.diffuse = uint32_t(__shfl(int(t.diffuse), int(l)));
		r.packed_normal_roughness = __shfl(t.packed_normal_roughness, int(l));
		return r;
	};
	return texel_mip(from(first), from(first + 2u * step), from(first + step), from(first + 3u * step));
}

// The wavy texture and its mips 1 .. 4 in one launch, a 16 x 16 tile of mip 0 per wave (a mip texel
// depends only on the square of mip 0 under it): a lane takes a 2 x 2 square of mip 0 and its mip 1 texel;
// the lanes lie in Morton order, so the block's first wave takes mip 2 of its four tiles from LDS (a
// texel's four parts follow each other), then mips 3 and 4 by lane exchanges. A square shares its field
// loads (12 values for four texels' 16). Bound by the correctly rounded roots and divisions of the normals:
// that is why the upper mips are gathered into one wave instead of costing every wave a pass each
// (1024 x 1024: 15.5 us with a texel per thread and the mips through LDS with barriers, 12.6 us with a pass
// per wave and mip, 9.9 us so; its 27 MB take 5.7 us at the rate of a large copy).
// PAIRS: the field is 8-byte aligned and the level starts on 16 bytes, so field values and texels move in
// pairs.
template <bool PAIRS>
__global__ __launch_bounds__(256) void k_water_texture(const float* __restrict__ field, uint32_t log2w, uint32_t log2h, uint32_t tiles,
	swk::WaterTexLaunch w, sw_texel* texels)
{
	__shared__ sw_texel mip1[256];
	const uint32_t lane = threadIdx.x & 63u;
	// past the last tile a wave redoes it (the same texels) for the barrier below
	const uint32_t tile = std::min(blockIdx.x * 4u + (threadIdx.x >> 6), tiles - 1u);
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	const uint32_t tx = tile & ((1u << (log2w - 4)) - 1u), ty = tile >> (log2w - 4);
	const uint32_t qx = (lane & 1u) | ((lane >> 1) & 2u) | ((lane >> 2) & 4u), qy = ((lane >> 1) & 1u) | ((lane >> 2) & 2u) | ((lane >> 3) & 4u);
	const uint32_t x = tx * 16u + qx * 2u, y = ty * 16u + qy * 2u;
	// rows y - 1 .. y + 2 at columns x, x + 1; rows y, y + 1 also at x - 1 and x + 2
	float f[4][4];
#pragma unroll
	for(uint32_t r = 0; r < 4; ++r)
	{
		const float* row = field + (((y + r - 1u) & my) << log2w);
		if(PAIRS)
		{
			const float2 p = *reinterpret_cast<const float2*>(row + x);
			f[r][1] = p.x;
			f[r][2] = p.y;
		}
		else
		{
			f[r][1] = row[x];
			f[r][2] = row[x + 1u];
		}
		if(r == 1 || r == 2)
		{
			f[r][0] = row[(x - 1u) & mx];
			f[r][3] = row[(x + 2u) & mx];
		}
	}
	const uint32_t i0 = x + (y << log2w), i1 = i0 + (1u << log2w);
	sw_texel* out = texels + w.dst_offset[0];
	sw_texel t[2][2]; // [y][x]
#pragma unroll
	for(uint32_t r = 0; r < 2; ++r)
#pragma unroll
		for(uint32_t c = 0; c < 2; ++c)
			t[r][c] = water_texel(f[r + 1][c + 2] - f[r + 1][c], f[r + 2][c + 1] - f[r][c + 1], log2w, log2h, w, texels, x + c, y + r);
	if(PAIRS)
	{
		*reinterpret_cast<uint4*>(out + i0) = make_uint4(t[0][0].diffuse, uint32_t(t[0][0].packed_normal_roughness), t[0][1].diffuse,
			uint32_t(t[0][1].packed_normal_roughness));
		*reinterpret_cast<uint4*>(out + i1) = make_uint4(t[1][0].diffuse, uint32_t(t[1][0].packed_normal_roughness), t[1][1].diffuse,
			uint32_t(t[1][1].packed_normal_roughness));
	}
	else
	{
		out[i0] = t[0][0];
		out[i0 + 1] = t[0][1];
		out[i1] = t[1][0];
		out[i1 + 1] = t[1][1];
	}
	sw_texel v = texel_mip(t[0][0], t[1][0], t[0][1], t[1][1]);
	texels[w.dst_offset[1] + (tx * 8u + qx) + ((ty * 8u + qy) << (log2w - 1))] = v;
	mip1[threadIdx.x] = v;
	__syncthreads();
	if(threadIdx.x >= 64u)
		return;
	// the first wave: lane 16 q + j takes mip 2 texel j (Morton order) of the block's tile q
	const uint32_t mt = blockIdx.x * 4u + (lane >> 4);
	const bool ok = mt < tiles;
	const uint32_t mtx = mt & ((1u << (log2w - 4)) - 1u), mty = mt >> (log2w - 4);
	const uint32_t jx = (lane & 1u) | ((lane >> 1) & 2u), jy = ((lane >> 1) & 1u) | ((lane >> 2) & 2u);
	v = texel_mip(mip1[lane * 4u], mip1[lane * 4u + 2u], mip1[lane * 4u + 1u], mip1[lane * 4u + 3u]);
	if(ok)
		texels[w.dst_offset[2] + (mtx * 4u + jx) + ((mty * 4u + jy) << (log2w - 2))] = v;
	v = quad_mip(v, lane, 1);
	if(ok && (lane & 3u) == 0)
		texels[w.dst_offset[3] + (mtx * 2u + (jx >> 1)) + ((mty * 2u + (jy >> 1)) << (log2w - 3))] = v;
	v = quad_mip(v, lane, 4);
	if(ok && (lane & 15u) == 0)
		texels[w.dst_offset[4] + mtx + (mty << (log2w - 4))] = v;
}

// The average of the lane's 2 x 2 square of texels, the square's lanes step apart in Morton order:
// its first lane, then x + 1 (step), y + 1 (2 * step) and both.
SW_DEV uint32_t quad_average(uint32_t v, uint32_t lane, uint32_t step)
{
	const uint32_t first = lane & ~(4u * step - 1u); // the square's (0, 0) lane
	return average_4(uint32_t(__shfl(int(v), int(first))), uint32_t(__shfl(int(v), int(first + 2u * step))),
		uint32_t(__shfl(int(v), int(first + step))), uint32_t(__shfl(int(v), int(first + 3u * step))));
}

// The palette texture (generate_emissive_texture_based_on_heat_map, :470-486) and its lite mips 1 .. 4
// (build_texture_lite_mip, textures.rs:385-415), a 16 x 16 tile per wave: a lane takes a 2 x 2 square of
// mip 0 and its mip 1 texel, the lanes lie in Morton order, so mips 2 .. 4 come from lane exchanges
// (no barriers). Bound by launch and memory latency: the palette travels in the kernel's arguments
// (no copy ahead of the launch), is staged in LDS once per block.
__global__ __launch_bounds__(256) void k_fire_texture(const uint8_t* heat, uint32_t log2w, uint32_t tiles, swk::FirePalette palette,
	uint32_t* lite, uint64_t o0, uint64_t o1, uint64_t o2, uint64_t o3, uint64_t o4)
{
	__shared__ uint32_t pal[256];
	pal[threadIdx.x] = palette.color[threadIdx.x];
	__syncthreads();
	const uint32_t tile = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
	if(tile >= tiles)
		return; // uniform over the wave
	const uint32_t tx = tile & ((1u << (log2w - 4)) - 1u), ty = tile >> (log2w - 4);
	const uint32_t qx = (lane & 1u) | ((lane >> 1) & 2u) | ((lane >> 2) & 4u), qy = ((lane >> 1) & 1u) | ((lane >> 2) & 2u) | ((lane >> 3) & 4u);
	const uint32_t x = tx * 16u + qx * 2u, y = ty * 16u + qy * 2u;
	const uint32_t i0 = x + (y << log2w), i1 = i0 + (1u << log2w);
	const uint32_t c00 = pal[heat[i0]], c10 = pal[heat[i0 + 1]], c01 = pal[heat[i1]], c11 = pal[heat[i1 + 1]];
	lite[o0 + i0] = c00;
	lite[o0 + i0 + 1] = c10;
	lite[o0 + i1] = c01;
	lite[o0 + i1 + 1] = c11;
	uint32_t v = average_4(c00, c01, c10, c11);
	lite[o1 + (tx * 8u + qx) + ((ty * 8u + qy) << (log2w - 1))] = v;
	v = quad_average(v, lane, 1);
	if((lane & 3u) == 0)
		lite[o2 + (tx * 4u + (qx >> 1)) + ((ty * 4u + (qy >> 1)) << (log2w - 2))] = v;
	v = quad_average(v, lane, 4);
	if((lane & 15u) == 0)
		lite[o3 + (tx * 2u + (qx >> 2)) + ((ty * 2u + (qy >> 2)) << (log2w - 3))] = v;
	v = quad_average(v, lane, 16);
	if(lane == 0)
		lite[o4 + tx + (ty << (log2w - 4))] = v;
}

} // namespace

namespace
{
// update_heat_map (:357-468), fast variant, and the step's set_heat points: row y < h - 2 from rows
// y + 1 (x - 1, x, x + 1, wrapped) and y + 2; row h - 2 takes row h - 1 twice; the last row is cleared.
// All reads see the old map (the reference walks rows downwards and reads only rows below). A block
// takes 1024 consecutive texels, four per thread; the points (packed as address and heat in the
// kernel's arguments) then raise the block's texels in LDS by atomic maxima, so a step is one launch
// with no copy ahead of it: bound by launch latency (a 64 x 64 map's step: 2.2 us of update, 9.4 us of
// points and 2.7 us of copy as three operations, 3 us as one). WORDS: both buffers are 4-byte
// aligned, texels move as words.
template <bool POINTS, bool WORDS>
SW_DEV void fire_step_fast(const uint8_t* src, uint8_t* dst, uint32_t log2w, uint32_t log2h, uint32_t att, const uint32_t* points,
	uint32_t num_points)
{
	__shared__ __align__(16) uint32_t cells[1024];
	const uint32_t w = 1u << log2w, h = 1u << log2h, mx = w - 1u;
	const uint32_t b0 = blockIdx.x * 1024u, i = b0 + threadIdx.x * 4u;
	const bool in = (i >> (log2w + log2h)) == 0;
	uint32_t v[4] = {0, 0, 0, 0};
	const uint32_t x = i & mx, y = i >> log2w;
	if(in && y != h - 1u)
	{
		const uint32_t r1 = (y + 1u) << log2w, r2 = (y + 2u < h ? y + 2u : y + 1u) << log2w;
		uint32_t a[6], c[4];
		a[0] = src[r1 + ((x - 1u) & mx)];
		a[5] = src[r1 + ((x + 4u) & mx)];
		if(WORDS)
		{
			const uint32_t wa = *reinterpret_cast<const uint32_t*>(src + r1 + x), wc = *reinterpret_cast<const uint32_t*>(src + r2 + x);
			for(uint32_t k = 0; k < 4; ++k)
			{
				a[k + 1] = (wa >> (8 * k)) & 0xFFu;
				c[k] = (wc >> (8 * k)) & 0xFFu;
			}
		}
		else
			for(uint32_t k = 0; k < 4; ++k)
			{
				a[k + 1] = src[r1 + x + k];
				c[k] = src[r2 + x + k];
			}
		for(uint32_t k = 0; k < 4; ++k)
			v[k] = ((a[k] + a[k + 1] + a[k + 2] + c[k]) * att) >> 20;
	}
	if constexpr(POINTS)
	{
		*reinterpret_cast<uint4*>(cells + threadIdx.x * 4u) = make_uint4(v[0], v[1], v[2], v[3]);
		__syncthreads();
		for(uint32_t k = threadIdx.x; k < num_points; k += 256u)
		{
			const uint32_t p = points[k], a = (p & swk::FIRE_POINT_ADDRESS) - b0;
			if(a < 1024u)
				atomicMax(&cells[a], p >> swk::FIRE_POINT_HEAT_SHIFT);
		}
		__syncthreads();
		const uint4 r = *reinterpret_cast<const uint4*>(cells + threadIdx.x * 4u);
		v[0] = r.x;
		v[1] = r.y;
		v[2] = r.z;
		v[3] = r.w;
	}
	if(!in)
		return;
	if(WORDS)
		*reinterpret_cast<uint32_t*>(dst + i) = v[0] | (v[1] << 8) | (v[2] << 16) | (v[3] << 24);
	else
		for(uint32_t k = 0; k < 4; ++k)
			dst[i + k] = uint8_t(v[k]);
}

template <uint32_t N, bool WORDS>
__global__ __launch_bounds__(256) void k_fire_step_fast(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t log2w,
	uint32_t log2h, uint32_t att, swk::FirePoints<N> pts)
{
	fire_step_fast<true, WORDS>(src, dst, log2w, log2h, att, pts.p, pts.n);
}
// A step without points, with no more arguments than it needs: queued steps of small maps are bound by the host's
// launches (4.3 us a step with the points' arguments, 3.6 so; the slow variant alike, at 256 x 256 13.1 us by its chain).
template <bool WORDS>
__global__ __launch_bounds__(256) void k_fire_update_fast(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t log2w,
	uint32_t log2h, uint32_t att)
{
	fire_step_fast<false, WORDS>(src, dst, log2w, log2h, att, nullptr, 0);
}

// The slow variant: each row is a chain (the left neighbour is the value just written; the last
// texel's right neighbour is the row's new first texel), from the row and the row below. A block
// takes 16 rows, 256 columns at a time: all threads sum what a texel reads besides its left neighbour
// (the loads do not depend on the chain, src and dst are distinct buffers) into LDS, one lane per row
// runs the chain there, and all threads store the texels, after the step's points raised them.
// Bound by the chain (an add, a multiply and a shift per texel); with each lane loading its own row's
// bytes the 64 x 64 step took 5.3 us of update beside the points' 9.4 us.
#define FIRE_SLOW_ROWS 16u
#define FIRE_SLOW_COLS 256u
template <bool POINTS>
SW_DEV void fire_step_slow(const uint8_t* src, uint8_t* dst, uint32_t log2w, uint32_t log2h, uint32_t att, const uint32_t* points,
	uint32_t num_points)
{
	// a row's cells: the sums, then the chain's values (a word between rows: the chain's lanes read 16
	// rows at one column, which then lie in 16 banks)
	__shared__ uint32_t cells[FIRE_SLOW_ROWS][FIRE_SLOW_COLS + 1];
	const uint32_t w = 1u << log2w, h = 1u << log2h;
	const uint32_t y0 = blockIdx.x * FIRE_SLOW_ROWS; // h is a multiple of 16
	const uint32_t cols = w < FIRE_SLOW_COLS ? w : FIRE_SLOW_COLS, log2c = log2w < 8 ? log2w : 8u;
	uint32_t prev = 0, first = 0;
	if(threadIdx.x < FIRE_SLOW_ROWS)
		prev = src[((y0 + threadIdx.x) << log2w) + w - 1u]; // the first texel's left neighbour
	for(uint32_t x0 = 0; x0 < w; x0 += cols)
	{
		for(uint32_t k = threadIdx.x; k < FIRE_SLOW_ROWS << log2c; k += 256u)
		{
			const uint32_t r = k >> log2c, x = x0 + (k & (cols - 1u)), row = (y0 + r) << log2w;
			uint32_t s = 0;
			if(y0 + r != h - 1u)
				s = uint32_t(src[row + x]) + (x + 1u < w ? src[row + x + 1u] : 0u) + src[row + w + x];
			cells[r][k & (cols - 1u)] = s;
		}
		__syncthreads();
		if(threadIdx.x < FIRE_SLOW_ROWS && y0 + threadIdx.x != h - 1u)
		{
			uint32_t* c = cells[threadIdx.x];
#pragma unroll 8
			for(uint32_t k = 0; k < cols; ++k)
			{
				uint32_t s = c[k];
				if(x0 + k == w - 1u)
					s += first;
				prev = ((prev + s) * att) >> 20;
				if(x0 + k == 0)
					first = prev;
				c[k] = prev;
			}
		}
		__syncthreads();
		if constexpr(POINTS)
		{
			for(uint32_t k = threadIdx.x; k < num_points; k += 256u)
			{
				const uint32_t p = points[k], a = p & swk::FIRE_POINT_ADDRESS;
				const uint32_t px = (a & (w - 1u)) - x0, py = (a >> log2w) - y0;
				if(px < cols && py < FIRE_SLOW_ROWS)
					atomicMax(&cells[py][px], p >> swk::FIRE_POINT_HEAT_SHIFT);
			}
			__syncthreads();
		}
		for(uint32_t k = threadIdx.x; k < FIRE_SLOW_ROWS << log2c; k += 256u)
		{
			const uint32_t r = k >> log2c, c = k & (cols - 1u);
			dst[((y0 + r) << log2w) + x0 + c] = uint8_t(cells[r][c]);
		}
		__syncthreads(); // the next columns rewrite the cells
	}
}

template <uint32_t N>
__global__ __launch_bounds__(256) void k_fire_step_slow(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t log2w,
	uint32_t log2h, uint32_t att, swk::FirePoints<N> pts)
{
	fire_step_slow<true>(src, dst, log2w, log2h, att, pts.p, pts.n);
}
__global__ __launch_bounds__(256) void k_fire_update_slow(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t log2w,
	uint32_t log2h, uint32_t att)
{
	fire_step_slow<false>(src, dst, log2w, log2h, att, nullptr, 0);
}

// set_heat (:80-86) for more points than a step's kernel arguments hold, 64 at a time: the first point
// of each address takes the maximum of the batch's heats for it (max is order-free)
__global__ __launch_bounds__(64) void k_fire_points(uint8_t* heat, const sw_heat_point* pts, uint32_t n, uint32_t log2w, uint32_t log2h)
{
	__shared__ uint32_t sa[64], sh[64];
	const uint32_t lane = threadIdx.x;
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	for(uint32_t base = 0; base < n; base += 64)
	{
		const uint32_t cnt = n - base < 64u ? n - base : 64u;
		uint32_t a = 0;
		if(lane < cnt)
		{
			const sw_heat_point p = pts[base + lane];
			a = (p.x & mx) + ((p.y & my) << log2w);
			sa[lane] = a;
			sh[lane] = p.heat & 0xFFu;
		}
		__syncthreads();
		if(lane < cnt)
		{
			bool first = true;
			for(uint32_t k = 0; k < lane; ++k)
				first = first && sa[k] != a;
			if(first)
			{
				uint32_t v = heat[a];
				for(uint32_t k = lane; k < cnt; ++k)
					if(sa[k] == a && sh[k] > v)
						v = sh[k];
				heat[a] = uint8_t(v);
			}
		}
		__syncthreads();
	}
}

} // namespace

namespace swk
{
static uint32_t water_blocks(uint32_t log2w, uint32_t log2h) { return ((1u << (log2w + log2h)) + WATER_BLOCK - 1u) / WATER_BLOCK; }
static bool water_aligned(const float* field, const float* field_old)
{
	return (reinterpret_cast<uintptr_t>(field) | reinterpret_cast<uintptr_t>(field_old)) % 16 == 0;
}

static void launch_water_step_alone(hipStream_t st, float* field, float* field_old, uint32_t log2w, uint32_t log2h, float attenuation)
{
	const dim3 grid(water_blocks(log2w, log2h));
	if(water_aligned(field, field_old))
		hipLaunchKernelGGL(k_water_step<true>, grid, dim3(256), 0, st, field_old, static_cast<const float*>(field), log2w, log2h, attenuation);
	else
		hipLaunchKernelGGL(k_water_step<false>, grid, dim3(256), 0, st, field_old, static_cast<const float*>(field), log2w, log2h, attenuation);
}

template <uint32_t N>
static void launch_water_step_n(hipStream_t st, float* field, float* field_old, uint32_t log2w, uint32_t log2h, float attenuation,
	const sw_wave_point* points, uint32_t num_points, uint32_t* ticket)
{
	WavePoints<N> p;
	p.n = num_points;
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	// sorted by address, an address's points in their order: only their own order matters to it
	uint64_t order[N];
	for(uint32_t k = 0; k < num_points; ++k)
		order[k] = (uint64_t((points[k].x & mx) + ((points[k].y & my) << log2w)) << 32) | k;
	std::sort(order, order + num_points);
	// the blocks that read a point's element: those of its four neighbours
	std::bitset<WATER_MAX_BLOCKS> readers;
	for(uint32_t k = 0; k < num_points; ++k)
	{
		p.address[k] = uint32_t(order[k] >> 32);
		p.value[k] = points[uint32_t(order[k])].value;
		for(uint32_t n = 0; n < 4; ++n)
			readers.set(water_neighbour(p.address[k], n, log2w, log2h) / WATER_BLOCK);
	}
	const uint32_t num_readers = uint32_t(readers.count());
	const dim3 grid(water_blocks(log2w, log2h));
	if(water_aligned(field, field_old))
		hipLaunchKernelGGL((k_water_step_points<N, true>), grid, dim3(256), 0, st, field_old, field, log2w, log2h, attenuation, p,
			num_readers, ticket);
	else
		hipLaunchKernelGGL((k_water_step_points<N, false>), grid, dim3(256), 0, st, field_old, field, log2w, log2h, attenuation, p,
			num_readers, ticket);
}

void launch_water_step(hipStream_t st, float* field, float* field_old, uint32_t log2w, uint32_t log2h, float attenuation,
	const sw_wave_point* points, uint32_t num_points, const sw_wave_point* points_dev, uint32_t* ticket)
{
	// the smallest argument block that holds the points: the runtime copies the whole block per launch
	if(num_points == 0)
		launch_water_step_alone(st, field, field_old, log2w, log2h, attenuation);
	else if(num_points <= WATER_ARG_POINTS_SMALL)
		launch_water_step_n<WATER_ARG_POINTS_SMALL>(st, field, field_old, log2w, log2h, attenuation, points, num_points, ticket);
	else if(num_points <= WATER_ARG_POINTS)
		launch_water_step_n<WATER_ARG_POINTS>(st, field, field_old, log2w, log2h, attenuation, points, num_points, ticket);
	else
	{
		hipLaunchKernelGGL(k_water_points, dim3(1), dim3(64), 0, st, field, field_old, points_dev, num_points, log2w, log2h);
		launch_water_step_alone(st, field, field_old, log2w, log2h, attenuation);
	}
}

void launch_water_texture(hipStream_t st, const float* field, uint32_t log2w, uint32_t log2h, const WaterTexLaunch& w, sw_texel* texels)
{
	const uint32_t tiles = 1u << (log2w + log2h - 8);
	const dim3 grid((tiles + 3u) / 4u);
	if(reinterpret_cast<uintptr_t>(field) % 8 == 0 && reinterpret_cast<uintptr_t>(texels + w.dst_offset[0]) % 16 == 0)
		hipLaunchKernelGGL(k_water_texture<true>, grid, dim3(256), 0, st, field, log2w, log2h, tiles, w, texels);
	else
		hipLaunchKernelGGL(k_water_texture<false>, grid, dim3(256), 0, st, field, log2w, log2h, tiles, w, texels);
}
static uint32_t fire_blocks(uint32_t log2w, uint32_t log2h) { return ((1u << (log2w + log2h)) + 1023u) / 1024u; }
static bool fire_aligned(const uint8_t* heat, const uint8_t* heat_old)
{
	return (reinterpret_cast<uintptr_t>(heat) | reinterpret_cast<uintptr_t>(heat_old)) % 4 == 0;
}

static void launch_fire_update(hipStream_t st, const uint8_t* heat, uint8_t* heat_old, uint32_t log2w, uint32_t log2h,
	uint32_t attenuation_i, bool slow)
{
	const dim3 grid(slow ? (1u << log2h) / FIRE_SLOW_ROWS : fire_blocks(log2w, log2h));
	if(slow)
		hipLaunchKernelGGL(k_fire_update_slow, grid, dim3(256), 0, st, heat, heat_old, log2w, log2h, attenuation_i);
	else if(fire_aligned(heat, heat_old))
		hipLaunchKernelGGL(k_fire_update_fast<true>, grid, dim3(256), 0, st, heat, heat_old, log2w, log2h, attenuation_i);
	else
		hipLaunchKernelGGL(k_fire_update_fast<false>, grid, dim3(256), 0, st, heat, heat_old, log2w, log2h, attenuation_i);
}

template <uint32_t N>
static void launch_fire_step_n(hipStream_t st, const uint8_t* heat, uint8_t* heat_old, uint32_t log2w, uint32_t log2h,
	uint32_t attenuation_i, bool slow, const sw_heat_point* points, uint32_t num_points)
{
	FirePoints<N> p;
	p.n = num_points;
	const uint32_t mx = (1u << log2w) - 1u, my = (1u << log2h) - 1u;
	for(uint32_t k = 0; k < num_points; ++k)
		p.p[k] = ((points[k].x & mx) + ((points[k].y & my) << log2w)) | ((points[k].heat & 0xFFu) << FIRE_POINT_HEAT_SHIFT);
	const dim3 grid(slow ? (1u << log2h) / FIRE_SLOW_ROWS : fire_blocks(log2w, log2h));
	if(slow)
		hipLaunchKernelGGL(k_fire_step_slow<N>, grid, dim3(256), 0, st, heat, heat_old, log2w, log2h, attenuation_i, p);
	else if(fire_aligned(heat, heat_old))
		hipLaunchKernelGGL((k_fire_step_fast<N, true>), grid, dim3(256), 0, st, heat, heat_old, log2w, log2h, attenuation_i, p);
	else
		hipLaunchKernelGGL((k_fire_step_fast<N, false>), grid, dim3(256), 0, st, heat, heat_old, log2w, log2h, attenuation_i, p);
}

void launch_fire_step(hipStream_t st, const uint8_t* heat, uint8_t* heat_old, uint32_t log2w, uint32_t log2h, uint32_t attenuation_i,
	bool slow, const sw_heat_point* points, uint32_t num_points, const sw_heat_point* points_dev)
{
	// the smallest argument block that holds the points: the runtime copies the whole block per launch
	if(num_points == 0)
		launch_fire_update(st, heat, heat_old, log2w, log2h, attenuation_i, slow);
	else if(num_points <= FIRE_ARG_POINTS_SMALL)
		launch_fire_step_n<FIRE_ARG_POINTS_SMALL>(st, heat, heat_old, log2w, log2h, attenuation_i, slow, points, num_points);
	else if(num_points <= FIRE_ARG_POINTS)
		launch_fire_step_n<FIRE_ARG_POINTS>(st, heat, heat_old, log2w, log2h, attenuation_i, slow, points, num_points);
	else
	{
		launch_fire_update(st, heat, heat_old, log2w, log2h, attenuation_i, slow);
		hipLaunchKernelGGL(k_fire_points, dim3(1), dim3(64), 0, st, heat_old, points_dev, num_points, log2w, log2h);
	}
}

void launch_fire_texture(hipStream_t st, const uint8_t* heat, uint32_t log2w, uint32_t log2h, const uint64_t dst_offset[5],
	const uint32_t palette[256], uint32_t* lite)
{
	FirePalette p;
	std::memcpy(p.color, palette, sizeof(p.color));
	const uint32_t tiles = 1u << (log2w + log2h - 8);
	hipLaunchKernelGGL(k_fire_texture, dim3((tiles + 3u) / 4u), dim3(256), 0, st, heat, log2w, tiles, p, lite, dst_offset[0],
		dst_offset[1], dst_offset[2], dst_offset[3], dst_offset[4]);
}

} // namespace swk
