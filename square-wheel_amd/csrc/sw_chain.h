// The end of a chain of float additions without walking it.
//
// The depth rasteriser steps 1 / z by additions along a span and along the rows of a polygon part
// (rasterizer.rs:1414-1474); float addition rounds at every step, so a value is defined by the whole chain.
// Between two powers of two, though, the floats are evenly spaced, and every addition of the same d moves a
// value there by the same multiple of the spacing: d rounded to it, or, when d lies half-way between two
// multiples, the choice that keeps the mantissa even, which repeats from the second step on. So the steps
// inside a binade are one exact multiply-add, and only the steps near the powers of two are walked.
//
// No HIP dependency: the kernels include this with SW_HD defined, a CPU check compiles it with a host
// compiler and compares it with the walked chain.
#pragma once

#include <stdint.h>

#ifndef SW_HD
#define SW_HD static inline
#endif

namespace swchain
{

SW_HD uint32_t float_bits(float x)
{
	uint32_t u;
	__builtin_memcpy(&u, &x, sizeof(u));
	return u;
}
SW_HD float bits_float(uint32_t u)
{
	float x;
	__builtin_memcpy(&x, &u, sizeof(x));
	return x;
}

// 0, infinite or NaN: one instruction of the device's (a mask of classes), which the kernels' inner loop notices.
SW_HD bool zero_or_not_finite(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
	return __builtin_amdgcn_classf(x, 0x267);
#else
	return (float_bits(x) << 1) - 1u >= 0xFEFFFFFFu;
#endif
}

// a and b, with their signs, strictly between the same two neighbouring powers of two (or both denormal);
// then so is every value of a monotonic chain from a to b.
SW_HD bool inside_one_binade(float a, float b)
{
	const uint32_t ua = float_bits(a), ub = float_bits(b);
	return ((ua ^ ub) & 0xFF800000u) == 0 && (ua & 0x007FFFFFu) != 0 && (ub & 0x007FFFFFu) != 0 && (ua & 0x7F800000u) != 0x7F800000u;
}

// v after n additions of d (n below 2^24).
SW_HD float chain_add(float v, float d, uint32_t n)
{
	while(n > 3u)
	{
		// v1, v2, v3 inside one binade: from v2 on (even, if the additions tie) every step is v3 - v2, exact
		// as a difference of neighbours, and so is a multiple of it added to v2 that stays in the binade.
		const float v1 = v + d, v2 = v1 + d, v3 = v2 + d;
		const float step = v3 - v2;
		const float end = __builtin_fmaf(float(n - 2u), step, v2);
		if(inside_one_binade(v1, end))
			return end;
		// a step of 0 (v2 + d rounds to v2 again and again), or an infinite one or NaN (so is v3, and stays so)
		if(zero_or_not_finite(step))
			return v3;
		v = v3;
		n -= 3u;
		if(inside_one_binade(v1, v3))
		{
			// jump close to the power of two that the chain crosses (kept only if it stays inside)
			const uint32_t edge = float_bits(v3) & 0xFF800000u;
			const float limit = bits_float((float_bits(step) ^ edge) >> 31 ? edge : edge + 0x00800000u);
			const float steps = (limit - v3) / step - 2.0f;
			const uint32_t k = steps >= 1.0f ? (steps < float(n) ? uint32_t(steps) : n) : 0u;
			const float near = __builtin_fmaf(float(k), step, v3);
			if(k != 0u && inside_one_binade(v1, near))
			{
				v = near;
				n -= k;
			}
		}
	}
	for(; n; --n)
		v += d;
	return v;
}

} // namespace swchain
