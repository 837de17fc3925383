// Host build of the kernels' addition-chain helper (csrc/sw_chain.h) against the walked chain.
#include "../../square-wheel_amd/csrc/sw_chain.h"

#include <cstring>

extern "C" {

// For each (start, step): every length 0 .. n of the chain; returns how many values differ in their bits
// (NaNs count as equal), and the first one in `first` (pair, length).
uint64_t check_chains(const float* start, const float* step, uint32_t count, uint32_t n, uint32_t* first)
{
	uint64_t bad = 0;
	for(uint32_t i = 0; i < count; ++i)
	{
		float v = start[i];
		for(uint32_t k = 0; k <= n; ++k)
		{
			const float got = swchain::chain_add(start[i], step[i], k);
			if(std::memcmp(&got, &v, 4) != 0 && !(got != got && v != v) && bad++ == 0)
			{
				first[0] = i;
				first[1] = k;
			}
			v += step[i];
		}
	}
	return bad;
}

// The same at one length only (long chains).
uint64_t check_chain_ends(const float* start, const float* step, uint32_t count, uint32_t n)
{
	uint64_t bad = 0;
	for(uint32_t i = 0; i < count; ++i)
	{
		float v = start[i];
		for(uint32_t k = 0; k < n; ++k)
			v += step[i];
		const float got = swchain::chain_add(start[i], step[i], n);
		bad += std::memcmp(&got, &v, 4) != 0 && !(got != got && v != v);
	}
	return bad;
}

// The chains' ends alone.
void chain_ends(const float* start, const float* step, uint32_t count, uint32_t n, float* out)
{
	for(uint32_t i = 0; i < count; ++i)
		out[i] = swchain::chain_add(start[i], step[i], n);
}
}
