// lookback.h -- running sums over the tiles of one launch (decoupled
// look-back): a tile posts its own sum, collects those of the tiles before it
// from the nearest that has its running sum, and posts its own running sum.
//
// A state word is 0 (nothing yet), kOwn | sum of the tile, or kAll | sum of
// the tile and all before it; words are 0 when the launch starts.  Tiles are
// numbered by tickets taken when a block starts, so the tiles before one's
// own belong to blocks that have started, and a block posts its own sum
// before it waits for anything: every wait ends.
#ifndef SF_LOOKBACK_H
#define SF_LOOKBACK_H

#include <hip/hip_runtime.h>

namespace look {

constexpr unsigned long long kOwn = 1ull << 62, kAll = 2ull << 62, kSum = kOwn - 1ull;

__device__ __forceinline__ unsigned long long peek(const unsigned long long* p) {
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void post(unsigned long long* p, unsigned long long v) {
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The next tile's number; every thread of the block calls it, s is shared.
__device__ __forceinline__ unsigned ticket(unsigned* counter, unsigned& s) {
	if (threadIdx.x == 0u) s = atomicAdd(counter, 1u);
	__syncthreads();
	return __builtin_amdgcn_readfirstlane(s);
}

// The sums over the tiles before `tile` of C components (C a power of two up
// to 64, state[tile * C + component]), with all 64 lanes of one wavefront:
// lane l looks at component l % C, 64 / C tiles at a time.  own: lane l < C's
// component of this tile.  Posts own and the running sum; returns the prior
// sum of component l % C.
template <int C>
__device__ __forceinline__ unsigned long long collect(unsigned long long* state, unsigned tile, unsigned long long own) {
	constexpr int W = 64 / C;
	const int lane = (int)(threadIdx.x & 63u), c = lane % C, q = lane / C;
	unsigned long long column = 0ull;   // the lanes of component 0
#pragma unroll
	for (int k = 0; k < W; ++k) column |= 1ull << (k * C);
	column <<= c;
	if (lane < C) post(state + (size_t)tile * C + lane, (tile ? kOwn : kAll) | own);
	unsigned long long prior = 0ull;
	bool open = tile != 0u;
	for (int j = (int)tile - 1; __ballot(open) != 0ull; j -= W) {
		unsigned long long v = kAll, all = 0ull;
		for (;;) {
			if (open && j - q >= 0) v = peek(state + (size_t)(j - q) * C + c);
			all = __ballot(v >= kAll) & column;
			// the lanes that count: those up to the nearest running sum
			const unsigned long long upto = all ? (2ull << __builtin_ctzll(all)) - 1ull : ~0ull;
			if (__ballot(v == 0ull && ((upto >> lane) & 1ull)) == 0ull) {
				if (!((upto >> lane) & 1ull)) v = 0ull;
				break;
			}
		}
		unsigned long long sum = open ? v & kSum : 0ull;
#pragma unroll
		for (int o = C; o < 64; o <<= 1) sum += __shfl_xor(sum, o);
		prior += sum;
		if (all) open = false;
	}
	if (tile && lane < C) post(state + (size_t)tile * C + lane, kAll | (prior + own));
	return prior;
}

}  // namespace look

#endif
