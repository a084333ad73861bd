// order_chain.h -- sums over j in index order for every particle i, as the
// reference adds them, with the terms made in parallel.
//
// Each sum is a chain: one lane, one (particle, component), four dependent
// additions a term where it is Kahan's.  A lane per particle with every term
// made in line left most of the card idle (64 blocks at N = 16384), each
// waiting for one division after another.  Here a block holds I = 64 or 32
// particles.  kMakers wavefronts make the terms of a tile of 64 bodies into
// LDS, a run of 8 bodies each, while the chain wavefronts add up the tile made
// before, 64 / I components each.
//
// Bound: a chain takes one wavefront's issue interval, 2.5 ns, per operation,
// 10 ns a body for Kahan's four; the makers take what their terms issue.  With
// I = 64 a run's bodies are uniform (scalar loads); with I = 32 a wavefront's
// halves take every second one each (vector loads), and half as many particles
// reach every CU.  So 32 up to 8192 particles (256 blocks), 64 above: exact PP
// at N = 6000 74 and 105 us, at 8193 190 and 150, at 16384 410 and 323.
//
// A model M has
//   kComps                 components per particle
//   Body, body(j, off)     what a term reads of body j + off; off is a constant, so that a
//                          run's loads share one address
//   Self, self(i)          and of particle i
//   Check                  what the makers' fast terms must be looked at for:
//                          Check{}.bad() after a run sends it through terms<false>
//   fast                   whether terms<true> may be used at all
//   terms<FAST>(Self, Body, float (&out)[kComps], Check&)
//   step(comp, s, c, x)    one addition of the chain
//   store(i, comp, s)
#ifndef SF_ORDER_CHAIN_H
#define SF_ORDER_CHAIN_H

#include <hip/hip_runtime.h>

namespace chain {

constexpr unsigned kFewN = 8192;             // up to here 32 particles a block
constexpr unsigned kJ = 64;                  // bodies per tile
constexpr unsigned kMakers = 8;              // wavefronts that make terms
constexpr unsigned kRun = kJ / kMakers;      // consecutive bodies per maker and tile
constexpr unsigned kAhead = 16;              // terms a chain has read ahead

template <unsigned I, unsigned COMPS>
constexpr unsigned chain_waves() { return (COMPS * I + 63u) / 64u; }
template <unsigned I, unsigned COMPS>
constexpr unsigned block_size() { return 64u * (kMakers + chain_waves<I, COMPS>()); }

// y = x - c; t = s + y; c = (t - s) - y; s = t (reference src/gravity.c:771-784)
__device__ __forceinline__ void kahan(float& s, float& c, float x) {
	const float y = x - c;
	const float t = s + y;
	const float z = t - s;
	c = z - y;
	s = t;
}

// WAVES: the block's wavefronts, where a launch runs models of different sizes;
// those that this one does not need wait.
template <unsigned I, unsigned WAVES = 0, class M>
__device__ __forceinline__ void run(const M& md, unsigned N) {
	constexpr unsigned kC = M::kComps, kChainWaves = chain_waves<I, kC>();
	static_assert(WAVES == 0 || WAVES >= kChainWaves + kMakers, "the model's wavefronts");
	constexpr unsigned kPer = 64u / I;           // bodies a wavefront takes at once
	constexpr unsigned kLane = kRun / kPer;      // bodies of a run per lane
	__shared__ float s_term[2][kC][kJ][I];
	const unsigned lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const unsigned part = I == 64u ? 0u : lane / I, il = lane % I;
	const unsigned i = blockIdx.x * I + il;
	const unsigned tiles = (N + kJ - 1u) / kJ;
	if (WAVES && wv >= kChainWaves + kMakers) {
		for (unsigned t = 0; t <= tiles; ++t) __syncthreads();
		return;
	}
	if (wv >= kChainWaves) {
		const typename M::Self me = md.self(min(i, N - 1u));
		const unsigned first = (wv - kChainWaves) * kRun;
		const bool fast = md.fast() && N >= kRun;
		// the lane's bodies, read one tile ahead from a clamped address (the
		// run that reaches past N takes the slow loop)
		typename M::Body b[kLane];
		auto read = [&](unsigned j0) {
			const unsigned jc = min(j0, N - kRun) + part;
#pragma unroll
			for (unsigned u = 0; u < kLane; ++u) b[u] = md.body(jc, kPer * u);
		};
		if (fast) read(first);
		for (unsigned t = 0; t < tiles; ++t) {
			float* out = &s_term[t & 1u][0][first][0] + lane;   // body kPer u + part, particle il: + 64 u
			const unsigned j0 = t * kJ + first;
			bool slow = true;
			if (fast) {
				typename M::Check chk;
#pragma unroll
				for (unsigned u = 0; u < kLane; ++u) {
					float v[kC];
					md.template terms<true>(me, b[u], v, chk);
#pragma unroll
					for (unsigned k = 0; k < kC; ++k) out[k * kJ * I + 64u * u] = v[k];
				}
				read(j0 + kJ);
				slow = __ballot(chk.bad()) != 0ull || j0 + kRun > N;
			}
			if (slow) {
#pragma unroll 1
				for (unsigned u = 0; u < kLane; ++u) {
					const unsigned j = j0 + kPer * u + part;
					if (j < N) {
						float v[kC];
						typename M::Check chk;
						md.template terms<false>(me, md.body(j, 0u), v, chk);
#pragma unroll
						for (unsigned k = 0; k < kC; ++k) out[k * kJ * I + 64u * u] = v[k];
					}
				}
			}
			__syncthreads();
		}
		__syncthreads();
		return;
	}
	const unsigned own = kPer * wv + part;
	const unsigned comp = min(own, kC - 1u);   // lanes left over repeat the last component
	float s = 0.0f, c = 0.0f;
	__syncthreads();
	for (unsigned t = 0; t < tiles; ++t) {
		const float* in = &s_term[t & 1u][comp][0][il];
		const unsigned n = min(N - t * kJ, kJ);
		if (n == kJ) {
			float v[kAhead], w[kAhead];
#pragma unroll
			for (unsigned u = 0; u < kAhead; ++u) v[u] = in[u * I];
#pragma unroll
			for (unsigned k = 0; k < kJ; k += kAhead) {
				if (k + kAhead < kJ) {
#pragma unroll
					for (unsigned u = 0; u < kAhead; ++u) w[u] = in[(k + kAhead + u) * I];
				}
#pragma unroll
				for (unsigned u = 0; u < kAhead; ++u) md.step(comp, s, c, v[u]);
#pragma unroll
				for (unsigned u = 0; u < kAhead; ++u) v[u] = w[u];
			}
		} else {
			for (unsigned k = 0; k < n; ++k) md.step(comp, s, c, in[k * I]);
		}
		__syncthreads();
	}
	if (i < N && own < kC) md.store(i, comp, s);
}

}  // namespace chain

#endif
