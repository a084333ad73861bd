// pp_sym.hip -- particle-particle gravity that evaluates each pair once.
//
// The distance, 1/s and 1/s^3 of a pair serve both of its bodies: with equal
// masses 16 VALU operations and one v_rsq_f32 for two interactions, where the
// one-sided kernel (pp.hip) takes 24 and two (general masses: 19 and one
// against 26 and two).  Every term has the one-sided kernel's bits.
//
// A body's sum.  In FP32 are added, plainly, its terms with the j of two tiles
// (128, the one-sided kernel's two), which Kahan's steps then collect, and as j
// its terms with a wavefront's 256 i: 64 sums of four at most, 67 roundings in a
// row.  Everything further is FP64: the wavefronts' sums, the planes, the
// combine.  With float4 planes a body's sum was rounded to 24 bits once per plane
// (193 of them at N = 262144); the FP64 ones cost 1 % there (12.71 -> 12.85 ms a
// step), 2.5 % at 65536, and 57 -> 60 us at 10007.
//
// What bounds it.  Measured on gfx950 with two or more wavefronts per SIMD:
// a wave64 FP32 operation on VGPRs issues every 0.95-1.05 ns (1.17 for the
// 8-byte v_fma_f32), v_rsq_f32 costs 5 to 6 in such a mix, and an
// instruction stream with a DPP operand falls to half that rate.  16
// operations and the rsq are 21 ns per pair and wavefront; the kernel takes
// 24 at N = 262144, against 2 x 15.8 for the one-sided kernel at its own
// bound.  So:
//  * i in registers, four per lane: the j side costs 4 adds and 3 LDS
//    accesses per four pairs.  Eight per lane (fewer wavefronts) and two
//    (more j work) were slower (12.7-13.7 and 15.4 ms against 12.7).
//  * the j sums move from lane to lane through LDS, one 16-byte read and
//    write a step.  Rotating them with DPP took 15.0 ms, adding them with
//    LDS atomics 171 ms (ds_add_f32 runs at a few lanes per cycle).
//  * a step's j record is read one step ahead: 12.9 -> 12.7 ms, and 8 % at
//    N = 10007, where fewer wavefronts hide the LDS latency.
//
// Kernel and combine, one-sided -> this, same box, with float4 planes (FP64 ones:
// above): N = 262144 17.3 -> 13.4 ms (another box 17.0 -> 12.7; general masses
// 18.0 -> 15.6), N = 65536 1085 -> 863 us, N = 16384 80 -> 67 us (general masses
// 83 -> 76), N = 10007 42 -> 35.
// The rest of its time at N = 16384 (54 us at the large-N rate) is the last
// wavefronts of 2112 blocks on 1024 slots, and the combine.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "bodies.h"
#include "force_epi.h"
#include "pp_sym.h"

namespace {

constexpr unsigned kBlock = 256;
constexpr unsigned kWaves = kBlock / 64;
constexpr int kPer = 4;                  // i per lane
constexpr unsigned kSet = 64u * kPer;    // i per wavefront
static_assert(kSet * kWaves == kSymWide && kSet == kSymNarrow, "the layouts' set sizes");
static_assert(kSymTile == 64u, "lane l starts at the tile's body l");

__device__ __forceinline__ void kahan_add(float& s, float& c, float x) {
	const float y = x - c;
	const float t = s + y;
	const float z = t - s;
	c = z - y;
	s = t;
}

// The lane's i and their plain FP32 sums over up to 128 j.
struct Set {
	float x[kPer], y[kPer], z[kPer], m[kPer];
	float tx[kPer], ty[kPer], tz[kPer], tp[kPer];

	__device__ __forceinline__ void clear() {
#pragma unroll
		for (int k = 0; k < kPer; ++k) tx[k] = ty[k] = tz[k] = tp[k] = 0.0f;
	}
	template <class L>
	__device__ __forceinline__ void load(const L& bodies, unsigned i0) {
#pragma unroll
		for (int k = 0; k < kPer; ++k) {
			const float4 b = bodies(i0 + 64u * k);
			x[k] = b.x;
			y[k] = b.y;
			z[k] = b.z;
			m[k] = b.w;
		}
		clear();
	}
	// every mass of the wavefront's i has the bits of mu
	__device__ __forceinline__ bool all_mass(float mu) const {
		bool d = false;
#pragma unroll
		for (int k = 0; k < kPer; ++k) d |= __float_as_uint(m[k]) != __float_as_uint(mu);
		return __ballot(d) == 0ull;
	}
};

// One tile: at step s, lane l meets body (l + s) mod 64.  sj holds the tile
// twice over, so that the address is the lane's own plus a constant; acc
// holds the running j sums the same way (the two copies are added at the
// end).  LDS operations of a wavefront complete in order, so a step's read of
// acc[l + s] follows the write that lane l + 1 made in the step before.
// SYM false leaves the j side out (pairs inside the i-block, seen from both
// ends).  UNIFORM: every mass is the same, and left out.
template <bool POT, bool UNIFORM, bool SYM>
__device__ __forceinline__ void sym_tile(const float4* __restrict__ sj, float4* __restrict__ acc, unsigned lane,
                                         float eps2, Set& a) {
	const float4* sl = sj + lane;
	float4* al = acc + lane;
	float4 nb = sl[0];
#pragma unroll 4
	for (unsigned s = 0; s < kSymTile; ++s) {
		float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		if (SYM) o = al[s];
		const float4 b = nb;
		nb = sl[s + 1u];   // s = 63: lane + 64, in the second copy
		float dx[kPer], dy[kPer], dz[kPer], inv[kPer];
#pragma unroll
		for (int k = 0; k < kPer; ++k) {
			dx[k] = b.x - a.x[k];
			dy[k] = b.y - a.y[k];
			dz[k] = b.z - a.z[k];
			inv[k] = __builtin_fmaf(dx[k], dx[k], eps2);
			inv[k] = __builtin_fmaf(dy[k], dy[k], inv[k]);
			inv[k] = __builtin_fmaf(dz[k], dz[k], inv[k]);
			inv[k] = __builtin_amdgcn_rsqf(inv[k]);
		}
		float px = 0.0f, py = 0.0f, pz = 0.0f, pp = 0.0f;
#pragma unroll
		for (int k = 0; k < kPer; ++k) {
			const float inv2 = inv[k] * inv[k];
			const float pj = UNIFORM ? inv[k] : b.w * inv[k];
			const float w = pj * inv2;
			a.tx[k] = __builtin_fmaf(w, dx[k], a.tx[k]);
			a.ty[k] = __builtin_fmaf(w, dy[k], a.ty[k]);
			a.tz[k] = __builtin_fmaf(w, dz[k], a.tz[k]);
			if (POT) a.tp[k] += pj;
			if (SYM) {
				const float pi = UNIFORM ? inv[k] : a.m[k] * inv[k];
				const float v = UNIFORM ? w : pi * inv2;
				px = k ? __builtin_fmaf(v, dx[k], px) : v * dx[k];
				py = k ? __builtin_fmaf(v, dy[k], py) : v * dy[k];
				pz = k ? __builtin_fmaf(v, dz[k], pz) : v * dz[k];
				if (POT) pp = k ? pp + pi : pi;
			}
		}
		if (SYM) {
			al[s] = make_float4(o.x + px, o.y + py, o.z + pz, o.w + pp);
			__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		}
	}
}

// Wide layout.  The block's four wavefronts hold a quarter each of its set
// of 1024 i and take the same tiles; their j sums meet in FP64 after each
// tile, in wavefront order.
template <bool POT>
__global__ __launch_bounds__(kBlock, 4) void k_pp_sym(const float4* __restrict__ body, unsigned n_pad, unsigned S,
                                                      unsigned d0, unsigned d1, unsigned tiles, unsigned chunks,
                                                      unsigned dchunks, float eps2, double4* __restrict__ part_i,
                                                      double* __restrict__ part_j) {
	__shared__ float4 s_j[2][2u * kSymTile];
	__shared__ float4 s_acc[2][kWaves][2u * kSymTile];
	const unsigned t = threadIdx.x, lane = t & 63u;
	const unsigned wv = __builtin_amdgcn_readfirstlane(t >> 6);
	// set ib against the bodies [t0, t1) counted from its first partner's
	// (or, in the blocks that come last, its own) first body, modulo n_pad
	const unsigned nsym = S * chunks;
	const bool sym = blockIdx.x < nsym;
	const unsigned e = sym ? blockIdx.x : blockIdx.x - nsym;
	const unsigned per = sym ? chunks : dchunks;
	const unsigned ib = e / per, c = e % per;
	const unsigned nd = S / 2u - (((S & 1u) || ib < S / 2u) ? 0u : 1u);
	const unsigned limit = sym ? (min(d1, nd) > d0 ? (min(d1, nd) - d0) * kSymWide : 0u) : kSymWide;
	const unsigned t0 = min(c * tiles * kSymTile, limit), t1 = min(t0 + tiles * kSymTile, limit);
	unsigned j = (sym ? (ib + 1u + d0) * kSymWide : ib * kSymWide) + t0;   // < 2 n_pad
	if (j >= n_pad) j -= n_pad;
	const unsigned i0 = ib * kSymWide + wv * kSet + lane;
	Set a;
	a.load(PackedBodies{body}, i0);
	float sum[kPer][4], com[kPer][4];
	bool pending = false, was_uni = false;   // plain sums not yet folded, and their kind
#pragma unroll
	for (int k = 0; k < kPer; ++k)
#pragma unroll
		for (int u = 0; u < 4; ++u) sum[k][u] = com[k][u] = 0.0f;
	const float mu = body[0].w;
	// one answer for the block: its wavefronts' j sums are added before they are scaled
	const bool i_uni = !__syncthreads_or(!a.all_mass(mu));
	for (unsigned u = t; u < 2u * kWaves * 2u * kSymTile; u += kBlock)
		(&s_acc[0][0][0])[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	if (t < kSymTile && t0 < t1) {
		const float4 v = body[j + t];
		s_j[0][t] = v;
		s_j[0][t + kSymTile] = v;
	}
	__syncthreads();
	auto fold = [&](bool uni) {
		const float sc = uni ? mu : 1.0f;
#pragma unroll
		for (int k = 0; k < kPer; ++k) {
			kahan_add(sum[k][0], com[k][0], sc * a.tx[k]);
			kahan_add(sum[k][1], com[k][1], sc * a.ty[k]);
			kahan_add(sum[k][2], com[k][2], sc * a.tz[k]);
			if (POT) kahan_add(sum[k][3], com[k][3], sc * a.tp[k]);
		}
		a.clear();
		pending = false;
	};
	unsigned buf = 0u;
	for (unsigned tt = t0; tt < t1; tt += kSymTile) {
		// the next tile, in flight during this one's arithmetic (past the
		// range's end it is not used, but in bounds)
		unsigned jn = j + kSymTile;
		if (jn >= n_pad) jn -= n_pad;
		float4 nv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		if (t < kSymTile) nv = body[jn + t];
		const bool uni = i_uni && __ballot(__float_as_uint(s_j[buf][lane].w) != __float_as_uint(mu)) == 0ull;
		if (pending && uni != was_uni) fold(was_uni);
		was_uni = uni;
		if (sym) {
			if (uni) sym_tile<POT, true, true>(s_j[buf], s_acc[buf][wv], lane, eps2, a);
			else sym_tile<POT, false, true>(s_j[buf], s_acc[buf][wv], lane, eps2, a);
		} else {
			if (uni) sym_tile<POT, true, false>(s_j[buf], s_acc[buf][wv], lane, eps2, a);
			else sym_tile<POT, false, false>(s_j[buf], s_acc[buf][wv], lane, eps2, a);
		}
		if (t < kSymTile) {
			s_j[buf ^ 1u][t] = nv;
			s_j[buf ^ 1u][t + kSymTile] = nv;
		}
		__syncthreads();
		if (sym) {
			// thread (j, component): the four wavefronts' sums, both copies,
			// cleared for the tile after next
			const unsigned comp = t & 3u, jl = t >> 2;
			float* r = reinterpret_cast<float*>(&s_acc[buf][0][jl]) + comp;
			double s = 0.0;
#pragma unroll
			for (unsigned w = 0; w < 2u * kWaves; ++w) {
				s += (double)r[4u * kSymTile * w];
				r[4u * kSymTile * w] = 0.0f;
			}
			// the j side of m w (r_j - r_i) has the opposite sign
			const double sc = uni ? (double)mu : 1.0;
			part_j[((size_t)(tt / kSymWide) * n_pad + j) * 4u + t] = comp < 3u ? -sc * s : sc * s;
		}
		// fold the i sums after two tiles of one kind
		pending = !pending;
		if (!pending) fold(uni);
		buf ^= 1u;
		j = jn;
	}
	if (pending) fold(was_uni);
	const unsigned plane = sym ? c : chunks + c;
#pragma unroll
	for (int k = 0; k < kPer; ++k)   // Kahan's compensation holds the negated lost low part
		part_i[(size_t)plane * n_pad + i0 + 64u * k] =
		    make_double4((double)sum[k][0] - (double)com[k][0], (double)sum[k][1] - (double)com[k][1],
		                 (double)sum[k][2] - (double)com[k][2], (double)sum[k][3] - (double)com[k][3]);
}

// Narrow layout.  The block's four wavefronts hold the same 256 i and take
// one tile each: chunk c < chunks is the set at offset d0 + c (a plane of
// zeros where an even S leaves it out), chunk `chunks` the set itself.  j and
// the j sums are each wavefront's own, so nothing waits until the four
// wavefronts' i sums meet in LDS at the end.
// One tile per wavefront needs no compensated sums: 94 VGPRs, 5 per SIMD (4
// and 6 measured the same).
template <bool POT, class L>
__global__ __launch_bounds__(kBlock, 5) void k_pp_sym_narrow(const L bodies, unsigned n_pad, unsigned S,
                                                             unsigned d0, unsigned chunks, unsigned dchunks,
                                                             float eps2, double4* __restrict__ part_i,
                                                             double4* __restrict__ part_j) {
	__shared__ float4 s_mem[kWaves][4u * kSymTile];   // a wavefront's j and j sums, then its i sums
	static_assert(kSet == 4u * kSymTile, "the i sums take the place of j and the j sums");
	const unsigned t = threadIdx.x, lane = t & 63u;
	const unsigned wv = __builtin_amdgcn_readfirstlane(t >> 6);
	const unsigned per = chunks + dchunks;
	const unsigned ib = blockIdx.x / per, c = blockIdx.x % per;
	const bool sym = c < chunks;
	const unsigned nd = S / 2u - (((S & 1u) || ib < S / 2u) ? 0u : 1u);
	const size_t out = (size_t)c * n_pad + ib * kSymNarrow + t;
	if (sym && d0 + c >= nd) {
		part_i[out] = make_double4(0.0, 0.0, 0.0, 0.0);
		return;
	}
	unsigned jb = sym ? ib + 1u + d0 + c : ib;
	if (jb >= S) jb -= S;
	const unsigned j = jb * kSymNarrow + wv * kSymTile;
	Set a;
	a.load(bodies, ib * kSymNarrow + lane);
	const float4 v = bodies(j + lane), zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	const float mu = bodies.mass(0u);
	const bool uni = a.all_mass(mu) && __ballot(__float_as_uint(v.w) != __float_as_uint(mu)) == 0ull;
	float4* sj = s_mem[wv];
	float4* acc = sj + 2u * kSymTile;
	sj[lane] = sj[lane + kSymTile] = v;
	acc[lane] = acc[lane + kSymTile] = zero;
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
	if (sym) {
		if (uni) sym_tile<POT, true, true>(sj, acc, lane, eps2, a);
		else sym_tile<POT, false, true>(sj, acc, lane, eps2, a);
		const float4 p = acc[lane], q = acc[lane + kSymTile];
		const double sc = uni ? (double)mu : 1.0;
		part_j[(size_t)c * n_pad + j + lane] =
		    make_double4(-sc * ((double)p.x + (double)q.x), -sc * ((double)p.y + (double)q.y),
		                 -sc * ((double)p.z + (double)q.z), sc * ((double)p.w + (double)q.w));
	} else {
		if (uni) sym_tile<POT, true, false>(sj, acc, lane, eps2, a);
		else sym_tile<POT, false, false>(sj, acc, lane, eps2, a);
	}
	// one tile: its plain sums need no compensation
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
	const float sc = uni ? mu : 1.0f;
#pragma unroll
	for (int k = 0; k < kPer; ++k)
		s_mem[wv][64u * k + lane] = make_float4(sc * a.tx[k], sc * a.ty[k], sc * a.tz[k], sc * a.tp[k]);
	__syncthreads();
	double sx = 0.0, sy = 0.0, sz = 0.0, sp = 0.0;
#pragma unroll
	for (unsigned w = 0; w < kWaves; ++w) {
		const float4 p = s_mem[w][t];
		sx += (double)p.x;
		sy += (double)p.y;
		sz += (double)p.z;
		sp += (double)p.w;
	}
	part_i[out] = make_double4(sx, sy, sz, sp);
}

// Fixed-order FP64 sum of a launch's planes (the i planes, then the j
// planes), added to the sums of the launches before it (run, when !first) and
// kept there or, at the last launch, written to acc and pot.  A block takes
// 64 particles; its wavefronts take every fourth plane each.
constexpr unsigned kCombI = 64;
template <class E, class L>
__global__ __launch_bounds__(kBlock) void k_sym_combine(const double4* __restrict__ part, unsigned n_pad,
                                                        unsigned planes, unsigned S, int last_offset, int first,
                                                        int last, double4* __restrict__ run, const L bodies,
                                                        float4* body, unsigned N, double G, int acc_phys, E epi) {
	__shared__ double red[kWaves][4][kCombI];
	const unsigned il = threadIdx.x % kCombI, g = threadIdx.x / kCombI;
	const unsigned i = blockIdx.x * kCombI + il;   // < n_pad: the grid covers N in kCombI steps
	// for even S the last offset's plane reaches the upper half of the blocks only
	if (last_offset && !(S & 1u) && i < n_pad / 2u) --planes;
	double sx = 0.0, sy = 0.0, sz = 0.0, sp = 0.0;
#pragma unroll 4
	for (unsigned s = g; s < planes; s += kWaves) {
		const double4 a = part[(size_t)s * n_pad + i];
		sx += a.x;
		sy += a.y;
		sz += a.z;
		sp += a.w;
	}
	red[g][0][il] = sx;
	red[g][1][il] = sy;
	red[g][2][il] = sz;
	red[g][3][il] = sp;
	__syncthreads();
	if (g != 0 || i >= N) return;
	for (unsigned q = 1; q < kWaves; ++q) {
		sx += red[q][0][il];
		sy += red[q][1][il];
		sz += red[q][2][il];
		sp += red[q][3][il];
	}
	if (!first) {
		const double4 r = run[i];
		sx += r.x;
		sy += r.y;
		sz += r.z;
		sp += r.w;
	}
	if (!last) {
		run[i] = make_double4(sx, sy, sz, sp);
		return;
	}
	const double f = acc_phys ? G : G * (double)bodies.mass(i);
	epi(i, (float)(f * sx), (float)(f * sy), (float)(f * sz), (float)(-G * sp), body);
}

struct CombineArgs {
	const double4* part;
	unsigned n_pad, planes, S;
	int first, last;
	double4* run;
	float4* body;
	unsigned N;
	double G;
	int acc_phys;
};
template <class E, class L>
void launch_combine(const CombineArgs& c, const L& bodies, const sf_force_epi& epi, hipStream_t s) {
	hipLaunchKernelGGL((k_sym_combine<E, L>), dim3((c.N + kCombI - 1u) / kCombI), dim3(kBlock), 0, s, c.part, c.n_pad,
	                   c.planes, c.S, c.last, c.first, c.last, c.run, bodies, c.body, c.N, c.G, c.acc_phys, E(epi));
}

}  // namespace

// The force of n_pad bodies (a multiple of 1024, at least 2048), ended by *epi:
// in the narrow layout SF_EPI_STORE's of the caller's arrays, else of the packed
// bodies (pos NULL); part holds sym_part_bytes(n_pad, sym_pp_wide(n_pad), kPpRecord).
extern "C" int sfd_pp_sym(const float* pos, const float* mas, float* body, unsigned N, unsigned n_pad, float eps2,
                          double G, int acc_phys, float* part, const sf_force_epi* epi, hipStream_t s) {
	if (N == 0) return 0;
	const bool wide = sym_pp_wide(n_pad);
	if (n_pad % kSymWide != 0 || n_pad < 2u * kSymWide || N > n_pad ||
	    (pos != nullptr) != (!wide && epi->kind == SF_EPI_STORE)) {
		sf_error("sfd_pp_sym", "n_pad %u does not fit N = %u, or the bodies what they are for", n_pad, N);
		return -1;
	}
	const SymGeometry g = sym_geometry(n_pad, wide, kPpRecord);
	float4* b4 = reinterpret_cast<float4*>(body);
	const PackedBodies packed{b4};
	const ArrayBodies arrays{pos, mas, N};
	const bool pot = epi->kind == SF_EPI_KICK || (epi->kind == SF_EPI_STORE && epi->pot);
	double4* p4 = reinterpret_cast<double4*>(part);
	double4* run = p4 + ((size_t)g.chunks + g.dchunks + g.per_launch) * n_pad;
	for (unsigned d0 = 0; d0 < g.offsets; d0 += g.per_launch) {
		const unsigned d1 = d0 + g.per_launch < g.offsets ? d0 + g.per_launch : g.offsets;
		const int first = d0 == 0u, last = d1 == g.offsets;
		const unsigned ch = wide ? g.chunks : d1 - d0;
		const unsigned dch = first ? g.dchunks : 0u;   // the sets themselves go with the first launch
		const unsigned pi = ch + dch;
		double4* pj = p4 + (size_t)pi * n_pad;
		const dim3 grid(g.blocks * pi);
		const int tok = sf_prof_begin("pp_fast", s);
		if (wide) {
			auto k = pot ? k_pp_sym<true> : k_pp_sym<false>;
			hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, s, b4, n_pad, g.blocks, d0, d1, g.tiles, ch, dch, eps2, p4,
			                   reinterpret_cast<double*>(pj));
		} else if (epi->kind == SF_EPI_STORE) {
			auto k = pot ? k_pp_sym_narrow<true, ArrayBodies> : k_pp_sym_narrow<false, ArrayBodies>;
			hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, s, arrays, n_pad, g.blocks, d0, ch, dch, eps2, p4, pj);
		} else {
			auto k = pot ? k_pp_sym_narrow<true, PackedBodies> : k_pp_sym_narrow<false, PackedBodies>;
			hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, s, packed, n_pad, g.blocks, d0, ch, dch, eps2, p4, pj);
		}
		sf_prof_end(tok, s);
		if (sf_hip_check(hipGetLastError(), "sfd_pp_sym", "k_pp_sym launch")) return -1;
		const int tok2 = sf_prof_begin("pp_combine", s);
		const CombineArgs ca{p4, n_pad, pi + (d1 - d0), g.blocks, first, last, run, b4, N, G, acc_phys};
		if (epi->kind == SF_EPI_KICK) launch_combine<EpiKick>(ca, packed, *epi, s);
		else if (epi->kind == SF_EPI_KDK) launch_combine<EpiKdk>(ca, packed, *epi, s);
		else if (pos) launch_combine<EpiStore>(ca, arrays, *epi, s);
		else launch_combine<EpiStore>(ca, packed, *epi, s);
		sf_prof_end(tok2, s);
		if (sf_hip_check(hipGetLastError(), "sfd_pp_sym", "k_sym_combine launch")) return -1;
	}
	return 0;
}
