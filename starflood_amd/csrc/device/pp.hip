// pp.hip -- particle-particle gravity on gfx950.
//
// Two kernels compute the same quantity as the reference's
// solve_gravity_part_part (src/gravity.c:666-819):
//   sum_i = sum_j m_j r_ij / (r_ij^2 + eps^2)^(3/2),  r_ij = r_i - r_j
//   acc_i = -G m_i sum_i   (SF_ACC_REFERENCE)   or  -G sum_i (SF_ACC_PHYSICAL)
//   pot_i = -G sum_j m_j / sqrt(r_ij^2 + eps^2)
// with the self pair included (its force term is zero, its potential term is
// -G m_i / eps), as the reference does.
//
// k_pp_exact keeps the reference's FP32 operation order (no contraction: the
// file is compiled with -ffp-contract=off; the IEEE quotients' and square
// root's bits; per-pair Kahan; j in index order), so its output is
// bit-identical to the CPU path.  The terms of a tile of j are made by some of
// a block's wavefronts while others run the chains of sums.
//
// k_pp_few is the throughput kernel of small states (from kSymMin bodies
// pp_sym.hip evaluates each pair once): 13 VALU operations plus one v_rsq_f32
// per interaction, one i per lane, tiles of 64 j staged in LDS, their plain
// partial sums folded into a Kahan-compensated running sum, and the j range
// split over wavefronts so that the grid fills the CUs.  Where a tile's masses
// all have the bits of the first body's, the per-pair mass product is left out
// and the tile's sums are scaled before the fold.  A block's four wavefronts
// hold the same 64 particles; their sums meet in LDS in FP64, in wavefront
// order, so a block writes one double4 per particle.
// A second kernel adds the slice partials per i in fixed order in FP64,
// which keeps the result deterministic.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "bodies.h"
#include "exact_pp.h"
#include "force_epi.h"
#include "pp_sym.h"

namespace {

constexpr unsigned kBlock = 256;

// One step of Kahan summation (reference src/gravity.c:771-784):
// y = x - c; t = s + y; c = (t - s) - y; s = t.
__device__ __forceinline__ void kahan_add(float& s, float& c, float x) {
	const float y = x - c;
	const float t = s + y;
	const float z = t - s;
	c = z - y;
	s = t;
}

template <unsigned I, bool KAHAN_ACC, bool KAHAN_POT, bool PHYS>
__global__ __launch_bounds__((chain::block_size<I, 4>())) void k_pp_exact(const float* __restrict__ pos,
                                                                        const float* __restrict__ mas, unsigned N,
                                                                        float eps2, float negG,
                                                                        float* __restrict__ acc,
                                                                        float* __restrict__ pot) {
	chain::run<I>(chain::ExactPP<KAHAN_ACC, KAHAN_POT, PHYS>{pos, mas, eps2, negG, acc, pot}, N);
}

template <unsigned I>
void launch_exact(int sel, const float* pos, const float* mas, unsigned N, float eps2, float negG, float* acc,
                  float* pot, hipStream_t s) {
	auto k = k_pp_exact<I, true, true, true>;
	switch (sel) {
	case 0: k = k_pp_exact<I, false, false, false>; break;
	case 1: k = k_pp_exact<I, false, false, true>; break;
	case 2: k = k_pp_exact<I, false, true, false>; break;
	case 3: k = k_pp_exact<I, false, true, true>; break;
	case 4: k = k_pp_exact<I, true, false, false>; break;
	case 5: k = k_pp_exact<I, true, false, true>; break;
	case 6: k = k_pp_exact<I, true, true, false>; break;
	default: break;
	}
	hipLaunchKernelGGL(k, dim3((N + I - 1) / I), dim3(chain::block_size<I, 4>()), 0, s, pos, mas, N, eps2, negG, acc,
	                   pot);
}

// Interactions with a tile's 64 bodies q in LDS, read by every lane.  UNIFORM:
// every mass is the same, and the sums leave it out.
template <bool WITH_POT, bool UNIFORM>
__device__ __forceinline__ void few_tile(const float4* __restrict__ q, float xi, float yi, float zi, float eps2,
                                         float& tx, float& ty, float& tz, float& tp) {
#pragma unroll 16
	for (unsigned k = 0; k < kSymTile; ++k) {
		const float4 bj = q[k];
		const float dx = bj.x - xi;
		const float dy = bj.y - yi;
		const float dz = bj.z - zi;
		float r2 = __builtin_fmaf(dx, dx, eps2);
		r2 = __builtin_fmaf(dy, dy, r2);
		r2 = __builtin_fmaf(dz, dz, r2);
		const float inv = __builtin_amdgcn_rsqf(r2);
		const float mi = UNIFORM ? inv : bj.w * inv;
		const float inv2 = inv * inv;
		const float w = mi * inv2;
		tx = __builtin_fmaf(w, dx, tx);
		ty = __builtin_fmaf(w, dy, ty);
		tz = __builtin_fmaf(w, dz, tz);
		if (WITH_POT) tp += mi;
	}
}

// Block b owns the 64 particles i of i-block b / slices (one per lane, the
// same in each of its wavefronts) and j slice b % slices, of which each
// wavefront takes `per` consecutive tiles.
// Bound by a wavefront's chain at small sizes (a lone wavefront issues one
// instruction in 2.5 ns) and by issue from about 6000 bodies on.  With the j
// stream in scalar loads, four bodies ahead of their use, each wavefront waited
// for most of them, 24 us whatever the size; now 6.7 us at 1000 bodies, 8.3 at
// 3000, 19.5 at 6000, 28 at 8192.  With the bodies read from the caller's arrays
// a force up to 1000 bodies takes 22.8 us instead of 44, 3000 24.6, 6000 34.1
// (42.8), 9216 47.6 (54.3).
constexpr unsigned kWavesPP = kBlock / 64;
template <bool WITH_POT, class L>
__global__ __launch_bounds__(kBlock) void k_pp_few(const L bodies, unsigned n_pad, unsigned slices, unsigned per,
                                                   float eps2, double4* __restrict__ part) {
	__shared__ float4 s_j[kWavesPP][2][kSymTile];
	__shared__ double red[kWavesPP][4][64];
	const unsigned s = blockIdx.x % slices;
	const unsigned lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const unsigned i = (blockIdx.x / slices) * 64u + lane;
	const unsigned j0 = min((s * kWavesPP + wv) * per * kSymTile, n_pad), j1 = min(j0 + per * kSymTile, n_pad);
	const float4 bi = bodies(i);
	float4 v = j0 < j1 ? bodies(j0 + lane) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	const float mu = bodies.mass(0u);
	float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f}, com[4] = {0.0f, 0.0f, 0.0f, 0.0f};
	unsigned buf = 0u;
	for (unsigned j = j0; j < j1; j += kSymTile) {
		s_j[wv][buf][lane] = v;
		const bool uni = __ballot(__float_as_uint(v.w) != __float_as_uint(mu)) == 0ull;
		if (j + kSymTile < j1) v = bodies(j + kSymTile + lane);
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
		if (uni) few_tile<WITH_POT, true>(s_j[wv][buf], bi.x, bi.y, bi.z, eps2, t[0], t[1], t[2], t[3]);
		else few_tile<WITH_POT, false>(s_j[wv][buf], bi.x, bi.y, bi.z, eps2, t[0], t[1], t[2], t[3]);
		const float sc = uni ? mu : 1.0f;
#pragma unroll
		for (int u = 0; u < (WITH_POT ? 4 : 3); ++u) kahan_add(sum[u], com[u], sc * t[u]);
		buf ^= 1u;
	}
	// Kahan's compensation c holds the negated lost low part: each sum is s - c
#pragma unroll
	for (int u = 0; u < 4; ++u) red[wv][u][lane] = (double)sum[u] - (double)com[u];
	__syncthreads();
	if (wv != 0) return;
	double4 t = make_double4(red[0][0][lane], red[0][1][lane], red[0][2][lane], red[0][3][lane]);
#pragma unroll
	for (unsigned q = 1; q < kWavesPP; ++q) {
		t.x += red[q][0][lane];
		t.y += red[q][1][lane];
		t.z += red[q][2][lane];
		t.w += red[q][3][lane];
	}
	part[(size_t)s * n_pad + i] = t;
}

// Fixed-order FP64 sum of the slice partials.  A block takes kCombI
// particles; its wavefronts take the slices s = g, g + kCombG, ... (g =
// wavefront), each lane one particle (coalesced loads), and wavefront 0
// adds the kCombG sums in order.  One lane per particle over all slices
// left most CUs idle at small N (64 blocks at N = 16384: 20 us).
constexpr unsigned kCombI = 64;
constexpr unsigned kCombG = kBlock / kCombI;
template <class E, class L>
__global__ __launch_bounds__(kBlock) void k_pp_combine(const double4* __restrict__ part, unsigned n_pad,
                                                       unsigned slices, const L bodies, float4* body, unsigned N,
                                                       double G, int acc_phys, E epi) {
	__shared__ double red[kCombG][4][kCombI];
	const unsigned il = threadIdx.x % kCombI, g = threadIdx.x / kCombI;
	const unsigned i = blockIdx.x * kCombI + il;   // < n_pad: the grid covers N in kCombI steps
	double sx = 0.0, sy = 0.0, sz = 0.0, sp = 0.0;
	for (unsigned s = g; s < slices; s += kCombG) {
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
	for (unsigned q = 1; q < kCombG; ++q) {
		sx += red[q][0][il];
		sy += red[q][1][il];
		sz += red[q][2][il];
		sp += red[q][3][il];
	}
	// sum_j m_j (r_j - r_i)/s^3 = -sum_j m_j r_ij/s^3, so acc = G (m_i) * sum
	const double f = acc_phys ? G : G * (double)bodies.mass(i);
	epi(i, (float)(f * sx), (float)(f * sy), (float)(f * sz), (float)(-G * sp), body);
}

// Packs (x, y, z, m) per body, padding with zeros to n_pad.  KICK: first the
// opening kick and drift of the fast step, with k_kick_drift_fast's operations
// (x64 restarts from pos where they differ).
template <bool KICK>
__global__ __launch_bounds__(kBlock) void k_pack_bodies(float* __restrict__ vel, const float* __restrict__ acc,
                                                        double* __restrict__ x64, float* __restrict__ pos,
                                                        const float* __restrict__ mas, unsigned N, unsigned n_pad,
                                                        float half_dt, double dt, float4* __restrict__ body) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n_pad) return;
	if (i >= N) {
		body[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		return;
	}
	float p[3] = {pos[3u * i], pos[3u * i + 1u], pos[3u * i + 2u]};
	if (KICK) {
#pragma unroll
		for (unsigned k = 0; k < 3u; ++k) {
			const float v = __builtin_fmaf(half_dt, acc[3u * i + k], vel[3u * i + k]);
			double x0 = x64[3u * i + k];
			if ((float)x0 != p[k]) x0 = (double)p[k];
			const double x = __builtin_fma(dt, (double)v, x0);
			vel[3u * i + k] = v;
			x64[3u * i + k] = x;
			p[k] = (float)x;
			pos[3u * i + k] = p[k];
		}
	}
	body[i] = make_float4(p[0], p[1], p[2], mas[i]);
}

// FP64 direct sum: one block per listed particle, lanes stride over j, then
// a fixed-shape tree reduction in LDS.
__global__ __launch_bounds__(kBlock) void k_pp_f64(const float* __restrict__ pos, const float* __restrict__ mas,
                                                   unsigned N, double eps2, double G, int acc_phys,
                                                   const unsigned* __restrict__ idx,
                                                   double* __restrict__ acc, double* __restrict__ pot) {
	__shared__ double red[4][kBlock];
	const unsigned i = idx[blockIdx.x];
	const double xi = pos[3u * i], yi = pos[3u * i + 1u], zi = pos[3u * i + 2u];
	double sx = 0.0, sy = 0.0, sz = 0.0, sp = 0.0;
	for (unsigned j = threadIdx.x; j < N; j += kBlock) {
		const double rx = xi - (double)pos[3u * j];
		const double ry = yi - (double)pos[3u * j + 1u];
		const double rz = zi - (double)pos[3u * j + 2u];
		const double s2 = rx * rx + ry * ry + rz * rz + eps2;
		const double inv1 = 1.0 / sqrt(s2);
		const double pj = (double)mas[j] * inv1;
		const double w = pj * inv1 * inv1;
		sx += w * rx;
		sy += w * ry;
		sz += w * rz;
		sp += pj;
	}
	red[0][threadIdx.x] = sx;
	red[1][threadIdx.x] = sy;
	red[2][threadIdx.x] = sz;
	red[3][threadIdx.x] = sp;
	__syncthreads();
	for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
		if (threadIdx.x < h) {
#pragma unroll
			for (int q = 0; q < 4; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + h];
		}
		__syncthreads();
	}
	if (threadIdx.x == 0) {
		const double f = acc_phys ? -G : -G * (double)mas[i];
		acc[3u * blockIdx.x + 0u] = f * red[0][0];
		acc[3u * blockIdx.x + 1u] = f * red[1][0];
		acc[3u * blockIdx.x + 2u] = f * red[2][0];
		pot[blockIdx.x] = -G * red[3][0];
	}
}


}  // namespace

template <bool KICK>
static void launch_pack(float* vel, const float* acc, double* x64, float* pos, const float* mas, unsigned N,
                        unsigned n_pad, float half_dt, double dt, float* body, hipStream_t s) {
	hipLaunchKernelGGL(k_pack_bodies<KICK>, dim3((n_pad + kBlock - 1) / kBlock), dim3(kBlock), 0, s, vel, acc, x64, pos,
	                   mas, N, n_pad, half_dt, dt, reinterpret_cast<float4*>(body));
}

extern "C" int sfd_pack_bodies(const float* pos, const float* mas, unsigned N, unsigned n_pad, float* body,
                               hipStream_t s) {
	launch_pack<false>(nullptr, nullptr, nullptr, const_cast<float*>(pos), mas, N, n_pad, 0.0f, 0.0, body, s);
	return sf_hip_check(hipGetLastError(), "sfd_pack_bodies", "k_pack_bodies launch");
}

extern "C" int sfd_kick_drift_pack(float* vel, const float* acc, double* x64, float* pos, const float* mas, unsigned N,
                                   unsigned n_pad, float half_dt, double dt, float* body, hipStream_t s) {
	const int tok = sf_prof_begin("kick_drift", s);
	launch_pack<true>(vel, acc, x64, pos, mas, N, n_pad, half_dt, dt, body, s);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_kick_drift_pack", "k_pack_bodies launch");
}

extern "C" int sfd_pp_exact(const float* pos, const float* mas, unsigned N, float eps2, float negG, int acc_phys,
                            int kahan_acc, int kahan_pot, float* acc, float* pot, hipStream_t s) {
	if (N == 0) return 0;
	const int sel = (kahan_acc ? 4 : 0) | (kahan_pot ? 2 : 0) | (acc_phys ? 1 : 0);
	const int tok = sf_prof_begin("pp_exact", s);
	if (N <= chain::kFewN) launch_exact<32>(sel, pos, mas, N, eps2, negG, acc, pot, s);
	else launch_exact<64>(sel, pos, mas, N, eps2, negG, acc, pot, s);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_pp_exact", "k_pp_exact launch");
}

extern "C" size_t sfd_pp_part_bytes(unsigned n_pad) { return pp_part_bytes(n_pad); }

// device/pp_sym.hip
extern "C" int sfd_pp_sym(const float* pos, const float* mas, float* body, unsigned N, unsigned n_pad, float eps2,
                          double G, int acc_phys, float* part, const sf_force_epi* epi, hipStream_t s);

extern "C" int sfd_pp_fast(const float* pos, const float* mas, float* body, unsigned N, unsigned n_pad, float eps2,
                           double G, int acc_phys, float* part, const sf_force_epi* epi, hipStream_t s) {
	if (N == 0) return 0;
	if (n_pad % 1024u != 0 || N > n_pad || (pos != nullptr) != (epi->kind == SF_EPI_STORE)) {
		sf_error("sfd_pp_fast", "n_pad %u does not fit N = %u, or the bodies what they are for", n_pad, N);
		return -1;
	}
	// part holds sfd_pp_part_bytes(n_pad)
	if (n_pad >= kSymMin) {
		if (pos && sym_pp_wide(n_pad)) {
			if (sfd_pack_bodies(pos, mas, N, n_pad, body, s)) return -1;
			pos = mas = nullptr;
		}
		return sfd_pp_sym(pos, mas, body, N, n_pad, eps2, G, acc_phys, part, epi, s);
	}
	const FewGeometry g = few_geometry(n_pad);
	const dim3 grid((n_pad / 64u) * g.bslices), cgrid((N + kCombI - 1) / kCombI);
	double4* p4 = reinterpret_cast<double4*>(part);
	float4* b4 = reinterpret_cast<float4*>(body);
	const PackedBodies packed{b4};
	const ArrayBodies arrays{pos, mas, N};
	const bool pot = epi->kind == SF_EPI_KICK || (epi->kind == SF_EPI_STORE && epi->pot);
	const int tok = sf_prof_begin("pp_fast", s);
	if (pos) {
		auto k = pot ? k_pp_few<true, ArrayBodies> : k_pp_few<false, ArrayBodies>;
		hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, s, arrays, n_pad, g.bslices, g.per, eps2, p4);
	} else {
		auto k = pot ? k_pp_few<true, PackedBodies> : k_pp_few<false, PackedBodies>;
		hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, s, packed, n_pad, g.bslices, g.per, eps2, p4);
	}
	sf_prof_end(tok, s);
	if (sf_hip_check(hipGetLastError(), "sfd_pp_fast", "k_pp_few launch")) return -1;
	const int tok2 = sf_prof_begin("pp_combine", s);
	if (epi->kind == SF_EPI_KICK)
		hipLaunchKernelGGL((k_pp_combine<EpiKick, PackedBodies>), cgrid, dim3(kBlock), 0, s, p4, n_pad, g.bslices, packed,
		                   b4, N, G, acc_phys, EpiKick(*epi));
	else if (epi->kind == SF_EPI_KDK)
		hipLaunchKernelGGL((k_pp_combine<EpiKdk, PackedBodies>), cgrid, dim3(kBlock), 0, s, p4, n_pad, g.bslices, packed,
		                   b4, N, G, acc_phys, EpiKdk(*epi));
	else
		hipLaunchKernelGGL((k_pp_combine<EpiStore, ArrayBodies>), cgrid, dim3(kBlock), 0, s, p4, n_pad, g.bslices, arrays,
		                   b4, N, G, acc_phys, EpiStore(*epi));
	sf_prof_end(tok2, s);
	return sf_hip_check(hipGetLastError(), "sfd_pp_fast", "k_pp_combine launch");
}

extern "C" int sfd_pp_f64(const float* pos, const float* mas, unsigned N, double eps2, double G, int acc_phys,
                          const unsigned* idx, unsigned n_idx, double* acc, double* pot, hipStream_t s) {
	if (n_idx == 0) return 0;
	const int tok = sf_prof_begin("pp_f64", s);
	hipLaunchKernelGGL(k_pp_f64, dim3(n_idx), dim3(kBlock), 0, s, pos, mas, N, eps2, G, acc_phys, idx, acc, pot);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_pp_f64", "k_pp_f64 launch");
}
