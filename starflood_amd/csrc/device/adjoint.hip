// adjoint.hip -- vector-Jacobian product of the softened PP force and the
// vector pieces of the adjoint KDK step (no reference counterpart).
//
// Force: a_i = c_i sum_j m_j (x_j - x_i) / s_ij^3, s^2 = |x_i - x_j|^2 + eps^2,
// with c_i = G (physical accelerations) or G m_i (the reference's
// force-like acc).  With d = x_k - x_j and K(d) = I/s^3 - 3 d d^T / s^5,
// the VJP g = (da/dx)^T mu is
//     g_k = G sum_j K(d_kj) (m_k nu_j - m_j nu_k),
// nu = mu (physical) or m mu (reference), since d a_i / d x_i =
// -c_i sum_j m_j K(d_ij) and d a_i / d x_k = c_i m_k K(d_ik).  The pair term
// w = m_k nu_j - m_j nu_k is formed from two rounded products, so the self
// pair (j = k, where K = I/eps^3 is largest) cancels exactly.
//
// Per pair: 26 VALU operations and one v_rsq_f32 (the force takes 13), with
// the same layout as pp.hip's kernel of small states: one lane per k, tiles of
// 64 j staged in LDS, j split over wavefronts, Kahan-folded sums per tile, and
// a fixed-order FP64 combine.  Tiles of one mass form w = m (nu_j - nu_k)
// instead (23 VALU operations; still exactly zero for j == k), scaling each
// tile's sums by m.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "pp_sym.h"

namespace {

constexpr unsigned kBlock = 256;

__device__ __forceinline__ void kahan_add(float& s, float& c, float x) {
	const float y = x - c;
	const float t = s + y;
	const float z = t - s;
	c = z - y;
	s = t;
}

// Pairs of k with a tile's 64 bodies and weights in LDS, read by every lane.
// UNIFORM: every mass of the tile and of k is the same, and the sums leave it
// out.
template <bool UNIFORM>
__device__ __forceinline__ void vjp_tile(const float4* __restrict__ body, const float4* __restrict__ nu,
                                         const float4& bk, const float4& nk, float eps2, float& tx, float& ty,
                                         float& tz) {
#pragma unroll 8
	for (unsigned j = 0; j < kSymTile; ++j) {
		const float4 bj = body[j], nj = nu[j];
		const float dx = bk.x - bj.x, dy = bk.y - bj.y, dz = bk.z - bj.z;
		float r2 = __builtin_fmaf(dx, dx, eps2);
		r2 = __builtin_fmaf(dy, dy, r2);
		r2 = __builtin_fmaf(dz, dz, r2);
		const float inv = __builtin_amdgcn_rsqf(r2);
		const float inv2 = inv * inv;
		const float inv3 = inv2 * inv;
		const float i5_3 = inv3 * (3.0f * inv2);
		// exactly zero when j == k: a difference of equal values, or of two
		// equal rounded products
		const float wx = UNIFORM ? nj.x - nk.x : bk.w * nj.x - bj.w * nk.x;
		const float wy = UNIFORM ? nj.y - nk.y : bk.w * nj.y - bj.w * nk.y;
		const float wz = UNIFORM ? nj.z - nk.z : bk.w * nj.z - bj.w * nk.z;
		const float dw = __builtin_fmaf(dz, wz, __builtin_fmaf(dy, wy, dx * wx));
		const float q = i5_3 * dw;
		tx = __builtin_fmaf(-q, dx, __builtin_fmaf(inv3, wx, tx));
		ty = __builtin_fmaf(-q, dy, __builtin_fmaf(inv3, wy, ty));
		tz = __builtin_fmaf(-q, dz, __builtin_fmaf(inv3, wz, tz));
	}
}

// body = (x, y, z, m) and nu = (nu, 0) for n_pad entries (m = nu = 0 past N).
// Block b owns 64 k (the same in its wavefronts) and a j slice, as k_pp_few.
// With the j stream in scalar loads a VJP with its launches and the wait for it
// took 64 us up to 1000 bodies, 54 at 3000 and 67 at 6000; now 33, 40 and 61.
constexpr unsigned kVjpWaves = kBlock / 64;
__global__ __launch_bounds__(kBlock) void k_vjp(const float4* __restrict__ body, const float4* __restrict__ nu,
                                                unsigned n_pad, unsigned slices, unsigned per, float eps2,
                                                double4* __restrict__ part) {
	__shared__ float4 s_body[kVjpWaves][2][kSymTile], s_nu[kVjpWaves][2][kSymTile];
	__shared__ double red[kVjpWaves][3][64];
	const unsigned sl = blockIdx.x % slices;
	const unsigned lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const unsigned k = (blockIdx.x / slices) * 64u + lane;
	const unsigned j0 = min((sl * kVjpWaves + wv) * per * kSymTile, n_pad), j1 = min(j0 + per * kSymTile, n_pad);
	const float4 bk = body[k], nk = nu[k], zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	float4 vb = j0 < j1 ? body[j0 + lane] : zero, vn = j0 < j1 ? nu[j0 + lane] : zero;
	const float mu = body[0].w;
	const bool k_uni = __ballot(__float_as_uint(bk.w) != __float_as_uint(mu)) == 0ull;
	float sum[3] = {0.0f, 0.0f, 0.0f}, com[3] = {0.0f, 0.0f, 0.0f};
	unsigned buf = 0u;
	for (unsigned j = j0; j < j1; j += kSymTile) {
		s_body[wv][buf][lane] = vb;
		s_nu[wv][buf][lane] = vn;
		const bool uni = k_uni && __ballot(__float_as_uint(vb.w) != __float_as_uint(mu)) == 0ull;
		if (j + kSymTile < j1) {
			vb = body[j + kSymTile + lane];
			vn = nu[j + kSymTile + lane];
		}
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		float t[3] = {0.0f, 0.0f, 0.0f};
		if (uni) vjp_tile<true>(s_body[wv][buf], s_nu[wv][buf], bk, nk, eps2, t[0], t[1], t[2]);
		else vjp_tile<false>(s_body[wv][buf], s_nu[wv][buf], bk, nk, eps2, t[0], t[1], t[2]);
		const float sc = uni ? mu : 1.0f;
#pragma unroll
		for (int u = 0; u < 3; ++u) kahan_add(sum[u], com[u], sc * t[u]);
		buf ^= 1u;
	}
	// Kahan's compensation holds the negated lost low part
#pragma unroll
	for (int u = 0; u < 3; ++u) red[wv][u][lane] = (double)sum[u] - (double)com[u];
	__syncthreads();
	if (wv != 0) return;
	double4 t = make_double4(red[0][0][lane], red[0][1][lane], red[0][2][lane], 0.0);
#pragma unroll
	for (unsigned q = 1; q < kVjpWaves; ++q) {
		t.x += red[q][0][lane];
		t.y += red[q][1][lane];
		t.z += red[q][2][lane];
	}
	part[(size_t)sl * n_pad + k] = t;
}

// ------------------------------------------------- each pair once (pp_sym.h)
// From kVjpSymMin bodies: w = m_k nu_j - m_j nu_k changes sign with the pair's
// order and K does not, so a pair's term goes to k as it is and to j negated:
// 29 VALU operations and one rsq with equal masses (35 with general ones) for
// both, where the one-sided kernel takes 46 and two (52).  The layout is
// pp_sym.hip's narrow one: 256 k per block, four per lane, the same in its
// four wavefronts, a 64-body tile each, the j sums passed from lane to lane
// through LDS.  Bound by issue: 32 operations and the rsq a pair and
// wavefront, 43 ns at N = 65536 (the model of pp_sym.hip says 38).  One-sided
// -> this, with the combine, us: N = 10007 75 -> 57, 16384 137 -> 110 (general
// masses 160 -> 125), 65536 1884 -> 1422; at 8192 the one-sided kernel's 49 is
// not beaten.  (With float4 planes.  A VJP call with general masses, float4
// planes -> FP64 ones: 10007 76.3 -> 77.7, 16384 137.8 -> 139.5, 65536 1610 ->
// 1647.)
constexpr int kPer = 4;
constexpr unsigned kWaves = kBlock / 64;

// a body's sums in a plane
struct Sum3 {
	double x, y, z;
};
static_assert(sizeof(Sum3) == kVjpRecord, "the planes' bytes");

struct KSet {
	float x[kPer], y[kPer], z[kPer], m[kPer], nx[kPer], ny[kPer], nz[kPer];
	float tx[kPer], ty[kPer], tz[kPer];
};

// At step s lane l meets body (l + s) mod 64; sb, sn and acc hold the tile
// twice over, as in pp_sym.hip.  SYM false: pairs inside the set.
template <bool UNIFORM, bool SYM>
__device__ __forceinline__ void vjp_sym_tile(const float4* __restrict__ sb, const float4* __restrict__ sn,
                                             float4* __restrict__ acc, unsigned lane, float eps2, KSet& a) {
	const float4* bl = sb + lane;
	const float4* nl = sn + lane;
	float4* al = acc + lane;
	float4 nb = bl[0], nn = nl[0];
#pragma unroll 2
	for (unsigned s = 0; s < kSymTile; ++s) {
		float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		if (SYM) o = al[s];
		const float4 b = nb, n = nn;
		nb = bl[s + 1u];   // s = 63: lane + 64, in the second copy
		nn = nl[s + 1u];
		float px = 0.0f, py = 0.0f, pz = 0.0f;
#pragma unroll
		for (int k = 0; k < kPer; ++k) {
			const float dx = a.x[k] - b.x, dy = a.y[k] - b.y, dz = a.z[k] - b.z;
			float r2 = __builtin_fmaf(dx, dx, eps2);
			r2 = __builtin_fmaf(dy, dy, r2);
			r2 = __builtin_fmaf(dz, dz, r2);
			const float inv = __builtin_amdgcn_rsqf(r2);
			const float inv2 = inv * inv;
			const float inv3 = inv2 * inv;
			const float i5_3 = inv3 * (-3.0f * inv2);   // -3 / s^5: every product below accumulates in place
			// exactly zero when j == k, as in vjp_tile
			const float wx = UNIFORM ? n.x - a.nx[k] : a.m[k] * n.x - b.w * a.nx[k];
			const float wy = UNIFORM ? n.y - a.ny[k] : a.m[k] * n.y - b.w * a.ny[k];
			const float wz = UNIFORM ? n.z - a.nz[k] : a.m[k] * n.z - b.w * a.nz[k];
			const float dw = __builtin_fmaf(dz, wz, __builtin_fmaf(dy, wy, dx * wx));
			const float q = i5_3 * dw;
			a.tx[k] = __builtin_fmaf(q, dx, __builtin_fmaf(inv3, wx, a.tx[k]));
			a.ty[k] = __builtin_fmaf(q, dy, __builtin_fmaf(inv3, wy, a.ty[k]));
			a.tz[k] = __builtin_fmaf(q, dz, __builtin_fmaf(inv3, wz, a.tz[k]));
			if (SYM) {   // k's sign; the tile's sums are negated at the end
				px = __builtin_fmaf(q, dx, k ? __builtin_fmaf(inv3, wx, px) : inv3 * wx);
				py = __builtin_fmaf(q, dy, k ? __builtin_fmaf(inv3, wy, py) : inv3 * wy);
				pz = __builtin_fmaf(q, dz, k ? __builtin_fmaf(inv3, wz, pz) : inv3 * wz);
			}
		}
		if (SYM) {
			al[s] = make_float4(o.x + px, o.y + py, o.z + pz, 0.0f);
			__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		}
	}
}

__global__ __launch_bounds__(kBlock, 4) void k_vjp_sym(const float4* __restrict__ body, const float4* __restrict__ nu,
                                                       unsigned n_pad, unsigned S, unsigned d0, unsigned chunks,
                                                       unsigned dchunks, float eps2, Sum3* __restrict__ part_i,
                                                       Sum3* __restrict__ part_j) {
	__shared__ float4 s_mem[kWaves][6u * kSymTile];   // a wavefront's bodies, nu and j sums, then its k sums
	const unsigned t = threadIdx.x, lane = t & 63u;
	const unsigned wv = __builtin_amdgcn_readfirstlane(t >> 6);
	const unsigned per = chunks + dchunks;
	const unsigned ib = blockIdx.x / per, c = blockIdx.x % per;
	const bool sym = c < chunks;
	const unsigned nd = S / 2u - (((S & 1u) || ib < S / 2u) ? 0u : 1u);
	const size_t out = (size_t)c * n_pad + ib * kSymNarrow + t;
	const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	if (sym && d0 + c >= nd) {
		part_i[out] = {0.0, 0.0, 0.0};
		return;
	}
	unsigned jb = sym ? ib + 1u + d0 + c : ib;
	if (jb >= S) jb -= S;
	const unsigned j = jb * kSymNarrow + wv * kSymTile;
	KSet a;
#pragma unroll
	for (int k = 0; k < kPer; ++k) {
		const float4 b = body[ib * kSymNarrow + 64u * k + lane], n = nu[ib * kSymNarrow + 64u * k + lane];
		a.x[k] = b.x;
		a.y[k] = b.y;
		a.z[k] = b.z;
		a.m[k] = b.w;
		a.nx[k] = n.x;
		a.ny[k] = n.y;
		a.nz[k] = n.z;
		a.tx[k] = a.ty[k] = a.tz[k] = 0.0f;
	}
	const float4 vb = body[j + lane], vn = nu[j + lane];
	const float mu = body[0].w;
	bool differs = __float_as_uint(vb.w) != __float_as_uint(mu);
#pragma unroll
	for (int k = 0; k < kPer; ++k) differs |= __float_as_uint(a.m[k]) != __float_as_uint(mu);
	const bool uni = __ballot(differs) == 0ull;
	float4* sb = s_mem[wv];
	float4* sn = sb + 2u * kSymTile;
	float4* acc = sn + 2u * kSymTile;
	sb[lane] = sb[lane + kSymTile] = vb;
	sn[lane] = sn[lane + kSymTile] = vn;
	acc[lane] = acc[lane + kSymTile] = zero;
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
	if (sym) {
		if (uni) vjp_sym_tile<true, true>(sb, sn, acc, lane, eps2, a);
		else vjp_sym_tile<false, true>(sb, sn, acc, lane, eps2, a);
		const float4 p = acc[lane], q = acc[lane + kSymTile];
		const double sc = uni ? -(double)mu : -1.0;
		part_j[(size_t)c * n_pad + j + lane] = {sc * ((double)p.x + (double)q.x), sc * ((double)p.y + (double)q.y),
		                                        sc * ((double)p.z + (double)q.z)};
	} else {
		if (uni) vjp_sym_tile<true, false>(sb, sn, acc, lane, eps2, a);
		else vjp_sym_tile<false, false>(sb, sn, acc, lane, eps2, a);
	}
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
	const float sc = uni ? mu : 1.0f;
#pragma unroll
	for (int k = 0; k < kPer; ++k)
		s_mem[wv][64u * k + lane] = make_float4(sc * a.tx[k], sc * a.ty[k], sc * a.tz[k], 0.0f);
	__syncthreads();
	double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
	for (unsigned w = 0; w < kWaves; ++w) {
		const float4 p = s_mem[w][t];
		sx += (double)p.x;
		sy += (double)p.y;
		sz += (double)p.z;
	}
	part_i[out] = {sx, sy, sz};
}

// What a combine does with g_k: store it, or take the adjoint one step
// further back (backward recursion of host/adjoint.c), which saves the three
// launches of 5 us each that the update, nu and the next bodies took.
struct VjpStore {
	float* g;
	explicit VjpStore(const sf_vjp_epi& e) : g(e.g) {}
	__device__ __forceinline__ void operator()(unsigned k, float gx, float gy, float gz) const {
		g[3u * k + 0u] = gx;
		g[3u * k + 1u] = gy;
		g[3u * k + 2u] = gz;
	}
};

__device__ __forceinline__ float4 weight(float coef, int acc_phys, float m, const float l[3]) {
	const float f = acc_phys ? coef : coef * m;
	return make_float4(f * l[0], f * l[1], f * l[2], 0.0f);
}

struct VjpStep {
	sf_vjp_epi e;
	explicit VjpStep(const sf_vjp_epi& v) : e(v) {}
	__device__ __forceinline__ void operator()(unsigned k, float gx, float gy, float gz) const {
		const float g[3] = {gx, gy, gz};
		float lx[3], lv[3];
#pragma unroll
		for (unsigned u = 0; u < 3u; ++u) {
			lx[u] = g[u] + e.lx[3u * k + u];
			lv[u] = e.lv[3u * k + u];
		}
		if (e.gx0) {   // x_0: done
#pragma unroll
			for (unsigned u = 0; u < 3u; ++u) {
				e.gx0[3u * k + u] = lx[u];
				e.gv0[3u * k + u] = lv[u];
			}
			return;
		}
#pragma unroll
		for (unsigned u = 0; u < 3u; ++u) {
			lv[u] = __builtin_fmaf(e.dt, lx[u], lv[u]);
			e.lx[3u * k + u] = lx[u];
			e.lv[3u * k + u] = lv[u];
		}
		float4* body = reinterpret_cast<float4*>(e.body);
		const float m = body[k].w;
		reinterpret_cast<float4*>(e.nu)[k] = weight(e.coef, e.acc_phys, m, lv);
		if (e.x) body[k] = make_float4(e.x[3u * k], e.x[3u * k + 1u], e.x[3u * k + 2u], m);
	}
};

// g_k = G * sum over slices, in FP64
// A block takes kCombI particles; its wavefronts take the slices s = w,
// w + kCombG, ... (w = wavefront) and wavefront 0 adds their sums in order
// (all lanes of one particle per slice would leave most CUs idle at small N).
constexpr unsigned kCombI = 64;
constexpr unsigned kCombG = kBlock / kCombI;
template <class E>
__global__ __launch_bounds__(kBlock) void k_vjp_combine(const double4* __restrict__ part, unsigned n_pad,
                                                        unsigned slices, unsigned N, double G, E epi) {
	__shared__ double red[kCombG][3][kCombI];
	const unsigned kl = threadIdx.x % kCombI, w = threadIdx.x / kCombI;
	const unsigned k = blockIdx.x * kCombI + kl;   // < n_pad: the grid covers N in kCombI steps
	double sx = 0.0, sy = 0.0, sz = 0.0;
	for (unsigned s = w; s < slices; s += kCombG) {
		const double4 a = part[(size_t)s * n_pad + k];
		sx += a.x;
		sy += a.y;
		sz += a.z;
	}
	red[w][0][kl] = sx;
	red[w][1][kl] = sy;
	red[w][2][kl] = sz;
	__syncthreads();
	if (w != 0 || k >= N) return;
	for (unsigned q = 1; q < kCombG; ++q) {
		sx += red[q][0][kl];
		sy += red[q][1][kl];
		sz += red[q][2][kl];
	}
	epi(k, (float)(G * sx), (float)(G * sy), (float)(G * sz));
}

// The same for a launch's planes of k_vjp_sym (one Sum3 per body and plane,
// the k planes, then the j planes), added to the sums of the launches before
// it (run, when !first), which all but the last keep there.
template <class E>
__global__ __launch_bounds__(kBlock) void k_vjp_sym_combine(const Sum3* __restrict__ part, unsigned n_pad,
                                                            unsigned planes, int first, int last,
                                                            double4* __restrict__ run, unsigned N, double G, E epi) {
	__shared__ double red[kCombG][3][kCombI];
	const unsigned kl = threadIdx.x % kCombI, w = threadIdx.x / kCombI;
	const unsigned k = blockIdx.x * kCombI + kl;   // < n_pad: the grid covers N in kCombI steps
	// the number of sets is even: the last offset's plane reaches the upper half only
	if (last && k < n_pad / 2u) --planes;
	double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll 4
	for (unsigned s = w; s < planes; s += kCombG) {
		const Sum3 a = part[(size_t)s * n_pad + k];
		sx += a.x;
		sy += a.y;
		sz += a.z;
	}
	red[w][0][kl] = sx;
	red[w][1][kl] = sy;
	red[w][2][kl] = sz;
	__syncthreads();
	if (w != 0 || k >= N) return;
	for (unsigned q = 1; q < kCombG; ++q) {
		sx += red[q][0][kl];
		sy += red[q][1][kl];
		sz += red[q][2][kl];
	}
	if (!first) {
		const double4 r = run[k];
		sx += r.x;
		sy += r.y;
		sz += r.z;
	}
	if (!last) {
		run[k] = make_double4(sx, sy, sz, 0.0);
		return;
	}
	epi(k, (float)(G * sx), (float)(G * sy), (float)(G * sz));
}

// nu_i = coef * mu_i (physical) or coef * m_i * mu_i (reference); zero past N
__global__ __launch_bounds__(kBlock) void k_pack_nu(const float* __restrict__ mu, const float* __restrict__ mas,
                                                    unsigned N, unsigned n_pad, float coef, int acc_phys,
                                                    float4* __restrict__ nu) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n_pad) return;
	float l[3] = {0.0f, 0.0f, 0.0f};
	float m = 1.0f;
	if (i < N) {
		m = mas[i];
#pragma unroll
		for (unsigned u = 0; u < 3u; ++u) l[u] = mu[3u * i + u];
	}
	nu[i] = i < N ? weight(coef, acc_phys, m, l) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// The state the forward integration starts from (positions into x too, when set)
__global__ __launch_bounds__(kBlock) void k_adjoint_init(const float* __restrict__ x0, const float* __restrict__ v0,
                                                         unsigned n3, double* __restrict__ x64,
                                                         float* __restrict__ v, float* __restrict__ x) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n3) return;
	const float p = x0[i];
	x64[i] = (double)p;
	v[i] = v0[i];
	if (x) x[i] = p;
}

// A segment from its checkpoint: x[0 .. 3N) its first positions; with steps,
// also the first step's opening kick and drift (EpiKdk's), its positions into
// x[3N .. 6N).  The last positions written go into the packed bodies.
__global__ __launch_bounds__(kBlock) void k_adjoint_reopen(const double* __restrict__ ck_x64,
                                                           const float* __restrict__ ck_v,
                                                           const float* __restrict__ ck_a, unsigned N, float h,
                                                           double dt, int steps, double* __restrict__ x64,
                                                           float* __restrict__ v, float* __restrict__ x,
                                                           float4* __restrict__ body) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= N) return;
	float p[3];
#pragma unroll
	for (unsigned u = 0; u < 3u; ++u) {
		const unsigned k = 3u * i + u;
		double y = ck_x64[k];
		p[u] = (float)y;
		x[k] = p[u];
		if (steps) {
			const float w = __builtin_fmaf(h, ck_a[k], ck_v[k]);
			y = __builtin_fma(dt, (double)w, y);
			p[u] = (float)y;
			v[k] = w;
			x64[k] = y;
			x[3u * (size_t)N + k] = p[u];
		}
	}
	body[i] = make_float4(p[0], p[1], p[2], body[i].w);
}

// The cotangents the backward starts from (NULL: zero), the first VJP's nu
// (zero past N) and its bodies.
__global__ __launch_bounds__(kBlock) void k_adjoint_begin(const float* __restrict__ gx, const float* __restrict__ gv,
                                                          const float* __restrict__ x, unsigned N, unsigned n_pad,
                                                          float coef, int acc_phys, float* __restrict__ lx,
                                                          float* __restrict__ lv, float4* __restrict__ body,
                                                          float4* __restrict__ nu) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n_pad) return;
	if (i >= N) {
		nu[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		return;
	}
	float l[3];
#pragma unroll
	for (unsigned u = 0; u < 3u; ++u) {
		lx[3u * i + u] = gx ? gx[3u * i + u] : 0.0f;
		l[u] = gv ? gv[3u * i + u] : 0.0f;
		lv[3u * i + u] = l[u];
	}
	const float m = body[i].w;
	nu[i] = weight(coef, acc_phys, m, l);
	body[i] = make_float4(x[3u * i], x[3u * i + 1u], x[3u * i + 2u], m);
}

__global__ __launch_bounds__(kBlock) void k_fill0(float* __restrict__ y, unsigned n) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i < n) y[i] = 0.0f;
}

inline dim3 grid(unsigned n) { return dim3((n + kBlock - 1u) / kBlock); }

}  // namespace

extern "C" {

// bytes of part for sfd_force_vjp: k_vjp_sym's planes, or below kVjpSymMin
// bodies k_vjp's
size_t sfd_vjp_part_bytes(unsigned n_pad) {
	return n_pad >= kVjpSymMin ? sym_part_bytes(n_pad, false, kVjpRecord) : (size_t)few_geometry(n_pad).bslices * n_pad * 32u;
}

int sfd_pack_nu(const float* mu, const float* mas, unsigned N, unsigned n_pad, float coef, int acc_phys, float* nu,
                hipStream_t s) {
	if (N == 0) return 0;
	hipLaunchKernelGGL(k_pack_nu, grid(n_pad), dim3(kBlock), 0, s, mu, mas, N, n_pad, coef, acc_phys,
	                   reinterpret_cast<float4*>(nu));
	return sf_hip_check(hipGetLastError(), "sfd_pack_nu", "launch");
}

// g = G sum_j K(d_kj) (m_k nu_j - m_j nu_k), then *epi: body is the packed
// (x, m) array of the force kernel, nu the packed weights (both n_pad float4),
// part scratch of sfd_vjp_part_bytes.
int sfd_force_vjp(const float* body, const float* nu, unsigned N, unsigned n_pad, float eps2, double G, float* part,
                  const sf_vjp_epi* epi, hipStream_t s) {
	if (N == 0) return 0;
	if (n_pad == 0 || n_pad % 1024u != 0) return -1;
	const float4* b4 = reinterpret_cast<const float4*>(body);
	const float4* nu4 = reinterpret_cast<const float4*>(nu);
	const dim3 cgrid((N + kCombI - 1) / kCombI);
	if (n_pad >= kVjpSymMin) {
		const SymGeometry q = sym_geometry(n_pad, false, kVjpRecord);
		Sum3* planes = reinterpret_cast<Sum3*>(part);
		double4* run = reinterpret_cast<double4*>(planes + ((size_t)q.chunks + q.dchunks + q.per_launch) * n_pad);
		for (unsigned d0 = 0; d0 < q.offsets; d0 += q.per_launch) {
			const unsigned ch = d0 + q.per_launch < q.offsets ? q.per_launch : q.offsets - d0;
			const int first = d0 == 0u, last = d0 + ch == q.offsets;
			const unsigned pi = ch + (first ? q.dchunks : 0u);
			const int tok = sf_prof_begin("force_vjp", s);
			hipLaunchKernelGGL(k_vjp_sym, dim3(q.blocks * pi), dim3(kBlock), 0, s, b4, nu4, n_pad, q.blocks, d0, ch,
			                   pi - ch, eps2, planes, planes + (size_t)pi * n_pad);
			sf_prof_end(tok, s);
			if (epi->step)
				hipLaunchKernelGGL(k_vjp_sym_combine<VjpStep>, cgrid, dim3(kBlock), 0, s, planes, n_pad, pi + ch, first,
				                   last, run, N, G, VjpStep(*epi));
			else
				hipLaunchKernelGGL(k_vjp_sym_combine<VjpStore>, cgrid, dim3(kBlock), 0, s, planes, n_pad, pi + ch, first,
				                   last, run, N, G, VjpStore(*epi));
		}
		return sf_hip_check(hipGetLastError(), "sfd_force_vjp", "launch");
	}
	const FewGeometry g = few_geometry(n_pad);
	double4* p8 = reinterpret_cast<double4*>(part);
	const int tok = sf_prof_begin("force_vjp", s);
	hipLaunchKernelGGL(k_vjp, dim3((n_pad / 64u) * g.bslices), dim3(kBlock), 0, s, b4, nu4, n_pad, g.bslices, g.per, eps2,
	                   p8);
	sf_prof_end(tok, s);
	if (epi->step)
		hipLaunchKernelGGL(k_vjp_combine<VjpStep>, cgrid, dim3(kBlock), 0, s, p8, n_pad, g.bslices, N, G,
		                   VjpStep(*epi));
	else
		hipLaunchKernelGGL(k_vjp_combine<VjpStore>, cgrid, dim3(kBlock), 0, s, p8, n_pad, g.bslices, N, G,
		                   VjpStore(*epi));
	return sf_hip_check(hipGetLastError(), "sfd_force_vjp", "launch");
}

int sfd_adjoint_init(const float* x0, const float* v0, unsigned N, double* x64, float* v, float* x, hipStream_t s) {
	hipLaunchKernelGGL(k_adjoint_init, grid(3u * N), dim3(kBlock), 0, s, x0, v0, 3u * N, x64, v, x);
	return sf_hip_check(hipGetLastError(), "sfd_adjoint_init", "launch");
}

int sfd_adjoint_reopen(const double* ck_x64, const float* ck_v, const float* ck_a, unsigned N, float h, double dt,
                       int steps, double* x64, float* v, float* x, float* body, hipStream_t s) {
	hipLaunchKernelGGL(k_adjoint_reopen, grid(N), dim3(kBlock), 0, s, ck_x64, ck_v, ck_a, N, h, dt, steps, x64, v, x,
	                   reinterpret_cast<float4*>(body));
	return sf_hip_check(hipGetLastError(), "sfd_adjoint_reopen", "launch");
}

int sfd_adjoint_begin(const float* gx, const float* gv, const float* x, unsigned N, unsigned n_pad, float coef,
                      int acc_phys, float* lx, float* lv, float* body, float* nu, hipStream_t s) {
	hipLaunchKernelGGL(k_adjoint_begin, grid(n_pad), dim3(kBlock), 0, s, gx, gv, x, N, n_pad, coef, acc_phys, lx, lv,
	                   reinterpret_cast<float4*>(body), reinterpret_cast<float4*>(nu));
	return sf_hip_check(hipGetLastError(), "sfd_adjoint_begin", "launch");
}

int sfd_fill0(float* y, unsigned n, hipStream_t s) {
	if (n == 0) return 0;
	hipLaunchKernelGGL(k_fill0, grid(n), dim3(kBlock), 0, s, y, n);
	return sf_hip_check(hipGetLastError(), "sfd_fill0", "launch");
}

}  // extern "C"
