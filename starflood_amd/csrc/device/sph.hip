// sph.hip -- smoothed-particle hydrodynamics sums, all pairs (PP SPH).
//
// SF_SPH_REFERENCE: the reference's model (src/sph.c:14-283) in its
// operation order -- Gaussian kernel W = (1/(sqrt(pi) h))^3 exp(-r^2/h^2),
// rho_i = sum_j 0.5 (W_i + W_j) m_j over every j, polytrope P = (0.1 rho)^2,
// and acc_i += -m_i sum_{r^2 <= 1} (P_i/rho_i^2 + P_j/rho_j^2) 0.5 (n_i + n_j) r_ij
// with n = -2 exp(-r^2/h^2) / (pi^{3/2} h^5).  The file is compiled with
// -ffp-contract=off, and every product, quotient and Kahan step rounds as the
// reference's does; the per-particle factors that do not depend on the pair
// ((a^2) a, h h, pi^{3/2} h^5 and P/rho^2) are computed once per particle with
// the same operations, which gives the same bits.  exp() is the device library's (faithfully rounded,
// like glibc's expf, but not always the same float) and (0.1 rho)^2 is the
// correctly rounded product where glibc's powf is off by one ulp in about
// 0.07% of cases: results agree with the reference to a few ulp, not bit
// for bit.
//
// SF_SPH_CUBIC_IDEAL: cubic spline W(r, h) = 8/(pi h^3) {1 - 6q^2 + 6q^3,
// q <= 1/2; 2 (1-q)^3, q <= 1} (support radius h, GADGET-2 convention), the
// symmetrised kernel 0.5 (W(r, h_i) + W(r, h_j)), ideal gas P = (gamma-1) rho u,
// acc_i += -s_i sum_j m_j (P_i/rho_i^2 + P_j/rho_j^2) grad_i W and
// du_i/dt = 0.5 sum_j m_j (P_i/rho_i^2 + P_j/rho_j^2) v_ij . grad_i W, where
// s_i = 1 for physical accelerations and m_i for the reference's force-like
// acc.  The j stream of packed records is wavefront-uniform, so the compiler
// reads it through scalar loads; lanes with no neighbour skip the kernel
// arithmetic.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "exact_pp.h"
#include "order_chain.h"

namespace {

constexpr unsigned kBlock = 256;
constexpr unsigned kTj = 128;   // j per unrolled tile of the cubic-model passes

// the reference's constants (src/common.h:18, :29), rounded to float as
// (real)INV_SQRT_PI and (real)INV_POW_PI_3_2 are; the second one's value
// is pi^{3/2}
constexpr float kInvSqrtPi = (float)0.56418958354775628694807945156077258584405062932900;
constexpr float kPiPow32 = (float)5.5683279968317078452848179821188357020136243902832;
constexpr float kPi = 3.14159265358979323846f;

// ------------------------------------------------------------ reference model
// The density and force sums run on order_chain.h: terms made in parallel,
// added in index order.  N = 6000 (us): density 1524 and force 2246 with one
// lane per particle and IEEE divisions in line, now 94 and 132.  Bound by the
// chains (12 ns a body for the density, 17 for the force, whose chains also
// test for skipped pairs) while the particles fit 32 to a CU, then by the
// makers.

// RN(a / b) from inv = RN(1 / b): the quotient's estimate corrected once by
// its residual (Markstein 1990), for normal b and quotients that neither
// overflow nor vanish.  Compared with a / b on 1.7e10 operand pairs.
__device__ __forceinline__ float divide_by(float a, float b, float inv) {
	const float q = a * inv;
	return __builtin_fmaf(__builtin_fmaf(-q, b, a), inv, q);
}
// the divisors for which that holds with room for every numerator here; the
// others' inverse is set to NaN, which sends their pairs to IEEE divisions
__device__ __forceinline__ bool divisor_ok(float b) { return b >= 0x1p-60f && b <= 0x1p60f; }
constexpr unsigned kQuotTop = 0x71800000u;    // 2^100: larger quotients, inf and NaN take IEEE divisions
constexpr unsigned kSkipBits = 0x7FBADBADu;   // a term that is not added (a NaN no operation returns)

// Records: a = (x, y, z, m), h = (h h, 1 / (h h), a3, -), d = (h h, 1 / (h h),
// den, 1 / den) with a3 = (a a) a, a = INV_SQRT_PI / h (src/sph.c:116-119) and
// den = INV_POW_PI_3_2 h h h h h evaluated left to right (src/sph.c:239-240).
__global__ __launch_bounds__(kBlock) void k_tables_ref(const float* __restrict__ pos, const float* __restrict__ mas,
                                                       const float* __restrict__ rad, unsigned N,
                                                       float4* __restrict__ ra, float4* __restrict__ rh,
                                                       float4* __restrict__ rd) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= N) return;
	const float h = rad[i];
	const float a = kInvSqrtPi / h;
	const float hh = h * h, den = kPiPow32 * h * h * h * h * h;
	const bool ok = divisor_ok(hh) && divisor_ok(den);
	const float ihh = ok ? 1.0f / hh : __builtin_nanf("");
	ra[i] = make_float4(pos[3u * i], pos[3u * i + 1u], pos[3u * i + 2u], mas[i]);
	rh[i] = make_float4(hh, ihh, a * a * a, 0.0f);
	rd[i] = make_float4(hh, ihh, den, 1.0f / den);
}

struct QuotCheck {
	unsigned top = 0u;
	__device__ bool bad() const { return top >= kQuotTop; }
};

// exp(-r2 / h h) for both smoothing lengths of a pair
template <bool FAST>
__device__ __forceinline__ void gauss_pair(float r2, float hi, float ihi, float hj, float ihj, float& ei, float& ej,
                                           QuotCheck& chk) {
	float qi, qj;
	if (FAST) {
		qi = divide_by(r2, hi, ihi);
		qj = divide_by(r2, hj, ihj);
		chk.top = max(chk.top, max(__float_as_uint(qi), __float_as_uint(qj)));   // r2 >= 0
	} else {
		qi = r2 / hi;
		qj = r2 / hj;
	}
	ei = expf(-qi);
	ej = expf(-qj);
}

// src/sph.c:35-145
template <bool KAHAN>
struct RhoRef {
	static constexpr unsigned kComps = 1;
	const float4* __restrict__ ra;
	const float4* __restrict__ rh;
	float* __restrict__ rho;
	struct Body {
		float4 a, h;
	};
	using Self = Body;
	using Check = QuotCheck;
	__device__ bool fast() const { return true; }
	__device__ Self self(unsigned i) const { return {ra[i], rh[i]}; }
	__device__ __forceinline__ Body body(unsigned j, unsigned off) const { return {(ra + j)[off], (rh + j)[off]}; }
	template <bool FAST>
	__device__ __forceinline__ void terms(const Self& i, const Body& j, float (&out)[1], Check& chk) const {
		const float rx = i.a.x - j.a.x, ry = i.a.y - j.a.y, rz = i.a.z - j.a.z;
		const float r2 = (rx * rx) + (ry * ry) + (rz * rz);
		float ei, ej;
		gauss_pair<FAST>(r2, i.h.x, i.h.y, j.h.x, j.h.y, ei, ej, chk);
		const float wi = i.h.z * ei, wj = j.h.z * ej;
		out[0] = 0.5f * (wi + wj) * j.a.w;
	}
	__device__ __forceinline__ void step(unsigned, float& s, float& c, float x) const {
		if (KAHAN) chain::kahan(s, c, x);
		else s += x;
	}
	__device__ void store(unsigned i, unsigned, float s) const { rho[i] = s; }
};

template <unsigned I, bool KAHAN>
__global__ __launch_bounds__((chain::block_size<I, 1>())) void k_rho_ref(const float4* __restrict__ ra,
                                                                       const float4* __restrict__ rh, unsigned N,
                                                                       float* __restrict__ rho) {
	chain::run<I>(RhoRef<KAHAN>{ra, rh, rho}, N);
}

// The density (blockIdx.y 0) beside the gravity that the force is added to
// (blockIdx.y 1), which do not need each other.  Up to 4096 particles their
// blocks fit one to a CU and overlap; a CU with one of each takes as long as
// one after the other.  Solve, apart -> together (us): 512 particles 50.7 ->
// 42.6, 2000 120 -> 95, 4096 214 -> 166, 4100 216 -> 207, 4600 239 -> 229, 5200
// 267 both, 6000 303 -> 305, 8192 403 -> 408.  Hence kTogetherN.
constexpr unsigned kTogetherN = 5120;
static_assert(kTogetherN <= chain::kFewN, "32 particles a block");

template <bool KAHAN_ACC, bool KAHAN_POT, bool PHYS>
__global__ __launch_bounds__((chain::block_size<32, 4>())) void k_rho_pp_ref(
    const float4* __restrict__ ra, const float4* __restrict__ rh, float* __restrict__ rho, const float* __restrict__ pos,
    const float* __restrict__ mas, unsigned N, float eps2, float negG, float* __restrict__ acc, float* __restrict__ pot) {
	constexpr unsigned kWaves = chain::block_size<32, 4>() / 64u;
	if (blockIdx.y == 0u) chain::run<32, kWaves>(RhoRef<KAHAN_ACC>{ra, rh, rho}, N);
	else chain::run<32>(chain::ExactPP<KAHAN_ACC, KAHAN_POT, PHYS>{pos, mas, eps2, negG, acc, pot}, N);
}

void launch_rho_pp(const sf_exact_pp* g, const float4* ra, const float4* rh, float* rho, const float* pos,
                   const float* mas, unsigned N, float* acc, hipStream_t s) {
	auto k = k_rho_pp_ref<true, true, true>;
	switch ((g->kahan_acc ? 4 : 0) | (g->kahan_pot ? 2 : 0) | (g->acc_phys ? 1 : 0)) {
	case 0: k = k_rho_pp_ref<false, false, false>; break;
	case 1: k = k_rho_pp_ref<false, false, true>; break;
	case 2: k = k_rho_pp_ref<false, true, false>; break;
	case 3: k = k_rho_pp_ref<false, true, true>; break;
	case 4: k = k_rho_pp_ref<true, false, false>; break;
	case 5: k = k_rho_pp_ref<true, false, true>; break;
	case 6: k = k_rho_pp_ref<true, true, false>; break;
	default: break;
	}
	hipLaunchKernelGGL(k, dim3((N + 31u) / 32u, 2), dim3(chain::block_size<32, 4>()), 0, s, ra, rh, rho, pos, mas, N,
	                   g->eps2, g->neg_g, acc, g->pot);
}

// P = (K rho)^(1/n + 1) with K = 0.1, n = 1 (src/sph.c:147-157), and the
// momentum-equation factor P / rho^2 (src/sph.c:189-192, :225-226), which
// takes the mass's place in the record
__global__ __launch_bounds__(kBlock) void k_eos_ref(const float* __restrict__ rho, unsigned N,
                                                    float* __restrict__ prs, float4* __restrict__ ra) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= N) return;
	const float x = 0.100f * rho[i];
	const float p = x * x;
	prs[i] = p;
	const float r2 = rho[i] * rho[i];
	ra[i].w = 0.0f < r2 ? p / r2 : 0.0f;
}

// src/sph.c:163-276.  Pairs with r2 > 1 are not added; their chains see
// kSkipBits.  2 exp / den: the numerator is scaled by 2^64 so that the
// residual of a tiny quotient does not vanish.
template <bool KAHAN>
struct ForceRef {
	static constexpr unsigned kComps = 3;
	const float4* __restrict__ ra;
	const float4* __restrict__ rd;
	const float* __restrict__ mas;
	float* __restrict__ acc;
	struct Body {
		float4 a, d;
	};
	using Self = Body;
	using Check = QuotCheck;
	__device__ bool fast() const { return true; }
	__device__ Self self(unsigned i) const { return {ra[i], rd[i]}; }
	__device__ __forceinline__ Body body(unsigned j, unsigned off) const { return {(ra + j)[off], (rd + j)[off]}; }
	template <bool FAST>
	__device__ __forceinline__ void terms(const Self& i, const Body& j, float (&out)[3], Check& chk) const {
		const float rx = i.a.x - j.a.x, ry = i.a.y - j.a.y, rz = i.a.z - j.a.z;
		const float r2 = (rx * rx) + (ry * ry) + (rz * rz);
		float ei, ej, ni, nj;
		gauss_pair<FAST>(r2, i.d.x, i.d.y, j.d.x, j.d.y, ei, ej, chk);
		if (FAST) {
			ni = divide_by(-0x1p65f * ei, i.d.z, i.d.w) * 0x1p-64f;
			nj = divide_by(-0x1p65f * ej, j.d.z, j.d.w) * 0x1p-64f;
		} else {
			ni = -2.0f * ei / i.d.z;
			nj = -2.0f * ej / j.d.z;
		}
		const float g = 0.5f * (ni + nj);
		const float cc = i.a.w + j.a.w;
		const float skip = __uint_as_float(kSkipBits);
		const bool far = r2 > 1.0f;
		out[0] = far ? skip : cc * (g * rx);
		out[1] = far ? skip : cc * (g * ry);
		out[2] = far ? skip : cc * (g * rz);
	}
	__device__ __forceinline__ void step(unsigned, float& s, float& c, float x) const {
		const bool add = __float_as_uint(x) != kSkipBits;
		float s1 = s, c1 = c;
		if (KAHAN) chain::kahan(s1, c1, x);
		else s1 += x;
		s = add ? s1 : s;
		c = add ? c1 : c;
	}
	__device__ void store(unsigned i, unsigned comp, float s) const { acc[3u * i + comp] += -mas[i] * s; }
};

template <unsigned I, bool KAHAN>
__global__ __launch_bounds__((chain::block_size<I, 3>())) void k_force_ref(const float4* __restrict__ ra,
                                                                         const float4* __restrict__ rd,
                                                                         const float* __restrict__ mas, unsigned N,
                                                                         float* __restrict__ acc) {
	chain::run<I>(ForceRef<KAHAN>{ra, rd, mas, acc}, N);
}

template <unsigned I, bool KAHAN>
void launch_ref(const sf_exact_pp* gravity, const float4* ra, const float4* rh, const float4* rd, const float* pos,
                const float* mas, unsigned N, float* rho, float* prs, float4* ra_con, float* acc, hipStream_t s) {
	const dim3 g((N + I - 1u) / I);
	if (gravity) launch_rho_pp(gravity, ra, rh, rho, pos, mas, N, acc, s);
	else hipLaunchKernelGGL((k_rho_ref<I, KAHAN>), g, dim3(chain::block_size<I, 1>()), 0, s, ra, rh, N, rho);
	hipLaunchKernelGGL(k_eos_ref, dim3((N + kBlock - 1u) / kBlock), dim3(kBlock), 0, s, rho, N, prs, ra_con);
	hipLaunchKernelGGL((k_force_ref<I, KAHAN>), g, dim3(chain::block_size<I, 3>()), 0, s, ra, rd, mas, N, acc);
}

// ---------------------------------------------------------------- cubic model
// Packed per-particle records (n_pad entries, zero past N):
//   q0 = (x, y, z, h^2), q1 = (m, 1/h, u_pred, P/rho^2), q2 = (v_pred, 0).
// v_pred = v + pred_dt acc and u_pred = u + pred_dt du/dt predict the
// half-kicked state to the end of the step (pred_dt = 0 takes it as it is).
__global__ __launch_bounds__(kBlock) void k_pack_cubic(const float* __restrict__ pos, const float* __restrict__ vel,
                                                       const float* __restrict__ acc, const float* __restrict__ mas,
                                                       const float* __restrict__ rad, const float* __restrict__ u,
                                                       const float* __restrict__ dudt, unsigned N, unsigned n_pad,
                                                       float pred_dt, float4* __restrict__ q0,
                                                       float4* __restrict__ q1, float4* __restrict__ q2) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n_pad) return;
	if (i >= N) {
		const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		q0[i] = z;
		q1[i] = z;
		q2[i] = z;
		return;
	}
	const float h = rad[i];
	q0[i] = make_float4(pos[3u * i], pos[3u * i + 1u], pos[3u * i + 2u], h * h);
	q1[i] = make_float4(mas[i], 1.0f / h, __builtin_fmaf(pred_dt, dudt[i], u[i]), 0.0f);
	q2[i] = make_float4(__builtin_fmaf(pred_dt, acc[3u * i], vel[3u * i]),
	                    __builtin_fmaf(pred_dt, acc[3u * i + 1u], vel[3u * i + 1u]),
	                    __builtin_fmaf(pred_dt, acc[3u * i + 2u], vel[3u * i + 2u]), 0.0f);
}

// W(r, h) and dW/dr(r, h) of the cubic spline for 0 <= q = r/h
__device__ __forceinline__ float cubic_w(float q, float inv_h) {
	const float k = (8.0f / kPi) * inv_h * inv_h * inv_h;
	const float t = 1.0f - q;
	const float inner = __builtin_fmaf(6.0f * q * q, q - 1.0f, 1.0f);
	return q <= 0.5f ? k * inner : (q <= 1.0f ? k * 2.0f * t * t * t : 0.0f);
}
__device__ __forceinline__ float cubic_dw(float q, float inv_h) {
	const float k = (8.0f / kPi) * inv_h * inv_h * inv_h * inv_h;
	const float t = 1.0f - q;
	const float inner = q * __builtin_fmaf(18.0f, q, -12.0f);
	return q <= 0.5f ? k * inner : (q <= 1.0f ? k * -6.0f * t * t : 0.0f);
}

// Both passes split j into slices over the grid (slice = blockIdx % slices,
// as the fast PP kernel does) so that a few thousand particles still give
// every SIMD several wavefronts; the neighbour test is 8 VALU operations per
// pair and the kernel arithmetic runs only for lanes with a neighbour.
__global__ __launch_bounds__(kBlock) void k_rho_cubic(const float4* __restrict__ q0, const float4* __restrict__ q1,
                                                      unsigned n_pad, unsigned slices, unsigned slice_len,
                                                      float* __restrict__ part) {
	const unsigned b = blockIdx.x;
	const unsigned sl = b % slices;
	const unsigned i = (b / slices) * kBlock + threadIdx.x;
	const float4 a = q0[i];
	const float inv_hi = q1[i].y;
	float s = 0.0f;
	const unsigned j0 = sl * slice_len;
	const unsigned j1 = min(j0 + slice_len, n_pad);
	for (unsigned jt = j0; jt < j1; jt += kTj) {
#pragma unroll 8
		for (unsigned j = jt; j < jt + kTj; ++j) {
			const float4 b4 = q0[j];
			const float dx = a.x - b4.x, dy = a.y - b4.y, dz = a.z - b4.z;
			const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
			if (r2 < fmaxf(a.w, b4.w)) {
				const float4 c = q1[j];
				const float r = __builtin_sqrtf(r2);
				const float w = cubic_w(r * inv_hi, inv_hi) + cubic_w(r * c.y, c.y);
				s = __builtin_fmaf(0.5f * c.x, w, s);
			}
		}
	}
	part[(size_t)sl * n_pad + i] = s;
}

// rho = sum of the slice partials in fixed order; P = (gamma - 1) rho u;
// P / rho^2 into q1.w for the force pass
__global__ __launch_bounds__(kBlock) void k_rho_cubic_combine(const float* __restrict__ part, unsigned n_pad,
                                                              unsigned slices, unsigned N, float gm1,
                                                              float4* __restrict__ q1, float* __restrict__ rho,
                                                              float* __restrict__ prs) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= N) return;
	double s = 0.0;
	for (unsigned k = 0; k < slices; ++k) s += (double)part[(size_t)k * n_pad + i];
	const float r = (float)s;
	float4 c = q1[i];
	const float p = gm1 * r * c.z;
	c.w = r > 0.0f ? p / (r * r) : 0.0f;
	q1[i] = c;
	rho[i] = r;
	prs[i] = p;
}

__global__ __launch_bounds__(kBlock) void k_force_cubic(const float4* __restrict__ q0, const float4* __restrict__ q1,
                                                        const float4* __restrict__ q2, unsigned n_pad, unsigned slices,
                                                        unsigned slice_len, float4* __restrict__ part) {
	const unsigned b = blockIdx.x;
	const unsigned sl = b % slices;
	const unsigned i = (b / slices) * kBlock + threadIdx.x;
	const float4 a = q0[i];
	const float4 ca = q1[i];
	const float4 va = q2[i];
	float ax = 0.0f, ay = 0.0f, az = 0.0f, du = 0.0f;
	const unsigned j0 = sl * slice_len;
	const unsigned j1 = min(j0 + slice_len, n_pad);
	for (unsigned jt = j0; jt < j1; jt += kTj) {
#pragma unroll 8
		for (unsigned j = jt; j < jt + kTj; ++j) {
			const float4 b4 = q0[j];
			const float dx = a.x - b4.x, dy = a.y - b4.y, dz = a.z - b4.z;
			const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
			if (r2 < fmaxf(a.w, b4.w) && r2 > 0.0f) {
				const float4 cb = q1[j];
				const float4 vb = q2[j];
				const float inv_r = __builtin_amdgcn_rsqf(r2);
				const float r = r2 * inv_r;
				const float dw = cubic_dw(r * ca.y, ca.y) + cubic_dw(r * cb.y, cb.y);
				const float f = 0.5f * cb.x * (ca.w + cb.w) * dw * inv_r;   // grad_i W = dW/dr d / r
				ax = __builtin_fmaf(-f, dx, ax);
				ay = __builtin_fmaf(-f, dy, ay);
				az = __builtin_fmaf(-f, dz, az);
				const float vd =
				    __builtin_fmaf(va.z - vb.z, dz, __builtin_fmaf(va.y - vb.y, dy, (va.x - vb.x) * dx));
				du = __builtin_fmaf(0.5f * f, vd, du);
			}
		}
	}
	part[(size_t)sl * n_pad + i] = make_float4(ax, ay, az, du);
}

__global__ __launch_bounds__(kBlock) void k_force_cubic_combine(const float4* __restrict__ part, unsigned n_pad,
                                                                unsigned slices, unsigned N, int acc_phys,
                                                                const float4* __restrict__ q1,
                                                                float* __restrict__ acc, float* __restrict__ dudt) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= N) return;
	double ax = 0.0, ay = 0.0, az = 0.0, du = 0.0;
	for (unsigned k = 0; k < slices; ++k) {
		const float4 p = part[(size_t)k * n_pad + i];
		ax += (double)p.x;
		ay += (double)p.y;
		az += (double)p.z;
		du += (double)p.w;
	}
	const double sc = acc_phys ? 1.0 : (double)q1[i].x;
	acc[3u * i + 0u] += (float)(sc * ax);
	acc[3u * i + 1u] += (float)(sc * ay);
	acc[3u * i + 2u] += (float)(sc * az);
	dudt[i] = (float)du;
}

__global__ __launch_bounds__(kBlock) void k_u_kick(float* __restrict__ u, const float* __restrict__ dudt, unsigned N,
                                                   float half_dt) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i < N) u[i] += half_dt * dudt[i];
}

inline dim3 grid(unsigned n) { return dim3((n + kBlock - 1u) / kBlock); }

}  // namespace

extern "C" {

size_t sfd_sph_tmp_floats(unsigned n_pad) { return 12u * (size_t)n_pad + 16u; }

int sfd_sph_ref(const float* pos, const float* mas, const float* rad, unsigned N, int kahan, const sf_exact_pp* gravity,
                float* rho, float* prs, float* acc, float* tmp, hipStream_t s) {
	if (N == 0) return 0;
	if (gravity && N > kTogetherN) {
		if (sfd_pp_exact(pos, mas, N, gravity->eps2, gravity->neg_g, gravity->acc_phys, gravity->kahan_acc,
		                 gravity->kahan_pot, acc, gravity->pot, s))
			return -1;
		gravity = nullptr;
	}
	float4* ra = reinterpret_cast<float4*>(tmp);
	float4* rh = ra + N;
	float4* rd = ra + 2u * (size_t)N;
	hipLaunchKernelGGL(k_tables_ref, grid(N), dim3(kBlock), 0, s, pos, mas, rad, N, ra, rh, rd);
	auto go = N <= chain::kFewN ? (kahan ? launch_ref<32, true> : launch_ref<32, false>)
	                            : (kahan ? launch_ref<64, true> : launch_ref<64, false>);
	go(gravity, ra, rh, rd, pos, mas, N, rho, prs, ra, acc, s);
	return sf_hip_check(hipGetLastError(), "solve_sph", "launch");
}

int sfd_sph_cubic_pack(const float* pos, const float* vel, const float* acc, const float* mas, const float* rad,
                       const float* u, const float* dudt, unsigned N, unsigned n_pad, float pred_dt, float* tmp,
                       hipStream_t s) {
	if (N == 0) return 0;
	float4* q0 = reinterpret_cast<float4*>(tmp);
	hipLaunchKernelGGL(k_pack_cubic, grid(n_pad), dim3(kBlock), 0, s, pos, vel, acc, mas, rad, u, dudt, N, n_pad,
	                   pred_dt, q0, q0 + n_pad, q0 + 2u * (size_t)n_pad);
	return sf_hip_check(hipGetLastError(), "solve_sph", "launch");
}

// part: slices x n_pad float4 of scratch
int sfd_sph_cubic(unsigned N, unsigned n_pad, float gamma, int acc_phys, float* rho, float* prs, float* acc,
                  float* dudt, float* tmp, float* part, unsigned slices, hipStream_t s) {
	if (N == 0) return 0;
	if (n_pad % kTj != 0 || n_pad % kBlock != 0 || slices == 0) return -1;
	float4* q0 = reinterpret_cast<float4*>(tmp);
	float4* q1 = q0 + n_pad;
	float4* q2 = q0 + 2u * (size_t)n_pad;
	const unsigned tiles = n_pad / kTj;
	if (slices > tiles) slices = tiles;
	const unsigned slice_len = (tiles + slices - 1u) / slices * kTj;
	slices = (n_pad + slice_len - 1u) / slice_len;
	const dim3 g((n_pad / kBlock) * slices);
	const int tok = sf_prof_begin("sph_rho_cubic", s);
	hipLaunchKernelGGL(k_rho_cubic, g, dim3(kBlock), 0, s, q0, q1, n_pad, slices, slice_len, part);
	hipLaunchKernelGGL(k_rho_cubic_combine, grid(N), dim3(kBlock), 0, s, part, n_pad, slices, N, gamma - 1.0f, q1,
	                   rho, prs);
	sf_prof_end(tok, s);
	const int tok2 = sf_prof_begin("sph_force_cubic", s);
	float4* p4 = reinterpret_cast<float4*>(part);
	hipLaunchKernelGGL(k_force_cubic, g, dim3(kBlock), 0, s, q0, q1, q2, n_pad, slices, slice_len, p4);
	hipLaunchKernelGGL(k_force_cubic_combine, grid(N), dim3(kBlock), 0, s, p4, n_pad, slices, N, acc_phys, q1, acc,
	                   dudt);
	sf_prof_end(tok2, s);
	return sf_hip_check(hipGetLastError(), "solve_sph", "launch");
}

int sfd_sph_u_kick(float* u, const float* dudt, unsigned N, float half_dt, hipStream_t s) {
	if (N == 0) return 0;
	hipLaunchKernelGGL(k_u_kick, grid(N), dim3(kBlock), 0, s, u, dudt, N, half_dt);
	return sf_hip_check(hipGetLastError(), "sim_step", "launch");
}

}  // extern "C"
