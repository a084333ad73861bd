// exact_sum.hip -- the reference's sequential FP64 Kahan sums (the energies,
// src/simulation.c:455-497, and the mean radius, src/simulation.c:245-277 and
// src/visualization.c:276-305) with the bits of the sequence, computed in
// parallel.
//
// A Kahan step is four dependent FP64 additions, 23 ns on one wavefront, and
// the sequence cannot be reordered step by step.  What it returns can be had
// without it:
//
// Energies (terms that are floats).  Let q be the last place of the smallest
// nonzero |x_i| and let every |x_i| < 2^51 q.  Then the running sum S and the
// compensation C satisfy, with X_i the exact partial sum,
//     S_i = RN(X_i),   C_i = S_i - X_i   (RN: rounding to 53 bits):
// x_i - C is a multiple of q below 2^52 q, so y = x_i - C is exact;
// S + y = X_i exactly, so t = RN(X_i); and (t - S) - y is the exact rounding
// error (Dekker's fast two-sum when |S| >= |y|; otherwise |S + y| < 2^53 q
// and nothing was rounded).  So the last S is RN of the exact sum, which
// integers give in any order.  Exponents that span more than 27 binary
// orders, and non-finite terms, take the sequence itself.
//
// Mean radius (terms that are doubles; their y is rounded).  Every use
// rounds the mean to a float, and the Kahan sum of N positive terms is
// within (2 u + O(N u^2)) of the exact one (u = 2^-53; Higham 2002, section
// 4.3).  A double-double sum and an interval of 16 u around it give the
// float unless the interval's ends round apart, which happens about once in
// 10^7 sums and takes the sequence.
//
// At N = 16384 the two energy sums took 2 x 866 us and take 8; the mean
// radius of 65536 particles 1.55 ms and 9 us.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "state_fold.h"
#include "tree_dev.h"

namespace {

constexpr unsigned kBlock = fold::kThreads;
constexpr unsigned kPer = 16;                  // terms per thread
constexpr unsigned kChunk = kBlock * kPer;     // terms per block
constexpr int kSpan = 27;                      // exponents kept in one integer: |m| 2^27 < 2^51

__device__ __forceinline__ void kahan_step(double& sum, double& com, double x) {
	const double y = x - com;
	const double t = sum + y;
	const double z = t - sum;
	com = z - y;
	sum = t;
}

// The sequence itself, its result in thread 0: 256 terms at a time through
// LDS.
template <class F>
__device__ double by_sequence(unsigned N, F&& term) {
	__shared__ double s_x[kBlock];
	double sum = 0.0, com = 0.0;
	for (unsigned b = 0; b < N; b += kBlock) {
		const unsigned n = min(kBlock, N - b);
		if (threadIdx.x < n) s_x[threadIdx.x] = term(b + threadIdx.x);
		__syncthreads();
		if (threadIdx.x == 0)
			for (unsigned k = 0; k < n; ++k) kahan_step(sum, com, s_x[k]);
		__syncthreads();
	}
	return sum;
}

// A chunk's exact sum in units of 2^(lo - 150): 4096 terms below 2^51 fit.
struct Partial {
	long long sum;
	int lo, hi;   // least and greatest biased exponent of the nonzero terms
};

__device__ __forceinline__ void wave_minmax(int& lo, int& hi) {
	for (int o = 32; o > 0; o >>= 1) {
		lo = min(lo, __shfl_xor(lo, o));
		hi = max(hi, __shfl_xor(hi, o));
	}
}

// the rounding to nearest, ties to even, of m 2^e
__device__ double round_i128(__int128 m, int e) {
	const bool neg = m < 0;
	unsigned __int128 a = neg ? (unsigned __int128)(-m) : (unsigned __int128)m;
	const unsigned long long top = (unsigned long long)(a >> 64);
	const int bits = top ? 128 - __clzll((long long)top) : 64 - __clzll((long long)(unsigned long long)a);
	if (bits > 53) {
		const int sh = bits - 53;
		const unsigned __int128 rest = a & (((unsigned __int128)1 << sh) - 1u), half = (unsigned __int128)1 << (sh - 1);
		a >>= sh;
		if (rest > half || (rest == half && (a & 1u))) a += 1u;   // 2^53 stays exact
		e += sh;
	}
	const double r = ldexp((double)(unsigned long long)a, e);
	return neg ? -r : r;
}

// The sum of a whole array from its chunks' partials (block-wide), or the
// sequence where they do not give it.
__device__ void finish_sum(const float* __restrict__ x, unsigned N, const Partial* __restrict__ part, unsigned np,
                           double* __restrict__ out) {
	__shared__ int s_lo[kBlock / 64], s_hi[kBlock / 64];
	__shared__ __int128 s_sum[kBlock];
	const unsigned t = threadIdx.x;
	int lo = 1 << 20, hi = -1;
	for (unsigned k = t; k < np; k += kBlock) {
		lo = min(lo, part[k].lo);
		hi = max(hi, part[k].hi);
	}
	wave_minmax(lo, hi);
	if ((t & 63u) == 0u) {
		s_lo[t >> 6] = lo;
		s_hi[t >> 6] = hi;
	}
	__syncthreads();
	for (unsigned w = 0; w < kBlock / 64; ++w) {
		lo = min(lo, s_lo[w]);
		hi = max(hi, s_hi[w]);
	}
	if (hi < 0) {   // no nonzero term
		if (t == 0) out[0] = 0.0;
		return;
	}
	if (hi >= 255 || hi - lo > kSpan) {
		const double s = by_sequence(N, [&](unsigned i) { return (double)x[i]; });
		if (t == 0) out[0] = s;
		return;
	}
	__int128 sum = 0;
	for (unsigned k = t; k < np; k += kBlock)
		if (part[k].hi >= 0) sum += (__int128)part[k].sum << (part[k].lo - lo);
	s_sum[t] = sum;
	__syncthreads();
	for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
		if (t < h) s_sum[t] += s_sum[t + h];
		__syncthreads();
	}
	if (t == 0) out[0] = round_i128(s_sum[0], lo - 150);
}

// Blocks (chunk, array): array 0 is x0, array 1 is x1.  A single chunk is
// finished here, more by k_exact_finish.  A block of a third row folds the
// partials of the state's reduction (a launch of its own took 3 us).
__global__ __launch_bounds__(kBlock) void k_exact_chunks(const float* __restrict__ x0, const float* __restrict__ x1,
                                                         unsigned N, Partial* __restrict__ part,
                                                         double* __restrict__ out, double* __restrict__ red,
                                                         unsigned red_blocks) {
	if (blockIdx.y == 2u) {
		if (blockIdx.x == 0u) fold::state(red, red_blocks);
		return;
	}
	__shared__ int s_lo[kBlock / 64], s_hi[kBlock / 64];
	__shared__ long long s_sum[kBlock / 64];
	const float* __restrict__ x = blockIdx.y ? x1 : x0;
	Partial* p = part + (size_t)blockIdx.y * gridDim.x;
	const unsigned t = threadIdx.x, base = blockIdx.x * kChunk + t;
	unsigned b[kPer];
	int lo = 1 << 20, hi = -1;
#pragma unroll
	for (unsigned r = 0; r < kPer; ++r) {
		const unsigned i = base + r * kBlock;
		b[r] = i < N ? __float_as_uint(x[i]) : 0u;
		if (b[r] & 0x7FFFFFFFu) {
			const int e = max((int)((b[r] >> 23) & 255u), 1);   // subnormals share the first binade's place
			lo = min(lo, e);
			hi = max(hi, e);
		}
	}
	wave_minmax(lo, hi);
	if ((t & 63u) == 0u) {
		s_lo[t >> 6] = lo;
		s_hi[t >> 6] = hi;
	}
	__syncthreads();
	for (unsigned w = 0; w < kBlock / 64; ++w) {
		lo = min(lo, s_lo[w]);
		hi = max(hi, s_hi[w]);
	}
	long long sum = 0;
	if (hi < 255 && hi - lo <= kSpan) {
#pragma unroll
		for (unsigned r = 0; r < kPer; ++r) {
			const int f = (int)((b[r] >> 23) & 255u);
			long long m = (long long)(b[r] & 0x7FFFFFu) | (f ? 0x800000ll : 0ll);
			if (m) m <<= max(f, 1) - lo;
			sum += (b[r] >> 31) ? -m : m;
		}
	}
	for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
	if ((t & 63u) == 0u) s_sum[t >> 6] = sum;
	__syncthreads();
	if (t == 0) {
		for (unsigned w = 1; w < kBlock / 64; ++w) sum += s_sum[w];
		p[blockIdx.x] = {sum, lo, hi};
	}
	if (gridDim.x > 1u) return;
	__syncthreads();
	finish_sum(x, N, p, 1u, out + blockIdx.y);
}

__global__ __launch_bounds__(kBlock) void k_exact_finish(const float* __restrict__ x0, const float* __restrict__ x1,
                                                         unsigned N, const Partial* __restrict__ part, unsigned np,
                                                         double* __restrict__ out) {
	finish_sum(blockIdx.x ? x1 : x0, N, part + (size_t)blockIdx.x * np, np, out + blockIdx.x);
}

// ------------------------------------------------------------ mean radius
// r_i = sqrt((x^2 + y^2) + z^2) in FP64 (src/simulation.c:256-262)
__device__ __forceinline__ double radius(const float* __restrict__ pos, unsigned i) {
	const double x = pos[3u * i], y = pos[3u * i + 1u], z = pos[3u * i + 2u];
	return sqrt((x * x + y * y) + z * z);
}

struct Dd {   // an unevaluated sum hi + lo
	double hi, lo;
};

__device__ __forceinline__ Dd dd_add(Dd a, Dd b) {
	const double s = a.hi + b.hi;
	const double v = s - a.hi;
	const double e = ((a.hi - (s - v)) + (b.hi - v)) + (a.lo + b.lo);
	const double h = s + e;
	return {h, e - (h - s)};
}

// The block's double-double sum of v, in thread 0.
__device__ Dd block_sum(Dd v) {
	__shared__ Dd sh[kBlock];
	const unsigned t = threadIdx.x;
	sh[t] = v;
	__syncthreads();
	for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
		if (t < h) sh[t] = dd_add(sh[t], sh[t + h]);
		__syncthreads();
	}
	return sh[0];
}

__global__ __launch_bounds__(kBlock) void k_radius_sums(const float* __restrict__ pos, unsigned N,
                                                        Dd* __restrict__ part) {
	Dd s = {0.0, 0.0};
	for (unsigned i = blockIdx.x * kBlock + threadIdx.x; i < N; i += gridDim.x * kBlock)
		s = dd_add(s, {radius(pos, i), 0.0});
	s = block_sum(s);
	if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// The mean of the reference's sequence, in thread 0.
__device__ double mean_by_sequence(const float* __restrict__ pos, unsigned N) {
	return by_sequence(N, [&](unsigned i) { return radius(pos, i); }) * (1.0 / (double)N);
}

// an interval that holds the sequence's mean: 2 u for the Kahan sum, 1 u for
// the product with 1 / N and 1 u for the sum here, rounded up to 16
constexpr double kMargin = 16.0 * 0x1p-53;

// The interval (block-wide); false when a radius is not finite.
__device__ bool mean_interval(const Dd* __restrict__ part, unsigned np, unsigned N, double& a_lo, double& a_hi) {
	Dd s = {0.0, 0.0};
	for (unsigned k = threadIdx.x; k < np; k += kBlock) s = dd_add(s, part[k]);
	s = block_sum(s);
	const double a = (s.hi + s.lo) * (1.0 / (double)N);
	a_lo = a * (1.0 - kMargin);
	a_hi = a * (1.0 + kMargin);
	return a <= 1e300;
}

// The jittered cube bounds (src/simulation.c:279-301) around the mean
// radius; jit[i] is 2 * (INV_PCG32_MAX * s[i]) - 1 from pcg4d of the step
// number.
__device__ __forceinline__ void cube_bounds(double avg, const double* jit, float* b) {
	for (int a = 0; a < 3; ++a) {
		b[a] = (float)(-2.000 * avg + 0.5 * jit[a] * avg);
		b[3 + a] = (float)(2.000 * avg + 0.5 * jit[a] * avg);
	}
}

__global__ __launch_bounds__(kBlock) void k_tree_bounds(const float* __restrict__ pos, unsigned N,
                                                        const Dd* __restrict__ part, unsigned np, double j0,
                                                        double j1, double j2, float* __restrict__ bounds) {
	const double jit[3] = {j0, j1, j2};
	double a_lo, a_hi;
	bool same = mean_interval(part, np, N, a_lo, a_hi);
	float b[6], c[6];
	cube_bounds(a_lo, jit, b);
	cube_bounds(a_hi, jit, c);
	for (int k = 0; k < 6; ++k) same &= b[k] == c[k];
	if (!same) cube_bounds(mean_by_sequence(pos, N), jit, b);
	if (threadIdx.x == 0)
		for (int k = 0; k < 6; ++k) bounds[k] = b[k];
}

__global__ __launch_bounds__(kBlock) void k_mean_interval(const Dd* __restrict__ part, unsigned np, unsigned N,
                                                          double* __restrict__ out) {
	double a_lo, a_hi;
	const bool ok = mean_interval(part, np, N, a_lo, a_hi);
	if (threadIdx.x != 0) return;
	out[0] = ok ? a_lo : __builtin_nan("");
	out[1] = a_hi;
}

__global__ __launch_bounds__(kBlock) void k_mean_sequence(const float* __restrict__ pos, unsigned N,
                                                          double* __restrict__ out) {
	const double a = mean_by_sequence(pos, N);
	if (threadIdx.x == 0) out[0] = out[1] = a;
}

unsigned radius_blocks(unsigned N) { return min((N + 2u * kBlock - 1u) / (2u * kBlock), SF_RADIUS_PARTIALS); }

void radius_sums(const float* pos, unsigned N, double* part, hipStream_t s) {
	hipLaunchKernelGGL(k_radius_sums, dim3(radius_blocks(N)), dim3(kBlock), 0, s, pos, N, reinterpret_cast<Dd*>(part));
}

}  // namespace

extern "C" size_t sfd_energy_scratch_bytes(unsigned N) {
	return 2u * sizeof(Partial) * (size_t)(N ? (N + kChunk - 1u) / kChunk : 1u);
}

extern "C" int sfd_energy_sums_exact(const float* ken, const float* pen, unsigned N, void* part, double* out,
                                     double* red, hipStream_t s) {
	const unsigned np = N ? (N + kChunk - 1u) / kChunk : 1u;
	Partial* p = static_cast<Partial*>(part);
	const int tok = sf_prof_begin("energy_sum_seq", s);
	hipLaunchKernelGGL(k_exact_chunks, dim3(np, pen ? (red ? 3 : 2) : 1), dim3(kBlock), 0, s, ken, pen, N, p, out, red,
	                   fold::blocks(N));
	if (np > 1u) hipLaunchKernelGGL(k_exact_finish, dim3(pen ? 2 : 1), dim3(kBlock), 0, s, ken, pen, N, p, np, out);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_energy_sums_exact", "launch");
}

extern "C" int sfd_mean_radius_interval(const float* pos, unsigned N, double* part, double* avg, hipStream_t s) {
	if (N == 0) return 0;
	radius_sums(pos, N, part, s);
	hipLaunchKernelGGL(k_mean_interval, dim3(1), dim3(kBlock), 0, s, reinterpret_cast<const Dd*>(part),
	                   radius_blocks(N), N, avg);
	return sf_hip_check(hipGetLastError(), "sfd_mean_radius_interval", "launch");
}

extern "C" int sfd_mean_radius_sequence(const float* pos, unsigned N, double* avg, hipStream_t s) {
	if (N == 0) return 0;
	hipLaunchKernelGGL(k_mean_sequence, dim3(1), dim3(kBlock), 0, s, pos, N, avg);
	return sf_hip_check(hipGetLastError(), "sfd_mean_radius_sequence", "launch");
}

extern "C" int sfd_tree_bounds_ref(const float* pos, unsigned N, const double jitter[3], double* part, float* bounds,
                                   hipStream_t s) {
	if (N == 0) return 0;
	radius_sums(pos, N, part, s);
	hipLaunchKernelGGL(k_tree_bounds, dim3(1), dim3(kBlock), 0, s, pos, N, reinterpret_cast<const Dd*>(part),
	                   radius_blocks(N), jitter[0], jitter[1], jitter[2], bounds);
	return sf_hip_check(hipGetLastError(), "sfd_tree_bounds_ref", "launch");
}
