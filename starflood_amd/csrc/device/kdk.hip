// kdk.hip -- kick-drift-kick pieces, per-particle energies and FP64
// reductions of the state (reference src/simulation.c:381-504).
//
// Exact policy: FP32 elementwise updates in the reference's operation order
// (file compiled with -ffp-contract=off); T and V are exact_sum.hip's.
// Fast policy: kick and FP64 drift fused in one pass over the state.  Both:
// tree-shaped FP64 block reductions with a fixed grid, which are
// deterministic and more accurate than a sequential sum.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "state_fold.h"

namespace {

constexpr unsigned kBlock = fold::kThreads;
using fold::kRedBlocks;
using fold::kRedQ;

inline unsigned grid_for(unsigned n) { return (n + kBlock - 1) / kBlock; }

// vel[k] += (0.5 dt) acc[k]  (src/simulation.c:382, :424)
__global__ __launch_bounds__(kBlock) void k_kick_exact(float* __restrict__ vel, const float* __restrict__ acc,
                                                       unsigned n3, float half_dt) {
	const unsigned k = blockIdx.x * kBlock + threadIdx.x;
	if (k < n3) vel[k] = vel[k] + half_dt * acc[k];
}

// Both, component by component: the same two roundings in one launch.  Here and
// in k_reduce_state the step's updates ride on other passes, 93 -> 84 us a step
// at 1000 bodies; the separate kernels serve the step times log, whose columns
// need them apart.
__global__ __launch_bounds__(kBlock) void k_kick_drift_exact(float* __restrict__ vel, const float* __restrict__ acc,
                                                             float* __restrict__ pos, unsigned n3, float half_dt,
                                                             float dt) {
	const unsigned k = blockIdx.x * kBlock + threadIdx.x;
	if (k >= n3) return;
	const float v = vel[k] + half_dt * acc[k];
	vel[k] = v;
	pos[k] = pos[k] + dt * v;
}

// pos[k] += dt vel[k]  (src/simulation.c:394)
__global__ __launch_bounds__(kBlock) void k_drift_exact(float* __restrict__ pos, const float* __restrict__ vel,
                                                        unsigned n3, float dt) {
	const unsigned k = blockIdx.x * kBlock + threadIdx.x;
	if (k < n3) pos[k] = pos[k] + dt * vel[k];
}

// ken_i = (0.5 m_i) * ((vx^2 + vy^2) + vz^2); pen_i = m_i pot_i  (src/simulation.c:434-451).
// KICK: the fast policy's closing kick first, for the step times log.
template <bool KICK>
__global__ __launch_bounds__(kBlock) void k_energy_terms(float* __restrict__ vel, const float* __restrict__ acc,
                                                         float half_dt, const float* __restrict__ mas,
                                                         const float* __restrict__ pot, unsigned N,
                                                         float* __restrict__ ken, float* __restrict__ pen) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= N) return;
	const float m = mas[i];
	float vx = vel[3u * i], vy = vel[3u * i + 1u], vz = vel[3u * i + 2u];
	if (KICK) {
		vx = __builtin_fmaf(half_dt, acc[3u * i], vx);
		vy = __builtin_fmaf(half_dt, acc[3u * i + 1u], vy);
		vz = __builtin_fmaf(half_dt, acc[3u * i + 2u], vz);
		vel[3u * i] = vx;
		vel[3u * i + 1u] = vy;
		vel[3u * i + 2u] = vz;
	}
	const float v2 = (vx * vx + vy * vy) + vz * vz;
	ken[i] = 0.5f * m * v2;
	pen[i] = m * pot[i];
}

// x64 follows pos unless it rounds to it: a host-side change of pos (or a
// first use) restarts the FP64 track from the FP32 value.
__global__ __launch_bounds__(kBlock) void k_x64_refresh(const float* __restrict__ pos, double* __restrict__ x64,
                                                        unsigned n3) {
	const unsigned k = blockIdx.x * kBlock + threadIdx.x;
	if (k >= n3) return;
	const float p = pos[k];
	if ((float)x64[k] != p) x64[k] = (double)p;
}

// k_x64_refresh's rule first, then kick and drift
__global__ __launch_bounds__(kBlock) void k_kick_drift_fast(float* __restrict__ vel, const float* __restrict__ acc,
                                                            double* __restrict__ x64, float* __restrict__ pos,
                                                            unsigned n3, float half_dt, double dt) {
	const unsigned k = blockIdx.x * kBlock + threadIdx.x;
	if (k >= n3) return;
	const float v = __builtin_fmaf(half_dt, acc[k], vel[k]);
	vel[k] = v;
	double x0 = x64[k];
	const float p = pos[k];
	if ((float)x0 != p) x0 = (double)p;
	const double x = __builtin_fma(dt, (double)v, x0);
	x64[k] = x;
	pos[k] = (float)x;
}

// Per-block partial sums with a fixed grid-stride assignment and a fixed
// LDS tree, so the result does not depend on scheduling.  KICK: first the
// closing kick (with the fast policy's rounding, or k_kick_exact's) and
// k_energy_terms, particle by particle, in the same pass (a launch of its own
// cost 5 us, 41 at 4M particles).
enum Kick { kNoKick, kFastKick, kExactKick };

template <Kick KICK>
__global__ __launch_bounds__(kBlock) void k_reduce_state(const float* __restrict__ pos, const double* __restrict__ x64,
                                                         float* __restrict__ vel, const float* __restrict__ mas,
                                                         const float* __restrict__ pot, float* __restrict__ ken,
                                                         float* __restrict__ pen, const float* __restrict__ u,
                                                         unsigned N, double G, double eps,
                                                         const float* __restrict__ acc, float half_dt,
                                                         double* __restrict__ red) {
	__shared__ double sh[kRedQ][kBlock];
	double q[kRedQ];
#pragma unroll
	for (int t = 0; t < kRedQ; ++t) q[t] = 0.0;
	const double self = eps > 0.0 ? G / eps : 0.0;
	for (unsigned i = blockIdx.x * kBlock + threadIdx.x; i < N; i += gridDim.x * kBlock) {
		const double m = mas[i];
		double x, y, z;
		if (x64) {
			x = x64[3u * i]; y = x64[3u * i + 1u]; z = x64[3u * i + 2u];
		} else {
			x = pos[3u * i]; y = pos[3u * i + 1u]; z = pos[3u * i + 2u];
		}
		float wx = vel[3u * i], wy = vel[3u * i + 1u], wz = vel[3u * i + 2u], ke, pe;
		if (KICK != kNoKick) {
			const float ax = acc[3u * i], ay = acc[3u * i + 1u], az = acc[3u * i + 2u];
			wx = KICK == kExactKick ? wx + half_dt * ax : __builtin_fmaf(half_dt, ax, wx);
			wy = KICK == kExactKick ? wy + half_dt * ay : __builtin_fmaf(half_dt, ay, wy);
			wz = KICK == kExactKick ? wz + half_dt * az : __builtin_fmaf(half_dt, az, wz);
			vel[3u * i] = wx;
			vel[3u * i + 1u] = wy;
			vel[3u * i + 2u] = wz;
			const float v2 = (wx * wx + wy * wy) + wz * wz;
			ke = 0.5f * mas[i] * v2;
			pe = mas[i] * pot[i];
			ken[i] = ke;
			pen[i] = pe;
		} else {
			ke = ken[i];
			pe = pen[i];
		}
		const double vx = wx, vy = wy, vz = wz;
		q[0] += (double)ke;
		q[1] += (double)pe;
		q[2] += 0.5 * m * ((double)pot[i] + self * m);
		if (u) q[3] += m * (double)u[i];
		q[4] += m * vx;
		q[5] += m * vy;
		q[6] += m * vz;
		q[7] += m * (y * vz - z * vy);
		q[8] += m * (z * vx - x * vz);
		q[9] += m * (x * vy - y * vx);
		q[10] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
	}
#pragma unroll
	for (int t = 0; t < kRedQ; ++t) sh[t][threadIdx.x] = q[t];
	__syncthreads();
	for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
		if (threadIdx.x < h) {
#pragma unroll
			for (int t = 0; t < kRedQ; ++t) sh[t][threadIdx.x] += sh[t][threadIdx.x + h];
		}
		__syncthreads();
	}
	if (threadIdx.x < kRedQ) red[(size_t)blockIdx.x * SF_RED_VALUES + threadIdx.x] = sh[threadIdx.x][0];
}

__global__ __launch_bounds__(kBlock) void k_reduce_final(double* __restrict__ red, unsigned nblocks) {
	fold::state(red, nblocks);
}

}  // namespace

extern "C" int sfd_kick_exact(float* vel, const float* acc, unsigned n3, float half_dt, hipStream_t s) {
	if (!n3) return 0;
	const int tok = sf_prof_begin("kick", s);
	hipLaunchKernelGGL(k_kick_exact, dim3(grid_for(n3)), dim3(kBlock), 0, s, vel, acc, n3, half_dt);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_kick_exact", "launch");
}

extern "C" int sfd_drift_exact(float* pos, const float* vel, unsigned n3, float dt, hipStream_t s) {
	if (!n3) return 0;
	const int tok = sf_prof_begin("drift", s);
	hipLaunchKernelGGL(k_drift_exact, dim3(grid_for(n3)), dim3(kBlock), 0, s, pos, vel, n3, dt);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_drift_exact", "launch");
}

extern "C" int sfd_kick_drift_exact(float* vel, const float* acc, float* pos, unsigned n3, float half_dt, float dt,
                                    hipStream_t s) {
	if (!n3) return 0;
	const int tok = sf_prof_begin("kick_drift", s);
	hipLaunchKernelGGL(k_kick_drift_exact, dim3(grid_for(n3)), dim3(kBlock), 0, s, vel, acc, pos, n3, half_dt, dt);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_kick_drift_exact", "launch");
}

extern "C" int sfd_energy_terms(const float* vel, const float* mas, const float* pot, unsigned N, float* ken,
                                float* pen, hipStream_t s) {
	if (!N) return 0;
	const int tok = sf_prof_begin("energy_terms", s);
	hipLaunchKernelGGL(k_energy_terms<false>, dim3(grid_for(N)), dim3(kBlock), 0, s, const_cast<float*>(vel), nullptr,
	                   0.0f, mas, pot, N, ken, pen);   // vel is not written without the kick
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_energy_terms", "launch");
}

extern "C" int sfd_kick_energy_fast(float* vel, const float* acc, const float* mas, const float* pot, unsigned N,
                                    float half_dt, float* ken, float* pen, hipStream_t s) {
	if (!N) return 0;
	const int tok = sf_prof_begin("kick", s);
	hipLaunchKernelGGL(k_energy_terms<true>, dim3(grid_for(N)), dim3(kBlock), 0, s, vel, acc, half_dt, mas, pot, N, ken,
	                   pen);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_kick_energy_fast", "launch");
}

extern "C" int sfd_x64_refresh(const float* pos, double* x64, unsigned n3, hipStream_t s) {
	if (!n3) return 0;
	hipLaunchKernelGGL(k_x64_refresh, dim3(grid_for(n3)), dim3(kBlock), 0, s, pos, x64, n3);
	return sf_hip_check(hipGetLastError(), "sfd_x64_refresh", "launch");
}

extern "C" int sfd_kick_drift_fast(float* vel, const float* acc, double* x64, float* pos, unsigned n3,
                                   float half_dt, double dt, hipStream_t s) {
	if (!n3) return 0;
	const int tok = sf_prof_begin("kick_drift", s);
	hipLaunchKernelGGL(k_kick_drift_fast, dim3(grid_for(n3)), dim3(kBlock), 0, s, vel, acc, x64, pos, n3, half_dt,
	                   dt);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_kick_drift_fast", "launch");
}

extern "C" unsigned sfd_reduce_scratch_doubles(unsigned N) {
	(void)N;
	return (kRedBlocks + 1u) * SF_RED_VALUES;
}

static int reduce(Kick kick, const float* pos, const double* x64, float* vel, const float* mas, const float* pot,
                  float* ken, float* pen, const float* u, unsigned N, double G, double eps, const float* acc,
                  float half_dt, double* red, hipStream_t s) {
	const unsigned nb = fold::blocks(N);
	const auto kernel = kick == kNoKick     ? k_reduce_state<kNoKick>
	                    : kick == kFastKick ? k_reduce_state<kFastKick>
	                                        : k_reduce_state<kExactKick>;
	const int tok = sf_prof_begin(kick == kNoKick ? "reduce_state" : "kick_reduce_state", s);
	hipLaunchKernelGGL(kernel, dim3(nb), dim3(kBlock), 0, s, pos, x64, vel, mas, pot, ken, pen, u, N, G, eps, acc,
	                   half_dt, red);
	// the exact policy's sums follow and fold the partials too
	if (kick != kExactKick) hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kBlock), 0, s, red, nb);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_reduce_state", "launch");
}

extern "C" int sfd_reduce_state(const float* pos, const double* x64, const float* vel, const float* mas,
                                const float* pot, const float* ken, const float* pen, const float* u, unsigned N,
                                double G, double eps, double* red, hipStream_t s) {
	// not written without the kick
	return reduce(kNoKick, pos, x64, const_cast<float*>(vel), mas, pot, const_cast<float*>(ken), const_cast<float*>(pen), u,
	              N, G, eps, nullptr, 0.0f, red, s);
}

extern "C" int sfd_kick_reduce_state(const float* pos, const double* x64, float* vel, const float* acc,
                                     const float* mas, const float* pot, float half_dt, float* ken, float* pen,
                                     const float* u, unsigned N, double G, double eps, double* red, hipStream_t s) {
	return reduce(kFastKick, pos, x64, vel, mas, pot, ken, pen, u, N, G, eps, acc, half_dt, red, s);
}

extern "C" int sfd_kick_reduce_exact(const float* pos, float* vel, const float* acc, const float* mas, const float* pot,
                                     float half_dt, float* ken, float* pen, const float* u, unsigned N, double G,
                                     double eps, double* red, hipStream_t s) {
	return reduce(kExactKick, pos, nullptr, vel, mas, pot, ken, pen, u, N, G, eps, acc, half_dt, red, s);
}
