// force_epi.h -- what the force's combine kernels do with a particle's
// acceleration once it is summed: store it, or finish the KDK step around it.
// A launch of its own for each of these passes costs 4 to 5 us on the
// stream, as much as a force of 2000 bodies: with these passes in the combine
// a step of the adjoint forward is two launches instead of five, its backward
// two instead of five, and 40 steps forward and back of 16384 bodies took
// 8.3 ms instead of 9.1 (8.4 since the planes are FP64).
#ifndef SF_FORCE_EPI_H
#define SF_FORCE_EPI_H

#include <hip/hip_runtime.h>

#include "../sf_internal.h"

struct EpiStore {
	float* acc;
	float* pot;   // may be NULL
	explicit EpiStore(const sf_force_epi& e) : acc(e.acc), pot(e.pot) {}
	__device__ __forceinline__ void operator()(unsigned i, float ax, float ay, float az, float p, float4*) const {
		acc[3u * i + 0u] = ax;
		acc[3u * i + 1u] = ay;
		acc[3u * i + 2u] = az;
		if (pot) pot[i] = p;
	}
};

// sim_step: the closing kick and the particle's energies as well, with the
// operations of kdk.hip's k_reduce_state<kFastKick> and k_energy_terms<true>
struct EpiKick {
	float *acc, *pot, *vel, *ken, *pen;
	float h;
	explicit EpiKick(const sf_force_epi& e) : acc(e.acc), pot(e.pot), vel(e.v), ken(e.ken), pen(e.pen), h(e.h) {}
	__device__ __forceinline__ void operator()(unsigned i, float ax, float ay, float az, float p, float4* body) const {
		const float m = body[i].w;
		const float vx = __builtin_fmaf(h, ax, vel[3u * i]);
		const float vy = __builtin_fmaf(h, ay, vel[3u * i + 1u]);
		const float vz = __builtin_fmaf(h, az, vel[3u * i + 2u]);
		acc[3u * i + 0u] = ax;
		acc[3u * i + 1u] = ay;
		acc[3u * i + 2u] = az;
		pot[i] = p;
		vel[3u * i] = vx;
		vel[3u * i + 1u] = vy;
		vel[3u * i + 2u] = vz;
		const float v2 = (vx * vx + vy * vy) + vz * vz;
		ken[i] = 0.5f * m * v2;
		pen[i] = m * p;
	}
};

// The adjoint's integration: close the step that the force ends (close), keep
// the state (ck_*, xN, vN, where set), and open the next one (open): kick and
// drift, the new position into x64, x and the packed body.
struct EpiKdk {
	sf_force_epi e;
	explicit EpiKdk(const sf_force_epi& v) : e(v) {}
	__device__ __forceinline__ void operator()(unsigned i, float ax, float ay, float az, float, float4* body) const {
		const float a[3] = {ax, ay, az};
		float v[3], x[3];
#pragma unroll
		for (unsigned k = 0; k < 3u; ++k) {
			v[k] = e.v[3u * i + k];
			if (e.close) v[k] = __builtin_fmaf(e.h, a[k], v[k]);
			double y = e.x64[3u * i + k];
			if (e.ck_x64) {
				e.ck_x64[3u * i + k] = y;
				e.ck_v[3u * i + k] = v[k];
				e.ck_a[3u * i + k] = a[k];
			}
			if (e.open) {
				v[k] = __builtin_fmaf(e.h, a[k], v[k]);
				y = __builtin_fma(e.dt, (double)v[k], y);
				e.x64[3u * i + k] = y;
			}
			x[k] = (float)y;
			e.v[3u * i + k] = v[k];
			if (e.x && e.open) e.x[3u * i + k] = x[k];
			if (e.xN) {
				e.xN[3u * i + k] = x[k];
				e.vN[3u * i + k] = v[k];
			}
		}
		if (e.open) body[i] = make_float4(x[0], x[1], x[2], body[i].w);
	}
};

#endif
