// bodies.h -- where the force kernels read a particle's (x, y, z, m): from
// bodies packed in a launch before (which the step's and the adjoint's
// launches leave behind anyway), or from the caller's arrays, which saves
// that launch.  Past the last particle both give a body at the origin of mass 0.
#ifndef SF_BODIES_H
#define SF_BODIES_H

#include <hip/hip_runtime.h>

struct PackedBodies {
	const float4* body;   // n_pad of them
	__device__ __forceinline__ float4 operator()(unsigned i) const { return body[i]; }
	__device__ __forceinline__ float mass(unsigned i) const { return body[i].w; }
};

struct ArrayBodies {
	const float* pos;
	const float* mas;
	unsigned N;
	__device__ __forceinline__ float4 operator()(unsigned i) const {
		if (i >= N) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		return make_float4(pos[3u * i], pos[3u * i + 1u], pos[3u * i + 2u], mas[i]);
	}
	__device__ __forceinline__ float mass(unsigned i) const { return mas[i]; }
};

#endif
