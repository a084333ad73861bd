// exact_pp.h -- the reference's particle-particle gravity as a model of
// order_chain.h (pp.hip, and sph.hip beside the reference model's density).
#ifndef SF_EXACT_PP_H
#define SF_EXACT_PP_H

#include "exact_inv.h"
#include "order_chain.h"

namespace chain {

// The terms of the reference's pair (src/gravity.c:709-769) and its sums:
// the model that order_chain.h runs, components x, y, z and the potential.
// Makers: 26 VALU operations, the rsq and 2 LDS writes a pair.  One lane per
// particle with IEEE divisions took 239 us at N = 1000, 1430 at 6000, 3918 at
// 16384 and 15.7 ms at 65536; this takes 14, 74, 323 and 4.5 ms.
template <bool KAHAN_ACC, bool KAHAN_POT, bool PHYS>
struct ExactPP {
	static constexpr unsigned kComps = 4;
	const float* __restrict__ pos;
	const float* __restrict__ mas;
	float eps2, negG;
	float* __restrict__ acc;
	float* __restrict__ pot;

	struct Self {
		float x, y, z;
	};
	struct Body {
		float x, y, z, m;
	};
	struct Check {
		unsigned top = 0u, edge = 0u;
		__device__ bool bad() const { return top >= kTopBits || edge >= kRootBits; }
	};
	__device__ bool fast() const { return eps2 >= kExactMinEps2; }
	__device__ Self self(unsigned i) const { return {pos[3u * i], pos[3u * i + 1u], pos[3u * i + 2u]}; }
	__device__ __forceinline__ Body body(unsigned j, unsigned off) const {
		const float* p = pos + 3u * (size_t)j;
		return {p[3u * off], p[3u * off + 1u], p[3u * off + 2u], (mas + j)[off]};
	}

	template <bool FAST>
	__device__ __forceinline__ void terms(const Self& a, const Body& b, float (&out)[4], Check& chk) const {
		const float rx = a.x - b.x, ry = a.y - b.y, rz = a.z - b.z;
		const float r2 = (rx * rx + ry * ry) + rz * rz;
		const float s = r2 + eps2;
		float inv_r2, inv_r1;
		if (FAST) {
			exact_inverses(s, inv_r2, inv_r1);
			const unsigned bits = __float_as_uint(s);
			chk.top = max(chk.top, bits);
			chk.edge = max(chk.edge, bits | 0xFF800000u);
		} else {
			inv_r2 = 1.0f / s;
			inv_r1 = 1.0f / sqrtf(s);
		}
		const float pj = b.m * inv_r1;
		const float w = pj * inv_r2;
		out[0] = w * rx;
		out[1] = w * ry;
		out[2] = w * rz;
		out[3] = pj;
	}
	__device__ __forceinline__ void step(unsigned comp, float& s, float& c, float x) const {
		if (KAHAN_ACC || KAHAN_POT) {
			kahan(s, c, x);
			// no compensation carried: the plain sum
			if (KAHAN_ACC != KAHAN_POT) c = (comp < 3u ? KAHAN_ACC : KAHAN_POT) ? c : 0.0f;
		} else {
			s += x;
		}
	}
	// reference src/gravity.c:808-811: ((-G) * m_i) * acc_sum, (-G) * pot_sum
	__device__ void store(unsigned i, unsigned comp, float s) const {
		if (comp == 3u) pot[i] = negG * s;
		else acc[3u * i + comp] = (PHYS ? negG : negG * mas[i]) * s;
	}
};

}  // namespace chain

#endif
