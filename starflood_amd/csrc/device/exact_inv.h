// exact_inv.h -- reciprocals with the IEEE operations' bits, in fewer of them.
#ifndef SF_EXACT_INV_H
#define SF_EXACT_INV_H

#include <hip/hip_runtime.h>

// 1 / s and 1 / sqrt(s) with the IEEE quotient's and square root's bits (each
// rounded to nearest, the second from the rounded root), in 11 operations and
// one v_rsq_f32 instead of two divisions and a square root of about 45:
// Newton steps whose last operation is an FMA (Markstein's scheme).
// Compared with 1.0f / s and 1.0f / sqrtf(s) on the device for every float
// in [2^-96, 2^97): they differ only where the significand of s is all ones
// or within one of it (1/s or 1/root then lies next to a rounding boundary).
// kRootBits tells those, and kTopBits the values above the range.
__device__ __forceinline__ void exact_inverses(float s, float& inv_s, float& inv_root) {
	const float r = __builtin_amdgcn_rsqf(s);
	const float g = s * r, h = 0.5f * r;
	const float root = __builtin_fmaf(__builtin_fmaf(-g, g, s), h, g);
	inv_root = __builtin_fmaf(r, __builtin_fmaf(-root, r, 1.0f), r);
	const float q = r * r;
	const float e = __builtin_fmaf(-s, q, 1.0f);
	inv_s = __builtin_fmaf(q, __builtin_fmaf(e, e, e), q);
}
constexpr unsigned kRootBits = 0xFFFFFFFEu;   // bits(s) | 0xFF800000 at or above this: IEEE operations
constexpr unsigned kTopBits = 0x6F800000u;    // bits(s) at or above this (2^96, inf, NaN): IEEE operations
constexpr float kExactMinEps2 = 0x1p-96f;     // s >= eps2: below this, IEEE operations throughout

// The same for one s at a time, with IEEE operations where they are needed.
__device__ __forceinline__ void checked_inverses(float s, float& inv_s, float& inv_root) {
	exact_inverses(s, inv_s, inv_root);
	const unsigned bits = __float_as_uint(s);
	if (!(s >= kExactMinEps2) || bits >= kTopBits || (bits | 0xFF800000u) >= kRootBits) {
		inv_s = 1.0f / s;
		inv_root = 1.0f / sqrtf(s);
	}
}

#endif
