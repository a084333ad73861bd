// state_fold.h -- the second stage of the state's FP64 reduction (kdk.hip),
// for a block of 256 threads of whichever launch follows the first.
#ifndef SF_STATE_FOLD_H
#define SF_STATE_FOLD_H

#include <hip/hip_runtime.h>

#include "../sf_internal.h"

namespace fold {

constexpr unsigned kThreads = 256;
constexpr unsigned kRedBlocks = 512;   // most blocks of the first stage, a fixed grid
constexpr int kRedQ = 11;              // T, V, W, U, Px, Py, Pz, Lx, Ly, Lz, K

inline unsigned blocks(unsigned N) {
	const unsigned nb = (N + kThreads - 1u) / kThreads;
	return nb > kRedBlocks ? kRedBlocks : (nb ? nb : 1u);
}

// Folds the blocks' partials in a fixed tree; the totals go to the first
// values of the region after the partials.
__device__ __forceinline__ void state(double* __restrict__ red, unsigned nblocks) {
	__shared__ double sh[kRedQ][kThreads];
	double q[kRedQ];
#pragma unroll
	for (int t = 0; t < kRedQ; ++t) q[t] = 0.0;
	for (unsigned b = threadIdx.x; b < nblocks; b += kThreads) {
#pragma unroll
		for (int t = 0; t < kRedQ; ++t) q[t] += red[(size_t)b * SF_RED_VALUES + t];
	}
#pragma unroll
	for (int t = 0; t < kRedQ; ++t) sh[t][threadIdx.x] = q[t];
	__syncthreads();
	for (unsigned h = kThreads / 2; h > 0; h >>= 1) {
		if (threadIdx.x < h) {
#pragma unroll
			for (int t = 0; t < kRedQ; ++t) sh[t][threadIdx.x] += sh[t][threadIdx.x + h];
		}
		__syncthreads();
	}
	if (threadIdx.x < (unsigned)kRedQ) red[(size_t)kRedBlocks * SF_RED_VALUES + threadIdx.x] = sh[threadIdx.x][0];
}

}  // namespace fold

#endif
