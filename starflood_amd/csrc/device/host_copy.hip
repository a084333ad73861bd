// host_copy.hip -- copies between page-locked host memory and device memory by
// a kernel, several ranges in one launch, in stream order with the kernels
// around them.
//
// Bound by the link (56 GB/s) and by latency.  A copy engine's transfer waits
// for the stream's kernels and they for it through signals, 10 us a copy; a
// launch costs 3 to 4.  The step of 1000 bodies in mirror mode took 85 us with
// ordinary memory (staged copies), 70 with page-locked memory and the copy
// engine, 47 here with the step's sums in the same launch as its blocks; of
// 16384 bodies 452, 401, 370.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"

namespace {

constexpr unsigned kBlock = 256;
constexpr unsigned kBlocks = 1024;

// `head` words up to a 16-byte boundary, n4 quads, `tail` words
struct Range {
	const unsigned* src;
	unsigned* dst;
	size_t n4;
	unsigned head, tail;
};

struct Ranges {
	Range r[SF_COPY_RANGES];
};

// blockIdx.y: the range
__global__ __launch_bounds__(kBlock) void k_copy_ranges(Ranges ranges) {
	const Range c = ranges.r[blockIdx.y];
	const unsigned t = blockIdx.x * kBlock + threadIdx.x;
	const uint4* __restrict__ s4 = reinterpret_cast<const uint4*>(c.src + c.head);
	uint4* __restrict__ d4 = reinterpret_cast<uint4*>(c.dst + c.head);
	for (size_t k = t; k < c.n4; k += gridDim.x * kBlock) d4[k] = s4[k];
	if (t < c.head) c.dst[t] = c.src[t];
	if (t < c.tail) c.dst[c.head + 4u * c.n4 + t] = c.src[c.head + 4u * c.n4 + t];
}

}  // namespace

extern "C" int sfd_copy_ranges(const sf_copy_range* range, unsigned count, hipStream_t s) {
	Ranges ranges = {};
	unsigned used = 0;
	size_t nb = 1;
	if (count > SF_COPY_RANGES) return -1;
	for (unsigned k = 0; k < count; ++k) {
		const size_t n = range[k].words;
		const uintptr_t from = (uintptr_t)range[k].src, to = (uintptr_t)range[k].dst;
		if (((from | to) & 3u) || ((from ^ to) & 15u)) return -1;
		if (!n) continue;
		size_t head = ((16u - (from & 15u)) & 15u) / 4u;
		if (head > n) head = n;
		ranges.r[used++] = {static_cast<const unsigned*>(range[k].src), static_cast<unsigned*>(range[k].dst),
		                    (n - head) / 4u, (unsigned)head, (unsigned)((n - head) % 4u)};
		const size_t b = ((n - head) / 4u + kBlock - 1u) / kBlock;
		if (b > nb) nb = b;
	}
	if (!used) return 0;
	if (nb > kBlocks) nb = kBlocks;
	hipLaunchKernelGGL(k_copy_ranges, dim3((unsigned)nb, used), dim3(kBlock), 0, s, ranges);
	return sf_hip_check(hipGetLastError(), "sfd_copy_ranges", "launch");
}
