// noalloc.hip -- sf_force_dev_noalloc: the PP force on caller device arrays
// (sf_force_dev's kernels and summation order) with its scratch memory in a
// static device array instead of hipMalloc'd buffers, for callers that
// cannot allocate (code under stream capture, allocation-free serving
// loops).  No counterpart in the reference.
//
// scratch holds the force kernels' partial sums.  It is sized for every N up to
// SF_NOALLOC_MAX_N: 32.5 MiB (65 planes of one double4 per body at the largest
// n_pad).  Each device holds its own copy; its address comes from
// hipGetSymbolAddress, once per device, on the first call with that device
// current.
#include <hip/hip_runtime.h>

#include <mutex>

#include "../sf_internal.h"
#include "pp_sym.h"

extern "C" {
size_t sf_pp_part_bytes(unsigned int n_pad);
int sf_pp_force_arrays(const sf_params_t* p, unsigned int N, unsigned int n_pad, const float* pos, const float* mas,
                       float* body, float* part, size_t part_bytes, float* acc, float* pot, hipStream_t s);
}

namespace {

constexpr unsigned kMaxN = SF_NOALLOC_MAX_N;
// the largest partial sums over the sizes
constexpr size_t max_part_bytes() {
	size_t most = 0;
	for (unsigned n = 1024u; n <= kMaxN; n += 1024u) {
		const size_t b = pp_part_bytes(n);
		if (b > most) most = b;
	}
	return most;
}
static_assert(!sym_pp_wide(kMaxN), "the kernels read the caller's arrays: no packed bodies");
constexpr size_t kPartBytes = max_part_bytes();

static __device__ __align__(256) unsigned char scratch[kPartBytes];

constexpr int kMaxDevices = 64;
std::mutex g_lock;
unsigned char* g_scratch[kMaxDevices];   // device address of scratch, per device

// The scratch address on the current device, looked up on first use.
unsigned char* scratch_ptr(const char* fn) {
	int dev = -1;
	if (sf_hip_check(hipGetDevice(&dev), fn, "hipGetDevice")) return nullptr;
	if (dev < 0 || dev >= kMaxDevices) {
		sf_error(fn, "device %d is beyond the %d this entry point serves", dev, kMaxDevices);
		return nullptr;
	}
	std::lock_guard<std::mutex> hold(g_lock);
	if (!g_scratch[dev]) {
		void* p = nullptr;
		if (sf_hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), fn, "hipGetSymbolAddress(scratch)"))
			return nullptr;
		g_scratch[dev] = static_cast<unsigned char*>(p);
	}
	return g_scratch[dev];
}

}  // namespace

extern "C" int sf_force_dev_noalloc(unsigned int N, const float* x, const float* m, float* acc, float* pot,
                                    void* stream) {
	const char* fn = "sf_force_dev_noalloc";
	if (N == 0) return STARFLOOD_SUCCESS;
	if (!x || !m || !acc) {
		sf_error(fn, "null array");
		return STARFLOOD_FAILURE;
	}
	if (N > kMaxN) {
		sf_error(fn, "N = %u exceeds the static scratch's maximum of %u particles", N, kMaxN);
		return STARFLOOD_FAILURE;
	}
	// the layout sf_force_dev allocates: n_pad a multiple of 1024
	const unsigned n_pad = (N + 1023u) / 1024u * 1024u;
	const size_t part_bytes = sf_pp_part_bytes(n_pad);
	if (part_bytes > sizeof(scratch)) {
		sf_error(fn, "N = %u needs %zu scratch bytes, more than the %zu available", N, part_bytes, sizeof(scratch));
		return STARFLOOD_FAILURE;
	}
	unsigned char* base = scratch_ptr(fn);
	if (!base) return STARFLOOD_FAILURE;
	return sf_pp_force_arrays(sf_params(), N, n_pad, x, m, nullptr, reinterpret_cast<float*>(base), part_bytes, acc, pot,
	                          static_cast<hipStream_t>(stream))
	           ? STARFLOOD_FAILURE
	           : STARFLOOD_SUCCESS;
}
