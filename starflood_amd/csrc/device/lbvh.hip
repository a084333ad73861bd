// lbvh.hip -- the SF_TREE_LBVH Barnes-Hut tree: build on gfx950 (the walk is
// in lbvh_walk.hip).
//
// Build (every step, O(N), bandwidth-bound):
//  1. FP64 bounding box (min/max are exact, so any reduction order gives the
//     same cube).
//  2. 63-bit Morton codes: q = floor((x - lo) * (2^21 / extent)) in FP64,
//     clamped to [0, 2^21), bits interleaved x-y-z from the top.  Exactly
//     reproducible by a CPU restatement.
//  3. Stable LSD radix sort of (code, index), 8 passes of 8-bit digits, one
//     launch each: a ballot-based stable local rank, and the tiles' offsets
//     by looking back.
//  4. Binary radix tree from the sorted codes (Karras 2012): internal node i
//     covers a contiguous range of the sorted particles; equal codes are
//     separated by their sorted position.
//  5. Monopoles from FP64 prefix sums of (m, m x, m y, m z) over the sorted
//     particles: a node's mass and moments are differences of two prefix
//     entries, so no bottom-up pass, atomics or cross-XCD fences are needed,
//     and the fixed-shape scan makes the result deterministic.  A node's size
//     in the opening test is its particles' bounding box when it holds at
//     most 64 particles, else its Morton cell: the cell fixed by the common
//     prefix of its first and last codes.
//
// Walk records (k_records) carry, per node, the squared critical radius for
// the current theta, either the particle range or the two children, and the
// size term of the relative opening test.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "lookback.h"
#include "tree_dev.h"

namespace {

constexpr unsigned kBlock = 256;
constexpr unsigned kTile = 4096;          // radix sorts take multiples of this

// ---------------------------------------------------------------- bbox
__global__ __launch_bounds__(kBlock) void k_bbox_partial(const float* __restrict__ pos, unsigned N,
                                                         double* __restrict__ part) {
	__shared__ double sh[6][kBlock];
	double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
	for (unsigned i = blockIdx.x * kBlock + threadIdx.x; i < N; i += gridDim.x * kBlock) {
		for (int a = 0; a < 3; ++a) {
			const double v = pos[3u * i + a];
			lo[a] = fmin(lo[a], v);
			hi[a] = fmax(hi[a], v);
		}
	}
	for (int a = 0; a < 3; ++a) {
		sh[a][threadIdx.x] = lo[a];
		sh[3 + a][threadIdx.x] = hi[a];
	}
	__syncthreads();
	for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
		if (threadIdx.x < h) {
			for (int a = 0; a < 3; ++a) {
				sh[a][threadIdx.x] = fmin(sh[a][threadIdx.x], sh[a][threadIdx.x + h]);
				sh[3 + a][threadIdx.x] = fmax(sh[3 + a][threadIdx.x], sh[3 + a][threadIdx.x + h]);
			}
		}
		__syncthreads();
	}
	if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = sh[threadIdx.x][0];
}

// box[0..2] = lo, box[3] = 2^21 / extent (extent = longest side, widened so
// the top cell is half-open)
__global__ __launch_bounds__(kBlock) void k_bbox_final(const double* __restrict__ part, unsigned nb,
                                                       double* __restrict__ box) {
	__shared__ double sh[6][kBlock];
	double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
	for (unsigned b = threadIdx.x; b < nb; b += kBlock)
		for (int a = 0; a < 3; ++a) {
			lo[a] = fmin(lo[a], part[b * 6 + a]);
			hi[a] = fmax(hi[a], part[b * 6 + 3 + a]);
		}
	for (int a = 0; a < 3; ++a) {
		sh[a][threadIdx.x] = lo[a];
		sh[3 + a][threadIdx.x] = hi[a];
	}
	__syncthreads();
	for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
		if (threadIdx.x < h) {
			for (int a = 0; a < 3; ++a) {
				sh[a][threadIdx.x] = fmin(sh[a][threadIdx.x], sh[a][threadIdx.x + h]);
				sh[3 + a][threadIdx.x] = fmax(sh[3 + a][threadIdx.x], sh[3 + a][threadIdx.x + h]);
			}
		}
		__syncthreads();
	}
	if (threadIdx.x != 0) return;
	double ext = 0.0;
	for (int a = 0; a < 3; ++a) ext = fmax(ext, sh[3 + a][0] - sh[a][0]);
	if (!(ext > 0.0)) ext = 1.0;
	ext *= 1.0 + 1.0e-9;
	for (int a = 0; a < 3; ++a) box[a] = sh[a][0];
	box[3] = 2097152.0 / ext;
}

// ---------------------------------------------------------------- Morton
__device__ __forceinline__ unsigned long long spread21(unsigned long long v) {
	v &= 0x1FFFFFull;
	v = (v | (v << 32)) & 0x1F00000000FFFFull;
	v = (v | (v << 16)) & 0x1F0000FF0000FFull;
	v = (v | (v << 8)) & 0x100F00F00F00F00Full;
	v = (v | (v << 4)) & 0x10C30C30C30C30C3ull;
	v = (v | (v << 2)) & 0x1249249249249249ull;
	return v;
}

// Keys, and (x, y, z, m) packed in index order, so that the gather after the
// sort reads one 16-byte record per particle instead of two cache lines.
__global__ __launch_bounds__(kBlock) void k_morton(const float* __restrict__ pos, const float* __restrict__ mas,
                                                   unsigned N, unsigned n_sort, const double* __restrict__ box,
                                                   unsigned long long* __restrict__ key, unsigned* __restrict__ val,
                                                   float4* __restrict__ packed) {
	const unsigned i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n_sort) return;
	if (i >= N) {
		key[i] = ~0ull;
		val[i] = i;
		return;
	}
	const double scale = box[3];
	const float x = pos[3u * i], y = pos[3u * i + 1u], z = pos[3u * i + 2u];
	const float c[3] = {x, y, z};
	unsigned long long q[3];
	for (int a = 0; a < 3; ++a) {
		double t = ((double)c[a] - box[a]) * scale;
		t = fmin(fmax(t, 0.0), 2097151.0);
		q[a] = (unsigned long long)t;
	}
	key[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
	val[i] = i;
	packed[i] = make_float4(x, y, z, mas[i]);
}

// ---------------------------------------------------------------- radix sort
// Stable LSD sort on 8-bit digits: k_radix_digits counts every pass's digits
// at once, k_radix_offsets turns the counts into each digit's first position,
// and one k_radix_pass per digit ranks, exchanges its tile counts and
// scatters.  A pass of histogram, scan and scatter launches took 20.3 us at
// 65536 pairs, 35 at 1M and 60 at 4M; k_radix_pass takes 8.1, 20 and 44, the
// two launches before the passes together 9, 16 and 29.  At 65536 pairs a pass
// is the latency of its chain (load, rank, post, collect, write); from 1M on
// the collection is a third of it: every tile running at once looks back at
// those before it (two at a time; 1 and 4 take 21 us at 1M, 8 take 21.3, 32
// take 27).

// A block's digit counts for the first `passes` digits, and the state of the
// first pass cleared.
constexpr unsigned kDigitBlocks = 256, kDigitThreads = 1024;
__global__ __launch_bounds__(kDigitThreads) void k_radix_digits(const unsigned long long* __restrict__ key, unsigned n,
                                                         unsigned passes, unsigned* __restrict__ part,
                                                         unsigned long long* __restrict__ state, unsigned state_len,
                                                         unsigned* __restrict__ tickets) {
	__shared__ unsigned h[8][256];
	const unsigned t = threadIdx.x, first = blockIdx.x * kDigitThreads + t, stride = gridDim.x * kDigitThreads;
	for (unsigned i = t; i < passes * 256u; i += kDigitThreads) (&h[0][0])[i] = 0u;
	if (blockIdx.x == 0u && t < 8u) tickets[t] = 0u;
	for (unsigned i = first; i < state_len; i += stride) state[i] = 0ull;
	__syncthreads();
	for (unsigned i = first; i < n; i += stride) {
		const unsigned long long k = key[i];
		for (unsigned p = 0; p < passes; ++p) {
			const unsigned d = (unsigned)(k >> (8u * p)) & 255u;
			// the high digits are often the same on every lane
			const unsigned long long on = __ballot(true);
			if (__ballot(d == __builtin_amdgcn_readfirstlane(d)) == on) {
				if (t % 64u == (unsigned)__builtin_ctzll(on)) atomicAdd(&h[p][d], (unsigned)__popcll(on));
			} else {
				atomicAdd(&h[p][d], 1u);
			}
		}
	}
	__syncthreads();
	for (unsigned i = t; i < passes * 256u; i += kDigitThreads)
		part[(i / 256u * gridDim.x + blockIdx.x) * 256u + i % 256u] = (&h[0][0])[i];
}

// One block per pass: the digits' exclusive prefix over all blocks' counts.
constexpr unsigned kOffsThreads = 1024;
__global__ __launch_bounds__(kOffsThreads) void k_radix_offsets(const unsigned* __restrict__ part, unsigned rows,
                                                                unsigned* __restrict__ offs) {
	__shared__ unsigned cnt[kOffsThreads], ws[4];
	const unsigned t = threadIdx.x, d = t % 256u, lane = t & 63u, w = t >> 6;
	unsigned n = 0;
#pragma unroll 8
	for (unsigned r = t / 256u; r < rows; r += kOffsThreads / 256u) n += part[(blockIdx.x * rows + r) * 256u + d];
	cnt[t] = n;
	__syncthreads();
	n = 0;
	for (unsigned q = d; q < kOffsThreads; q += 256u) n += cnt[q];
	unsigned inc = n;
	for (int o = 1; o < 64; o <<= 1) {
		const unsigned v = __shfl_up(inc, (unsigned)o);
		if ((int)lane >= o) inc += v;
	}
	if (lane == 63u && w < 4u) ws[w] = inc;
	__syncthreads();
	if (w >= 4u) return;
	unsigned excl = inc - n;
	for (unsigned q = 0; q < w; ++q) excl += ws[q];
	offs[blockIdx.x * 256u + t] = excl;
}

// One digit's pass over a tile of 256 PER pairs.  Each wavefront ranks its
// consecutive elements in index order (a 64-lane match mask from eight
// ballots per round, and per-wave running digit counts in LDS); the tile's
// counts are posted, the counts of the tiles before it collected (thread t:
// digit t), the tile is staged in LDS in sorted order and written out by
// consecutive threads, so that each digit's run goes to consecutive global
// addresses.
// State words and tickets as in lookback.h.
template <unsigned PER>
__global__ __launch_bounds__(kBlock) void k_radix_pass(const unsigned long long* __restrict__ key_in,
                                                       const unsigned* __restrict__ val_in, unsigned shift,
                                                       const unsigned* __restrict__ offs,
                                                       unsigned long long* state, unsigned long long* state_next,
                                                       unsigned* tickets, unsigned long long* __restrict__ key_out,
                                                       unsigned* __restrict__ val_out) {
	constexpr unsigned kLook = 2;   // tiles looked back at once
	__shared__ unsigned long long s_key[kBlock * PER];
	__shared__ unsigned s_val[kBlock * PER];
	__shared__ unsigned s_wcnt[kBlock / 64][256];   // running counts, then each wave's prefix
	__shared__ unsigned s_start[256];               // the digit's first slot in the tile
	__shared__ unsigned s_base[256];                // the digit's first global position of this tile
	__shared__ unsigned s_wsum[kBlock / 64];
	__shared__ unsigned s_tile;
	const unsigned t = threadIdx.x, lane = t & 63u, w = t >> 6;
	for (unsigned q = 0; q < kBlock / 64; ++q) s_wcnt[q][t] = 0u;
	const unsigned tile = look::ticket(tickets, s_tile);   // past its barrier s_wcnt is clear
	state_next[(size_t)tile * 256u + t] = 0ull;
	// rank: element r of this thread is tile element (w PER + r) 64 + lane
	const unsigned long long lt = (1ull << lane) - 1ull;
	const size_t g0 = (size_t)tile * (kBlock * PER) + w * (64u * PER) + lane;
	unsigned long long kr[PER];
	unsigned vr[PER], pk[PER];
#pragma unroll
	for (unsigned r = 0; r < PER; ++r) {
		kr[r] = key_in[g0 + 64u * r];
		vr[r] = val_in[g0 + 64u * r];
	}
#pragma unroll
	for (unsigned r = 0; r < PER; ++r) {
		const unsigned d = (unsigned)(kr[r] >> shift) & 255u;
		unsigned long long match = ~0ull;
		for (int bit = 0; bit < 8; ++bit) {
			const unsigned long long b = __ballot((d >> bit) & 1u);
			match &= ((d >> bit) & 1u) ? b : ~b;
		}
		const unsigned before = s_wcnt[w][d];
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		const unsigned rank = __popcll(match & lt);
		if (rank == 0u) s_wcnt[w][d] = before + (unsigned)__popcll(match);
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		pk[r] = (d << 16) | (before + rank);   // before + rank < 64 PER
	}
	__syncthreads();
	// each wave's offset within every digit, and the tile's count
	unsigned cnt = 0;
	for (unsigned q = 0; q < kBlock / 64; ++q) {
		const unsigned c = s_wcnt[q][t];
		s_wcnt[q][t] = cnt;
		cnt += c;
	}
	unsigned long long* mine = state + (size_t)tile * 256u + t;
	look::post(mine, (tile ? look::kOwn : look::kAll) | cnt);
	// exclusive scan of the tile's 256 digit counts
	unsigned inc = cnt;
	for (int k = 1; k < 64; k <<= 1) {
		const unsigned v = __shfl_up(inc, (unsigned)k);
		if ((int)lane >= k) inc += v;
	}
	if (lane == 63u) s_wsum[w] = inc;
	unsigned prior = 0;
	for (int j = (int)tile - 1; j >= 0;) {
		unsigned long long v[kLook];
#pragma unroll
		for (unsigned q = 0; q < kLook; ++q)
			v[q] = j >= (int)q ? look::peek(state + (size_t)(j - (int)q) * 256u + t) : look::kAll;
		bool done = false;
#pragma unroll
		for (unsigned q = 0; q < kLook; ++q) {
			if (done || j < (int)q) continue;
			while (v[q] == 0ull) v[q] = look::peek(state + (size_t)(j - (int)q) * 256u + t);
			prior += (unsigned)v[q];
			done = v[q] >= look::kAll;
		}
		if (done) break;
		j -= (int)kLook;
	}
	if (tile) look::post(mine, look::kAll | (unsigned long long)(prior + cnt));
	s_base[t] = offs[t] + prior;
	__syncthreads();
	unsigned excl = inc - cnt;
	for (unsigned q = 0; q < w; ++q) excl += s_wsum[q];
	s_start[t] = excl;
	__syncthreads();
#pragma unroll
	for (unsigned r = 0; r < PER; ++r) {
		const unsigned d = pk[r] >> 16;
		const unsigned slot = s_start[d] + s_wcnt[w][d] + (pk[r] & 0xFFFFu);
		s_key[slot] = kr[r];
		s_val[slot] = vr[r];
	}
	__syncthreads();
#pragma unroll
	for (unsigned r = 0; r < PER; ++r) {
		const unsigned slot = r * kBlock + t;
		const unsigned long long k = s_key[slot];
		const unsigned d = (unsigned)(k >> shift) & 255u;
		const unsigned dst = s_base[d] + slot - s_start[d];
		key_out[dst] = k;
		val_out[dst] = s_val[slot];
	}
}

// ---------------------------------------------------------------- tree
__global__ __launch_bounds__(kBlock) void k_gather_sorted(const float4* __restrict__ packed,
                                                          const unsigned* __restrict__ order, unsigned N,
                                                          float4* __restrict__ body,
                                                          unsigned long long* __restrict__ start, unsigned words) {
	const unsigned p = blockIdx.x * kBlock + threadIdx.x;
	if (p < words) start[p] = 0ull;   // for k_group_flags (words <= the grid's threads)
	if (p >= N) return;
	body[p] = packed[order[p]];
}

__device__ __forceinline__ int delta(const unsigned long long* __restrict__ key, int N, int i, int j) {
	if (j < 0 || j >= N) return -1;
	const unsigned long long a = key[i], b = key[j];
	if (a != b) return __clzll((long long)(a ^ b));
	return 64 + __clz((int)((unsigned)i ^ (unsigned)j));
}

// delta(i, j) > d as two comparisons, for -1 <= d <= 95: the keys (63 bits)
// agree in more than d bits, and if d >= 64 so do the indexes.
struct Longer {
	unsigned long long key_i, below;
	unsigned i, upto;
	int N;
	__device__ __forceinline__ Longer(unsigned long long key_i_, int i_, int N_, int d)
	    : key_i(key_i_), below(d < 0 ? ~0ull : (d < 64 ? 1ull << (63 - d) : 1ull)), i((unsigned)i_),
	      upto(d < 64 ? ~0u : (1u << (95 - d)) - 1u), N(N_) {}
	__device__ __forceinline__ bool operator()(const unsigned long long* __restrict__ key, int j) const {
		return j >= 0 && j < N && (key[j] ^ key_i) < below && (i ^ (unsigned)j) <= upto;
	}
};

// Internal nodes 0..N-2; node id >= N-1 is the leaf of sorted particle
// id - (N-1).  node_lr holds (left, right), node_range (first, count).
// Bound by issue: a wavefront takes as many probes as its largest node, a
// couple of dozen.  Comparisons in place of a count of leading bits per probe:
// 65537 particles 17.3 -> 14.0 us, 1M 45 -> 36, 4M 132 -> 105.  Keeping the keys
// around a block in LDS changed nothing.
__global__ __launch_bounds__(kBlock) void k_karras(const unsigned long long* __restrict__ key, int N,
                                                   int2* __restrict__ node_lr, int2* __restrict__ node_range) {
	const int i = (int)(blockIdx.x * kBlock + threadIdx.x);
	if (i >= N - 1) return;
	const unsigned long long ki = key[i];
	const int up = delta(key, N, i, i + 1), down = delta(key, N, i, i - 1);
	const int d = up - down >= 0 ? 1 : -1;
	const Longer of_node(ki, i, N, min(up, down));
	int lmax = 2;
	while (of_node(key, i + lmax * d)) lmax <<= 1;
	int l = 0;
	for (int t = lmax >> 1; t >= 1; t >>= 1)
		if (of_node(key, i + (l + t) * d)) l += t;
	const int j = i + l * d;
	const Longer of_child(ki, i, N, delta(key, N, i, j));
	int s = 0;
	for (int k = 1;; ++k) {
		const int t = (l + (1 << k) - 1) >> k;
		if (of_child(key, i + (s + t) * d)) s += t;
		if (t <= 1) break;
	}
	const int gamma = i + s * d + min(d, 0);
	const int lo = min(i, j), hi = max(i, j);
	const int left = (lo == gamma) ? (N - 1) + gamma : gamma;
	const int right = (hi == gamma + 1) ? (N - 1) + gamma + 1 : gamma + 1;
	node_lr[i] = make_int2(left, right);
	node_range[i] = make_int2(lo, hi - lo + 1);
}

// ---- FP64 inclusive prefix sums over the sorted particles of (m, m x, m y,
// m z) and, for quadrupoles, of m x' x'^T (x' = x - ref, six components).
// Fixed shape: spans of 1024 elements, summed by a wavefront each, 64 consecutive
// elements at a time; tiles of four spans, whose sums one block scans; then
// every span scanned in 64s from what lies before it.
struct d4 {
	double m, x, y, z;
	__device__ static d4 zero() { return {0.0, 0.0, 0.0, 0.0}; }
	__device__ static d4 of(float4 b, const double*) {
		const double m = b.w;
		return {m, m * (double)b.x, m * (double)b.y, m * (double)b.z};
	}
	__device__ d4 operator+(const d4& o) const { return {m + o.m, x + o.x, y + o.y, z + o.z}; }
	__device__ d4 shfl_up(unsigned o) const {
		return {__shfl_up(m, o), __shfl_up(x, o), __shfl_up(y, o), __shfl_up(z, o)};
	}
};
struct d6 {   // xx, xy, xz, yy, yz, zz
	double v[6];
	__device__ static d6 zero() { return {{0.0, 0.0, 0.0, 0.0, 0.0, 0.0}}; }
	__device__ static d6 of(float4 b, const double* ref) {
		const double m = b.w, x = (double)b.x - ref[0], y = (double)b.y - ref[1], z = (double)b.z - ref[2];
		return {{m * x * x, m * x * y, m * x * z, m * y * y, m * y * z, m * z * z}};
	}
	__device__ d6 operator+(const d6& o) const {
		d6 r;
		for (int k = 0; k < 6; ++k) r.v[k] = v[k] + o.v[k];
		return r;
	}
	__device__ d6 shfl_up(unsigned o) const {
		d6 r;
		for (int k = 0; k < 6; ++k) r.v[k] = __shfl_up(v[k], o);
		return r;
	}
};

constexpr unsigned kScanPer = 16;
constexpr unsigned kScanSpan = 64 * kScanPer;   // consecutive elements summed by a wavefront
constexpr unsigned kScanSpans = 4;              // in a tile
constexpr unsigned kScanTile = kScanSpans * kScanSpan;

template <class R>
__device__ R block_exclusive_scan(R v, R* sh) {
	const unsigned t = threadIdx.x;
	sh[t] = v;
	__syncthreads();
	for (unsigned off = 1; off < kBlock; off <<= 1) {
		const R o = t >= off ? sh[t - off] : R::zero();
		__syncthreads();
		sh[t] = sh[t] + o;
		__syncthreads();
	}
	const R excl = t ? sh[t - 1] : R::zero();
	__syncthreads();
	return excl;
}

// Span sums, and tile sums from them: a wavefront reads its span 64
// consecutive elements at a time and adds its lanes in a fixed order, then
// wave 0 adds the tile's spans in order.
template <class R>
__global__ __launch_bounds__(kBlock) void k_scan_tiles(const float4* __restrict__ body, unsigned N,
                                                       const double* __restrict__ ref, R* __restrict__ tile_sum,
                                                       R* __restrict__ span_sum) {
	static_assert(kScanSpans == kBlock / 64, "a wavefront per span");
	__shared__ R sh[kScanSpans];
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned first = blockIdx.x * kScanTile + w * kScanSpan;
	R s = R::zero();
	for (unsigned r = 0; r < kScanPer; ++r) {
		const unsigned i = first + 64u * r + lane;
		if (i < N) s = s + R::of(body[i], ref);
	}
	for (unsigned o = 1; o < 64; o <<= 1) {
		const R t = s.shfl_up(o);
		if (lane >= o) s = s + t;
	}
	if (lane == 63u) {
		sh[w] = s;
		span_sum[blockIdx.x * kScanSpans + w] = s;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		R t = sh[0];
		for (unsigned q = 1; q < kScanSpans; ++q) t = t + sh[q];
		tile_sum[blockIdx.x] = t;
	}
}

template <class R>
__global__ __launch_bounds__(kBlock) void k_scan_tile_sums(R* __restrict__ tile_sum, unsigned ntiles) {
	__shared__ R sh[kBlock];
	const unsigned chunk = (ntiles + kBlock - 1) / kBlock;
	const unsigned b = threadIdx.x * chunk, e = min(b + chunk, ntiles);
	R s = R::zero();
	for (unsigned k = b; k < e; ++k) s = s + tile_sum[k];
	R run = block_exclusive_scan(s, sh);
	for (unsigned k = b; k < e; ++k) {
		const R v = tile_sum[k];
		tile_sum[k] = run;       // exclusive offset of tile k
		run = run + v;
	}
}

// Inclusive prefix of a span: each wavefront scans four of its sixteen 64s
// (interleaved: a lane scan is a chain of six exchanges), which start from the
// tile's offset, the spans before and the 64s before, added in order.  (One
// wavefront taking all sixteen in turn, after summing the span again for the
// offsets, took 18.4 us at 65537 particles and 56 at 4M, 83 with second
// moments; this 7.0, 45 and 67.)
template <class R>
__global__ __launch_bounds__(kBlock) void k_scan_write(const float4* __restrict__ body, unsigned N,
                                                       const double* __restrict__ ref, const R* __restrict__ tile_off,
                                                       const R* __restrict__ span_sum, R* __restrict__ prefix) {
	constexpr unsigned kRounds = kScanPer / (kBlock / 64);
	__shared__ R sh[kScanPer];
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned tile = blockIdx.x / kScanSpans, span = blockIdx.x % kScanSpans;
	const unsigned first = blockIdx.x * kScanSpan + w * 64u * kRounds + lane;
	R v[kRounds];
#pragma unroll
	for (unsigned k = 0; k < kRounds; ++k) v[k] = first + 64u * k < N ? R::of(body[first + 64u * k], ref) : R::zero();
	for (unsigned o = 1; o < 64; o <<= 1) {
#pragma unroll
		for (unsigned k = 0; k < kRounds; ++k) {
			const R t = v[k].shfl_up(o);
			if (lane >= o) v[k] = v[k] + t;
		}
	}
	if (lane == 63u)
		for (unsigned k = 0; k < kRounds; ++k) sh[w * kRounds + k] = v[k];
	R run = tile_off[tile];
	for (unsigned q = 0; q < span; ++q) run = run + span_sum[tile * kScanSpans + q];
	__syncthreads();
	for (unsigned q = 0; q < w * kRounds; ++q) run = run + sh[q];
#pragma unroll
	for (unsigned k = 0; k < kRounds; ++k) {
		if (first + 64u * k < N) prefix[first + 64u * k] = run + v[k];   // inclusive
		run = run + sh[w * kRounds + k];
	}
}

// Reference point of the second-moment prefix sums: the global centre of
// mass (the last first-moment prefix), so that the sums stay of the order of
// the system's own second moment (a point far from the mass, such as the
// centre of a bounding cube stretched by one distant particle, would make
// them large and the differences S - M c c^T of small nodes meaningless).
__global__ void k_quad_ref(const d4* __restrict__ prefix, unsigned N, double* __restrict__ ref) {
	if (threadIdx.x >= 3) return;
	const d4 t = prefix[N - 1];
	const double c = threadIdx.x == 0 ? t.x : (threadIdx.x == 1 ? t.y : t.z);
	ref[threadIdx.x] = t.m > 0.0 ? c / t.m : 0.0;
}

// Traceless quadrupole Qt = 3 Q - tr(Q) I of every internal node about its
// centre of mass, Q = sum m (x - c)(x - c)^T; stored as q0 = (Qxx, Qxy, Qxz,
// Qyy), q1 = Qyz (Qzz = -Qxx - Qyy).  Nodes of at most kQuadDirect particles
// sum directly in FP64, in one pass over offsets from their first particle
// (Q = S' - M c' c'^T with S' and c' about that particle, whose terms are of
// the node's own size); larger nodes use the prefix differences S - M c c^T.
// In FP64 the prefix rounding measured at most 1.2e-6 of M l^2 (l the
// node's longest side) for nodes of 16 particles and 3.5e-7 for 32, on a
// Plummer sphere of 4M particles with outliers at up to 1000 scale radii
// (sequential prefix sums, which round worse than this blocked scan).  Each thread sums its own node, so a
// wavefront takes as long as its largest node: with 256 here the kernel took
// 0.74 ms at 4M particles.  Single-particle leaves have Qt = 0.
constexpr int kQuadDirect = 16;

__global__ __launch_bounds__(kBlock) void k_node_quad(int N, const int2* __restrict__ node_range,
                                                      const float4* __restrict__ body, const d4* __restrict__ prefix,
                                                      const d6* __restrict__ prefix2, const double* __restrict__ ref,
                                                      float4* __restrict__ q0, float* __restrict__ q1) {
	const int n = (int)(blockIdx.x * kBlock + threadIdx.x);
	if (n >= 2 * N - 1) return;
	if (n >= N - 1) {
		q0[n] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		q1[n] = 0.0f;
		return;
	}
	const int2 rg = node_range[n];
	const int f = rg.x, l = rg.x + rg.y - 1;
	const d4 a = f > 0 ? prefix[f - 1] : d4::zero();
	const d4 b = prefix[l];
	const double M = b.m - a.m;
	if (!(M > 0.0)) {
		q0[n] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		q1[n] = 0.0f;
		return;
	}
	double qxx, qxy, qxz, qyy, qyz, qzz;
	if (rg.y <= kQuadDirect) {
		const float4 p0 = body[f];
		double sm = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
		qxx = qxy = qxz = qyy = qyz = qzz = 0.0;
		for (int k = f; k <= l; ++k) {
			const float4 p = body[k];
			const double m = p.w, x = (double)p.x - (double)p0.x, y = (double)p.y - (double)p0.y,
			             z = (double)p.z - (double)p0.z;
			sm += m;
			sx += m * x;
			sy += m * y;
			sz += m * z;
			qxx += m * x * x;
			qxy += m * x * y;
			qxz += m * x * z;
			qyy += m * y * y;
			qyz += m * y * z;
			qzz += m * z * z;
		}
		const double cx = sx / sm, cy = sy / sm, cz = sz / sm;
		qxx -= sm * cx * cx;
		qxy -= sm * cx * cy;
		qxz -= sm * cx * cz;
		qyy -= sm * cy * cy;
		qyz -= sm * cy * cz;
		qzz -= sm * cz * cz;
	} else {
		const d6 a2 = f > 0 ? prefix2[f - 1] : d6::zero(), b2 = prefix2[l];
		// centre of mass relative to ref
		const double cx = (b.x - a.x) / M - ref[0], cy = (b.y - a.y) / M - ref[1], cz = (b.z - a.z) / M - ref[2];
		qxx = (b2.v[0] - a2.v[0]) - M * cx * cx;
		qxy = (b2.v[1] - a2.v[1]) - M * cx * cy;
		qxz = (b2.v[2] - a2.v[2]) - M * cx * cz;
		qyy = (b2.v[3] - a2.v[3]) - M * cy * cy;
		qyz = (b2.v[4] - a2.v[4]) - M * cy * cz;
		qzz = (b2.v[5] - a2.v[5]) - M * cz * cz;
	}
	const double tr = qxx + qyy + qzz;
	q0[n] = make_float4((float)(3.0 * qxx - tr), (float)(3.0 * qxy), (float)(3.0 * qxz), (float)(3.0 * qyy - tr));
	q1[n] = (float)(3.0 * qyz);
	(void)qzz;
}

__device__ __forceinline__ unsigned compact21(unsigned long long v) {
	v &= 0x1249249249249249ull;
	v = (v | (v >> 2)) & 0x10C30C30C30C30C3ull;
	v = (v | (v >> 4)) & 0x100F00F00F00F00Full;
	v = (v | (v >> 8)) & 0x1F0000FF0000FFull;
	v = (v | (v >> 16)) & 0x1F00000000FFFFull;
	v = (v | (v >> 32)) & 0x1FFFFFull;
	return (unsigned)v;
}

// Nodes of at most this many particles take their particles' bounding box as
// their size in the opening test; larger ones their Morton cell.  Each
// thread scans its node's range, so a wavefront takes as long as its largest
// node: 64 kept the build at ~0.15 ms more than Morton cells alone, where 256
// cost ~0.3 ms, for 0.7 % more interactions (a CPU model of the walk).
constexpr int kAabbNode = 64;

// Monopole (node_cm) of every node, and the box of its opening test
// (node_cell: centre, longest side): the bounding box of its particles for
// nodes of at most kAabbNode particles (a point for a leaf), its Morton cell
// above.  For small nodes the particles' box is often much smaller than the
// Morton cell, so at equal accuracy the walk accepts cells sooner (a CPU model
// of the walk at N = 1M: 15 % fewer interactions and 12 % fewer node visits
// for the same 99th-percentile force error).
__global__ __launch_bounds__(kBlock) void k_node_moments(const float4* __restrict__ body, int N,
                                                         const unsigned long long* __restrict__ key,
                                                         const int2* __restrict__ node_range,
                                                         const d4* __restrict__ prefix, const double* __restrict__ box,
                                                         float4* __restrict__ node_cm, float4* __restrict__ node_cell) {
	const int n = (int)(blockIdx.x * kBlock + threadIdx.x);
	if (n >= 2 * N - 1) return;
	if (n >= N - 1) {
		const float4 b = body[n - (N - 1)];
		node_cm[n] = b;
		node_cell[n] = make_float4(b.x, b.y, b.z, 0.0f);
		return;
	}
	const int2 rg = node_range[n];
	const int f = rg.x, l = rg.x + rg.y - 1;
	const d4 hi = prefix[l];
	const d4 lo = f > 0 ? prefix[f - 1] : d4::zero();
	const double M = hi.m - lo.m;
	// cell of the common code prefix: p leading bits of the 63-bit code
	const unsigned long long ka = key[f], kb = key[l];
	const int p = ka == kb ? 63 : __clzll((long long)(ka ^ kb)) - 1;
	const double inv_scale = 1.0 / box[3];
	double centre[3];
	int bmin = 21;
	for (int a = 0; a < 3; ++a) {
		const int bits = max(p - a + 2, 0) / 3;   // code bits fixed on this axis
		bmin = min(bmin, bits);
		const unsigned q = compact21(ka >> (2 - a));
		const unsigned span = 1u << (21 - bits);
		const unsigned q0 = bits == 0 ? 0u : (q & ~(span - 1u));
		centre[a] = box[a] + ((double)q0 + 0.5 * (double)span) * inv_scale;
	}
	const double side = (double)(1u << (21 - bmin)) * inv_scale;
	float4 cm;
	if (M > 0.0) {
		cm = make_float4((float)((hi.x - lo.x) / M), (float)((hi.y - lo.y) / M), (float)((hi.z - lo.z) / M),
		                 (float)M);
	} else {
		cm = make_float4((float)centre[0], (float)centre[1], (float)centre[2], 0.0f);
	}
	node_cm[n] = cm;
	if (rg.y <= kAabbNode) return;   // its particles' box: k_group_boxes
	node_cell[n] = make_float4((float)centre[0], (float)centre[1], (float)centre[2], (float)side);
}

// The opening-test boxes of the internal nodes of at most kAabbNode
// particles: their particles' bounding box (centre, longest side).  These
// are the internal nodes of the walk groups, the maximal subtrees of at most
// 64 particles, and a radix-tree node's index is one end of its range, so a
// group's internal nodes are the indices of its sorted range whose range
// lies inside it.  One wavefront per group: a sparse table of min and max
// over the group's particles (windows of 2^k particles, k = 0 .. 6) in LDS,
// then one lane per internal node combines the two windows that cover its
// range.  Min and max are exact, so each box equals a scan over the node's
// range.
constexpr int kBoxLevels = 7;
constexpr unsigned kBoxWaves = kBlock / 64;
static_assert(kAabbNode == 64, "the walk groups hold at most 64 particles");
__global__ __launch_bounds__(kBlock) void k_group_boxes(const float4* __restrict__ body, int N,
                                                        const unsigned long long* __restrict__ start,
                                                        const int2* __restrict__ node_range,
                                                        float4* __restrict__ node_cell) {
	// one table at a time (the minima, then the maxima): 7 KiB per wavefront
	__shared__ float s_tab[kBoxWaves][kBoxLevels][3][64];
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned c = blockIdx.x * kBoxWaves + w;   // chunk of 64 sorted positions
	if (c >= ((unsigned)N + 63u) / 64u) return;
	// the groups that start in the chunk; each ends at the next start flag,
	// at most 64 positions later (start[N] is set)
	const unsigned at = 64u * c + lane;
	const unsigned long long e1 = start[c], e2 = start[c + 1u];
	unsigned long long rem = e1 & __ballot(at < (unsigned)N);
	if (!rem) return;
	// the bodies and node ranges of the chunk and of the part of the next one
	// that its last group reaches, loaded once and handed to each group by
	// lane shuffles
	const int over = e2 ? __builtin_ctzll(e2) : 64;
	const int p0 = (int)at, p1 = p0 + 64;
	const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
	const float4 b0 = p0 < N ? body[p0] : zero4;
	const float4 b1 = ((int)lane < over && p1 < N) ? body[p1] : zero4;
	const int2 r0 = p0 < N - 1 ? node_range[p0] : make_int2(0, 0);
	const int2 r1 = ((int)lane < over && p1 < N - 1) ? node_range[p1] : make_int2(0, 0);
	while (rem) {
		const int s0 = __builtin_ctzll(rem);
		rem &= rem - 1ull;
		const unsigned long long above = s0 < 63 ? e1 & (~0ull << (s0 + 1)) : 0ull;
		const int e0 = above ? __builtin_ctzll(above) : (e2 ? 64 + __builtin_ctzll(e2) : 128);
		const int base = 64 * (int)c + s0;
		const int cnt = min(min(e0 - s0, 64), N - base);
		if (cnt < 2) continue;   // a single particle: no internal node
		const bool live = (int)lane < cnt;
		// position base + lane: lane s0 + lane of the chunk's loads, or of the
		// next chunk's.  Every lane takes part in every shuffle (a lane left
		// out of a shuffle does not provide its value to the others), and
		// then picks its half.
		const int src = (s0 + (int)lane) & 63;
		const bool hi_half = s0 + (int)lane >= 64;
		const float x0 = __shfl(b0.x, src), y0 = __shfl(b0.y, src), z0 = __shfl(b0.z, src);
		const float x1 = __shfl(b1.x, src), y1 = __shfl(b1.y, src), z1 = __shfl(b1.z, src);
		const int f0 = __shfl(r0.x, src), n0 = __shfl(r0.y, src);
		const int f1 = __shfl(r1.x, src), n1 = __shfl(r1.y, src);
		const float4 b = hi_half ? make_float4(x1, y1, z1, 0.f) : make_float4(x0, y0, z0, 0.f);
		const int2 rg = hi_half ? make_int2(f1, n1) : make_int2(f0, n0);
		const int idx = base + (int)lane;
		// an internal node of this group: its range lies inside the group
		const bool node = live && idx < N - 1 && rg.x >= base && rg.x + rg.y <= base + cnt;
		const int a0 = rg.x - base, len = max(rg.y, 1);
		const int k = 31 - __clz(len);
		const int a1 = a0 + len - (1 << k);
		float l3[3], h3[3];
#pragma unroll
		for (int pass = 0; pass < 2; ++pass) {
			float v[3] = {b.x, b.y, b.z};
#pragma unroll
			for (int lv = 0; lv < kBoxLevels; ++lv) {
				if (lv > 0) {
					// window [j, j + 2^lv) from [j, j + 2^(lv-1)) and the next one;
					// the windows that run past the group are never read
					const unsigned d = 1u << (lv - 1);
#pragma unroll
					for (int a = 0; a < 3; ++a) {
						const float o = __shfl_down(v[a], d);
						v[a] = pass ? fmaxf(v[a], o) : fminf(v[a], o);
					}
				}
#pragma unroll
				for (int a = 0; a < 3; ++a) s_tab[w][lv][a][lane] = v[a];
			}
			__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
			if (node) {
#pragma unroll
				for (int a = 0; a < 3; ++a) {
					const float x0 = s_tab[w][k][a][a0], x1 = s_tab[w][k][a][a1];
					if (pass) h3[a] = fmaxf(x0, x1);
					else l3[a] = fminf(x0, x1);
				}
			}
			__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		}
		if (node) {
			const float side_box = fmaxf(fmaxf(h3[0] - l3[0], h3[1] - l3[1]), h3[2] - l3[2]);
			node_cell[idx] =
			    make_float4(0.5f * (l3[0] + h3[0]), 0.5f * (l3[1] + h3[1]), 0.5f * (l3[2] + h3[2]), side_box);
		}
	}
}

// Walk records: (r_crit^2, a, b, q) with r_crit = side / theta +
// |com - box centre| (node_cell's box).  Nodes of at most leaf_size particles
// carry (a, b) = (first, count) and the sign bit of the r_crit^2 word set;
// larger ones (left, right).  q is the node's size l = side (float bits),
// which the relative opening test takes to M l^2 and M l^3.
__global__ __launch_bounds__(kBlock) void k_records(int N, const int2* __restrict__ node_lr,
                                                    const int2* __restrict__ node_range,
                                                    const float4* __restrict__ node_cm,
                                                    const float4* __restrict__ node_cell, float inv_theta,
                                                    int leaf_size, int4* __restrict__ rec_b,
                                                    unsigned long long* __restrict__ counters) {
	const int n = (int)(blockIdx.x * kBlock + threadIdx.x);
	// the walk's counters, but the fifth, which lasts until the host clears it
	if (blockIdx.x == 0u && threadIdx.x < 6u && threadIdx.x != 4u) counters[threadIdx.x] = 0ull;
	if (n >= 2 * N - 1) return;
	int first, count, l = -1, r = -1;
	if (n < N - 1) {
		const int2 rg = node_range[n];
		first = rg.x;
		count = rg.y;
		l = node_lr[n].x;
		r = node_lr[n].y;
	} else {
		first = n - (N - 1);
		count = 1;
	}
	const float4 cm = node_cm[n], cell = node_cell[n];
	const float ox = cm.x - cell.x, oy = cm.y - cell.y, oz = cm.z - cell.z;
	const float rc = cell.w * inv_theta + sqrtf(ox * ox + oy * oy + oz * oz);
	const bool leafy = count <= leaf_size;
	const int rc2 = __float_as_int(rc * rc) | (leafy ? (int)0x80000000u : 0);
	rec_b[n] = make_int4(rc2, leafy ? first : l, leafy ? count : r, __float_as_int(cell.w));
}

// Walk groups: the maximal subtrees holding at most `cap` particles.  They
// partition the sorted order into runs of at most cap particles that each lie
// inside one Morton cell; bit p of start is set where a run begins, bit N ends
// the last run.  `start` is zero beforehand.
__global__ __launch_bounds__(kBlock) void k_group_flags(int N, const int2* __restrict__ node_lr,
                                                        const int2* __restrict__ node_range, int cap,
                                                        unsigned long long* __restrict__ start) {
	const int i = (int)(blockIdx.x * kBlock + threadIdx.x);
	if (i == 0) {
		atomicOr(&start[N >> 6], 1ull << (N & 63));
		if (N <= cap) atomicOr(&start[0], 1ull);   // the root (a single leaf when N == 1) is the only group
	}
	if (i >= N - 1) return;
	if (node_range[i].y <= cap) return;
	const int2 lr = node_lr[i];
	const int child[2] = {lr.x, lr.y};
	for (int k = 0; k < 2; ++k) {
		const int c = child[k];
		const int2 rg = c >= N - 1 ? make_int2(c - (N - 1), 1) : node_range[c];
		if (rg.y <= cap) atomicOr(&start[rg.x >> 6], 1ull << (rg.x & 63));
	}
}

// The set bits of start in order, as a list (the last is N, the end of the last
// group), and the number of groups.  A block takes 1024 words; each adds up the
// words before its own itself, 256 KiB on average at 4M particles, instead of a
// scan in launches of its own.
constexpr unsigned kListBlock = 1024;
__global__ __launch_bounds__(kListBlock) void k_group_list(const unsigned long long* __restrict__ start,
                                                           unsigned words, unsigned* __restrict__ list,
                                                           unsigned* __restrict__ n_groups) {
	__shared__ unsigned s_sum[2][kListBlock / 64];
	const unsigned t = threadIdx.x, lane = t & 63u, w = t >> 6, first = blockIdx.x * kListBlock;
	unsigned before = 0;
	for (unsigned i = t; i < first; i += kListBlock) before += (unsigned)__popcll(start[i]);
	const unsigned long long v = first + t < words ? start[first + t] : 0ull;
	const unsigned n = (unsigned)__popcll(v);
	unsigned incl = n;
#pragma unroll
	for (int o = 1; o < 64; o <<= 1) {
		const unsigned up = __shfl_up(incl, (unsigned)o);
		if ((int)lane >= o) incl += up;
	}
	for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
	if (lane == 63u) s_sum[0][w] = incl;
	if (lane == 0u) s_sum[1][w] = before;
	__syncthreads();
	unsigned at = incl - n;
	for (unsigned k = 0; k < kListBlock / 64; ++k) at += s_sum[1][k] + (k < w ? s_sum[0][k] : 0u);
	for (unsigned long long rem = v; rem; rem &= rem - 1ull) list[at++] = 64u * (first + t) + (unsigned)__builtin_ctzll(rem);
	if (v && first + t + 1u == words) *n_groups = at - 1u;   // the last word holds bit N alone or last
}

}  // namespace

extern "C" {

unsigned sfd_lbvh_group_words(unsigned N) { return N / 64u + 2u; }

int sfd_lbvh_groups(unsigned N, const void* node_lr, const void* node_range, int cap,
                    unsigned long long* start, hipStream_t s) {
	if (N == 0 || cap < 1 || cap > 64) return -1;
	const unsigned threads = N > 1 ? N - 1 : 1;
	hipLaunchKernelGGL(k_group_flags, dim3((threads + kBlock - 1) / kBlock), dim3(kBlock), 0, s, (int)N,
	                   static_cast<const int2*>(node_lr), static_cast<const int2*>(node_range), cap, start);
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_groups", "launch");
}

int sfd_lbvh_group_list(unsigned N, const unsigned long long* start, unsigned* list, unsigned* n_groups,
                        hipStream_t s) {
	if (N == 0) return 0;
	const unsigned words = N / 64u + 1u;   // bit N is in the last of them
	hipLaunchKernelGGL(k_group_list, dim3((words + kListBlock - 1u) / kListBlock), dim3(kListBlock), 0, s, start, words,
	                   list, n_groups);
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_group_list", "launch");
}

int sfd_lbvh_group_boxes(unsigned N, const void* body, const unsigned long long* start, const void* node_range,
                         void* node_cell, hipStream_t s) {
	if (N < 2) return 0;
	const unsigned chunks = (N + 63u) / 64u;
	hipLaunchKernelGGL(k_group_boxes, dim3((chunks + kBoxWaves - 1) / kBoxWaves), dim3(kBlock), 0, s,
	                   static_cast<const float4*>(body), (int)N, start, static_cast<const int2*>(node_range),
	                   static_cast<float4*>(node_cell));
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_group_boxes", "launch");
}

unsigned sfd_lbvh_bbox_blocks(void) { return 256u; }

int sfd_lbvh_keys(const float* pos, const float* mas, unsigned N, unsigned n_sort, double* bbox_part, double* box,
                  unsigned long long* key, unsigned* val, void* packed, hipStream_t s) {
	const unsigned nb = sfd_lbvh_bbox_blocks();
	if (N == 0 || n_sort % kTile != 0) return -1;
	hipLaunchKernelGGL(k_bbox_partial, dim3(nb), dim3(kBlock), 0, s, pos, N, bbox_part);
	hipLaunchKernelGGL(k_bbox_final, dim3(1), dim3(kBlock), 0, s, bbox_part, nb, box);
	hipLaunchKernelGGL(k_morton, dim3((n_sort + kBlock - 1) / kBlock), dim3(kBlock), 0, s, pos, mas, N, n_sort, box,
	                   key, val, static_cast<float4*>(packed));
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_keys", "launch");
}

unsigned sfd_radix_tile(void) { return kTile; }

// Tiles of 1024 pairs up to this many, for sorts that leave most CUs idle (a
// pass over 65536 pairs: 512 pairs 10.7 us, 1024 9.2, 2048 9.1), and of 4096
// above, where each tile's collection costs more (1M: 1024 pairs 38 us, 2048
// 26, 4096 21, 6144 21; 4M: 101, 64, 47, 44; the choices compared at 8 tiles
// looked back).
constexpr unsigned kSmallSort = 1u << 19, kPerSmall = 4, kPerLarge = 16;
static unsigned radix_tiles(unsigned n_sort) { return n_sort / (kBlock * (n_sort <= kSmallSort ? kPerSmall : kPerLarge)); }

// two passes' state words, the blocks' digit counts and offsets of 8 passes, tickets
unsigned sfd_radix_hist_entries(unsigned n_sort) {
	// no fewer than any smaller sort's
	const unsigned ntiles = max(radix_tiles(n_sort), radix_tiles(min(n_sort, kSmallSort)));
	return 2u * 2u * 256u * ntiles + 8u * 256u * (kDigitBlocks + 1u) + 8u;
}

static unsigned scan_tiles(unsigned N) { return (N + kScanTile - 1) / kScanTile; }
unsigned sfd_lbvh_scan_records(unsigned N) { return (1u + kScanSpans) * scan_tiles(N); }

// Sorts n_sort (a multiple of the tile) pairs on the low 8 * passes key bits;
// the result ends in (key0, val0) after an even number of passes and in
// (key1, val1) after an odd one.  hist: sfd_radix_hist_entries(n_sort), 8-byte
// aligned.
int sfd_radix_sort_passes(unsigned long long* key0, unsigned* val0, unsigned long long* key1, unsigned* val1,
                          unsigned n_sort, unsigned* hist, unsigned passes, hipStream_t s) {
	if (n_sort % kTile != 0 || passes > 8u) return -1;
	if (n_sort == 0 || passes == 0) return 0;
	const unsigned ntiles = radix_tiles(n_sort), len = 256u * ntiles;
	unsigned long long* state = reinterpret_cast<unsigned long long*>(hist);
	unsigned* part = hist + 4u * (size_t)len;
	const unsigned rows = min(kDigitBlocks, (n_sort + kDigitThreads - 1u) / kDigitThreads);
	unsigned* offs = part + 8u * 256u * kDigitBlocks;
	unsigned* tickets = offs + 8u * 256u;
	hipLaunchKernelGGL(k_radix_digits, dim3(rows), dim3(kDigitThreads), 0, s, key0, n_sort, passes, part, state, len, tickets);
	hipLaunchKernelGGL(k_radix_offsets, dim3(passes), dim3(kOffsThreads), 0, s, part, rows, offs);
	for (unsigned pass = 0; pass < passes; ++pass) {
		const bool odd = pass & 1u;
		hipLaunchKernelGGL((n_sort <= kSmallSort ? k_radix_pass<kPerSmall> : k_radix_pass<kPerLarge>), dim3(ntiles), dim3(kBlock), 0, s,
		                   odd ? key1 : key0, odd ? val1 : val0, 8u * pass, offs + 256u * pass,
		                   state + (odd ? len : 0u), state + (odd ? 0u : len), tickets + pass, odd ? key0 : key1,
		                   odd ? val0 : val1);
	}
	return sf_hip_check(hipGetLastError(), "sfd_radix_sort", "launch");
}

int sfd_radix_sort(unsigned long long* key0, unsigned* val0, unsigned long long* key1, unsigned* val1,
                   unsigned n_sort, unsigned* hist, hipStream_t s) {
	return sfd_radix_sort_passes(key0, val0, key1, val1, n_sort, hist, 8u, s);
}

// prefix: N records of 4 doubles; tile_sum: sfd_lbvh_scan_records(N) records
int sfd_lbvh_topology(const unsigned long long* key, const unsigned* order, unsigned N, const double* box, void* body,
                      void* node_lr, void* node_range, void* prefix, void* tile_sum, void* node_cm, void* node_cell,
                      unsigned long long* start, hipStream_t s) {
	const unsigned g = (N + kBlock - 1) / kBlock;
	float4* b4 = static_cast<float4*>(body);
	int2* rg = static_cast<int2*>(node_range);
	d4* pre = static_cast<d4*>(prefix);
	d4* ts = static_cast<d4*>(tile_sum);
	const unsigned ntiles = scan_tiles(N), nspans = (N + kScanSpan - 1u) / kScanSpan;
	const int tok = sf_prof_begin("lbvh_topology", s);
	// the packed records of sfd_lbvh_keys, in the prefix buffer until the scan overwrites it
	hipLaunchKernelGGL(k_gather_sorted, dim3(g), dim3(kBlock), 0, s, reinterpret_cast<const float4*>(prefix), order, N,
	                   b4, start, sfd_lbvh_group_words(N));
	if (N > 1)
		hipLaunchKernelGGL(k_karras, dim3((N - 1 + kBlock - 1) / kBlock), dim3(kBlock), 0, s, key, (int)N,
		                   static_cast<int2*>(node_lr), rg);
	hipLaunchKernelGGL(k_scan_tiles<d4>, dim3(ntiles), dim3(kBlock), 0, s, b4, N, (const double*)nullptr, ts,
	                   ts + ntiles);
	hipLaunchKernelGGL(k_scan_tile_sums<d4>, dim3(1), dim3(kBlock), 0, s, ts, ntiles);
	hipLaunchKernelGGL(k_scan_write<d4>, dim3(nspans), dim3(kBlock), 0, s, b4, N, (const double*)nullptr, ts,
	                   ts + ntiles, pre);
	const unsigned nn = 2u * N - 1u;
	hipLaunchKernelGGL(k_node_moments, dim3((nn + kBlock - 1) / kBlock), dim3(kBlock), 0, s, b4, (int)N, key, rg, pre,
	                   box, static_cast<float4*>(node_cm), static_cast<float4*>(node_cell));
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_topology", "launch");
}

// Traceless quadrupoles of every node (after sfd_lbvh_topology): prefix2 is
// N records of 6 doubles, tile_sum2 sfd_lbvh_scan_records(N) of them, ref 3
// doubles; node_q0 / node_q1 are 2N-1 float4 / float.
int sfd_lbvh_quadrupoles(unsigned N, const void* body, const void* node_range, const void* prefix, const double* box,
                         void* prefix2, void* tile_sum2, double* ref, void* node_q0, float* node_q1, hipStream_t s) {
	(void)box;
	if (N == 0) return 0;
	const float4* b4 = static_cast<const float4*>(body);
	d6* pre2 = static_cast<d6*>(prefix2);
	d6* ts2 = static_cast<d6*>(tile_sum2);
	const unsigned ntiles = scan_tiles(N), nspans = (N + kScanSpan - 1u) / kScanSpan;
	hipLaunchKernelGGL(k_quad_ref, dim3(1), dim3(64), 0, s, static_cast<const d4*>(prefix), N, ref);
	hipLaunchKernelGGL(k_scan_tiles<d6>, dim3(ntiles), dim3(kBlock), 0, s, b4, N, (const double*)ref, ts2,
	                   ts2 + ntiles);
	hipLaunchKernelGGL(k_scan_tile_sums<d6>, dim3(1), dim3(kBlock), 0, s, ts2, ntiles);
	hipLaunchKernelGGL(k_scan_write<d6>, dim3(nspans), dim3(kBlock), 0, s, b4, N, (const double*)ref, ts2,
	                   ts2 + ntiles, pre2);
	const unsigned nn = 2u * N - 1u;
	hipLaunchKernelGGL(k_node_quad, dim3((nn + kBlock - 1) / kBlock), dim3(kBlock), 0, s, (int)N,
	                   static_cast<const int2*>(node_range), b4, static_cast<const d4*>(prefix), pre2,
	                   (const double*)ref, static_cast<float4*>(node_q0), node_q1);
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_quadrupoles", "launch");
}

int sfd_lbvh_records(unsigned N, const void* node_lr, const void* node_range, const void* node_cm,
                     const void* node_cell, float theta, int leaf_size, void* rec_b,
                     unsigned long long* counters, hipStream_t s) {
	const unsigned nn = 2u * N - 1u;
	const float inv_theta = theta > 0.0f ? 1.0f / theta : 3.0e38f;
	hipLaunchKernelGGL(k_records, dim3((nn + kBlock - 1) / kBlock), dim3(kBlock), 0, s, (int)N,
	                   static_cast<const int2*>(node_lr), static_cast<const int2*>(node_range),
	                   static_cast<const float4*>(node_cm), static_cast<const float4*>(node_cell), inv_theta,
	                   leaf_size, static_cast<int4*>(rec_b), counters);
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_records", "launch");
}

}  // extern "C"
