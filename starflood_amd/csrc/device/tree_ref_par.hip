// tree_ref_par.hip -- the reference's octree (src/tree.c:120-296) built level
// by level in parallel, node for node and bit for bit equal to the serial
// insertion of tree_ref.hip.
//
// Why the serial insertion can be replayed one depth at a time:
//  * particles reach a node in index order (each insertion ends before the
//    next begins, and a split hands its eight bodies down in index order),
//    so a node's body count, leaf list and FP32 moment sums depend only on
//    its member set taken in index order;
//  * a node splits when its ninth member arrives.  Its first eight members
//    are redistributed with '<' (src/tree.c:244-247), the ninth and every
//    later member descends with '<=' (src/tree.c:282-285): the rule follows
//    from the member's rank at the node;
//  * node X splits while its rank-8 member i9 is inserted, at X's depth, so
//    the serial order of the splits is the order of (i9, depth), and the
//    k-th split (from 0) creates nodes 1 + 8k ... 1 + 8k + 7.
// Each level holds the particles still descending slot by slot, in index order
// within a slot.  A level is three launches: its slots (leaf lists, splits and
// their numbers, children), its particles (mass-moment products, octants by
// rank, running counts of each octant), and their move to the child slots; the
// sums over blocks that each needs are collected by looking back (lookback.h).
// Nodes are numbered level-major while building.  Every node's moments are
// summed in index order, sequentially as the reference adds them, on a second
// stream as soon as the node's level is finished (the root's chain, the
// longest, beside the deeper levels); the split events, ordered by (i9, depth),
// map the level-major numbering onto the reference's.
//
// Bound by launches and their latency.  With ten launches a level (marks,
// flags, scan, routing and a two-pass radix sort) and the events sorted by four
// more passes, the solve of a Plummer sphere of 65536 took 1.87 ms; now 1.12,
// 0.31 of it the walk.
//
// The level sizes live on the device (lv[]), so the host queues several
// levels at a time and synchronises once per batch.  A build that would run
// out of nodes or past depth_max is reported to the caller, which runs the
// serial build: that one stops where the reference stops and leaves the same
// partial tree.
#include <hip/hip_runtime.h>

#include <cstring>

#include "../sf_internal.h"
#include "lookback.h"
#include "tree_dev.h"

namespace {

constexpr unsigned kBlock = 256;
constexpr unsigned kNone = ~0u;               // a particle that descends no further, a leaf's split number
constexpr unsigned kAlign = 256;
constexpr unsigned kMaxLevels = 17;           // depths 0..16: tree_depth_max is at most 16
constexpr unsigned kFirstBatch = 6, kNextBatch = 3;   // levels queued per host synchronisation
constexpr unsigned kPer = 4;                  // particles per thread of a tile
constexpr unsigned kTileP = kBlock * kPer;    // consecutive particles per block
static_assert(kBlock / 64u == 4u, "k_level_particles: two octants per wavefront of the block");

enum Status { RUNNING = 0, DONE = 1, FALLBACK = 2 };
// A level: its slots, the level-major id of the first, splits of the shallower
// levels, particles that reached it, members of the shallower leaves, first
// archive entry, status, depth.
struct LevelRec {
	unsigned m, base, evoff, n, done, aoff, status, depth;
};
static_assert(sizeof(LevelRec) <= SF_TREE_PAR_STATE * sizeof(unsigned), "the host mirror holds a level");
// Level 0 is lv[0]; each level's last block of slots writes the next.
struct State {
	LevelRec lv[kMaxLevels + 1];
	unsigned ticket[2 * kMaxLevels + 2];
};

__device__ __forceinline__ void child_bounds(const float* bmin, const float* bmax, const float* mid, int o, float* out) {
	for (int a = 0; a < 3; ++a) {
		out[a] = ((o >> a) & 1) ? mid[a] : bmin[a];
		out[3 + a] = ((o >> a) & 1) ? bmax[a] : mid[a];
	}
}

__device__ __forceinline__ void clear_node(sf_node& n, unsigned parent, const float* b) {
	n.parent = parent;
	n.bodies = 0u;
	for (int k = 0; k < 8; ++k) n.branch[k] = 0u;
	for (int k = 0; k < 6; ++k) n.bounds[k] = b[k];
	for (int k = 0; k < 4; ++k) n.params[k] = 0.0f;
}

// The root record as the reference purges it, the build state, and the state
// words of every look-back.
__global__ __launch_bounds__(kBlock) void k_par_state(const float* __restrict__ tb, sf_node* __restrict__ tnode,
                                                      State* __restrict__ st, unsigned long long* __restrict__ words,
                                                      size_t n_words) {
	for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n_words; i += (size_t)gridDim.x * kBlock)
		words[i] = 0ull;
	if (blockIdx.x != 0 || threadIdx.x != 0) return;
	float b[6];
	for (int k = 0; k < 6; ++k) b[k] = tb[k];
	clear_node(tnode[0], 0u, b);
	for (unsigned k = 0; k < sizeof(State) / sizeof(unsigned); ++k) reinterpret_cast<unsigned*>(st)[k] = 0u;
	st->lv[0].m = 1u;
}

// The particles inside the tree bounds (the test of src/tree.c:147-152, so NaN
// coordinates are inside) become the root's, in index order; those outside
// take the back of the walk order.
__global__ __launch_bounds__(kBlock) void k_par_init(const float* __restrict__ pos, unsigned N,
                                                     const float* __restrict__ tb, State* st,
                                                     unsigned long long* words, uint2* __restrict__ seg,
                                                     unsigned* __restrict__ slot, unsigned* __restrict__ val,
                                                     unsigned* __restrict__ evmask, unsigned* __restrict__ order) {
	__shared__ unsigned s_ticket, s_cnt[kTileP / 64];
	__shared__ unsigned long long s_prior;
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned tile = look::ticket(&st->ticket[0], s_ticket);
	const float b[6] = {tb[0], tb[1], tb[2], tb[3], tb[4], tb[5]};
	unsigned long long in[kPer];
#pragma unroll
	for (unsigned k = 0; k < kPer; ++k) {
		const unsigned i = tile * kTileP + (w * kPer + k) * 64u + lane;
		bool inside = false;
		if (i < N) {
			const float px = pos[3u * i], py = pos[3u * i + 1u], pz = pos[3u * i + 2u];
			inside = !(b[0] > px || px > b[3] || b[1] > py || py > b[4] || b[2] > pz || pz > b[5]);
			evmask[i] = 0u;
		}
		in[k] = __ballot(inside);
		if (lane == 0u) s_cnt[w * kPer + k] = (unsigned)__popcll(in[k]);
	}
	__syncthreads();
	unsigned before = 0, total = 0;
	for (unsigned k = 0; k < kTileP / 64; ++k) {
		if (k < w * kPer) before += s_cnt[k];
		total += s_cnt[k];
	}
	if (w == 0u) {
		const unsigned long long prior = look::collect<1>(words, tile, total);
		if (lane == 0u) s_prior = prior;
	}
	__syncthreads();
	unsigned at = (unsigned)s_prior + before;
#pragma unroll
	for (unsigned k = 0; k < kPer; ++k) {
		const unsigned i = tile * kTileP + (w * kPer + k) * 64u + lane;
		const unsigned q = at + (unsigned)__popcll(in[k] & ((1ull << lane) - 1ull));
		if ((in[k] >> lane) & 1ull) {
			slot[q] = 0u;
			val[q] = i;
		} else if (i < N) {
			order[N - 1u - (i - q)] = i;
		}
		at += (unsigned)__popcll(in[k]);
	}
	if (threadIdx.x == 0u && (tile + 1u) * kTileP >= N) {
		const unsigned n = (unsigned)s_prior + total;
		st->lv[0].n = n;
		seg[0] = make_uint2(0u, n);
	}
}

// The slots of level L: body counts, leaf lists and archive ranges (trange) of
// their nodes; a splitting slot's number within the level (split; kNone for a
// leaf), its children at level-major ids 1 + 8 g + octant (g = splits before
// this one, in level-major order), its branches and its split event (i9 =
// the slot's rank-8 member, depth).  A leaf's members take the next places of
// the walk order, so that a wavefront of the walk holds particles of
// neighbouring leaves (any order gives the same per-particle results).  Writes
// stay inside the node and event capacities; the last block of slots decides
// whether the build stops (no split), falls back (a split at depth_max, or more
// than max_nodes nodes) or goes on.
__global__ __launch_bounds__(kBlock) void k_level_slots(State* st, unsigned L, unsigned long long* words,
                                                        const unsigned* __restrict__ val,
                                                        const uint2* __restrict__ seg, unsigned depth_max,
                                                        unsigned node_cap, unsigned ev_cap,
                                                        sf_node* __restrict__ tnode, uint2* __restrict__ trange,
                                                        unsigned* __restrict__ split, uint2* __restrict__ event,
                                                        unsigned* __restrict__ evmask, unsigned* __restrict__ order) {
	__shared__ unsigned s_ticket, s_split[kBlock / 64], s_next[kBlock / 64];
	__shared__ unsigned long long s_prior;
	const LevelRec r = st->lv[L];
	if (r.status != RUNNING) {
		if (blockIdx.x == 0u && threadIdx.x == 0u) st->lv[L + 1u] = r;
		return;
	}
	if (blockIdx.x * kBlock >= r.m) return;
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned tile = look::ticket(&st->ticket[1u + 2u * L], s_ticket);
	const unsigned s = tile * kBlock + threadIdx.x;
	const bool live = s < r.m;
	uint2 g = make_uint2(0u, 0u);
	if (live) g = seg[s];
	const unsigned c = g.y - g.x, t = r.base + s;
	const bool splits = c >= 9u;
	if (live) {
		sf_node& nd = tnode[t];
		nd.bodies = c;
		trange[t] = make_uint2(r.aoff + g.x, r.aoff + g.y);
	}
	const unsigned long long m = __ballot(splits);
	unsigned down = splits ? c : 0u;   // particles that descend from this slot and those before
#pragma unroll
	for (int o = 1; o < 64; o <<= 1) {
		const unsigned v = __shfl_up(down, (unsigned)o);
		if ((int)lane >= o) down += v;
	}
	if (lane == 63u) {
		s_split[w] = (unsigned)__popcll(m);
		s_next[w] = down;
	}
	__syncthreads();
	unsigned before = (unsigned)__popcll(m & ((1ull << lane) - 1ull)), n_split = 0, n_next = 0;
	for (unsigned q = 0; q < kBlock / 64; ++q) {
		if (q < w) {
			before += s_split[q];
			down += s_next[q];
		}
		n_split += s_split[q];
		n_next += s_next[q];
	}
	// splits (below 2^30) in the upper half, the particles that descend in the lower
	const unsigned long long own = ((unsigned long long)n_split << 32) | n_next;
	if (w == 0u) {
		const unsigned long long prior = look::collect<1>(words, tile, own);
		if (lane == 0u) s_prior = prior;
	}
	__syncthreads();
	before += (unsigned)(s_prior >> 32);
	down += (unsigned)s_prior;
	if (live && !splits) {   // its place: after the members of all leaves before it
		const unsigned at = r.done + g.x - down;
		for (unsigned k = 0; k < c; ++k) {
			const unsigned i = val[g.x + k];
			tnode[t].branch[k] = i;
			order[at + k] = i;
		}
	}
	if (live) split[s] = splits ? before : kNone;
	if (splits) {
		const unsigned k = r.evoff + before;
		if (k < ev_cap && 9ull + 8ull * k <= (unsigned long long)node_cap) {
			sf_node& nd = tnode[t];
			const unsigned child0 = 1u + 8u * k, i9 = val[g.x + 8u];
			float bmin[3], bmax[3], mid[3];
			for (int a = 0; a < 3; ++a) {
				bmin[a] = nd.bounds[a];
				bmax[a] = nd.bounds[3 + a];
				mid[a] = 0.5f * (bmin[a] + bmax[a]);
			}
			for (int o = 0; o < 8; ++o) {
				float b[6];
				child_bounds(bmin, bmax, mid, o, b);
				clear_node(tnode[child0 + (unsigned)o], t, b);
				nd.branch[o] = child0 + (unsigned)o;
			}
			event[k] = make_uint2(i9, r.depth);
			atomicOr(&evmask[i9], 1u << r.depth);
		}
	}
	if (threadIdx.x == 0u && (tile + 1u) * kBlock >= r.m) {
		const unsigned long long sum = s_prior + own;
		const unsigned all = (unsigned)(sum >> 32);
		LevelRec q = r;
		if ((all && r.depth >= depth_max) || 1ull + 8ull * ((unsigned long long)r.evoff + all) >= (unsigned long long)node_cap) {
			q.status = FALLBACK;
		} else if (all == 0u) {
			q.status = DONE;
		} else {
			q.m = 8u * all;
			q.base += r.m;
			q.evoff += all;
			q.n = (unsigned)sum;
			q.done += r.n - q.n;
			q.aoff += r.n;
			q.depth += 1u;
		}
		st->lv[L + 1u] = q;
	}
}

// The particles of level L: their products (m x, m y, m z, m), one component
// per archive plane of a_cap floats from entry aoff; for those of splitting
// slots the octant, by '<' for the slot's first eight members and '<=' after
// them, and the number of particles before it that take the same octant of
// their slots (move = octant << 28 | number; kNone for members of leaves).
// first and last of a slot's members leave all eight octants' numbers at the
// slot's ends (ends: 16 per slot).
__global__ __launch_bounds__(kBlock) void k_level_particles(State* st, unsigned L, unsigned long long* words,
                                                            const float* __restrict__ pos,
                                                            const float* __restrict__ mas,
                                                            const unsigned* __restrict__ slot,
                                                            const unsigned* __restrict__ val,
                                                            const uint2* __restrict__ seg,
                                                            const unsigned* __restrict__ split,
                                                            const sf_node* __restrict__ tnode, size_t a_cap,
                                                            float* __restrict__ arch, unsigned* __restrict__ move,
                                                            unsigned* __restrict__ ends) {
	__shared__ unsigned s_ticket, s_cnt[kTileP / 64][8];
	const LevelRec r = st->lv[L];
	if (r.status != RUNNING || blockIdx.x * kTileP >= r.n) return;
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned tile = look::ticket(&st->ticket[2u + 2u * L], s_ticket);
	int oct[kPer];
	unsigned sl[kPer];
	bool first[kPer], last[kPer];
#pragma unroll
	for (unsigned k = 0; k < kPer; ++k) {
		const unsigned p = tile * kTileP + (w * kPer + k) * 64u + lane;
		oct[k] = -1;
		sl[k] = 0u;
		first[k] = last[k] = false;
		if (p < r.n) {
			const unsigned s = slot[p], i = val[p];
			const float x[3] = {pos[3u * i], pos[3u * i + 1u], pos[3u * i + 2u]}, pm = mas[i];
			const size_t q = (size_t)r.aoff + p;
			arch[q] = pm * x[0];
			arch[a_cap + q] = pm * x[1];
			arch[2u * a_cap + q] = pm * x[2];
			arch[3u * a_cap + q] = pm;
			if (split[s] != kNone) {
				const uint2 g = seg[s];
				const sf_node& nd = tnode[r.base + s];
				oct[k] = 0;
				for (int a = 0; a < 3; ++a) {
					const float mid = 0.5f * (nd.bounds[a] + nd.bounds[3 + a]);
					if (p - g.x < 8u ? mid < x[a] : mid <= x[a]) oct[k] += 1 << a;
				}
				sl[k] = s;
				first[k] = p == g.x;
				last[k] = p + 1u == g.y;
			}
		}
#pragma unroll
		for (int o = 0; o < 8; ++o) {
			const unsigned n = (unsigned)__popcll(__ballot(oct[k] == o));
			if ((int)lane == o) s_cnt[w * kPer + k][o] = n;
		}
	}
	__syncthreads();
	{
		// wavefront w: octants 2 w and 2 w + 1; the rounds' counts become the
		// numbers before them
		const unsigned o = 2u * w + (lane & 1u);
		unsigned own = 0;
		for (unsigned q = 0; q < kTileP / 64; ++q) own += s_cnt[q][o];
		unsigned run = (unsigned)look::collect<2>(words + (size_t)w * 2u * ((r.n + kTileP - 1u) / kTileP), tile, own);
		if (lane < 2u)
			for (unsigned q = 0; q < kTileP / 64; ++q) {
				const unsigned n = s_cnt[q][o];
				s_cnt[q][o] = run;
				run += n;
			}
	}
	__syncthreads();
	const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
	for (unsigned k = 0; k < kPer; ++k) {
		const unsigned p = tile * kTileP + (w * kPer + k) * 64u + lane;
		unsigned out = kNone;
#pragma unroll
		for (int o = 0; o < 8; ++o) {
			const unsigned long long b = __ballot(oct[k] == o);
			const unsigned n = s_cnt[w * kPer + k][o] + (unsigned)__popcll(b & lt);
			if (oct[k] == o) out = ((unsigned)o << 28) | n;
			if (first[k]) ends[16u * sl[k] + (unsigned)o] = n;
			if (last[k]) ends[16u * sl[k] + 8u + (unsigned)o] = n + (oct[k] == o ? 1u : 0u);
		}
		if (p < r.n) move[p] = out;
	}
}

// The particles of level L that descend, to their places in level L + 1: slot
// by slot, octant by octant, in index order; and that level's segments.
__global__ __launch_bounds__(kBlock) void k_level_move(const State* __restrict__ st, unsigned L,
                                                       const unsigned* __restrict__ move,
                                                       const unsigned* __restrict__ ends,
                                                       const uint2* __restrict__ seg,
                                                       const unsigned* __restrict__ split,
                                                       const unsigned* __restrict__ slot,
                                                       const unsigned* __restrict__ val, unsigned* __restrict__ slot_out,
                                                       unsigned* __restrict__ val_out, uint2* __restrict__ seg_out) {
	const unsigned p = blockIdx.x * kBlock + threadIdx.x;
	if (st->lv[L + 1u].status != RUNNING || p >= st->lv[L].n) return;
	const unsigned mv = move[p];
	if (mv == kNone) return;
	const unsigned s = slot[p], o = mv >> 28, c0 = 8u * split[s];
	const unsigned* e = ends + 16u * s;
	unsigned at = 0;   // the particles that descend from the slots before
#pragma unroll
	for (int k = 0; k < 8; ++k) at += e[k];
	const bool lead = p == seg[s].x;
#pragma unroll
	for (unsigned k = 0; k < 8u; ++k) {
		const unsigned n = e[8u + k] - e[k];
		if (lead) seg_out[c0 + k] = make_uint2(at, at + n);
		if (k == o) {
			const unsigned q = at + (mv & 0x0FFFFFFFu) - e[k];
			slot_out[q] = c0 + o;
			val_out[q] = val[p];
		}
		at += n;
	}
}

// Moment sums params[c] = (((0 + q_0) + q_1) + ...) over each node's members
// in index order: the FP32 chain of the serial insertion (src/tree.c:205-208).
// Nodes of more than min_size members: one wavefront per (node, component);
// waves stride over the (node, component) items.  The products go through LDS
// in chunks of 256, loaded two chunks ahead, and come back four at a time to
// every lane: 1.25 instructions a link of the chain, which a lone wavefront
// issues in 2.5 ns each (lanes loading 64 products that the chain reads back
// lane by lane, two: the root of 65536 485 -> 225 us beside the levels; scalar
// loads, which cannot be far enough ahead, 637).  Products past the last are
// zeros, which leave a sum as it is (it is never -0).
constexpr unsigned kSumSmall = 256;   // larger nodes are summed by a wavefront

__global__ __launch_bounds__(64) void k_node_sums(const float* __restrict__ arch, size_t a_cap,
                                                  const uint2* __restrict__ trange, unsigned first, unsigned count,
                                                  unsigned min_size, sf_node* __restrict__ tnode) {
	constexpr unsigned kChunk = 256, kLoads = kChunk / 64, kRead = 8;
	__shared__ float4 s_chunk[2][kChunk / 4];
	const unsigned lane = threadIdx.x;
	for (unsigned item = blockIdx.x; item < 4u * count; item += gridDim.x) {
		const unsigned t = first + (item >> 2), comp = item & 3u;
		const uint2 r = trange[t];
		const unsigned n = r.y - r.x;
		if (n <= min_size || n == 0u) continue;
		const float* __restrict__ a = arch + comp * a_cap + r.x;
		auto load = [&](unsigned c, float v[kLoads]) {
#pragma unroll
			for (unsigned q = 0; q < kLoads; ++q) {
				const unsigned k = c + 64u * q + lane;
				v[q] = k < n ? a[k] : 0.0f;
			}
		};
		auto store = [&](unsigned buf, const float v[kLoads]) {
#pragma unroll
			for (unsigned q = 0; q < kLoads; ++q) reinterpret_cast<float*>(s_chunk[buf])[64u * q + lane] = v[q];
		};
		float va[kLoads], vb[kLoads], sum = 0.0f;
		load(0u, va);
		store(0u, va);
		load(kChunk, va);
		load(2u * kChunk, vb);
		unsigned buf = 0u;
		for (unsigned c = 0; c < n; c += kChunk) {
			__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
			store(buf ^ 1u, va);
#pragma unroll
			for (unsigned q = 0; q < kLoads; ++q) va[q] = vb[q];
			load(c + 3u * kChunk, vb);
			const float4* __restrict__ p = s_chunk[buf];
			float4 x[kRead];
#pragma unroll
			for (unsigned q = 0; q < kRead; ++q) x[q] = p[q];
			for (unsigned k = 0; k < kChunk / 4; k += kRead) {
				float4 y[kRead];
				const unsigned at = k + kRead < kChunk / 4 ? k + kRead : 0u;
#pragma unroll
				for (unsigned q = 0; q < kRead; ++q) y[q] = p[at + q];
#pragma unroll
				for (unsigned q = 0; q < kRead; ++q) {
					sum = (((sum + x[q].x) + x[q].y) + x[q].z) + x[q].w;
					x[q] = y[q];
				}
			}
			buf ^= 1u;
		}
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
		if (lane == 0u) tnode[t].params[comp] = sum;
	}
}

// The same sums for nodes of 1..kSumSmall members, one lane per
// (node, component).
__global__ __launch_bounds__(kBlock) void k_node_sums_small(const float* __restrict__ arch, size_t a_cap,
                                                            const uint2* __restrict__ trange, unsigned first,
                                                            unsigned count, sf_node* __restrict__ tnode) {
	const unsigned item = blockIdx.x * kBlock + threadIdx.x;
	if (item >= 4u * count) return;
	const unsigned t = first + (item >> 2), comp = item & 3u;
	const uint2 r = trange[t];
	if (r.y == r.x || r.y - r.x > kSumSmall) return;
	const float* __restrict__ a = arch + comp * a_cap;
	float sum = 0.0f;
	for (unsigned i = r.x; i < r.y; ++i) sum = sum + a[i];
	tnode[t].params[comp] = sum;
}

// pre[i] = split events of the particles before i (evmask: one bit per depth)
__global__ __launch_bounds__(kBlock) void k_event_scan(const unsigned* __restrict__ evmask, unsigned N, State* st,
                                                       unsigned long long* words, unsigned* __restrict__ pre) {
	__shared__ unsigned s_ticket, s_cnt[kTileP / 64];
	__shared__ unsigned long long s_prior;
	const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
	const unsigned tile = look::ticket(&st->ticket[2u * kMaxLevels + 1u], s_ticket);
	unsigned n[kPer], incl[kPer];
#pragma unroll
	for (unsigned k = 0; k < kPer; ++k) {
		const unsigned i = tile * kTileP + (w * kPer + k) * 64u + lane;
		incl[k] = n[k] = i < N ? (unsigned)__popc(evmask[i]) : 0u;
#pragma unroll
		for (int o = 1; o < 64; o <<= 1) {
			const unsigned v = __shfl_up(incl[k], (unsigned)o);
			if ((int)lane >= o) incl[k] += v;
		}
		if (lane == 63u) s_cnt[w * kPer + k] = incl[k];
	}
	__syncthreads();
	unsigned before = 0, total = 0;
	for (unsigned k = 0; k < kTileP / 64; ++k) {
		if (k < w * kPer) before += s_cnt[k];
		total += s_cnt[k];
	}
	if (w == 0u) {
		const unsigned long long prior = look::collect<1>(words, tile, total);
		if (lane == 0u) s_prior = prior;
	}
	__syncthreads();
	before += (unsigned)s_prior;
#pragma unroll
	for (unsigned k = 0; k < kPer; ++k) {
		const unsigned i = tile * kTileP + (w * kPer + k) * 64u + lane;
		if (i < N) pre[i] = before + incl[k] - n[k];
		before += s_cnt[w * kPer + k];
	}
}

// perm[g] = position of split g in (i9, depth) order
__global__ __launch_bounds__(kBlock) void k_ev_perm(const uint2* __restrict__ event, const unsigned* __restrict__ evmask,
                                                    const unsigned* __restrict__ pre, unsigned S,
                                                    unsigned* __restrict__ perm) {
	const unsigned g = blockIdx.x * kBlock + threadIdx.x;
	if (g >= S) return;
	const uint2 e = event[g];
	perm[g] = pre[e.x] + (unsigned)__popc(evmask[e.x] & ((1u << e.y) - 1u));
}

__device__ __forceinline__ unsigned final_id(unsigned t, const unsigned* __restrict__ perm) {
	return t == 0u ? 0u : 1u + 8u * perm[(t - 1u) >> 3] + ((t - 1u) & 7u);
}

// node[final(t)] = tnode[t] with parent and child ids renumbered and the
// centre of mass, as k_tree_com_ref (src/tree.c:302-310)
__global__ __launch_bounds__(kBlock) void k_final_nodes(const sf_node* __restrict__ tnode, unsigned num_nodes,
                                                        const unsigned* __restrict__ perm, sf_node* __restrict__ node,
                                                        unsigned* __restrict__ meta) {
	const unsigned t = blockIdx.x * kBlock + threadIdx.x;
	if (t == 0u) {
		meta[0] = num_nodes;
		meta[1] = 0u;
	}
	if (t >= num_nodes) return;
	sf_node rec = tnode[t];
	rec.parent = final_id(rec.parent, perm);
	if (rec.bodies > 8u)
		for (int o = 0; o < 8; ++o) rec.branch[o] = final_id(rec.branch[o], perm);
	const float mass = rec.params[3];
	const float inv = 0.0f < mass ? 1.0f / mass : 1.0f;
	for (int k = 0; k < 3; ++k) rec.params[k] = rec.params[k] * inv;
	node[final_id(t, perm)] = rec;
}

inline unsigned blocks(unsigned n) { return (n + kBlock - 1u) / kBlock; }
inline size_t align_up(size_t n) { return (n + kAlign - 1u) / kAlign * kAlign; }

// Scratch planes, each 256-byte aligned.
enum Plane { SLOT0, SLOT1, VAL0, VAL1, MOVE, EVMASK, PRE, SEG0, SEG1, SPLIT, ENDS, EVENT, PERM, TNODE, TRANGE, STATE, WORDS,
             ARCH, kPlanes };

struct Layout {
	unsigned ev_cap, slot_cap, tiles, slot_tiles;
	size_t n_words;   // of look-backs: the first tiles', then each level's slots and particles, then the events'
	size_t a_cap;     // floats per product plane
	size_t off[kPlanes];
	size_t bytes;
};

Layout layout(unsigned N, unsigned max_nodes) {
	Layout L;
	const size_t nodes = max_nodes ? max_nodes : 1u, n = N ? N : 1u;
	L.ev_cap = max_nodes / 8u + 1u;
	L.slot_cap = 8u * L.ev_cap + 8u;
	L.a_cap = (size_t)kMaxLevels * n;
	L.tiles = (unsigned)((n + kTileP - 1u) / kTileP);
	// at most N particles descend, and a level has at most 8 (N / 9) + 1 slots
	L.slot_tiles = (8u * (N / 9u) + 1u + kBlock - 1u) / kBlock;
	L.n_words = 2u * (size_t)L.tiles + kMaxLevels * ((size_t)L.slot_tiles + 8u * (size_t)L.tiles);
	size_t sz[kPlanes];
	sz[SLOT0] = sz[SLOT1] = sz[VAL0] = sz[VAL1] = sz[MOVE] = sz[EVMASK] = sz[PRE] = 4u * n;
	sz[SEG0] = sz[SEG1] = 8u * (size_t)L.slot_cap;
	sz[SPLIT] = 4u * (size_t)L.slot_cap;
	sz[ENDS] = 64u * (size_t)L.slot_cap;
	sz[EVENT] = 8u * (size_t)L.ev_cap;
	sz[PERM] = 4u * (size_t)L.ev_cap;
	sz[TNODE] = sizeof(sf_node) * nodes;
	sz[TRANGE] = 8u * nodes;
	sz[STATE] = sizeof(State);
	sz[WORDS] = 8u * L.n_words;
	sz[ARCH] = 4u * 4u * L.a_cap;
	size_t o = 0;
	for (int k = 0; k < kPlanes; ++k) {
		L.off[k] = o;
		o += align_up(sz[k]);
	}
	L.bytes = o;
	return L;
}

template <class T>
T* plane(void* scratch, const Layout& L, Plane k) {
	return reinterpret_cast<T*>(static_cast<char*>(scratch) + L.off[k]);
}

// The level-synchronous build applies when the tree can hold N bodies (at
// most 8 per leaf, so N <= 8 max_nodes) and archive offsets fit 32 bits
// (particle numbers then fit the 28 bits of move).
bool par_applies(unsigned N, unsigned max_nodes) {
	return max_nodes >= 2u && (unsigned long long)N <= 8ull * max_nodes &&
	       (unsigned long long)kMaxLevels * N < (1ull << 32);
}

// Moment sums of nodes [first, first + count): lanes for the small ones,
// wavefronts for the others.
void launch_sums(const float* arch, size_t a_cap, const uint2* trange, unsigned first, unsigned count, sf_node* tnode,
                 hipStream_t s) {
	const unsigned items = 4u * count;
	hipLaunchKernelGGL(k_node_sums_small, dim3(blocks(items)), dim3(kBlock), 0, s, arch, a_cap, trange, first, count,
	                   tnode);
	hipLaunchKernelGGL(k_node_sums, dim3(items < 4096u ? items : 4096u), dim3(64), 0, s, arch, a_cap, trange, first,
	                   count, kSumSmall, tnode);
}

int build_par(const sf_tree_par_ctx* x, const float* pos, const float* mas, unsigned N, const float* bounds,
              unsigned max_nodes, int depth_max, sf_node* node, unsigned* meta, unsigned* order, hipStream_t s) {
	if (!par_applies(N, max_nodes) || depth_max < 0 || depth_max >= (int)kMaxLevels) return 1;
	const Layout L = layout(N, max_nodes);
	void* scr = x->scratch;
	unsigned* slot[2] = {plane<unsigned>(scr, L, SLOT0), plane<unsigned>(scr, L, SLOT1)};
	unsigned* val[2] = {plane<unsigned>(scr, L, VAL0), plane<unsigned>(scr, L, VAL1)};
	uint2* seg[2] = {plane<uint2>(scr, L, SEG0), plane<uint2>(scr, L, SEG1)};
	unsigned* move = plane<unsigned>(scr, L, MOVE);
	unsigned* evmask = plane<unsigned>(scr, L, EVMASK);
	unsigned* pre = plane<unsigned>(scr, L, PRE);
	unsigned* split = plane<unsigned>(scr, L, SPLIT);
	unsigned* ends = plane<unsigned>(scr, L, ENDS);
	uint2* event = plane<uint2>(scr, L, EVENT);
	sf_node* tnode = plane<sf_node>(scr, L, TNODE);
	uint2* trange = plane<uint2>(scr, L, TRANGE);
	unsigned* perm = plane<unsigned>(scr, L, PERM);
	State* st = plane<State>(scr, L, STATE);
	float* arch = plane<float>(scr, L, ARCH);
	unsigned long long* words = plane<unsigned long long>(scr, L, WORDS);
	unsigned long long* level_words = words + L.tiles;
	const size_t per_level = (size_t)L.slot_tiles + 8u * (size_t)L.tiles;

	const size_t fill = (L.n_words + kBlock - 1u) / kBlock;
	hipLaunchKernelGGL(k_par_state, dim3((unsigned)(fill < 1024u ? fill : 1024u)), dim3(kBlock), 0, s, bounds, tnode, st,
	                   words, L.n_words);
	hipLaunchKernelGGL(k_par_init, dim3(L.tiles), dim3(kBlock), 0, s, pos, N, bounds, st, words, seg[0], slot[0], val[0],
	                   evmask, order);
	LevelRec rec;
	unsigned levels = 0;
	unsigned summed = 1u;   // nodes [1, summed) have their sums queued on the side stream
	for (;;) {
		unsigned batch = levels ? kNextBatch : kFirstBatch;
		if (batch > kMaxLevels - levels) batch = kMaxLevels - levels;
		for (unsigned b = 0; b < batch; ++b, ++levels) {
			const unsigned cur = levels & 1u;
			unsigned long long* wd = level_words + levels * per_level;
			hipLaunchKernelGGL(k_level_slots, dim3(L.slot_tiles), dim3(kBlock), 0, s, st, levels, wd, val[cur], seg[cur],
			                   (unsigned)depth_max, max_nodes, L.ev_cap, tnode, trange, split, event, evmask, order);
			hipLaunchKernelGGL(k_level_particles, dim3(L.tiles), dim3(kBlock), 0, s, st, levels, wd + L.slot_tiles, pos,
			                   mas, slot[cur], val[cur], seg[cur], split, tnode, L.a_cap, arch, move, ends);
			if (levels == 0) {
				// the root's sums, the longest chain, run beside the deeper levels
				if (sf_hip_check(hipEventRecord(x->ev[0], s), "sfd_tree_build_ref_par", "event") ||
				    sf_hip_check(hipStreamWaitEvent(x->side, x->ev[0], 0), "sfd_tree_build_ref_par", "wait"))
					return -1;
				hipLaunchKernelGGL(k_node_sums, dim3(4), dim3(64), 0, x->side, arch, L.a_cap, trange, 0u, 1u, 0u, tnode);
				if (sf_hip_check(hipEventRecord(x->ev[1], x->side), "sfd_tree_build_ref_par", "event")) return -1;
			}
			hipLaunchKernelGGL(k_level_move, dim3(blocks(N ? N : 1u)), dim3(kBlock), 0, s, st, levels, move, ends, seg[cur],
			                   split, slot[cur], val[cur], slot[cur ^ 1u], val[cur ^ 1u], seg[cur ^ 1u]);
		}
		if (sf_hip_check(hipMemcpyAsync(x->h_state, &st->lv[levels], sizeof(LevelRec), hipMemcpyDeviceToHost, s),
		                 "sfd_tree_build_ref_par", "state copy") ||
		    sf_hip_check(hipStreamSynchronize(s), "sfd_tree_build_ref_par", "levels"))
			return -1;
		memcpy(&rec, x->h_state, sizeof(rec));
		if (rec.status != RUNNING || levels == kMaxLevels) break;
		// nodes of the finished levels (all before the current level's first
		// slot) are complete: their sums run beside the next levels
		if (rec.base > summed) {
			launch_sums(arch, L.a_cap, trange, summed, rec.base - summed, tnode, x->side);
			if (sf_hip_check(hipEventRecord(x->ev[1], x->side), "sfd_tree_build_ref_par", "event")) return -1;
			summed = rec.base;
		}
	}
	if (rec.status != DONE) {
		// sums on the side stream may still read the archive: finish them first
		if (sf_hip_check(hipStreamSynchronize(x->side), "sfd_tree_build_ref_par", "side")) return -1;
		return 1;
	}

	const unsigned S = rec.evoff;
	const unsigned num_nodes = 1u + 8u * S;
	if (num_nodes > summed) launch_sums(arch, L.a_cap, trange, summed, num_nodes - summed, tnode, s);
	if (S) {
		hipLaunchKernelGGL(k_event_scan, dim3(L.tiles), dim3(kBlock), 0, s, evmask, N, st,
		                   level_words + kMaxLevels * per_level, pre);
		hipLaunchKernelGGL(k_ev_perm, dim3(blocks(S)), dim3(kBlock), 0, s, event, evmask, pre, S, perm);
	}
	if (sf_hip_check(hipStreamWaitEvent(s, x->ev[1], 0), "sfd_tree_build_ref_par", "wait")) return -1;
	hipLaunchKernelGGL(k_final_nodes, dim3(blocks(num_nodes)), dim3(kBlock), 0, s, tnode, num_nodes, perm, node, meta);
	return sf_hip_check(hipGetLastError(), "sfd_tree_build_ref_par", "launch") ? -1 : 0;
}

}  // namespace

extern "C" size_t sfd_tree_par_bytes(unsigned N, unsigned max_nodes) {
	return par_applies(N, max_nodes) ? layout(N, max_nodes).bytes : 0u;
}

extern "C" int sfd_tree_build_ref_par(const sf_tree_par_ctx* x, const float* pos, const float* mas, unsigned N,
                                      const float* bounds, unsigned max_nodes, int depth_max, sf_node* node,
                                      unsigned* meta, unsigned* order, hipStream_t s) {
	const int tok = sf_prof_begin("tree_build_ref_par", s);
	const int rc = build_par(x, pos, mas, N, bounds, max_nodes, depth_max, node, meta, order, s);
	sf_prof_end(tok, s);
	return rc;
}
