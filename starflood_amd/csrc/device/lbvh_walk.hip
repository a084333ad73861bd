// lbvh_walk.hip -- the SF_TREE_LBVH walk: one wavefront per walk group, a
// maximal subtree of at most 64 particles (a run of consecutive sorted
// particles inside one Morton cell).  Groups are not fixed runs of 64 sorted
// particles: a run that crosses a high-level Morton boundary (the octant
// planes through the centre of a cluster) has a bounding box the size of the
// whole core and would open nearly every node.
//
// Each step pops up to 64 pending nodes, one per lane, and classifies them
// against the group's bounding box: a monopole "cell" when the box stays
// outside the node's critical radius r = l/theta + |com - centre| (l = longest
// side of the node's particle box), a "leaf" summed particle by particle when
// the node holds at most leaf_size particles, otherwise opened (its two
// children are pushed).  Cells and leaf particles are queued in LDS and
// evaluated 64 at a time with a 14-VALU + rsqrt interaction; leaf particles
// are gathered 64 at a time with one vector load, so the tree logic and
// memory latency are amortised over 64 interactions.
//
// The evaluation is bound by VALU issue.  Groups hold 44 particles on
// average, so with one particle per lane a third of it went to idle lanes.
// Instead each row of 16 lanes takes every fourth entry and each lane up to
// four particles (Slots): (cnt + 15) / 16 interactions per lane for four
// entries, 0.8 of the work on average, a quarter of the LDS reads and four
// independent chains.  KDK step, before -> after: 65537 particles (monopole,
// theta 0.5) 266 -> 236 us, 1M 2116 -> 1876 us; 4M quadrupoles under the
// relative test, more of it tree logic, 5474 -> 5300 us.
//
// Options: quadrupole cells (the 34-VALU interact_quad), and the relative
// opening test, which also requires G M l^p <= alpha |a|min d^(p+2) of a
// cell (|a|min the group's smallest previous acceleration); a quadrupole
// walk then sums the cells that meet the monopole form of that bound (scaled
// by kMonoBeta) as monopoles, through the leaf particles' queue.
//
// The grid is persistent and sized to the wavefronts resident at once, or to
// N / 32 if that is less.  Each wavefront walks the group of its own rank and
// then takes further ones from a shared counter, and owns a node stack: its top
// in LDS, the rest in global memory (deep enough that the 64-wide pops rarely
// have to narrow).  Groups are taken one by one from a list of them: taken by
// runs of 64 sorted positions, a wavefront had up to three in series while
// others had none, which at 65537 particles (1570 groups on 1024 SIMDs) was
// most of the walk: 394 -> 222 us (step 646 -> 487 us alone); 1M step 2661 ->
// 2518 us alone, 4M quadrupole walk 4 % faster.  A block walking a group
// together (shared frontier, two barriers a round) took 273 us at 65537 and
// half as long again at 1M.  The self pair is included in leaf sums, as in the
// reference's PP sum.
#include <hip/hip_runtime.h>

#include "../sf_internal.h"
#include "tree_dev.h"

namespace {

constexpr unsigned kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr unsigned kSpan = 32;      // particles per wavefront of the grid: fewer than an average group's 44
constexpr int kList = 128;          // queued cells / leaves / particle ids per wavefront
constexpr int kStack = 8192;        // node ids per wavefront (global memory)
constexpr int kHead = 160;          // room for a depth-first descent (tree depth <= 96)
// The top of each wavefront's node stack lives in LDS: a batch's children
// are pushed there and the next batch pops them without a round trip to L2.
// Children that do not fit go to the global stack, which is popped when the
// LDS top holds fewer than a batch.  The quadrupole walk's LDS (its cells
// carry 24 more bytes) leaves room for a smaller top at 5 wavefronts per SIMD.
constexpr int kTopMono = 256;
constexpr int kTopQuad = 128;
// A quadrupole walk under the relative opening test takes a cell as a
// monopole when G M l^2 <= kMonoBeta alpha |a| d^4.  The factor calibrates
// the two size terms against each other.  Swept at 4M particles (quadrupole
// walk, theta 1.15, alpha 2e-3 to 4e-3): up to 0.2 the 99th-percentile force
// error rises by under 3 % while the walk gets 18 % faster; 0.5 raises it by
// half, 1 more than quadruples it.
constexpr float kMonoBeta = 0.2f;

__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// the same on every lane: kept in a scalar register
__device__ __forceinline__ float uniform(float v) {
	return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

__device__ __forceinline__ float wave_min(float v) {
	for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
	return uniform(v);
}
__device__ __forceinline__ float wave_max(float v) {
	for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
	return uniform(v);
}

// The lists' entries are taken four at a time, one by each row of 16 lanes;
// lane 16 r + p sums entries 4 k + r for the particles p, p + 16, p + 32 and
// p + 48 of the group, as many of these slots as the group fills.
constexpr int kWays = 4;

struct Slots {
	float x[kWays], y[kWays], z[kWays];
	float t[kWays][4];   // plain sums of at most 64 terms
	double s[4];         // running sums of particle `lane`
	int terms;           // in t, per lane
};

// a of the upper 32 lanes with b of the lower ones, and the same for odd and even rows
__device__ __forceinline__ double swap_add32(float a, float b) {
	const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
	return (double)__uint_as_float(v[0]) + (double)__uint_as_float(v[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b) {
	const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
	const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
	return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Adds t over the rows, slot r's sum to row r: lane l then holds particle l's.
// In FP64: added plainly in FP32 the rows would make one sum of up to 256 terms
// before the running sum sees it (the 1M step 1753 -> 1761 us).
__device__ __forceinline__ void fold(Slots& a) {
#pragma unroll
	for (int u = 0; u < 4; ++u) {
		const double lo = swap_add32(a.t[0][u], a.t[2][u]);   // lower half: slot 0, upper: slot 2
		const double hi = swap_add32(a.t[1][u], a.t[3][u]);
		a.s[u] += swap_add16(lo, hi);
#pragma unroll
		for (int j = 0; j < kWays; ++j) a.t[j][u] = 0.0f;
	}
	a.terms = 0;
}

__device__ __forceinline__ void interact(float t[4], float xi, float yi, float zi, float4 bj, float eps2) {
	const float dx = bj.x - xi, dy = bj.y - yi, dz = bj.z - zi;
	float r2 = __builtin_fmaf(dx, dx, eps2);
	r2 = __builtin_fmaf(dy, dy, r2);
	r2 = __builtin_fmaf(dz, dz, r2);
	const float inv = __builtin_amdgcn_rsqf(r2);
	const float mi = bj.w * inv;
	const float w = mi * (inv * inv);
	t[0] = __builtin_fmaf(w, dx, t[0]);
	t[1] = __builtin_fmaf(w, dy, t[1]);
	t[2] = __builtin_fmaf(w, dz, t[2]);
	t[3] += mi;
}

// Monopole plus traceless quadrupole of a cell with e = com - x:
//   acc += M e / r^3 - Qt e / r^5 + (5/2) (e^T Qt e) e / r^7
//   pot += M / r + (1/2) (e^T Qt e) / r^5
// (the potential -G [M/r + (1/2) d^T Qt d / r^5] with d = -e and its
// gradient), Plummer-softened through r^2 = |e|^2 + eps^2.  Qt is
// (q0 = Qxx, Qxy, Qxz, Qyy; q1 = Qyz, Qzz), Qzz = -Qxx - Qyy stored with the
// queued cell.  34 VALU operations plus the rsqrt.
__device__ __forceinline__ void interact_quad(float t[4], float xi, float yi, float zi, float4 c, float4 q0, float2 q1,
                                              float eps2) {
	const float ex = c.x - xi, ey = c.y - yi, ez = c.z - zi;
	float r2 = __builtin_fmaf(ex, ex, eps2);
	r2 = __builtin_fmaf(ey, ey, r2);
	r2 = __builtin_fmaf(ez, ez, r2);
	const float inv = __builtin_amdgcn_rsqf(r2);
	const float inv2 = inv * inv;
	const float mi = c.w * inv;
	const float m3 = mi * inv2;
	const float inv5 = (inv * inv2) * inv2;
	const float qx = __builtin_fmaf(q0.x, ex, __builtin_fmaf(q0.y, ey, q0.z * ez));
	const float qy = __builtin_fmaf(q0.y, ex, __builtin_fmaf(q0.w, ey, q1.x * ez));
	const float qz = __builtin_fmaf(q0.z, ex, __builtin_fmaf(q1.x, ey, q1.y * ez));
	const float eqe = __builtin_fmaf(ex, qx, __builtin_fmaf(ey, qy, ez * qz));
	const float v = eqe * inv5;
	const float w = __builtin_fmaf(2.5f, v * inv2, m3);
	t[0] = __builtin_fmaf(w, ex, __builtin_fmaf(-inv5, qx, t[0]));
	t[1] = __builtin_fmaf(w, ey, __builtin_fmaf(-inv5, qy, t[1]));
	t[2] = __builtin_fmaf(w, ez, __builtin_fmaf(-inv5, qz, t[2]));
	t[3] = __builtin_fmaf(0.5f, v, t[3]) + mi;
}

// Interactions of P slots with the entries q[0 .. n), n <= 64, read from LDS.
template <int P>
__device__ __forceinline__ void eval_slots(Slots& a, const float4* q, int n, int row, float eps2) {
	if (n == 64) {
#pragma unroll (8 / P)
		for (int k = 0; k < 64; k += kWays) {
			const float4 b = q[k + row];
#pragma unroll
			for (int j = 0; j < P; ++j) interact(a.t[j], a.x[j], a.y[j], a.z[j], b, eps2);
		}
	} else {
		for (int k = row; k < n; k += kWays) {
			const float4 b = q[k];
#pragma unroll
			for (int j = 0; j < P; ++j) interact(a.t[j], a.x[j], a.y[j], a.z[j], b, eps2);
		}
	}
}

template <int P>
__device__ __forceinline__ void eval_slots_quad(Slots& a, const float4* c, const float4* q0, const float2* q1, int n,
                                                int row, float eps2) {
	if (n == 64) {
#pragma unroll 2
		for (int k = 0; k < 64; k += kWays) {
			const float4 b = c[k + row], r0 = q0[k + row];
			const float2 r1 = q1[k + row];
#pragma unroll
			for (int j = 0; j < P; ++j) interact_quad(a.t[j], a.x[j], a.y[j], a.z[j], b, r0, r1, eps2);
		}
		return;
	}
	for (int k = row; k < n; k += kWays) {
		const float4 b = c[k], r0 = q0[k];
		const float2 r1 = q1[k];
#pragma unroll
		for (int j = 0; j < P; ++j) interact_quad(a.t[j], a.x[j], a.y[j], a.z[j], b, r0, r1, eps2);
	}
}

// slots: (particles of the group + 15) / 16
__device__ __forceinline__ void eval_list(Slots& a, int slots, const float4* q, int n, int row, float eps2) {
	switch (slots) {
	case 1: eval_slots<1>(a, q, n, row, eps2); break;
	case 2: eval_slots<2>(a, q, n, row, eps2); break;
	case 3: eval_slots<3>(a, q, n, row, eps2); break;
	default: eval_slots<4>(a, q, n, row, eps2);
	}
	a.terms += (n + kWays - 1) / kWays;
	if (a.terms > 48) fold(a);
}

__device__ __forceinline__ void eval_list_quad(Slots& a, int slots, const float4* c, const float4* q0,
                                               const float2* q1, int n, int row, float eps2) {
	switch (slots) {
	case 1: eval_slots_quad<1>(a, c, q0, q1, n, row, eps2); break;
	case 2: eval_slots_quad<2>(a, c, q0, q1, n, row, eps2); break;
	case 3: eval_slots_quad<3>(a, c, q0, q1, n, row, eps2); break;
	default: eval_slots_quad<4>(a, c, q0, q1, n, row, eps2);
	}
	a.terms += (n + kWays - 1) / kWays;
	if (a.terms > 48) fold(a);
}

// Quadrupole lists take two entries at a time (4M step 4936 -> 4863 us).
// Monopole walk: 5 wavefronts per SIMD (96 VGPRs, no spills) run the 1M step
// in 1876 us, 4 in 2016.  Quadrupole walk: 4 (128 VGPRs) and 5 (34 spilled)
// measure the same.
// QUAD: cells carry traceless quadrupoles (node_q0, node_q1).
template <bool QUAD>
__global__ __launch_bounds__(kBlock, QUAD ? 4 : 5) void k_walk(const float4* __restrict__ body, const unsigned* __restrict__ order,
                                                 int N, const unsigned* __restrict__ groups,
                                                 const unsigned* __restrict__ group_count,
                                                 const float4* __restrict__ rec_a,
                                                 const float4* __restrict__ node_q0, const float* __restrict__ node_q1,
                                                 const int4* __restrict__ rec_b, float alpha_g, float eps2, double G, int acc_phys,
                                                 float* __restrict__ acc, float* __restrict__ pot,
                                                 unsigned long long* __restrict__ counters,
                                                 int* __restrict__ gstack) {
	__shared__ float4 s_cell[kWaves][kList];
	__shared__ int2 s_leaf[kWaves][kList];
	__shared__ int s_pid[kWaves][kList];
	__shared__ float4 s_part[kWaves][64];
	__shared__ float4 s_q0[kWaves][QUAD ? kList : 1];
	__shared__ float2 s_q1[kWaves][QUAD ? kList : 1];
	constexpr int kTop = QUAD ? kTopQuad : kTopMono;
	__shared__ int s_top[kWaves][kTop];
	const unsigned lane = threadIdx.x & 63u, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int row = (int)(lane >> 4);
	float4* cq0 = s_q0[w];
	float2* cq1 = s_q1[w];
	int* stack = gstack + (size_t)(blockIdx.x * kWaves + w) * kStack;
	int* top = s_top[w];
	float4* cells = s_cell[w];
	int2* leaves = s_leaf[w];
	int* pid = s_pid[w];
	float4* part = s_part[w];
	const unsigned long long lt = (1ull << lane) - 1ull;
	const int n_nodes = 2 * N - 1;
	const unsigned budget = 2u * (unsigned)n_nodes + 64u;
	unsigned long long n_cell_tot = 0, n_part_tot = 0, n_batch = 0;
	unsigned bad = 0;

	// Each wavefront has a first group of its own and takes further ones from
	// a shared counter: groups differ in cost (more so under the relative
	// opening test), and a static split leaves wavefronts idle at the end.
	const unsigned n_waves = gridDim.x * kWaves, n_groups = *group_count;
	for (unsigned g = blockIdx.x * kWaves + w; g < n_groups;) {
		const int base = (int)groups[g];
		int cnt = (int)groups[g + 1u] - base;
		if (cnt < 1 || cnt > 64 || base + cnt > N) {   // only a malformed list gets here
			bad = 1u;
			break;
		}
		const int p = base + (int)lane;
		const bool live = (int)lane < cnt;
		const int slots = (cnt + 15) / 16;
		Slots a;
		float gx0, gy0, gz0, gx1, gy1, gz1;   // the group's box
#pragma unroll
		for (int j = 0; j < kWays; ++j) {
			const float4 b = body[base + min(16 * j + (int)(lane & 15u), cnt - 1)];
			a.x[j] = b.x;
			a.y[j] = b.y;
			a.z[j] = b.z;
			gx0 = j ? fminf(gx0, b.x) : b.x;
			gy0 = j ? fminf(gy0, b.y) : b.y;
			gz0 = j ? fminf(gz0, b.z) : b.z;
			gx1 = j ? fmaxf(gx1, b.x) : b.x;
			gy1 = j ? fmaxf(gy1, b.y) : b.y;
			gz1 = j ? fmaxf(gz1, b.z) : b.z;
#pragma unroll
			for (int u = 0; u < 4; ++u) a.t[j][u] = 0.0f;
		}
#pragma unroll
		for (int u = 0; u < 4; ++u) a.s[u] = 0.0;
		a.terms = 0;
		gx0 = wave_min(gx0);
		gy0 = wave_min(gy0);
		gz0 = wave_min(gz0);
		gx1 = wave_max(gx1);
		gy1 = wave_max(gy1);
		gz1 = wave_max(gz1);
		// relative opening test: am = alpha / G times the smallest previous
		// |a| of the group (0: theta test alone; also when no particle has a
		// positive finite previous acceleration)
		float am = 0.0f;
		if (alpha_g > 0.0f) {
			float amag = 3.0e38f;
			if (live) {
				const unsigned i0 = order[p];
				const float ax = acc[3u * i0], ay = acc[3u * i0 + 1u], az = acc[3u * i0 + 2u];
				const float a = sqrtf(ax * ax + ay * ay + az * az);
				amag = acc_phys ? a : a / body[p].w;   // the reference's acc is m a
			}
			amag = wave_min(amag);   // fminf drops NaN
			am = (amag > 0.0f && amag < 3.0e38f) ? alpha_g * amag : 0.0f;
		}

		unsigned long long n_cell = 0, n_part = 0, n_mono = 0;
		unsigned popped = 0;
		// pending nodes: nt in the LDS top, ng in the global stack
		int nt = 1, ng = 0, nc = 0, nl = 0, npid = 0;
		if (lane == 0) top[0] = 0;   // root: internal node 0, or the only leaf when N == 1
		wave_fence();

		while (nt + ng > 0 || nc > 0 || nl > 0 || npid > 0) {
			if (nt + ng > 0) {
				// pops come from the LDS top first; the global stack grows by at
				// most 2 k per batch, and by one per batch in the narrow regime
				const int k = (ng + 128 <= kStack - kHead) ? min(64, nt + ng) : 1;
				const int kt = min(k, nt);
				int node = -1;
				if ((int)lane < kt) node = top[nt - 1 - (int)lane];
				else if ((int)lane < k) node = stack[ng - 1 - ((int)lane - kt)];
				nt -= kt;
				ng -= k - kt;
				popped += (unsigned)k;
				++n_batch;
				wave_fence();
				if (node >= n_nodes) {
					node = -1;   // only a malformed tree gets here
					bad = 1u;
				}
				int cls = 0;   // 0 none, 1 cell, 2 leaf, 3 open, 4 monopole of a quadrupole walk
				float4 ra = make_float4(0.f, 0.f, 0.f, 0.f);
				int4 rb = make_int4(0, 0, 0, 0);
				if (node >= 0) {
					ra = rec_a[node];
					rb = rec_b[node];
					const float dx = fmaxf(fmaxf(gx0 - ra.x, ra.x - gx1), 0.0f);
					const float dy = fmaxf(fmaxf(gy0 - ra.y, ra.y - gy1), 0.0f);
					const float dz = fmaxf(fmaxf(gz0 - ra.z, ra.z - gz1), 0.0f);
					const float d2 = dx * dx + dy * dy + dz * dz;
					// the sign bit of the r_crit^2 word marks a (first, count) record
					const bool leafy = rb.x < 0;
					// relative test: G M l^p <= alpha |a| d^(p+2), p = 2 for a
					// monopole and 3 for a quadrupole (l = the record's size).  A
					// quadrupole walk takes a cell that meets the p = 2 bound
					// (scaled by kMonoBeta) as a monopole, for 13 VALU instead of 34.
					bool rel = true, mono = false;
					if (am > 0.0f) {
						const float l = __int_as_float(rb.w), d4 = d2 * d2;
						const float ml2 = ra.w * l * l;
						mono = ml2 <= (QUAD ? kMonoBeta : 1.0f) * am * d4;
						rel = QUAD ? ml2 * l <= am * d4 * sqrtf(d2) : mono;
					}
					// a cell holds at least two particles (every internal node does)
					if (d2 > __int_as_float(rb.x & 0x7fffffff) && (!leafy || rb.z > 1) && rel)
						cls = (QUAD && mono) ? 4 : 1;
					else if (leafy) cls = 2;
					else cls = 3;
				}
				const unsigned long long m_cell = __ballot(cls == 1);
				const unsigned long long m_leaf = __ballot(cls == 2);
				const unsigned long long m_open = __ballot(cls == 3);
				// monopoles of a quadrupole walk join the particle queue as
				// negative ids (npid < 64 here, so 64 more fit in pid[])
				const unsigned long long m_mono = QUAD ? __ballot(cls == 4) : 0ull;
				if (QUAD && cls == 4) pid[npid + __popcll(m_mono & lt)] = ~node;
				if (cls == 1) {
					const int at = nc + __popcll(m_cell & lt);
					cells[at] = ra;
					if (QUAD) {
						const float4 q0 = node_q0[node];
						cq0[at] = q0;
						cq1[at] = make_float2(node_q1[node], -q0.x - q0.w);
					}
				}
				if (cls == 2) leaves[nl + __popcll(m_leaf & lt)] = make_int2(rb.y, rb.z);
				if (cls == 3) {
					// children fill the LDS top; what does not fit goes to the
					// global stack
					const int at = nt + 2 * __popcll(m_open & lt);
#pragma unroll
					for (int h = 0; h < 2; ++h) {
						const int child = h ? rb.z : rb.y;
						if (at + h < kTop) {
							top[at + h] = child;
						} else {
							const int gi = ng + at + h - kTop;
							if (gi < kStack) stack[gi] = child;   // always: see kHead
							else bad = 1u;
						}
					}
				}
				nc += __popcll(m_cell);
				nl += __popcll(m_leaf);
				npid += __popcll(m_mono);
				n_mono += (unsigned long long)__popcll(m_mono);
				const int pushed = nt + 2 * __popcll(m_open);
				ng = min(ng + max(pushed - kTop, 0), kStack);
				nt = min(pushed, kTop);
				wave_fence();
				if (popped > budget) {   // a tree visits each node at most once per group
					bad = 1u;
					nt = ng = 0;
				}
			}
			const bool drain = nt + ng == 0;
			// monopoles
			if (nc >= 64 || (drain && nc > 0)) {
				const int take = min(nc, 64);
				if (QUAD) eval_list_quad(a, slots, cells, cq0, cq1, take, row, eps2);
				else eval_list(a, slots, cells, take, row, eps2);
				n_cell += (unsigned long long)take;
				wave_fence();
				if ((int)lane < nc - take) {
					cells[lane] = cells[take + lane];
					if (QUAD) {
						cq0[lane] = cq0[take + lane];
						cq1[lane] = cq1[take + lane];
					}
				}
				nc -= take;
				wave_fence();
			}
			// leaves: expand into particle ids, then gather and sum 64 at a time
			if (nl >= 64 || npid >= 64 || (drain && (nl > 0 || npid > 0))) {
				int q = 0;
				while (q < nl || npid >= 64 || (drain && npid > 0)) {
					if (q < nl && npid < 64) {
						// up to 64 leaves at once, one per lane: an inclusive scan of
						// their counts places each leaf's particle ids after the
						// previous ones; the leaves that fit in pid[] (a prefix, the
						// scan being nondecreasing, and at least the first: counts
						// are at most 64 and npid < 64) are taken
						const int li = q + (int)lane;
						const int2 lf = li < nl ? leaves[li] : make_int2(0, 0);
						int incl = lf.y;
#pragma unroll
						for (int o = 1; o < 64; o <<= 1) {
							const int v = __shfl_up(incl, (unsigned)o);
							if ((int)lane >= o) incl += v;
						}
						const bool fits = li < nl && npid + incl <= kList;
						const int k = __popcll(__ballot(fits));
						const int total = __builtin_amdgcn_readlane(incl, k - 1);
						if (fits) {
							const int at = npid + incl - lf.y;
							for (int j = 0; j < lf.y; ++j) pid[at + j] = lf.x + j;
						}
						npid += total;
						q += k;
					}
					wave_fence();
					if (npid >= 64 || (drain && q == nl && npid > 0)) {
						const int take = min(npid, 64);
						if ((int)lane < take) {
							const int id = pid[lane];
							part[lane] = (!QUAD || id >= 0) ? body[id] : rec_a[~id];
						}
						wave_fence();
						eval_list(a, slots, part, take, row, eps2);
						n_part += (unsigned long long)take;
						wave_fence();
						if ((int)lane < npid - take) pid[lane] = pid[take + (int)lane];
						npid -= take;
						wave_fence();
					} else {
						break;
					}
				}
				wave_fence();
				if ((int)lane < nl - q) leaves[lane] = leaves[q + (int)lane];
				nl -= q;
				wave_fence();
			}
		}
		fold(a);
		if (live) {
			const unsigned i = order[p];
			const double f = acc_phys ? G : G * (double)body[p].w;
			acc[3u * i + 0u] = (float)(f * a.s[0]);
			acc[3u * i + 1u] = (float)(f * a.s[1]);
			acc[3u * i + 2u] = (float)(f * a.s[2]);
			pot[i] = (float)(-G * a.s[3]);
		}
		n_cell_tot += (n_cell + n_mono) * (unsigned long long)cnt;
		n_part_tot += (n_part - n_mono) * (unsigned long long)cnt;
		if (n_groups <= n_waves) break;
		if (lane == 0) g = n_waves + (unsigned)atomicAdd(&counters[5], 1ull);
		g = __builtin_amdgcn_readfirstlane(g);
	}
	const bool any_bad = __ballot(bad != 0u) != 0ull;
	if (counters && lane == 0) {
		atomicAdd(&counters[0], n_cell_tot);
		atomicAdd(&counters[1], n_part_tot);
		if (any_bad) {
			atomicAdd(&counters[2], 1ull);
			atomicAdd(&counters[4], 1ull);   // sticky: cleared when the host checks it
		}
		atomicAdd(&counters[3], n_batch);
	}
}

// Blocks that are resident at once, the size of the persistent grid: every
// wavefront runs from the start and takes chunks until none are left
// (cached after the first call).
template <bool QUAD>
unsigned resident_blocks_of(void) {
	static unsigned cached = 0;
	if (cached) return cached;
	int per_cu = 0, cus = 0, dev = 0;
	if (hipGetDevice(&dev) != hipSuccess ||
	    hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_walk<QUAD>, kBlock, 0) != hipSuccess ||
	    hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu < 1 ||
	    cus < 1) {
		(void)hipGetLastError();
		per_cu = 4;
		cus = 256;
	}
	cached = (unsigned)per_cu * (unsigned)cus;
	return cached;
}

// the node stacks are sized for the larger of the two variants' grids
unsigned resident_blocks(void) { return max(resident_blocks_of<false>(), resident_blocks_of<true>()); }

}  // namespace

extern "C" {

size_t sfd_lbvh_walk_stack_bytes(void) { return (size_t)resident_blocks() * kWaves * kStack * sizeof(int); }

int sfd_lbvh_walk(const void* body, const unsigned* order, unsigned N, const unsigned* groups, const unsigned* n_groups,
                  const void* node_cm, const void* node_q0, const float* node_q1, const void* rec_b,
                  float alpha_g, float eps2, double G, int acc_phys, float* acc, float* pot,
                  unsigned long long* counters, int* gstack, hipStream_t s) {
	if (N == 0) return 0;
	if (!counters || !gstack || !groups || !n_groups) return -1;
	const bool quad = node_q0 && node_q1;
	const unsigned resident = quad ? resident_blocks_of<true>() : resident_blocks_of<false>();
	unsigned blocks = (N + kWaves * kSpan - 1u) / (kWaves * kSpan);
	if (blocks > resident) blocks = resident;   // gstack holds resident_blocks() >= resident slots
	const int tok = sf_prof_begin("lbvh_walk", s);
	if (quad)
		hipLaunchKernelGGL(k_walk<true>, dim3(blocks), dim3(kBlock), 0, s, static_cast<const float4*>(body), order,
		                   (int)N, groups, n_groups, static_cast<const float4*>(node_cm),
		                   static_cast<const float4*>(node_q0), node_q1, static_cast<const int4*>(rec_b),
		                   alpha_g, eps2, G, acc_phys, acc, pot, counters, gstack);
	else
		hipLaunchKernelGGL(k_walk<false>, dim3(blocks), dim3(kBlock), 0, s, static_cast<const float4*>(body), order,
		                   (int)N, groups, n_groups, static_cast<const float4*>(node_cm), (const float4*)nullptr,
		                   (const float*)nullptr, static_cast<const int4*>(rec_b), alpha_g, eps2, G, acc_phys,
		                   acc, pot, counters, gstack);
	sf_prof_end(tok, s);
	return sf_hip_check(hipGetLastError(), "sfd_lbvh_walk", "launch");
}

}  // extern "C"
