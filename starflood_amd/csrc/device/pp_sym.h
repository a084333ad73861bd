// pp_sym.h -- the work split of the kernels that evaluate each pair once
// (pp_sym.hip, adjoint.hip): which pairs a block takes, and the planes of
// partial sums it writes.
//
// The n_pad bodies form S sets.  Set b meets the sets b + 1 .. b + S / 2
// (modulo S), which covers every unordered pair of sets once; for even S the
// last of these, b + S / 2, is taken by b < S / 2 only.  The offset d = 0 ..
// S / 2 - 1 names the pair of b with b + 1 + d.  Pairs inside a set are
// summed one-sided, after the others.
//
// A block takes one set of i against a run of 64-body tiles of j.  It
// writes the sums of its i to an i plane (one plane per run) and those of
// each tile's j to the j plane of the offset: a body gets one contribution
// per offset.  Planes hold one record per body, in FP64: nothing is rounded
// between a block and the combine.
//
// Two layouts.  Narrow: a set is 256 bodies, held by each of the block's
// four wavefronts, which take a tile each.  Wide: a set is 1024 bodies, 256
// per wavefront, and the four wavefronts take the same tile, so that a body
// gets a quarter of the j contributions (N / 2048 of them instead of N / 512)
// at the price of a barrier per tile and of coarser items.
#ifndef SF_PP_SYM_H
#define SF_PP_SYM_H

#include <stddef.h>

constexpr unsigned kSymTile = 64;                      // j per tile
constexpr unsigned kSymNarrow = 256, kSymWide = 1024;  // bodies per set
// Below kSymMin bodies the one-sided kernel (k_pp_few).  A force with its combine
// and the wait for it, general masses: 10240 bodies one-sided 53.5 us, each pair
// once 53.4; 11264 58.7 and 54.4; 12288 68.7 and 62.0 (with float4 planes 9216
// 47.6 and 52.6).
constexpr unsigned kSymMin = 10240;
// The same line for the force VJP (k_vjp, k_vjp_sym).
constexpr unsigned kVjpSymMin = 10240;
// The wide layout from here.  The line was drawn where the two met with float4
// planes and packed bodies (kernels alone: 24576 bodies wide 146 us, narrow 140;
// 32768 226 and 230).  With FP64 planes they meet higher: a step with equal masses
// 26624 195 and 184, 32768 274 and 257, 49152 519 and 518, 57344 681 and 711, 65536
// 875 and 920; general masses 32768 300 and 288, 65536 1046 and 1054.
constexpr unsigned kSymWideMin = 25600;
constexpr size_t kSymPlaneBytes = (size_t)512 << 20;   // j planes of one launch, at most
constexpr unsigned kPpRecord = 32;                     // bytes of a body in a plane: the force's
constexpr unsigned kVjpRecord = 24;                    // and its VJP's

struct SymGeometry {
	unsigned set;          // bodies per set
	unsigned blocks;       // S
	unsigned offsets;      // S / 2
	unsigned per_launch;   // offsets taken by one launch
	unsigned tiles;        // tiles per block (wide layout)
	unsigned chunks;       // i planes: blocks per set, off the diagonal
	unsigned dchunks;      // and on it (first launch; narrow: one plane)
};

// Blocks of the wide layout's first launch at `tiles` tiles each.
constexpr unsigned sym_items(unsigned S, unsigned offsets, unsigned tiles) {
	constexpr unsigned per = kSymWide / kSymTile;
	return S * ((offsets * per + tiles - 1u) / tiles + (per + tiles - 1u) / tiles);
}

// Wide layout: the fewest tiles per block that leave at most ~4500 blocks,
// four to five times what is resident (1024), up to 32.  Fewer, longer
// blocks leave compute units idle at the end; more of them write and read
// more i planes.  Measured with float4 planes, tiles: microseconds -- 32768 bodies 1: 247, 2:
// 226, 4: 233; 65536 2: 885, 8: 882, 16: 939; 131072 8: 3438, 32: 3410, 64:
// 3592; 262144 16: 13619, 32: 13429, 64: 13630.
constexpr SymGeometry sym_geometry(unsigned n_pad, bool wide, unsigned record) {
	SymGeometry g{};
	g.set = wide ? kSymWide : kSymNarrow;
	g.blocks = n_pad / g.set;
	g.offsets = g.blocks / 2u;
	size_t fit = kSymPlaneBytes / ((size_t)n_pad * record);
	if (fit < 1u) fit = 1u;
	g.per_launch = fit < g.offsets ? (unsigned)fit : g.offsets;
	g.tiles = 1u;
	if (wide) {
		constexpr unsigned per = kSymWide / kSymTile;
		while (g.tiles < 32u && sym_items(g.blocks, g.per_launch, g.tiles) > 4500u) ++g.tiles;
		g.chunks = (g.per_launch * per + g.tiles - 1u) / g.tiles;
		g.dchunks = (per + g.tiles - 1u) / g.tiles;
	} else {
		// a block's wavefronts take one tile each: as many tiles as a set has
		g.chunks = g.per_launch;
		g.dchunks = 1u;
	}
	return g;
}

// Bytes of all planes, and of the FP64 running sums (one double4 per body)
// that several launches need.
constexpr size_t sym_part_bytes(unsigned n_pad, bool wide, unsigned record) {
	const SymGeometry g = sym_geometry(n_pad, wide, record);
	const size_t planes = (size_t)g.chunks + g.dchunks + g.per_launch;
	return planes * n_pad * record + (g.per_launch < g.offsets ? (size_t)n_pad * 32u : 0u);
}

// the layout of the force kernel
constexpr bool sym_pp_wide(unsigned n_pad) { return n_pad >= kSymWideMin; }

// k_pp_few: 64 i and 64 per j per wavefront, four wavefronts to a block; as many
// j tiles per wavefront as leave about eight wavefronts per SIMD (a force of
// 9216 bodies: four 54.1 us, eight 47.7, sixteen 48.8).
struct FewGeometry {
	unsigned per;       // j tiles per wavefront
	unsigned bslices;   // blocks (planes of partial sums) per 64 i
};
constexpr FewGeometry few_geometry(unsigned n_pad) {
	const unsigned long long t = n_pad / kSymTile;
	const unsigned per = (unsigned)((t * t + 8191u) / 8192u);
	const unsigned waves = (unsigned)((t + per - 1u) / per), slices = (waves + 3u) / 4u;
	return {(unsigned)((t + 4u * slices - 1u) / (4u * slices)), slices};
}
// bytes of partial sums of the fast PP force
constexpr size_t pp_part_bytes(unsigned n_pad) {
	return n_pad == 0u ? 0u : (n_pad >= kSymMin ? sym_part_bytes(n_pad, sym_pp_wide(n_pad), kPpRecord)
	                                            : (size_t)few_geometry(n_pad).bslices * n_pad * 32u);
}

#endif
