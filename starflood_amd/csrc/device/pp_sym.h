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
// per offset.  Planes hold one float4 per body.
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
// Below 10240 bodies the one-sided kernel (k_pp_fast) is as fast: at 8192 it
// takes 29.8 us with its combine, the narrow layout 30.8 (its 544 blocks
// leave half of the wavefront slots empty); at 9217 43.6 and 36.7 us, at
// 10007 41.9 and 35.1, at 16384 80 and 67.
constexpr unsigned kSymMin = 10240;
// The wide layout from here: at 16384 bodies it takes 75.5 us and the narrow
// one 73.9, at 24576 146 and 140, at 32768 226 and 230, at 65536 832 and 845.
constexpr unsigned kSymWideMin = 25600;
constexpr size_t kSymPlaneBytes = (size_t)512 << 20;   // j planes of one launch, at most

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
// more i planes.  Measured, tiles: microseconds -- 32768 bodies 1: 247, 2:
// 226, 4: 233; 65536 2: 885, 8: 882, 16: 939; 131072 8: 3438, 32: 3410, 64:
// 3592; 262144 16: 13619, 32: 13429, 64: 13630.
constexpr SymGeometry sym_geometry(unsigned n_pad, bool wide) {
	SymGeometry g{};
	g.set = wide ? kSymWide : kSymNarrow;
	g.blocks = n_pad / g.set;
	g.offsets = g.blocks / 2u;
	size_t fit = kSymPlaneBytes / ((size_t)n_pad * 16u);
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
constexpr size_t sym_part_bytes(unsigned n_pad, bool wide) {
	const SymGeometry g = sym_geometry(n_pad, wide);
	const size_t planes = (size_t)g.chunks + g.dchunks + g.per_launch;
	return planes * n_pad * 16u + (g.per_launch < g.offsets ? (size_t)n_pad * 32u : 0u);
}

// the layout of the force kernel
constexpr bool sym_pp_wide(unsigned n_pad) { return n_pad >= kSymWideMin; }

#endif
