// Sizes of launches, and how their workgroups share the work, as functions of nothing but numbers: they also compile without
// HIP, so that they can be checked on their own.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define N2_HD __host__ __device__
#else
#define N2_HD
#endif

// Whether what a training step passes over between two uses of an optimiser's moment is more than the last-level cache holds, so that moments do not stay there and only push
// out what the next kernels read.  That is the optimiser's state and, for each sample of the batch, about 1600 bytes of coordinates, network rows, slopes and scatter records.
constexpr uint64_t N2_LAST_LEVEL_CACHE_BYTES = 256ull << 20, N2_STEP_BYTES_PER_SAMPLE = 1600;
static inline bool n2_moments_stream(uint64_t state_bytes, uint64_t batch) {
	return state_bytes + N2_STEP_BYTES_PER_SAMPLE * batch > N2_LAST_LEVEL_CACHE_BYTES;
}

// Whether a training step's optimiser makes lists of the parameters that have a gradient before it steps them (adam_step_kernel): in small batches on large tables, whose
// samples, with eight entries of two parameters on every level each, meet at most a sixth of the parameters.  Beyond, what a step takes is its lines, which lists meet in
// smaller pieces; small tables have most of their parameters met at any batch.  Steps in us, without | with lists:
//   table of 2^19 entries a level (12.6 M parameters): batch 2048 97.4 | 79.3, 4096 106.2 | 94, 6144 110.8 | 99.6, 8192 116.8 | 108.1, 12 288 121.6 | 119.5, 16 384 131.1 | 134.2
//   2^20 (24 M): 4096 145.7 | 124.2, 8192 180.5 | 160.1, 16 384 232.3 | 230.8, 20 480 259.5 | 266.4      2^22 (85 M): 8192 291 | 234, 16 384 373 | 307, 32 768 496 | 473, 65 536 724 | 765
//   2^17 (3.5 M): 2048 65.5 to 73 | 65.3, 4096 68 to 77 | 69, 8192 74.5 | 75 to 84                         2^14 (0.5 M): 256 52 to 58 | 59 to 62, 4096 59 to 62 | 65
constexpr uint64_t N2_LIST_PARAMS_MIN = 1u << 21, N2_LIST_BATCH_MAX = 40960;
static inline bool n2_adam_lists(uint64_t n_params, uint32_t n_levels, uint64_t batch) {
	return n_params >= N2_LIST_PARAMS_MIN && batch <= N2_LIST_BATCH_MAX && batch * n_levels * 16u * 6u <= n_params;
}

// Whether the optimiser's state is streamed past that cache (adam_step_kernel).  Where whole pieces of 64 bytes are written that pays long before all is full: a sample counts
// twice, and the line is 96 MiB lower.  Lists are written in pieces, and of them only the moments are streamed; their batches are small.  Steps in us, plain | streamed:
//   state 227 MB (table of 2^19 entries a level): batch 9088 117.6 | 113.4, 16 384 130.4 | 122.2, 24 576 148.7 | 132.3, 2^15 163.8 | 143.6, 2^16 202.5 | 178.8, 2^18 351 | 337.7; with lists 1024
//   75.7 | 76.0, 2048 79.1 | 79.1, 4096 85 to 95 | 83.4, 8192 107.9 | 102.4
//   434 MB (2^20): 16 384 240.6 | 228, 2^16 554 | 527; with lists 4096 125.7 | 124.2      1.5 GB (2^22): 2^16 745 | 719, 2^18 2000 | 1921; with lists 16 384 308.5 | 306.7
//   120 MB (2^18): 8192 83.1 | 87 to 95, 16 384 105.7 | 104.4, 2^15 124.3 | 119.8, 2^16 160.6 | 150; with lists 4096 73.3 | 75.9
//   63 MB (2^17): 16 384 81.3 | 83 to 91, 2^15 103.5 | 103.2, 2^16 138.5 | 134.7, 2^18 293.7 | 289.2
//   33 MB (2^16): 16 384 73.2 | 75.8, 2^16 127.0 | 127.0, 2^18 293.2 | 291.7        9 MB (2^14): 2^15 95.9 | 97.3, 2^18 270.2 | 270.0
static inline bool n2_optimiser_streams(uint64_t state_bytes, uint64_t batch, bool listed) {
	return listed ? n2_moments_stream(state_bytes, 8u * batch) : n2_moments_stream(state_bytes + (96ull << 20), 2u * batch);
}

// The encoding's Jacobian (384 bytes per point of sixteen levels) is streamed from 64 MiB on.  Forward, scatter and input gradient in
// us with nothing | the loads | the stores | both streamed: 2^18 uniform points (96 MiB) 219 | 203 | 204 | 195, along rays 169 | 165 | 163 | 157;
// 2^19 434 | 430 | 430 | 423; 2^17 (48 MiB) 108 in all four, along rays 92.  The SDF network with the eikonal term, 2^18: uniform 283 | 285 | 288 | 287,
// along rays 244 | 236 | 241 | 235; 2^17 155 | 154 | 155 | 153.
static inline bool n2_jacobian_streams(uint32_t n_points, uint32_t rows) { return 12ull * n_points * rows >= (64ull << 20); }
// Whether n elements to a row leave every row at the start of a line of 128 bytes (of an array that starts there).
static inline bool n2_rows_of_whole_lines(uint32_t n, uint32_t bytes) { return (uint64_t)n * bytes % 128u == 0u; }
// In the SDF network's step it is read once, by the launch right behind the one that writes it (n2_fused_sdf_eikonal): the stores stay in the last-level cache up to where
// that is full, and the loads, which nothing follows, are streamed much earlier.  Step in us, by the rule above | this one: 32 768 uniform 68.3 | 66.3, 65 536 along rays 83.2 | 81.8, 2^17
// 124.7 | 124.1 (uniform 144.4 | 145.0), 180 000 159.0 | 154.4, 2^18 209.6 | 204.6 (uniform 257.2 | 253.2), 393 216 uniform 377.4 | 364.5; with the stores cached beyond 2^19 along rays
// 380.6 | 385.0 (uniform 489.9 | 479.2), 2^20 752.9 | 771.8; with the loads streamed 8192 37.6 | 37.9.
static inline bool n2_step_jacobian_stores_stream(uint32_t n_points, uint32_t rows) { return 12ull * n_points * rows >= (160ull << 20); }
// Rows that do not start lines are streamed from 64 MiB on as above: where two waves share a line, the first one's streamed load costs the second one the line.  Along rays, streamed earlier all
// the same | not: 72 008 97.2 | 96.3, 100 008 115.2 | 112.4, 150 008 149.9 | 147.3; streamed | not at all: 262 136 217.0 | 219.9.
static inline bool n2_step_jacobian_loads_stream(uint32_t n_points, uint32_t rows) {
	return n2_rows_of_whole_lines(n_points, 12u) ? 12ull * n_points * rows >= (12ull << 20) : n2_jacobian_streams(n_points, rows);
}

// Points per thread of the scatter's sorting kernel.  Three of its workgroups share a CU, 768 run at a time.  One point per thread where all workgroups
// (levels x tiles) then start together: the launch takes one workgroup's chain of round trips, which is shorter for one point.  Beyond, a
// workgroup of two points per thread takes less than two of one, and the summing kernel finds half as many runs.  Both kernels in us, one | two:
//   16 levels (768: 24 576 points): uniform 8192 21.7 | 25.2, 16 384 25.1 | 26.8, 20 480 28.7 | 28.9, 24 576 30.0 | 30.0, 32 768 33.4 | 31.8, 52 344 40.4 | 38.0, 2^17 63 | 56
//     rays 8192 20.3 | 22.2, 16 384 23.3 | 23.5, 20 480 25.8 | 25.4, 24 576 27.2 | 26.8, 32 768 31.7 | 29.0; training step 16 384 134.7 | 135.9, 24 576 154.0 | 153.7,
//     32 768 153.7 | 151.6; field 16 384 55.8 | 57.2, 24 576 62.5 | 62.8, 32 768 68.4 | 67.6, 49 152 85.8 | 82.9
//   8 levels (49 152): uniform 32 768 21.4 | 22.2, 49 152 25.3 | 24.9, 52 344 26.5 | 25.5, 2^17 40 | 37; rays 24 576 15.0 | 15.7, 32 768 16.7 | 16.2, 49 152 18.9 | 17.8
//   4 levels (98 304): uniform 65 536 20.3 | 20.9, 98 304 24.4 | 24.8, 2^17 28.7 | 28.6; rays 65 536 12.6 | 12.9, 98 304 14.8 | 15.9, 2^17 18.2 | 18.0
constexpr uint32_t N2_BIN_AT_A_TIME = 768;
// the largest batch that takes one
static inline uint32_t n2_bin_single_points(uint32_t n_levels, uint32_t block) { return N2_BIN_AT_A_TIME / n_levels * block; }
static inline uint32_t n2_bin_points_per_thread(uint32_t n_levels, uint32_t n_points, uint32_t block) { return n_points <= n2_bin_single_points(n_levels, block) ? 1u : 2u; }

// Where the summing kernel finds a bucket's runs (grid_reduce_items).  Run r of a bucket, of which a workgroup has the tiles group, group + groups, ..., is a part of
// this tile (runs behind the last one: of the last tile).
static inline N2_HD uint32_t n2_run_tile(uint32_t group, uint32_t groups, uint32_t run, uint32_t part_shift, uint32_t tiles) {
	const uint32_t tile = group + groups * (run >> part_shift);
	return tile < tiles ? tile : tiles - 1u;
}
// A level's records are up to 2^33 (2^30 points, eight each), more than 32 bits count.  The 64 runs that a wave has at hand, every `stride`-th one, lie in at most
// 63 * 16 * 32 tiles behind the first one's: the wave's two addresses stand at that tile, and a lane counts from there.
static inline N2_HD uint64_t n2_run_base(uint32_t first_tile, uint32_t tile_records) { return (uint64_t)first_tile * tile_records; }
static inline N2_HD uint32_t n2_run_place(uint32_t first_tile, uint32_t tile, uint32_t tile_records) { return (tile - first_tile) * tile_records; }

// Whether the SDF network's step takes its one-pass kernel (sdf_eikonal_forward_kernel): a lane keeps its place in a matrix as a 32-bit number of bytes, 12 for each row and
// point of the Jacobian, of which the last lane starts at 60 n - 12 (row 4 of a scalar base).  Larger batches take the single kernels, whose places are 64-bit.  (In 64 bits per
// lane the kernel's registers spill: 56 us instead of 38.7 for 2^18 points.)
static inline bool n2_sdf_one_pass(uint32_t n) { return 60ull * n <= 1ull << 32; }

// The part of a lattice that one launch of its kernels takes: columns, rows and planes (lattice.hip).
struct N2LatticeSlab {
	uint32_t nx, ny, nz;
};
// Runs of 64 points along x that a slab may have: a launch has at most 2^32 - 1 threads, and the one for the fine levels has 64
// per run and level, of eleven levels at most.
constexpr uint32_t N2_LATTICE_RUNS = 1u << 22;
// Whole planes where `points` of them fit, else whole rows of one plane, else (few points, or rows of more than 2^28) a piece of one row.
static inline N2LatticeSlab n2_lattice_slab(const uint32_t res[3], uint64_t points) {
	const uint64_t longest = points < N2_LATTICE_RUNS * 64ull ? points : N2_LATTICE_RUNS * 64ull;
	const uint32_t nx = res[0] <= longest ? res[0] : longest >= 64u ? (uint32_t)longest / 64u * 64u : (uint32_t)longest;
	const uint32_t most = N2_LATTICE_RUNS / ((nx + 63u) / 64u);
	const uint32_t rows = points / nx < most ? (uint32_t)(points / nx) : most;
	if (nx < res[0]) return {nx, 1u, 1u};
	if (rows < res[1]) return {nx, rows, 1u};
	return {nx, res[1], rows / res[1] < res[2] ? rows / res[1] : res[2]};
}

// A slab's features, a 4-byte word per point and fine level, lie in the scratch (of `words` words) and, where a lattice has large slabs, in the output
// behind the slab's own points too, where nothing has been written yet.  A slab ends with workgroups that have most of a CU to themselves, which takes
// its two launches 33 us together.  On the other hand the scratch of a chunk of 2^22 points is 176 MiB, and features of more than that no longer stay in the 256 MiB
// behind the L2s: the line is for such chunks, where it makes a difference of 4 % at most.  Smaller chunks' scratches are far below that; there a line at four slabs would serve
// lattices of four to eight better.  In us, scratch alone | both (slabs that the scratch alone takes):
//   chunk 2^22: 64 x 512 x 512 1555 | 1576 (2.2), 320^3 1480 | 1473 (5.7), 384^3 2205 | 2172 (8.6), 400^3 2699 | 2630 (9.7), 464^3 4127 | 4025 (15), 512^3 4472 | 4290 (17)
//   chunk 2^20: 160^3 345 | 347 (3.2), 192^3 506 | 482 (5.5), 224^3 736 | 730 (7.8), 512 x 64 x 512 682 | 642 (8.7), 256^3 1039 | 977 (12), 320^3 1856 | 1661 (23), 400^3 3273 | 2831 (39)
//   chunk 2^18: 96^3 187 | 183 (3.4), 112^3 271 | 238 (4.9), 128^3 344 | 321 (7.3), 160^3 572 | 451 (13), 192^3 971 | 662 (22), 256^3 1752 | 1142 (47)
static inline bool n2_lattice_large_slabs(uint64_t all, uint64_t words, uint32_t n_fine) { return n_fine != 0 && all > words / n_fine * 8u; }
// Points that the next slab may have, `rest` of the lattice's being left, and how many levels' features go to the scratch.
static inline uint64_t n2_lattice_slab_points(uint64_t rest, uint64_t words, uint32_t n_fine, bool large, uint32_t& in_scratch) {
	in_scratch = n_fine ? n_fine : 1u;  // (without fine levels the walk reads, and does not use, a row of the scratch)
	uint64_t most = words / in_scratch < rest ? words / in_scratch : rest;
	for (uint32_t k = n_fine; large && k-- > 0;) {
		const uint64_t here = k ? words / k : rest, there = rest / (n_fine - k + 1u), points = here < there ? here : there;
		if (points > most) { most = points; in_scratch = k; }
	}
	return most;
}

// Planes that a wave of a lattice's kernels walks, of nz with `runs` runs of 64 points each; parts of equal length.
static inline uint32_t n2_lattice_part(uint32_t nz, uint32_t most) {
	const uint32_t parts = (nz - 1u) / most + 1u;
	return (nz - 1u) / parts + 1u;
}
// Fine levels: few enough that the last waves are done soon, fewer still where a SIMD would not get several waves
// (256^3, 208^3, 320^3 in us with 16 | 12 planes: 892 | 873, 572 | 565, 1547 | 1536; 96^3 with 8 | 4: 122 | 106).
static inline uint32_t n2_lattice_fine_walk(uint32_t runs, uint32_t nz) {
	const uint64_t waves = (uint64_t)runs * nz / 4096u;
	return n2_lattice_part(nz, waves >= 16u ? 12u : waves <= 4u ? 4u : (uint32_t)waves);
}
// The waves that a SIMD holds of its kernel, which has the registers for six (66; 87 and five for every lattice when it had two copies of the loop over the longest rows): five
// where a launch is small, by measurement.  Lattices in us, five | six: 48^3 47.3 | 46.9, 32 x 64 x 64 45.6 | 47.5, 64^3 53.9 | 55.5, 64 x 64 x 80 58.3 | 60.4,
// 96 x 64 x 64 57.1 | 58.6, 64 x 64 x 128 69.2 | 69.4, 80 x 96 x 64 68.9 | 69.0, 96^3 92.8 | 91.1; slabs of a chunk of 2^20 points 512 x 256 x 64 530 | 508, 512 x 512 x 64 929 | 902, 448 x 448 x 64 859 |
// 822; 200^3 in a box of a tenth 306 | 293, 304 x 256 x 128 627 | 609, 256^3 904 | 915, 512^3 the same; of 2^22 128^3 152 | 155, 400 x 80 x 240 330 | 323.  (Seven: 512 x 256 x 64 3 % and 200^3 3 % faster, 256^3 and 512^3 1 % slower.)
static inline uint32_t n2_lattice_fine_waves(uint32_t runs, uint32_t nz) { return (uint64_t)runs * nz <= 10240u ? 5u : 6u; }
// The walk, `per_simd` of whose waves a SIMD holds: the 1024 SIMDs take the waves in rounds, of which each costs a wave's planes and a start as long
// as two of them.  (By eye, up to 16 planes where there are many | by this count: 96^3 101 | 97, 128^3 174 | 171, 320^3 1547 | 1524, 512 x 64 x 512 623 | 600; with up to
// 30 planes 96^3 to 320^3 lose up to 1.5 %.)
static inline uint32_t n2_lattice_walk(uint32_t runs, uint32_t nz, uint32_t per_simd) {
	const uint64_t at_a_time = 1024u * per_simd;
	uint64_t least = ~0ull;
	uint32_t walk = 1;
	for (uint32_t most = 4; most <= 24u; ++most) {
		const uint32_t part = n2_lattice_part(nz, most);
		const uint64_t waves = (uint64_t)runs * ((nz - 1u) / part + 1u), cost = ((waves - 1u) / at_a_time + 1u) * (part + 2u);
		if (cost < least) { least = cost; walk = part; }
	}
	return walk;
}

// The chunks of four entries along x that the cells c_first .. c_last of a run and their neighbours at +1 lie in (either end may be
// the larger one): `chunks` of them from cell c_lo on.  Cells are signed: a box far outside the unit cube has them saturated at
// the ends of the 32-bit range, 2^32 apart.
N2_HD inline void n2_lattice_chunks(uint32_t c_first, uint32_t c_last, uint32_t& c_lo, uint32_t& chunks) {
	const int64_t a = (int32_t)c_first, b = (int32_t)c_last, lo = (a < b ? a : b) & ~(int64_t)3, hi = (a < b ? b : a) + 1;
	c_lo = (uint32_t)lo;
	chunks = (uint32_t)((hi - lo) >> 2) + 1u;
}

// Levels that the lattice's walk keeps planes of where its points gather for themselves (lattice_gather_walk_kernel), by the step along z.
// It is right for any level and step.  A level whose cells are larger than a step crosses into a new plane less than once per step; of one
// whose cells are smaller every step meets two planes and nothing is kept, but up to about 1.15 cells per step that costs less than its
// features' way through memory.  (Call in us with 6 | 8 | 10 levels walked, the default table, when every lattice took this kernel and it was a
// tenth slower: 128^3 187 | 190 | 197, 176^3 438 | 407 | 427, 208^3 647 | 679 | 675, 256^3 1056 | 1001 | 1010, 272^3 1335 | 1273 | 1257, 384^3 3097 | 2858 | 2706,
// 512^3 6783 | 6220 | 5745; 512 x 512 x 128 1777 | 1726 | 1789, 128 x 128 x 512 692 | 668 | 664.)
static inline uint32_t n2_lattice_walked_levels(const float scale[16], float step) {
	return scale[8] * step < 1.15f ? 10u : scale[7] * step < 0.95f ? 8u : 6u;
}
// The levels that lattice_walk_kernel can take, by where their vertices lie: a run of up to 64 points that are `step_x` apart meets at most
// 62 vertices of a row, which stand in the wave's lanes then, and a step along z (step_z >= 0) never leaves out a plane.  reach: the
// largest coordinate along x; where it is too large for a cell's number to be exact in fp32 nothing is known about a run's vertices.
// At most ten: a wave has registers for no more.
static inline uint32_t n2_lattice_row_levels(const float scale[16], uint32_t nx, float step_x, float reach, float step_z) {
	const float points = (float)(nx < 64u ? nx : 64u) - 1.f;
	uint32_t l = 0;
	while (l < 10u && points * scale[l] * step_x <= 60.f && scale[l] * reach < 4194304.f && step_z >= 0.f && scale[l] * step_z < 0.95f) ++l;
	return l;
}
// Which of the two.  A plane costs lattice_walk_kernel half the loads, but it walks fewer levels where the points are further apart along x
// than along z.  Call in us, gathering | by rows, (levels): 64^3 60 (6) | 81 (4), 80^3 83 (6) | 81 (5), 512 x 64 x 64 121 (6) | 128 (4),
// 512 x 512 x 64 913 (6) | 840 (4), 512 x 512 x 128 1604 (6) | 1495 (6), 256 x 256 x 512 1782 (10) | 1725 (8), 96 x 304 x 304 859 (10) | 852 (5),
// 128 x 512 x 512 2420 (10) | 2536 (6), 80 x 512 x 400 1638 (10) | 1703 (5), 64 x 512 x 512 1624 (10) | 1799 (4), 512^3 5219 (10) | 4802 (10).
// (With four levels walked, the other twelve levels' features of a small lattice do not fit the scratch at once.)
static inline bool n2_lattice_by_rows(uint32_t rows, uint32_t walked, uint64_t points) {
	return rows + 2u >= walked && (rows >= 5u || (rows == 4u && points >= 1u << 23));
}

// ----------------------------------------------------------------------------
// Which (level, tile of points) is this workgroup?  The hardware deals consecutive workgroup ids round-robin over the XCDs,
// each with an L2 of its own: id b runs on XCD b % 8.  Every XCD gets whole levels, so that its L2 fetches only those levels'
// tables and not all of them (24 MiB, eight times over).  Their cost per point differs by how the points lie (on points in
// ray order a fine level costs two and a half times a coarse one, on scattered ones about the same), so no plan by fixed costs is
// even on both; dealing the levels out in rounds of eight, forwards and backwards in turn from the finest down (XCD 0: 15 and
// 0, XCD 1: 14 and 1, ...), is within a tenth on both.  A last round of fewer than eight levels, the coarsest, is cut evenly.
// ----------------------------------------------------------------------------
constexpr uint32_t N2_XCDS = 8;
N2_HD inline uint32_t n2_xcd_blocks(uint32_t n_levels, uint32_t tiles) {
	return N2_XCDS * ((n_levels / N2_XCDS) * tiles + ((n_levels % N2_XCDS) * tiles + N2_XCDS - 1u) / N2_XCDS);
}
N2_HD inline bool n2_xcd_level_tile(uint32_t block, uint32_t n_levels, uint32_t tiles, uint32_t& level, uint32_t& tile) {
	const uint32_t xcd = block % N2_XCDS, j = block / N2_XCDS, round = j / tiles, rest = n_levels % N2_XCDS;
	if (round < n_levels / N2_XCDS) {
		tile = j - round * tiles;
		level = n_levels - N2_XCDS * (round + 1u) + ((round & 1u) ? xcd : N2_XCDS - 1u - xcd);
		return true;
	}
	const uint32_t share = (rest * tiles + N2_XCDS - 1u) / N2_XCDS, k = j - (n_levels / N2_XCDS) * tiles, item = xcd * share + k;
	if (k >= share || item >= rest * tiles) return false;
	level = item / tiles;
	tile = item - level * tiles;
	return true;
}

// The launch of a kernel that takes (level, tile of points) items: workgroups in x and y.  Up to `by_xcd_max` points the levels are
// dealt to the XCDs (y is 1); beyond, y counts the levels: the workgroups that run at one time then work on one or two
// levels, whose tables stay in every L2, and what reading the tables into every L2 costs is less than what the uneven XCDs
// lose.  (y, because a launch has at most 2^32 - 1 threads along x: 2^28 points of sixteen levels.)
// Call in us, level-major | by XCD:
//   field, points along rays: 2^14 12.4 | 9.9 and 52 000 24.8 | 19 (gather alone), 2^18 279 | 271, 2^19 507 | 502, 3 * 2^18 734 | 735, 2^20 961 | 969, 2^21 1917 | 1954
//   query, uniform points: 2^17 52.8 | 47.9, 2^18 87.8 | 86.6, 5 * 2^16 105.4 | 105.6, 3 * 2^17 123.4 | 125.3, 2^19 159 | 164, 2^20 301 | 314, 2^21 594 | 617
//   encoding alone, with the Jacobian and the backward: uniform 2^18 202 | 196, 2^19 421 | 422, 3 * 2^18 618 | 627, 2^20 819 | 834, 2^21 1708 | 1743;
//   rays 2^18 165 | 158, 2^19 334 | 329, 2^20 654 | 655, 2^21 1333 | 1349
// A listed pass of the field is dealt to the XCDs at any size (trained training step: 2^17 364 | 363, 2^18 559 | 530, 2^19 947 | 929, 2^20 1749 | 1726).
constexpr uint32_t N2_FIELD_XCD_MAX = 1u << 19, N2_QUERY_XCD_MAX = 5u << 16, N2_ENCODING_XCD_MAX = 1u << 19;
struct N2GatherGrid {
	uint32_t x, y;
};
static inline N2GatherGrid n2_gather_grid(uint32_t by_xcd_max, uint32_t n, uint32_t n_levels, uint32_t points_per_block) {
	const uint32_t tiles = n / points_per_block + (n % points_per_block != 0u);
	if (n <= by_xcd_max || n_levels == 1u) return {n2_xcd_blocks(n_levels, tiles), 1u};
	return {tiles, n_levels};
}
// the item of workgroup (x, y) of such a launch of `height` workgroups in y; false: none
N2_HD inline bool n2_gather_item(uint32_t x, uint32_t y, uint32_t height, uint32_t n_levels, uint32_t tiles, uint32_t& level, uint32_t& tile) {
	if (height == 1u) return n2_xcd_level_tile(x, n_levels, tiles, level, tile);
	level = y;
	tile = x;
	return true;
}

// A launch of two kinds of work in turn: `every` groups of workgroups of the first kind, then one group of the second, each `group` workgroups long.
struct N2Turns {
	uint32_t every, blocks;
};
static inline N2Turns n2_turns(uint32_t first, uint32_t second, uint32_t group) {
	const uint32_t every = (first + second - 1u) / second, a = (first + every * group - 1u) / (every * group), b = (second + group - 1u) / group;
	return {every, (a > b ? a : b) * (every + 1u) * group};
}
// The number of a workgroup among those of its kind, which may be past the last one.
N2_HD inline uint32_t n2_turn(uint32_t block, uint32_t every, uint32_t group, bool& second) {
	const uint32_t g = block / group, lane = block - g * group, q = g / (every + 1u), m = g - q * (every + 1u);
	second = m == every;
	return (second ? q : q * every + m) * group + lane;
}

// Workgroups beyond what a launch can count along x (2^32 - 1 threads) go into further rows in y, numbered through: row by row, each a multiple of the
// XCDs long, so that a number keeps its XCD.  The last ones may be past `blocks`.  (With the second order's output gathered beside it the sorting launch
// has 24 threads a point of sixteen levels: 2^28 points and less than 2^32 / 24 do not go together.)
static inline N2GatherGrid n2_rows_of_blocks(uint32_t blocks, uint32_t threads) {
	const uint32_t most = 0xFFFFFFFFu / threads / N2_XCDS * N2_XCDS;
	if (blocks <= most) return {blocks, 1u};
	const uint32_t y = blocks / most + (blocks % most != 0u), x = blocks / y + (blocks % y != 0u);
	return {(x + N2_XCDS - 1u) / N2_XCDS * N2_XCDS, y};
}
