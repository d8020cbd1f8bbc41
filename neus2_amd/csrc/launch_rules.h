// Sizes of launches that depend on nothing but numbers: host code without HIP, so that they can be checked on their own.
#pragma once
#include <cstdint>

// Whether a training step streams its optimiser's moments past the last-level cache (n2_adam_step_gated): when what the step
// passes over between two uses of a moment is more than the cache holds, the moments do not stay there and only push out
// what the next kernels read.  That is the optimiser's state and, for each sample of the batch, about 1600 bytes of coordinates,
// network rows, slopes and scatter records.  Steps in us, plain | streamed:
//   state 227 MB (table of 2^19 entries a level): batch 4096 113 | 120, 20 480 140 | 142, 24 576 147 | 146, 28 672 154 | 152, 2^16 198 | 187, 2^18 381 | 373
//   434 MB (2^20): 4096 149 | 148, 8192 187 | 180, 2^15 349 | 335        1.5 GB (2^22): 4096 236 | 234, 2^14 385 | 379
//   63 MB (2^17): 2^14 100 | 102, 2^16 141 | 143, 2^17 201 | 199, 2^18 325 | 323        9 MB (2^14): 2^17 184 | 184, 2^18 305 | 304
constexpr uint64_t N2_LAST_LEVEL_CACHE_BYTES = 256ull << 20, N2_STEP_BYTES_PER_SAMPLE = 1600;
static inline bool n2_moments_stream(uint64_t state_bytes, uint64_t batch) {
	return state_bytes + N2_STEP_BYTES_PER_SAMPLE * batch > N2_LAST_LEVEL_CACHE_BYTES;
}

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
