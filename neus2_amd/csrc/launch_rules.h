// Sizes of launches that depend on nothing but numbers: host code without HIP, so that they can be checked on their own.
#pragma once
#include <cstdint>

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
