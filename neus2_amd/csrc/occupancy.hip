// Occupancy-grid update: the running 128^3 (x cascades) density estimate, its
// decayed-maximum merge with fresh field densities, the mean threshold, the
// 1-bit-per-cell morton bitfield the ray marcher reads and its 8 mip levels
// (Testbed::update_density_grid_nerf and update_density_grid_mean_and_bitfield,
// src/testbed_nerf.cu:3286-3391, kernels at :630-786).
//
// Sample positions and cell indices are part of the bit-exact contract with
// the CPU oracle, so floating-point contraction is off for this file.
#include "n2_common.h"

#include <new>

#pragma clang fp contract(off)

typedef _Float16 hf;

constexpr uint32_t OCC_GRIDSIZE = 128;
constexpr uint32_t OCC_CELLS = OCC_GRIDSIZE * OCC_GRIDSIZE * OCC_GRIDSIZE;
constexpr uint32_t OCC_LEVELS = 8;                          // NERF_CASCADES()
constexpr uint32_t OCC_LEVEL_BYTES = OCC_CELLS / 8;
constexpr float OCC_MIN_OPTICAL_THICKNESS = 0.1f;           // NERF_MIN_OPTICAL_THICKNESS(), SDF_GRID 0
constexpr uint32_t OCC_BLOCK = 256;
constexpr uint32_t OCC_MEAN_BLOCKS = OCC_CELLS / (OCC_BLOCK * 32);  // 256 partial sums of 8192 cells each

struct n2_occupancy {
	uint32_t n_cascades;
	uint64_t rng_state, rng_inc;
	uint32_t ema_step;
	unsigned char* ws;
	uint32_t max_samples, chunk;
	float* grid;         // [n_cascades][128^3]
	float* tmp;          // same
	float* positions;    // [max_samples + 8][3]
	uint32_t* indices;   // [max_samples + 8]
	hf* mlp_out;         // [16][chunk] fp16 (the field's full output, unfused path only), then [chunk] fp32: the density row
	uint8_t* bitfield;   // [8][128^3 / 8]
	float* partial;      // [OCC_MEAN_BLOCKS]
	float* mean;         // [1]
	uint32_t last_n, last_n_uniform;
};

// ---------------------------------------------------------------------------
// PCG32 (XSH-RR 64/32) as tiny-cuda-nn ships it: the reference hands the generator to the kernel by value,
// every thread skips 4*i draws ahead and takes four floats.
// ---------------------------------------------------------------------------
constexpr uint64_t PCG32_MULT = 0x5851f42d4c957f2dULL;

struct Pcg32 {
	uint64_t state, inc;
	__host__ __device__ uint32_t next_uint() {
		const uint64_t old = state;
		state = old * PCG32_MULT + inc;
		const uint32_t xorshifted = (uint32_t)(((old >> 18u) ^ old) >> 27u);
		const uint32_t rot = (uint32_t)(old >> 59u);
		return (xorshifted >> rot) | (xorshifted << ((~rot + 1u) & 31));
	}
	__device__ float next_float() { return __uint_as_float((next_uint() >> 9) | 0x3f800000u) - 1.0f; }
	__host__ __device__ void advance(uint64_t delta) {
		uint64_t cur_mult = PCG32_MULT, cur_plus = inc, acc_mult = 1u, acc_plus = 0u;
		while (delta > 0) {
			if (delta & 1) {
				acc_mult *= cur_mult;
				acc_plus = acc_plus * cur_mult + cur_plus;
			}
			cur_plus = (cur_mult + 1) * cur_plus;
			cur_mult *= cur_mult;
			delta /= 2;
		}
		state = acc_mult * state + acc_plus;
	}
};

__device__ __forceinline__ uint32_t occ_expand_bits(uint32_t v) {
	v = (v * 0x00010001u) & 0xFF0000FFu;
	v = (v * 0x00000101u) & 0x0F00F00Fu;
	v = (v * 0x00000011u) & 0xC30C30C3u;
	v = (v * 0x00000005u) & 0x49249249u;
	return v;
}
__device__ __forceinline__ uint32_t occ_morton3d(uint32_t x, uint32_t y, uint32_t z) {
	return occ_expand_bits(x) | (occ_expand_bits(y) << 1) | (occ_expand_bits(z) << 2);
}
__device__ __forceinline__ uint32_t occ_morton3d_invert(uint32_t x) {
	x = x & 0x49249249u;
	x = (x | (x >> 2)) & 0xc30c30c3u;
	x = (x | (x >> 4)) & 0x0f00f00fu;
	x = (x | (x >> 8)) & 0xff0000ffu;
	x = (x | (x >> 16)) & 0x0000ffffu;
	return x;
}

// generate_grid_samples_nerf_nonuniform (:630-660), unit aabb.  Slots [n, n_pad) are filled with the cube centre
// so that the field can run on a multiple of 8 points.
//
// Which sample a slot holds.  The first candidate cell of sample i is ((i + step n) P + R) mod 128^3 with P = 56924617: a
// pseudo-random walk over the cells, so that consecutive samples would splat their maxima into unrelated memory lines
// (one atomic request per sample).  The samples are independent of each other, so the order they are generated and
// evaluated in is free: when n is a power of two, slot t holds sample i(t) = t P^-1 mod n (P^-1 mod 2^32, masked), whose
// candidate cell is t + const mod n: consecutive slots splat into consecutive cells of (at most 128^3 / n) runs, and a
// wave's 64 atomics fall into a few lines.  Other n: slot t holds sample t.
constexpr uint32_t OCC_WALK = 56924617u, OCC_FIRST = 96925573u;
constexpr uint32_t occ_inverse_mod_2_32(uint32_t a) {  // a odd; Newton's iteration doubles the number of correct low bits
	uint32_t x = a;                                     // a * a = 1 mod 8
	for (int k = 0; k < 5; ++k) x *= 2u - a * x;
	return x;
}
constexpr uint32_t OCC_WALK_INV = occ_inverse_mod_2_32(OCC_WALK);
static_assert(OCC_WALK * OCC_WALK_INV == 1u, "inverse of the walk's multiplier");
static inline uint32_t occ_order_mul(uint32_t n) { return (n >= 2 && (n & (n - 1)) == 0) ? OCC_WALK_INV : 0u; }

// The rows of positions that the encoding's gather reads, and with them the densities, stand in another order yet where n is a power of two: a wave's 64
// cells are a brick of 16 x 2 x 2 along x instead of 4 x 4 x 4, because a line of the encoding's tables is 32 vertices along x, and a load is served
// in fewer clocks when neighbouring lanes ask for the same line.  The bricks lie on the cells' grid: a row's place gives its cell (of n, modulo n), the cell
// its slot.  Gather and whole update of 128^3 cells in us: slots' order 381 | 468, the same laid on the cells' grid - | 458, bricks 353 | 430.
// Where there are fewer samples than cells, 2 x 2 x 2 cells stay together in a brick: 2^20 samples 270 | 258, 2^19 161 | 157 (whole bricks along
// x 262 and 163), 2^19 and 2^19 others 286 | 282.  Samples that look for an occupied cell end up anywhere: their rows are in the slots' order (2^19 of either
// kind 289 with the others' in bricks, too).
struct OccOrder {
	uint32_t mul;    // slot -> sample (0: the same)
	uint32_t shift;  // a slot's first candidate cell is slot + shift mod n
	uint32_t mask;   // n - 1 where the rows have an order of their own, else 0
};
// Bit of the cell's number (x, y, z interleaved) that each bit of the row's place is, for samples of all cells and of fewer
constexpr uint32_t OCC_BRICK_BITS = 15;
constexpr uint8_t OCC_BRICK_ALL[OCC_BRICK_BITS] = {0, 3, 6, 9, 1, 2, 12, 4, 5, 7, 8, 10, 11, 13, 14};
constexpr uint8_t OCC_BRICK_SOME[OCC_BRICK_BITS] = {0, 3, 1, 2, 6, 9, 4, 5, 7, 8, 10, 11, 12, 13, 14};
__device__ __forceinline__ uint32_t occ_row_place(const OccOrder& o, uint32_t slot) {
	if (o.mask == 0u) return slot;
	const uint32_t cell = (slot + o.shift) & o.mask;
	const bool all = o.mask >= OCC_CELLS - 1u;
	uint32_t at = cell & ~((1u << OCC_BRICK_BITS) - 1u);
#pragma unroll
	for (uint32_t b = 0; b < OCC_BRICK_BITS; ++b) at |= ((cell >> (all ? OCC_BRICK_ALL[b] : OCC_BRICK_SOME[b])) & 1u) << b;
	return at;
}
__device__ __forceinline__ uint32_t occ_row_slot(const OccOrder& o, uint32_t at) {
	if (o.mask == 0u) return at;
	const bool all = o.mask >= OCC_CELLS - 1u;
	uint32_t cell = at & ~((1u << OCC_BRICK_BITS) - 1u);
#pragma unroll
	for (uint32_t b = 0; b < OCC_BRICK_BITS; ++b) cell |= ((at >> b) & 1u) << (all ? OCC_BRICK_ALL[b] : OCC_BRICK_SOME[b]);
	return (cell - o.shift) & o.mask;
}

// The generator skips 4 i draws ahead for sample i: state -> mult^(4 i) state + inc (1 + mult + .. + mult^(4 i - 1)).  The skip is
// composed from the hexadecimal digits of i, whose two factors are a table of constants: a multiply-add per digit instead of
// a loop over the bits of 4 i with three 64-bit products each (2^21 samples, one cascade: 33 us and 5.6 us for the clearing -> 15.6 us for
// all of it; 42 us when every workgroup works the factors out itself).
// The launch also clears tmp (n_tmp floats, a multiple of 4), which the samples' densities are splatted into, and leaves the
// positions as three rows of n_rows floats beside the [n][3] array (rows: null or these): the encoding's gather reads them.
constexpr uint32_t OCC_DIGITS = 8;
struct OccSkips {
	uint64_t mult[OCC_DIGITS * 16], plus[OCC_DIGITS * 16];  // [digit's place][digit]; plus for an increment of one
};
constexpr OccSkips occ_build_skips() {
	OccSkips t{};
	uint64_t m = 1, s = 0;  // the skip by one unit of the place: 4 draws at first
	for (int k = 0; k < 4; ++k) {
		s = s * PCG32_MULT + 1u;
		m *= PCG32_MULT;
	}
	for (uint32_t p = 0; p < OCC_DIGITS; ++p) {
		uint64_t cm = 1, cs = 0;
		for (uint32_t d = 0; d < 16; ++d) {
			t.mult[p * 16 + d] = cm;
			t.plus[p * 16 + d] = cs;
			cs = cs * m + s;
			cm *= m;
		}
		m = cm;
		s = cs;
	}
	return t;
}
static __device__ const OccSkips OCC_SKIPS = occ_build_skips();

// EACH samples to a thread.  With more than one, for samples of all cells (n is a power of two then, and nothing is padded), a workgroup takes 1024 consecutive cells and their rows go
// through LDS: positions and indices are written in the slots' order, rows in theirs, all in whole lines.  (Each sample's row from the lane that has it is sixteen
// pieces of 16 bytes a store, whose lines other XCDs complete: 2^21 samples 25.3 us, now 21.8, and 20.5 with the rows in the slots' order.  Of fewer samples the four
// behind one another take longer than that saves: updates of 2^17 63.9 | 66.6, 2^20 234.8 | 234.5, 2^21 398.8 | 394.4.)
constexpr uint32_t OCC_SPREAD_BITS = 10, OCC_SPREAD = 1u << OCC_SPREAD_BITS;
static_assert(OCC_SPREAD_BITS <= OCC_BRICK_BITS, "whole groups of cells");
__host__ __device__ __forceinline__ bool occ_all_cells(const OccOrder& o) { return o.mask >= OCC_CELLS - 1u; }
// The cell within its 1024 of the q-th of their rows: the bits of the rows' order that lie within them, in its sequence
__device__ __forceinline__ uint32_t occ_spread_cell(uint32_t q) {
	uint32_t cell = 0u, b = 0u;
#pragma unroll
	for (uint32_t k = 0; k < OCC_BRICK_BITS; ++k)
		if (OCC_BRICK_ALL[k] < OCC_SPREAD_BITS) cell |= ((q >> b++) & 1u) << OCC_BRICK_ALL[k];
	return cell;
}
template <uint32_t EACH>
__global__ void __launch_bounds__(OCC_BLOCK) occ_generate_kernel(uint32_t n, uint32_t n_pad, Pcg32 first, uint32_t n_digits, uint32_t step, const float* __restrict__ grid,
                                                                 uint32_t n_cascades, float thresh, OccOrder order,
                                                                 float* __restrict__ positions, uint32_t* __restrict__ indices, float* __restrict__ rows, uint32_t n_rows,
                                                                 float* __restrict__ tmp, uint32_t n_tmp) {
	constexpr bool SPREAD = EACH > 1;
	static_assert(!SPREAD || EACH * OCC_BLOCK == OCC_SPREAD, "a workgroup takes the cells that it spreads");
	__shared__ ulonglong2 skip[OCC_DIGITS][16];
	__shared__ float spread[3][SPREAD ? OCC_SPREAD : 1];
	if (threadIdx.x < n_digits * 16u) {
		skip[threadIdx.x >> 4][threadIdx.x & 15u] = make_ulonglong2(OCC_SKIPS.mult[threadIdx.x], OCC_SKIPS.plus[threadIdx.x] * first.inc);
	}
	for (uint64_t k = blockIdx.x * OCC_BLOCK + threadIdx.x; k * 4u < n_tmp; k += (uint64_t)gridDim.x * OCC_BLOCK)
		reinterpret_cast<float4*>(tmp)[k] = make_float4(0.f, 0.f, 0.f, 0.f);
	__syncthreads();
	const uint32_t cell0 = blockIdx.x * OCC_SPREAD;  // SPREAD: the workgroup's first cell, modulo n
#pragma unroll
	for (uint32_t e = 0; e < EACH; ++e) {
		const uint32_t local = e * OCC_BLOCK + threadIdx.x, slot = SPREAD ? (cell0 + local - order.shift) & order.mask : blockIdx.x * OCC_BLOCK + threadIdx.x;
		if (slot >= n_pad) return;  // (without SPREAD: all slots are there)
		float pos[3] = {0.5f, 0.5f, 0.5f};
		if (slot < n) {
			Pcg32 rng = first;
			const uint32_t i = order.mul ? (slot * order.mul) & (n - 1u) : slot;
			for (uint32_t p = 0; p < n_digits; ++p) {
				const ulonglong2 f = skip[p][(i >> (4u * p)) & 15u];
				rng.state = f.x * rng.state + f.y;
			}
			const uint32_t level = (uint32_t)(rng.next_float() * n_cascades) % n_cascades;
			uint32_t idx = 0;
			for (uint32_t j = 0; j < 10; ++j) {
				idx = ((i + step * n) * OCC_WALK + j * 19349663u + OCC_FIRST) % OCC_CELLS;
				idx += level * OCC_CELLS;
				if (grid[idx] > thresh) break;
			}
			const uint32_t pos_idx = idx % OCC_CELLS;
			const float scale = scalbnf(1.0f, (int)level);
#pragma unroll
			for (int d = 0; d < 3; ++d) {
				const float c = (float)occ_morton3d_invert(pos_idx >> d);
				const float u = rng.next_float();
				pos[d] = ((c + u) / (float)OCC_GRIDSIZE - 0.5f) * scale + 0.5f;
			}
			indices[slot] = idx;
		}
		const uint32_t at = rows && slot < n ? occ_row_place(order, slot) : slot;
#pragma unroll
		for (int d = 0; d < 3; ++d) {
			positions[(size_t)slot * 3 + d] = pos[d];
			if (SPREAD) spread[d][local] = pos[d];
			else if (rows) rows[(size_t)d * n_rows + at] = pos[d];
		}
	}
	if constexpr (SPREAD) {
		__syncthreads();
#pragma unroll
		for (uint32_t e = 0; e < EACH; ++e) {
			const uint32_t local = occ_spread_cell(e * OCC_BLOCK + threadIdx.x), at = occ_row_place(order, (cell0 + local - order.shift) & order.mask);
#pragma unroll
			for (int d = 0; d < 3; ++d) rows[(size_t)d * n_rows + at] = spread[d][local];
		}
	}
}

// splat_grid_samples_nerf_max_nearest_neighbor (:662-680): positive floats order like their bit patterns.  Density i is that of row i.
__global__ void __launch_bounds__(OCC_BLOCK) occ_splat_kernel(uint32_t n, const uint32_t* __restrict__ indices, const float* __restrict__ density,
                                                              float* __restrict__ tmp, uint32_t n_uniform, OccOrder uniform, OccOrder others) {
	const uint32_t i = blockIdx.x * OCC_BLOCK + threadIdx.x;
	if (i >= n) return;
	const uint32_t slot = i < n_uniform ? occ_row_slot(uniform, i) : n_uniform + occ_row_slot(others, i - n_uniform);
	atomicMax(reinterpret_cast<uint32_t*>(tmp) + indices[slot], __float_as_uint(density[i]));
}

// ema_grid_samples_nerf (:698-727), fused with the partial sums of max(v, 0) over the first cascade (:3383).
// A block covers 8192 consecutive cells; its partial sum is built in a fixed order, so the mean is reproducible.
// MERGE false: only the partial sums (the grid was written from outside).  Bound by the trip to memory: a thread has its eight cells under way at once, the block
// is as many waves as a CU's share (four waves of 32 cells a thread in two batches 7.5 us for 128^3 cells, now 6.1).
constexpr uint32_t OCC_EMA_BLOCK = 1024, OCC_EMA_EACH = 8;
static_assert(OCC_EMA_BLOCK * OCC_EMA_EACH == OCC_BLOCK * 32 && OCC_CELLS % (OCC_BLOCK * 32) == 0, "whole blocks");
template <bool MERGE>
__global__ void __launch_bounds__(OCC_EMA_BLOCK) occ_ema_kernel(float decay, float4* __restrict__ grid, const float4* __restrict__ tmp, float* __restrict__ partial) {
	__shared__ float red[OCC_EMA_BLOCK / 64];
	constexpr uint32_t QUADS = OCC_EMA_EACH / 4;
	const size_t at = (size_t)blockIdx.x * (OCC_EMA_BLOCK * QUADS) + threadIdx.x;
	float4 val[QUADS], fresh[QUADS];
#pragma unroll
	for (uint32_t q = 0; q < QUADS; ++q) {
		val[q] = grid[at + q * OCC_EMA_BLOCK];
		if (MERGE) fresh[q] = tmp[at + q * OCC_EMA_BLOCK];
	}
	float sum = 0.f;
#pragma unroll
	for (uint32_t q = 0; q < QUADS; ++q) {
		const auto merged = [&](float v, float f) { return !MERGE || v < 0.f ? v : fmaxf(v * decay, f); };
		val[q] = make_float4(merged(val[q].x, fresh[q].x), merged(val[q].y, fresh[q].y), merged(val[q].z, fresh[q].z), merged(val[q].w, fresh[q].w));
		if (MERGE) grid[at + q * OCC_EMA_BLOCK] = val[q];
		sum += (fmaxf(val[q].x, 0.f) + fmaxf(val[q].y, 0.f)) + (fmaxf(val[q].z, 0.f) + fmaxf(val[q].w, 0.f));
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o);
	if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
	__syncthreads();
	if (threadIdx.x == 0 && blockIdx.x < OCC_MEAN_BLOCKS) {
		float all = 0.f;
#pragma unroll
		for (uint32_t w = 0; w < OCC_EMA_BLOCK / 64; ++w) all += red[w];
		partial[blockIdx.x] = all;
	}
}

// The mean over the first cascade from its partial sums: every workgroup adds them up again, in the same order, instead of
// waiting for a launch that does.  All OCC_BLOCK lanes take part.
static_assert(OCC_MEAN_BLOCKS == OCC_BLOCK, "one partial sum per lane");
__device__ __forceinline__ float occ_mean(const float* __restrict__ partial, float* red) {
	float sum = partial[threadIdx.x];
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o);
	if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
	__syncthreads();
	return ((red[0] + red[1]) + (red[2] + red[3])) / (float)OCC_CELLS;
}

// bitfield_max_pool (:766-786): a byte of the next level collects "any bit set" of 8 bytes (8 blocks of 2^3 cells) of
// the previous one ...
__device__ __forceinline__ uint32_t occ_pool_byte(const uint2 p) {
	uint32_t bits = 0;
#pragma unroll
	for (uint32_t j = 0; j < 4; ++j) {
		bits |= ((p.x >> (8 * j)) & 0xFFu) ? (1u << j) : 0u;
		bits |= ((p.y >> (8 * j)) & 0xFFu) ? (16u << j) : 0u;
	}
	return bits;
}
// ... and lands in the central half of the next level's grid: byte i of 8-byte groups -> byte of the next level
__device__ __forceinline__ uint32_t occ_pool_target(uint32_t i) {
	return occ_morton3d(occ_morton3d_invert(i >> 0) + OCC_GRIDSIZE / 8, occ_morton3d_invert(i >> 1) + OCC_GRIDSIZE / 8, occ_morton3d_invert(i >> 2) + OCC_GRIDSIZE / 8);
}

// grid_to_bitfield (:738-764): one byte = 8 consecutive (morton-ordered) cells, a lane works out eight of them and writes them
// as one store; levels beyond the scene's cascades are cleared.  With one cascade a lane's eight bytes also are all that
// goes into one byte of level 1: it writes that too, and the lanes that clear level 1 leave the central half alone.
__global__ void __launch_bounds__(OCC_BLOCK) occ_bitfield_kernel(uint32_t n_cascades, const float* __restrict__ grid, uint8_t* __restrict__ bitfield,
                                                                 const float* __restrict__ partial, float* __restrict__ mean) {
	__shared__ float red[OCC_BLOCK / 64];
	const float m = occ_mean(partial, red);
	if (blockIdx.x == 0 && threadIdx.x == 0) mean[0] = m;
	const uint32_t i = blockIdx.x * OCC_BLOCK + threadIdx.x;  // group of eight bytes
	uint2* out = reinterpret_cast<uint2*>(bitfield) + i;
	constexpr uint32_t GROUPS = OCC_LEVEL_BYTES / 8;
	if (i >= n_cascades * GROUPS) {
		if (n_cascades == 1 && i < 2u * GROUPS) {
			const uint32_t g = i - GROUPS, x = occ_morton3d_invert(g), y = occ_morton3d_invert(g >> 1), z = occ_morton3d_invert(g >> 2);  // 2^3 bytes each
			constexpr uint32_t LO = OCC_GRIDSIZE / 16, HI = LO + OCC_GRIDSIZE / 8;
			if (x >= LO && x < HI && y >= LO && y < HI && z >= LO && z < HI) return;
		}
		*out = make_uint2(0u, 0u);
		return;
	}
	const float thresh = fminf(OCC_MIN_OPTICAL_THICKNESS, m);
	uint32_t bytes[2] = {0u, 0u};
#pragma unroll
	for (uint32_t q = 0; q < 16; ++q) {
		const float4 a = reinterpret_cast<const float4*>(grid)[(size_t)i * 16 + q];
		const uint32_t bits = (a.x > thresh ? 1u : 0u) | (a.y > thresh ? 2u : 0u) | (a.z > thresh ? 4u : 0u) | (a.w > thresh ? 8u : 0u);
		bytes[q >> 3] |= bits << (4 * (q & 7u));
	}
	*out = make_uint2(bytes[0], bytes[1]);
	if (n_cascades == 1) bitfield[OCC_LEVEL_BYTES + occ_pool_target(i)] = (uint8_t)occ_pool_byte(make_uint2(bytes[0], bytes[1]));
}

// One level of pooling, for levels that have cells of their own or lie right above one that has.  Distinct i write distinct bytes.
__global__ void __launch_bounds__(OCC_BLOCK) occ_pool_kernel(const uint8_t* __restrict__ prev, uint8_t* __restrict__ next) {
	const uint32_t i = blockIdx.x * OCC_BLOCK + threadIdx.x;
	if (i >= OCC_CELLS / 64) return;
	next[occ_pool_target(i)] |= (uint8_t)occ_pool_byte(reinterpret_cast<const uint2*>(prev)[i]);
}

// The pooling of all levels from `first` on, by one workgroup: level first - 1 has nothing outside its central half, so level
// `first` has nothing outside its central quarter, and so on: 16^3 groups of bytes for the first level, an eighth for each
// level after it.  A level's bytes stay in LDS for the next one: bound by the chain of levels, each a trip to memory before.  (128^3 cells, one cascade: mean,
// bitfield and seven launches for the levels 42 us -> 13.3 us in two launches, this one 8.6; with the bytes in LDS 5.6.)
__global__ void __launch_bounds__(1024) occ_pool_upper_kernel(uint32_t first, uint8_t* __restrict__ bitfield) {
	constexpr uint32_t SIDE_LOG = 4, SIDE = 1u << SIDE_LOG, EACH = SIDE * SIDE * SIDE / 1024;  // groups of eight bytes along a side of the first level's central half
	static_assert(OCC_GRIDSIZE == 8 * SIDE, "half of 64 bytes along a side");
	__shared__ uint8_t own[2][SIDE * SIDE * SIDE];
	{
		const uint2* prev = reinterpret_cast<const uint2*>(bitfield + (size_t)(first - 1) * OCC_LEVEL_BYTES);
		uint2 p[EACH];
		uint32_t at[EACH];
#pragma unroll
		for (uint32_t q = 0; q < EACH; ++q) {
			const uint32_t k = q * 1024u + threadIdx.x;
			at[q] = occ_morton3d(SIDE / 2 + k % SIDE, SIDE / 2 + (k / SIDE) % SIDE, SIDE / 2 + k / (SIDE * SIDE));
			p[q] = prev[at[q]];
		}
#pragma unroll
		for (uint32_t q = 0; q < EACH; ++q) {
			const uint8_t byte = (uint8_t)occ_pool_byte(p[q]);
			bitfield[(size_t)first * OCC_LEVEL_BYTES + occ_pool_target(at[q])] = byte;
			own[0][q * 1024u + threadIdx.x] = byte;
		}
	}
	uint32_t lo = SIDE / 2 + SIDE, log = SIDE_LOG;  // the level below has bytes lo .. lo + 2^log - 1 along each axis
	for (uint32_t level = first + 1, q = 0; level < OCC_LEVELS; ++level, q ^= 1u) {
		__syncthreads();
		// (16, 8, 4 bytes from an even one on are half as many groups; so are two, from an odd one on, two groups)
		const uint32_t width = 1u << log, g = lo / 2, side_log = log > 1u ? log - 1u : 1u, side = 1u << side_log;
		for (uint32_t k = threadIdx.x; k < side * side * side; k += 1024) {
			const uint32_t x = g + (k & (side - 1u)), y = g + ((k >> side_log) & (side - 1u)), z = g + (k >> (2 * side_log));
			uint32_t byte = 0;
#pragma unroll
			for (uint32_t j = 0; j < 8; ++j) {
				const uint32_t bx = 2 * x + (j & 1u) - lo, by = 2 * y + ((j >> 1) & 1u) - lo, bz = 2 * z + (j >> 2) - lo;
				const bool inside = bx < width && by < width && bz < width;
				byte |= (own[q][inside ? (bz << 2 * log) + (by << log) + bx : 0u] != 0 && inside ? 1u : 0u) << j;
			}
			bitfield[(size_t)level * OCC_LEVEL_BYTES + occ_pool_target(occ_morton3d(x, y, z))] = (uint8_t)byte;
			own[q ^ 1u][k] = (uint8_t)byte;
		}
		lo = g + SIDE;
		log = side_log;
	}
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline uint64_t o256(uint64_t x) { return (x + 255) / 256 * 256; }

struct OccCarve {
	uint64_t grid, tmp, positions, indices, mlp_out, bitfield, partial, mean, total;
};
static OccCarve occ_carve(uint32_t n_cascades, uint32_t max_samples, uint32_t chunk) {
	OccCarve c{};
	uint64_t o = 0;
	auto take = [&](uint64_t bytes) { const uint64_t at = o; o = o256(o + bytes); return at; };
	c.grid = take(4ull * n_cascades * OCC_CELLS);
	c.tmp = take(4ull * n_cascades * OCC_CELLS);
	c.positions = take(12ull * ((uint64_t)max_samples + 8));
	c.indices = take(4ull * ((uint64_t)max_samples + 8));
	c.mlp_out = take(32ull * chunk + 4ull * chunk);
	c.bitfield = take((uint64_t)OCC_LEVELS * OCC_LEVEL_BYTES);
	c.partial = take(4ull * OCC_MEAN_BLOCKS);
	c.mean = take(4);
	c.total = o;
	return c;
}

N2_API int n2_occupancy_create(uint32_t n_cascades, uint64_t seed, n2_occupancy_t** out) {
	N2_REQUIRE(out != nullptr, "n2_occupancy_create: out is null");
	*out = nullptr;
	N2_REQUIRE(n_cascades >= 1 && n_cascades <= OCC_LEVELS, "n2_occupancy_create: n_cascades %u outside [1, %u]", n_cascades, OCC_LEVELS);
	n2_occupancy* o = new (std::nothrow) n2_occupancy();
	N2_REQUIRE(o != nullptr, "n2_occupancy_create: out of host memory");
	o->n_cascades = n_cascades;
	// pcg32(initstate = seed, initseq = 1)
	Pcg32 r{0u, (1ull << 1u) | 1u};
	r.next_uint();
	r.state += seed;
	r.next_uint();
	o->rng_state = r.state; o->rng_inc = r.inc;
	o->ema_step = 0;
	o->ws = nullptr;
	*out = o;
	return N2_OK;
}

N2_API void n2_occupancy_destroy(n2_occupancy_t* occ) { delete occ; }

static uint32_t occ_chunk(uint32_t max_samples, uint32_t max_chunk) {
	uint32_t c = (max_samples + 7) / 8 * 8;
	if (c > max_chunk) c = max_chunk / 8 * 8;
	return c;
}

N2_API uint64_t n2_occupancy_workspace_bytes(const n2_occupancy_t* occ, uint32_t max_samples, uint32_t max_chunk) {
	if (!occ || max_chunk < 8 || max_samples == 0) return 0;
	return occ_carve(occ->n_cascades, max_samples, occ_chunk(max_samples, max_chunk)).total;
}

N2_API int n2_occupancy_set_workspace(n2_occupancy_t* occ, void* d_workspace, uint64_t n_bytes, uint32_t max_samples, uint32_t max_chunk) {
	N2_REQUIRE(occ != nullptr && d_workspace != nullptr, "n2_occupancy_set_workspace: null argument");
	N2_REQUIRE(reinterpret_cast<uintptr_t>(d_workspace) % 256 == 0, "n2_occupancy_set_workspace: workspace must be 256-byte aligned");
	N2_REQUIRE(max_samples >= 1 && max_chunk >= 8, "n2_occupancy_set_workspace: max_samples >= 1 and max_chunk >= 8 required");
	const uint32_t chunk = occ_chunk(max_samples, max_chunk);
	const OccCarve c = occ_carve(occ->n_cascades, max_samples, chunk);
	N2_REQUIRE(n_bytes >= c.total, "n2_occupancy_set_workspace: %llu bytes given, %llu needed", (unsigned long long)n_bytes, (unsigned long long)c.total);
	unsigned char* b = reinterpret_cast<unsigned char*>(d_workspace);
	occ->ws = b; occ->max_samples = max_samples; occ->chunk = chunk;
	occ->grid = reinterpret_cast<float*>(b + c.grid);
	occ->tmp = reinterpret_cast<float*>(b + c.tmp);
	occ->positions = reinterpret_cast<float*>(b + c.positions);
	occ->indices = reinterpret_cast<uint32_t*>(b + c.indices);
	occ->mlp_out = reinterpret_cast<hf*>(b + c.mlp_out);
	occ->bitfield = b + c.bitfield;
	occ->partial = reinterpret_cast<float*>(b + c.partial);
	occ->mean = reinterpret_cast<float*>(b + c.mean);
	occ->last_n = 0;
	occ->last_n_uniform = 0;
	return N2_OK;
}

N2_API int n2_occupancy_reset(n2_occupancy_t* occ, n2_stream_t stream) {
	N2_REQUIRE(occ != nullptr && occ->ws != nullptr, "n2_occupancy_reset: no workspace");
	occ->ema_step = 0;
	if (int rc = n2_fill_zero_u32(n2_stream(stream), occ->grid, 4ull * occ->n_cascades * OCC_CELLS)) return rc;
	if (int rc = n2_fill_zero_u32(n2_stream(stream), occ->bitfield, (uint64_t)OCC_LEVELS * OCC_LEVEL_BYTES)) return rc;
	return n2_fill_zero_u32(n2_stream(stream), occ->mean, 4);
}

static inline dim3 ogrid(uint64_t n) { return dim3((uint32_t)((n + OCC_BLOCK - 1) / OCC_BLOCK)); }

static int occ_bitfield_from_partials(n2_occupancy_t* occ, hipStream_t s);

N2_API int n2_occupancy_update_bitfield(n2_occupancy_t* occ, n2_stream_t stream) {
	N2_REQUIRE(occ != nullptr && occ->ws != nullptr, "n2_occupancy_update_bitfield: no workspace");
	hipStream_t s = n2_stream(stream);
	const uint32_t n_elements = occ->n_cascades * OCC_CELLS;
	occ_ema_kernel<false><<<dim3(n_elements / (OCC_BLOCK * 32)), dim3(OCC_EMA_BLOCK), 0, s>>>(1.f, reinterpret_cast<float4*>(occ->grid), nullptr, occ->partial);
	N2_LAUNCH_CHECK();
	return occ_bitfield_from_partials(occ, s);
}

static int occ_bitfield_from_partials(n2_occupancy_t* occ, hipStream_t s) {
	occ_bitfield_kernel<<<ogrid(OCC_LEVELS * OCC_LEVEL_BYTES / 8), dim3(OCC_BLOCK), 0, s>>>(occ->n_cascades, occ->grid, occ->bitfield, occ->partial, occ->mean);
	N2_LAUNCH_CHECK();
	if (occ->n_cascades > 1) {
		for (uint32_t level = 1; level <= occ->n_cascades && level < OCC_LEVELS; ++level) {
			occ_pool_kernel<<<ogrid(OCC_CELLS / 64), dim3(OCC_BLOCK), 0, s>>>(occ->bitfield + (size_t)(level - 1) * OCC_LEVEL_BYTES,
			                                                                  occ->bitfield + (size_t)level * OCC_LEVEL_BYTES);
			N2_LAUNCH_CHECK();
		}
	}
	if (occ->n_cascades + 1 < OCC_LEVELS) {
		occ_pool_upper_kernel<<<dim3(1), dim3(1024), 0, s>>>(occ->n_cascades + 1, occ->bitfield);
		N2_LAUNCH_CHECK();
	}
	return N2_OK;
}

N2_API int n2_occupancy_update(n2_occupancy_t* occ, n2_field_t* field, n2_stream_t stream, float decay, uint32_t n_uniform,
                               uint32_t n_nonuniform) {
	N2_REQUIRE(occ != nullptr && occ->ws != nullptr, "n2_occupancy_update: n2_occupancy_set_workspace has not been called");
	N2_REQUIRE(field != nullptr, "n2_occupancy_update: field is null");
	const uint64_t n64 = (uint64_t)n_uniform + n_nonuniform;
	N2_REQUIRE(n64 <= occ->max_samples, "n2_occupancy_update: %llu samples exceed the workspace's %u", (unsigned long long)n64, occ->max_samples);
	hipStream_t s = n2_stream(stream);
	const uint32_t n = (uint32_t)n64, n_elements = occ->n_cascades * OCC_CELLS;
	Pcg32 rng{occ->rng_state, occ->rng_inc};
	// when one chunk holds all samples, their positions also go out as rows, into the fp16 scratch (which the unfused field
	// path writes only after it has read them)
	const uint32_t n8 = (n + 7) / 8 * 8;
	float* rows = n8 <= occ->chunk ? reinterpret_cast<float*>(occ->mlp_out) : nullptr;
	auto order_of = [&](uint32_t count) {
		return OccOrder{occ_order_mul(count), occ->ema_step * count * OCC_WALK + OCC_FIRST, 0u};
	};
	OccOrder uniform = order_of(n_uniform), others = order_of(n_nonuniform);
	if (rows != nullptr && uniform.mul != 0u && n_uniform >= (1u << OCC_BRICK_BITS)) uniform.mask = n_uniform - 1u;
	auto generate = [&](uint32_t count, uint32_t pad, uint32_t first, float thresh, bool clear, const OccOrder& order) -> int {
		uint32_t digits = 1;
		while (digits < OCC_DIGITS && (count >> (4u * digits)) != 0) ++digits;
		constexpr uint32_t EACH = OCC_SPREAD / OCC_BLOCK;
		const bool spread = occ_all_cells(order);
		auto* const kernel = spread ? occ_generate_kernel<EACH> : occ_generate_kernel<1>;
		kernel<<<ogrid(spread ? pad / EACH : pad), dim3(OCC_BLOCK), 0, s>>>(count, pad, rng, digits, occ->ema_step, occ->grid, occ->n_cascades, thresh, order,
		                                                                        occ->positions + (size_t)first * 3, occ->indices + first, rows ? rows + first : nullptr, n8,
		                                                                        occ->tmp, clear ? n_elements : 0u);
		N2_LAUNCH_CHECK();
		return N2_OK;
	};
	if (n == 0) {
		if (int rc = n2_fill_zero_u32(s, occ->tmp, 4ull * n_elements)) return rc;
	}
	if (n_uniform) {
		// slots of the second group are written by the second launch; only the last launch pads
		if (int rc = generate(n_uniform, n_nonuniform ? n_uniform : n8, 0, -0.01f, true, uniform)) return rc;
	}
	rng.advance(1ull << 32);
	if (n_nonuniform) {
		if (int rc = generate(n_nonuniform, n8 - n_uniform, n_uniform, OCC_MIN_OPTICAL_THICKNESS, n_uniform == 0, others)) return rc;
	}
	rng.advance(1ull << 32);
	occ->rng_state = rng.state;
	// densities, a chunk at a time (row 0 of the field's 16 x chunk output)
	for (uint32_t a = 0; a < n; a += occ->chunk) {
		const uint32_t m = (n - a < occ->chunk) ? n - a : occ->chunk, m8 = (m + 7) / 8 * 8;
		// only the density row is kept, as fp32 (the fp16 output widened); the row sits behind the fp16 scratch the unfused path needs
		float* row0 = reinterpret_cast<float*>(occ->mlp_out + (size_t)16 * occ->chunk);
		if (int rc = n2_field_sdf_row0(field, stream, rows ? rows : occ->positions + (size_t)a * 3, rows ? 1u : 3u, rows ? n8 : 1u, m8, m8, row0,
		                               reinterpret_cast<n2_half*>(occ->mlp_out), true)) return rc;
		occ_splat_kernel<<<ogrid(m), dim3(OCC_BLOCK), 0, s>>>(m, occ->indices + a, row0, occ->tmp, n_uniform, uniform, others);
		N2_LAUNCH_CHECK();
	}
	occ_ema_kernel<true><<<dim3(n_elements / (OCC_BLOCK * 32)), dim3(OCC_EMA_BLOCK), 0, s>>>(decay, reinterpret_cast<float4*>(occ->grid),
	                                                                                          reinterpret_cast<const float4*>(occ->tmp), occ->partial);
	N2_LAUNCH_CHECK();
	occ->ema_step += 1;
	occ->last_n = n;
	occ->last_n_uniform = n_uniform;
	return occ_bitfield_from_partials(occ, s);
}

N2_API int n2_occupancy_view(n2_occupancy_t* occ, n2_occupancy_buffers* out) {
	N2_REQUIRE(occ != nullptr && out != nullptr, "n2_occupancy_view: null argument");
	N2_REQUIRE(occ->ws != nullptr, "n2_occupancy_view: n2_occupancy_set_workspace has not been called");
	out->density_grid = occ->grid;
	out->density_grid_tmp = occ->tmp;
	out->bitfield = occ->bitfield;
	out->mean = occ->mean;
	out->positions = occ->positions;
	out->indices = occ->indices;
	out->n_samples = occ->last_n;
	out->n_uniform = occ->last_n_uniform;
	out->n_cascades = occ->n_cascades;
	out->ema_step = occ->ema_step;
	out->rng_state = occ->rng_state;
	out->rng_inc = occ->rng_inc;
	return N2_OK;
}

N2_API int n2_occupancy_set_state(n2_occupancy_t* occ, uint32_t ema_step, uint64_t rng_state, uint64_t rng_inc) {
	N2_REQUIRE(occ != nullptr, "n2_occupancy_set_state: occupancy is null");
	N2_REQUIRE((rng_inc & 1u) == 1u, "n2_occupancy_set_state: a PCG32 increment is odd");
	occ->ema_step = ema_step; occ->rng_state = rng_state; occ->rng_inc = rng_inc;
	return N2_OK;
}
