// The field's SDF on a regular lattice (Testbed::get_density_on_grid, src/testbed_nerf.cu:4082-4133): what mesh extraction
// evaluates, up to 2^31 points at a time.
//
// On a lattice everything that a point's place in the encoding depends on is separable: cell and weight along an axis are
// functions of one index.  A wave takes a run of 64 points along x at one y and walks along z, so y and z quantities are
// wave-uniform (scalar registers) and a lane keeps only what depends on its x.  Two kinds of levels:
//  * coarse levels, whose cells are larger than the steps (lattice_walk_kernel): the values of the two z planes of vertices
//    round the walk's position stay in registers, already interpolated in x and y; a step only interpolates in z, and a
//    plane is loaded when the walk crosses into it (once per cell, loads issued one step ahead).
//  * fine levels (lattice_fine_kernel): nothing is shared between steps.  They run level by level over a slab of planes, so
//    that the 2 MiB table being read stays in every XCD's L2, and leave their features in the caller's scratch; the walk
//    picks them up.  (Point by point through all levels, 10 MiB of fine tables compete for 4 MiB of L2: 44 % of the requests
//    missed, 1.4 GB per 2^22 points through the fabric.)
// The walk hands its 64 points to the SDF network as two MFMA tiles: v_permlane32_swap_b32 turns "lane = point, register =
// level" into the operand layout "lane = (point, level group)" without touching LDS.
// 512^3 lattice in ten slabs: 3.86 to 3.98 ms on four cards; under the profiler 2.30 ms for six fine levels and 1.75 ms for the walk.  The fine levels are held by lines (one of 128 bytes into an L1
// in every 2.8 clocks; 2.3 at best) beside vector issue (83 %), the walk by vector instructions (69 %), waits of three waves per SIMD and
// the features, which come from beyond the L2 (37 % hits).  (On the same cards 4.25 to 4.32 ms with 2.46 and 1.98, before what stands at the two kernels; 4.80 in 18 slabs, when a walk's start waited
// for its planes one after the other and then for the fine features; 5.76 before that, with vertices picked out of LDS row by row, and four gathers per point and plane by two waves per SIMD.  One launch
// for a slab's walk and the next one's fine levels, in any mixture, or the two on two streams: 5.3 ms and more, the two hold each other up.)
// Features and SDF are written, and features read, as streams that pass by the caches: each is met once, and the tables stay where they are (by that alone 512^3 takes 1.7 % less, with the walk's
// alone 2.3; 464^3 2.3 %, 400^3 2.2, 192^3 1.8, 128^3 0.8; 448 x 512 x 96 0.2 %, with the walk's alone 0.9 more).
// Rows that are no multiple of 64 leave lanes idle in their last run.  Other lattices, before what stands at the two kernels | now, us: 64^3 59.2 | 54.3, 80^3 72.8 | 69.5, 96^3 96.0 | 91.3, 128^3 168.6 | 156.4,
// 208^3 563 | 509, 256^3 843 | 775, 320^3 1484 | 1348, 400^3 2634 | 2383, 464^3 4049 | 3605, 512 x 64 x 512 583 | 535, 64 x 512 x 512 1555 | 1425; with a chunk of 2^20 points 128^3 189 | 176, 256^3 971 | 918,
// 400^3 2839 | 2561, 512^3 4557 | 4203.
#include "n2_common.h"

#include "grid_device.h"
#include "launch_rules.h"
#include "mlp_device.h"
#include "sdf_frags.h"

#include <type_traits>

constexpr uint32_t LT_LEVELS = 16;
constexpr uint32_t LT_BLOCK = 256;
constexpr uint32_t LT_MAX_FINE = 11;  // feature rows of 4 bytes per point of a chunk that the scratch holds (n2_density_on_grid_scratch_bytes)

struct LatticeArgs {
	float scale[LT_LEVELS];
	uint32_t res[LT_LEVELS], entries[LT_LEVELS], offset[LT_LEVELS];
	uint32_t hash_mask, active_levels, n_levels;
	const __half2* table;
	hf* frags;                // fragment image of the SDF network, and what it is made of
	const hf* sdf_w;
	uint32_t sdf_in_w;
	float sdf_bias;
	N2Lattice lat;
	uint32_t y0, ny, z0, nz;  // the slab: rows y0 .. y0 + ny of planes z0 .. z0 + nz,
	uint32_t x_runs, walk;    // runs of 64 points per row of the slab; planes per wave of this launch
	uint32_t first_fine;      // levels first_fine .. n_levels - 1 come from `features`
	// [nz ny nx] half2 for each of the levels from first_fine on: rows of one buffer for the first `near_levels` of them, of another for the rest
	uint32_t *near, *beyond;  // (`beyond` counts its rows from first_fine on, too)
	uint32_t near_levels;
	uint64_t points;          // of the slab
	float* out;               // row 0 of point (x0, y0, z0)
	uint32_t x0, nx;          // columns x0 .. x0 + nx of the slab
};

// the features of the slab's points on level first_fine + f
__device__ __forceinline__ uint32_t* lattice_features(const LatticeArgs& a, uint32_t f) {
	return (f < a.near_levels ? a.near : a.beyond) + f * a.points;
}
// coordinate of lattice index c on axis d: each step rounded on its own (positions are part of a bit-exact contract)
__device__ __forceinline__ float lattice_coord(const N2Lattice& lat, int d, uint32_t c) {
	return __fadd_rn(__fmul_rn(__fmul_rn((float)c, lat.inv_res[d]), lat.extent[d]), lat.corner[d]);
}
__device__ __forceinline__ uint32_t lane_u32(uint32_t v, uint32_t lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane); }
__device__ __forceinline__ float lane_f32(float v, uint32_t lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)lane)); }

// A vertex's byte offset in its level's table is  xo ^ row  on a hashed level and  xo + row  (minus the table's size if that
// is past its end) on a dense one, xo the part of x and row the part of (y, z).
__device__ __forceinline__ uint32_t x_part(bool hashed, uint32_t entries, uint32_t res, uint32_t gx) {
	return (hashed ? gx & (entries - 1u) : min(gx, res)) << 2;
}
__device__ __forceinline__ uint32_t row_part(bool hashed, uint32_t entries, uint32_t res, uint32_t gy, uint32_t gz) {
	return (hashed ? ((gy * 2654435761u) ^ (gz * 805459861u)) & (entries - 1u) : min(gy, res) * res + min(gz, res) * res * res) << 2;
}
__device__ __forceinline__ uint32_t vertex(bool hashed, uint32_t table_bytes, uint32_t xo, uint32_t row) {
	if (hashed) return xo ^ row;
	const uint32_t at = xo + row;
	return min(at, at - table_bytes);  // one conditional subtraction stands in for the modulo (unsigned wrap-around)
}
__device__ __forceinline__ float2 lt_h2f(uint32_t raw) {
	const half2v h = __builtin_bit_cast(half2v, raw);
	return make_float2((float)h[0], (float)h[1]);
}
__device__ __forceinline__ uint32_t lt_pack(float a, float b) {
	const half2v h = {(hf)a, (hf)b};
	return __builtin_bit_cast(uint32_t, h);
}

// The wave's run: the lane's column of the slab (past the last one in a run that is not full), y, first plane.  False: nothing to do.
__device__ __forceinline__ bool lattice_run(const LatticeArgs& a, uint32_t wave, uint32_t& x, uint32_t& y, uint32_t& z, uint32_t& nz) {
	const uint32_t xr = wave % a.x_runs, rest = wave / a.x_runs, yy = rest % a.ny, zz = rest / a.ny;
	if (zz * a.walk >= a.nz) return false;
	x = xr * 64u + (threadIdx.x & 63u);
	y = a.y0 + yy;
	z = a.z0 + zz * a.walk;
	nz = min(a.walk, a.nz - zz * a.walk);
	return true;
}

// The SDF network's fragments as one image (SDF_FRAG_COUNT KiB): workgroup `block` of FRAG_BLOCKS
constexpr uint32_t FRAG_BLOCKS = SDF_FRAG_COUNT * 64u / LT_BLOCK + (SDF_FRAG_COUNT * 64u % LT_BLOCK != 0u);
__device__ __forceinline__ void lattice_write_frags(const LatticeArgs& a, uint32_t block) {
	const uint32_t i = block * LT_BLOCK + threadIdx.x;
	if (i < SDF_FRAG_COUNT * 64u) *reinterpret_cast<half8*>(a.frags + i * 8u) = sdf_forward_frag(a.sdf_w, (int)a.sdf_in_w, a.n_levels * 2u, (int)(i >> 6), (int)(i & 63u));
}
__global__ void __launch_bounds__(LT_BLOCK) lattice_frags_kernel(const LatticeArgs a) { lattice_write_frags(a, blockIdx.x); }

// Fine levels, level-major workgroup ids; the workgroups behind those write the fragments (a launch for them alone was 5 us of the 60
// that a lattice of 64^3 takes).  A run needs eight vertices per point, on four rows (y, z), (y + 1, z), (y, z + 1),
// (y + 1, z + 1).  On a hashed level a row's neighbours in x stand in one aligned 128-byte line per 32, permuted; a load of four bytes per lane costs the L1 one clock per
// group of four lanes at least, and up to four where the lanes' spacing makes their banks collide (spacing 8, the finest level of a 512^3 lattice: 65 clocks).  So the wave
// loads the rows as a whole and weighs the four rows against each other where they are, in
// registers; what remains is one row, which goes through LDS (in fp32, a slot left out after every 32 entries so that lanes any
// number of entries apart meet different banks), and every point picks its two neighbours (LDS active in 34 % of the
// clocks; 73 % when the eight vertices were picked there).  Runs longer than that (coarse lattices) and dense levels gather from memory.
//  * Rows of up to 384 entries come a word per lane (walk_words).  64 words of which sixteen lanes each meet aligned 64 bytes, in any order, take an L1 4.4 clocks; a load of 8
//    or 16 bytes per lane takes it 16.5 however few lanes take part, and a row seldom fills the last of those.
//  * Longer ones, 16 bytes per lane (walk_wide): eight words a lane and row would be as many clocks and four times the instructions.
//  * The waves of a small lattice, of four planes at most, take 8 or 16 bytes per lane always: there the number of a plane's loads counts and not what an L1 makes of them (64^3
//    60 us with wide loads, 65 with words).
// The kernel's launches for 512^3, wide loads alone | this, five waves per SIMD: 2.57 | 2.44 ms; lattices 256^3 935 | 910 us, 320^3 1605 | 1534, 400^3 2706 | 2624, 464^3 4047 | 3850, 512 x 64 x 512 680 | 655.
// It takes a line of 128 bytes in every 2.8 clocks (3.1 with wide loads alone; 2.3 at best, 216 lines for 64 points on six levels), beside vector issue (83 % of the clocks).  Each point taking the
// aligned 8 bytes round its corners by itself, without LDS, is slower where rows are of 64 entries and more (finest levels of 512^3 527 -> 575 and 690 -> 750 us).
constexpr uint32_t FINE_CHUNKS = 128;  // chunks of four entries a row may have
constexpr uint32_t FINE_SLOTS = FINE_CHUNKS * 4u + FINE_CHUNKS / 8u;
__device__ __forceinline__ uint32_t fine_slot(uint32_t entry) { return entry + (entry >> 5); }

// EACH entries per lane: of the rows at byte offsets row[q] (on a hashed level: entry x is at x's bytes ^ row[q]), weighed by
// weight[q], the sums, W of them at a time to put(h, sums).  off: the lane's places in a row, of W entries each; have: whether there is one.
// (A part's sums are put down before the next part's are formed, which takes eight registers less; the loads are under way together.)
template <uint32_t EACH, uint32_t W, class Put>
__device__ __forceinline__ void fine_sum_rows(const char* __restrict__ base, const uint32_t (&off)[2], const bool (&have)[2], const uint32_t (&row)[4],
                                              const float (&weight)[4], Put put) {
	constexpr uint32_t H = EACH / W;  // loads per row
	typedef uint32_t words __attribute__((ext_vector_type(W)));
	words v[4][H];  // (a lane without a place holds anything: its slots are not read)
#pragma unroll
	for (uint32_t h = 0; h < H; ++h)
		if (have[h]) {
#pragma unroll
			for (uint32_t q = 0; q < 4; ++q) v[q][h] = *reinterpret_cast<const words*>(base + (off[h] ^ (row[q] & ~(4u * W - 1u))));
		}
#pragma unroll
	for (uint32_t h = 0; h < H; ++h) {
		float2 sum[W];
#pragma unroll
		for (uint32_t e = 0; e < W; ++e) sum[e] = make_float2(0.f, 0.f);
#pragma unroll
		for (uint32_t q = 0; q < 4; ++q) {
			// the entries of a load are permuted by the row's low bits, the same for the whole wave
			auto add = [&](auto flip) __attribute__((always_inline)) {
				constexpr uint32_t F = decltype(flip)::value;
#pragma unroll
				for (uint32_t e = 0; e < W; ++e) {
					const float2 f = lt_h2f(v[q][h][e ^ F]);
					sum[e].x = fmaf(weight[q], f.x, sum[e].x);
					sum[e].y = fmaf(weight[q], f.y, sum[e].y);
					asm volatile("; permutation %2" : "+v"(sum[e].x), "+v"(sum[e].y) : "n"(F));  // (the cases stay apart: merged, each entry is picked by selects)
				}
			};
			if (W > 2u && (row[q] & 8u)) {
				if (row[q] & 4u) add(std::integral_constant<uint32_t, 3 % W>());
				else add(std::integral_constant<uint32_t, 2 % W>());
			} else {
				if (row[q] & 4u) add(std::integral_constant<uint32_t, 1>());
				else add(std::integral_constant<uint32_t, 0>());
			}
			// (here the row's load has arrived, whichever case was taken; without saying so the next plane's loads wait for the store)
			asm volatile("" ::"v"(v[q][h]));
		}
		put(h, sum);
	}
}

// WAVES per SIMD at most (n2_lattice_fine_waves, launch_rules.h).
template <uint32_t WAVES>
__global__ void __launch_bounds__(LT_BLOCK) __attribute__((amdgpu_waves_per_eu(1, WAVES))) lattice_fine_kernel(const LatticeArgs a, uint32_t blocks_per_level) {
	if (blockIdx.x >= blocks_per_level * (a.n_levels - a.first_fine)) {
		lattice_write_frags(a, blockIdx.x - blocks_per_level * (a.n_levels - a.first_fine));
		return;
	}
	__shared__ float2 staged[LT_BLOCK / 64][FINE_SLOTS];
	const uint32_t level = a.first_fine + blockIdx.x / blocks_per_level;
	const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x % blocks_per_level) * (LT_BLOCK / 64) + (threadIdx.x >> 6));
	uint32_t x, y, z, nz;
	if (!lattice_run(a, wave, x, y, z, nz)) return;
	const bool inside = x < a.nx;
	const uint32_t lane = threadIdx.x & 63u, plane = a.nx * a.ny;
	uint32_t* out = lattice_features(a, level - a.first_fine) + (size_t)(z - a.z0) * plane + (size_t)(y - a.y0) * a.nx + x;
	if (level >= a.active_levels) {
		for (uint32_t k = 0; k < nz; ++k)
			if (inside) out[(size_t)k * plane] = 0u;
		return;
	}
	const float scale = a.scale[level];
	const uint32_t res = a.res[level], entries = a.entries[level], bytes = entries << 2;
	const bool hashed = (a.hash_mask >> level) & 1u;
	float wx, wy, wz;
	uint32_t cx, cy, cz;
	n2_locate(lattice_coord(a.lat, 0, a.x0 + min(x, a.nx - 1u)), scale, wx, cx);
	n2_locate(lattice_coord(a.lat, 1, y), scale, wy, cy);
	n2_locate(lattice_coord(a.lat, 2, z + min(lane, nz - 1u)), scale, wz, cz);  // lane k: plane z + k (at most 64 of them)
	// lane k: the four rows of vertices of plane z + k and their weights
	uint32_t rows[4];
	float weights[4];
#pragma unroll
	for (uint32_t q = 0; q < 4; ++q) {
		rows[q] = row_part(hashed, entries, res, cy + (q & 1u), cz + (q >> 1));
		weights[q] = ((q & 1u) ? wy : 1.f - wy) * ((q >> 1) ? wz : 1.f - wz);
	}
	const char* base = reinterpret_cast<const char*>(a.table + a.offset[level]);
	const float ux = 1.f - wx;
	auto finish = [&](uint32_t k, const uint32_t (&raw)[8]) {
		float s[2][2] = {};
#pragma unroll
		for (uint32_t q = 0; q < 4; ++q) {
			const float w = lane_f32(weights[q], k);
#pragma unroll
			for (uint32_t b = 0; b < 2; ++b) {
				const float2 v = lt_h2f(raw[2 * q + b]);
				s[b][0] = fmaf(w, v.x, s[b][0]);
				s[b][1] = fmaf(w, v.y, s[b][1]);
			}
		}
		if (inside) __builtin_nontemporal_store(lt_pack(fmaf(ux, s[0][0], wx * s[1][0]), fmaf(ux, s[0][1], wx * s[1][1])), out);
		out += plane;
	};
	// chunks of four entries that the run meets: from c_lo's to the one behind c_hi's
	uint32_t c_lo, chunks;
	n2_lattice_chunks(lane_u32(cx, 0), lane_u32(cx, 63), c_lo, chunks);
	if (hashed && chunks <= FINE_CHUNKS) {
		float2* st = staged[threadIdx.x >> 6];
		const uint32_t at0 = fine_slot(cx - c_lo), at1 = fine_slot(cx - c_lo + 1u);
		// a plane's sums stand in LDS: from the lanes' places in the row to the points
		auto finish_row = [&]() __attribute__((always_inline)) {
			__builtin_amdgcn_wave_barrier();
			const float2 lo = st[at0], hi = st[at1];
			if (inside) __builtin_nontemporal_store(lt_pack(fmaf(ux, lo.x, wx * hi.x), fmaf(ux, lo.y, wx * hi.y)), out);
			out += plane;
		};
		auto plane_rows = [&](uint32_t k, uint32_t (&row)[4], float (&weight)[4]) __attribute__((always_inline)) {
#pragma unroll
			for (uint32_t q = 0; q < 4; ++q) {
				row[q] = lane_u32(rows[q], k);
				weight[q] = lane_f32(weights[q], k);
			}
		};
		auto walk_words = [&](auto loads) __attribute__((always_inline)) {
			constexpr uint32_t LOADS = decltype(loads)::value;
			// The run's entries start anywhere in 64 bytes: the lanes are turned so that sixteen of them meet one aligned 64 bytes.  (Lanes behind the last entry
			// load that again: behind a branch the loads would be waited for one by one.)
			uint32_t off[LOADS], slot[LOADS];
#pragma unroll
			for (uint32_t h = 0; h < LOADS; ++h) {
				uint32_t at = lane + 64u * h - c_lo % 16u;
				if (h == 0u && (int32_t)at < 0) at += 64u * LOADS;
				off[h] = ((c_lo + min(at, chunks * 4u - 1u)) & (entries - 1u)) << 2;
				slot[h] = fine_slot(at);
			}
			for (uint32_t k = 0; k < nz; ++k) {
				uint32_t row[4], v[4][LOADS];
				float weight[4];
				plane_rows(k, row, weight);
#pragma unroll
				for (uint32_t q = 0; q < 4; ++q)
#pragma unroll
					for (uint32_t h = 0; h < LOADS; ++h) v[q][h] = *reinterpret_cast<const uint32_t*>(base + (off[h] ^ row[q]));
				float2 sum[LOADS];
#pragma unroll
				for (uint32_t h = 0; h < LOADS; ++h) sum[h] = make_float2(0.f, 0.f);
#pragma unroll
				for (uint32_t q = 0; q < 4; ++q)
#pragma unroll
					for (uint32_t h = 0; h < LOADS; ++h) {
						const float2 f = lt_h2f(v[q][h]);
						sum[h].x = fmaf(weight[q], f.x, sum[h].x);
						sum[h].y = fmaf(weight[q], f.y, sum[h].y);
					}
				__builtin_amdgcn_wave_barrier();
#pragma unroll
				for (uint32_t h = 0; h < LOADS; ++h) st[slot[h]] = sum[h];
				finish_row();
			}
		};
		auto walk_wide = [&](auto each) __attribute__((always_inline)) {
			constexpr uint32_t EACH = decltype(each)::value, W = EACH < 4u ? EACH : 4u, H = EACH / W;
			// The run's places, of W entries each, start anywhere in 64 bytes.  The lanes are turned so that those of a group meet one
			// aligned 64 bytes (permuted), which the address unit takes at once; a group across two of them costs twice the time.
			uint32_t off[2], slot[2];
			bool have[2];
#pragma unroll
			for (uint32_t h = 0; h < H; ++h) {
				const uint32_t at = (lane + 64u * h - c_lo / W % (16u / W)) % (64u * H);
				have[h] = at < chunks * (4u / W);
				off[h] = ((c_lo + W * at) & (entries - 1u)) << 2;
				slot[h] = fine_slot(W * at);
			}
			for (uint32_t k = 0; k < nz; ++k) {
				uint32_t row[4];
				float weight[4];
				plane_rows(k, row, weight);
				fine_sum_rows<EACH, W>(base, off, have, row, weight, [&](uint32_t h, const float2 (&sum)[W]) __attribute__((always_inline)) {
					if (h == 0u) __builtin_amdgcn_wave_barrier();
#pragma unroll
					for (uint32_t e = 0; e < W; ++e) st[slot[h] + e] = sum[e];
				});
				finish_row();
			}
		};
		// (walk_wide<8> once: what two copies of it keep for their loops takes a wave per SIMD)
		if (chunks > 96u || (chunks > 64u && a.walk <= 4u)) walk_wide(std::integral_constant<uint32_t, 8>());
		else if (a.walk > 4u) {
			if (chunks > 64u) walk_words(std::integral_constant<uint32_t, 6>());
			else if (chunks > 48u) walk_words(std::integral_constant<uint32_t, 4>());
			else if (chunks > 32u) walk_words(std::integral_constant<uint32_t, 3>());
			else walk_words(std::integral_constant<uint32_t, 2>());
		} else if (chunks > 32u) walk_wide(std::integral_constant<uint32_t, 4>());
		else walk_wide(std::integral_constant<uint32_t, 2>());
		return;
	}
	const uint32_t x0 = x_part(hashed, entries, res, cx), x1 = x_part(hashed, entries, res, cx + 1u);
	auto load = [&](uint32_t k, uint32_t (&raw)[8]) __attribute__((always_inline)) {
#pragma unroll
		for (uint32_t q = 0; q < 4; ++q) {
			const uint32_t row = lane_u32(rows[q], k);
			raw[2 * q] = *reinterpret_cast<const uint32_t*>(base + vertex(hashed, bytes, x0, row));
			raw[2 * q + 1] = *reinterpret_cast<const uint32_t*>(base + vertex(hashed, bytes, x1, row));
		}
	};
	// The next plane's vertices are asked for in front of a plane's store: behind it, the wait for them is one for the store as well, which passes by the caches.  Lattices whose runs
	// are longer than a row of LDS, in us, behind | in front: 64 x 512 x 512 1518 | 1423, 64 x 480 x 304 919 | 866, 80 x 512 x 512 1860 | 1808, 160 x 320 x 480 1538 | 1507, 64^3 56.1 | 54.0, 96^3 95.3 |
	// 94.0, 128^3 161.3 | 158.8; others as before.
	uint32_t raw[8], next[8];
	load(0, raw);
	for (uint32_t k = 1; k < nz; ++k) {
		load(k, next);
		finish(k - 1u, raw);
#pragma unroll
		for (uint32_t q = 0; q < 8; ++q) raw[q] = next[q];
	}
	finish(nz - 1u, raw);
}

// exchange of the upper 32 lanes of `a` with the lower 32 of `b`
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
	const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
	a = r[0];
	b = r[1];
}

// The SDF of the wave's 64 points from their features (enc: one word per level), two tiles of the network.  Tile 0 works for lanes
// 0..31, tile 1 for lanes 32..63; at: the coordinates for either, x and y in word 0, in the lanes that need them (the lower half), z written here.
__device__ __forceinline__ void lattice_xy(float px, float py, uint32_t g, uint32_t& xc0, uint32_t& xc1) {
	xc0 = xc1 = lt_pack((float)((hf)px - (hf)0.5f), (float)((hf)py - (hf)0.5f));
	swap_halves(xc0, xc1);
	xc0 = g == 0u ? xc0 : 0u;
	xc1 = g == 0u ? xc1 : 0u;
}
__device__ __forceinline__ hf lattice_network(const hf* F, uint32_t lane, uint32_t (&enc)[LT_LEVELS], uint4v (&at)[2], float pz, float bias) {
	// (the fence keeps the network's fragments in LDS: hoisted out of the walk's loop they would take 40 registers)
	tile_fence();
	half8 xs[2][3];
#pragma unroll
	for (int c = 0; c < 2; ++c) {
		uint4v t[2];
#pragma unroll
		for (int q = 0; q < 4; ++q) {
			constexpr int first[4] = {0, 1, 4, 5};
			uint32_t p0 = enc[8 * c + first[q]], p1 = enc[8 * c + first[q] + 2];
			swap_halves(p0, p1);
			t[0][q] = p0;
			t[1][q] = p1;
		}
		xs[0][c] = __builtin_bit_cast(half8, t[0]);
		xs[1][c] = __builtin_bit_cast(half8, t[1]);
	}
	const half2v zc = {(hf)pz - (hf)0.5f, (hf)0};
	const uint32_t zcm = lane < 32u ? __builtin_bit_cast(uint32_t, zc) : 0u;
#pragma unroll
	for (int t = 0; t < 2; ++t) {
		at[t][1] = zcm;
		asm("" : "+v"(at[t]));  // (one set of registers for the whole walk: otherwise a second one, and eight moves a step)
		xs[t][2] = __builtin_bit_cast(half8, at[t]);
	}
	// The second layer, of which only row 0 is wanted: a lane holds half of its sample's hidden values (the other group the
	// other half), and a product of sixteen 4 x 4 blocks takes four of them with the weights that the lanes of a block share; all four rows come out alike.  (Dot
	// products on the vector unit, which the walk has least to spare of: 1.88 ms for 512^3, now 1.81; four more of the large products per tile took longer than those.)
	// (one tile after the other: side by side they take 32 registers more, and a third wave has no room; the weights of 32 rows serve both: read for each
	// tile anew, and with registers spilled whose return waits for the loads of two steps, the walk took 4.2 us a plane of 512^2, then 3.9; 3.5 with what depends on x in LDS)
	typedef float float4v __attribute__((ext_vector_type(4)));
	float4v dot[2] = {float4v(0.f), float4v(0.f)};
#pragma unroll
	for (int mt = 0; mt < 2; ++mt) {
		half8 w[3];
#pragma unroll
		for (int c = 0; c < 3; ++c) w[c] = frag(F, SDF_FRAG_W0 + mt * 3 + c, lane);
#pragma unroll
		for (int t = 0; t < 2; ++t) {
			float16v acc = zero16();
#pragma unroll
			for (int c = 0; c < 3; ++c) acc = N2_MFMA(w[c], xs[t][c], acc);
			half8 h[2];
			relu_pack(acc, h[0], h[1]);
#pragma unroll
			for (int c = 0; c < 2; ++c) {
				const half8 wv = frag(F, SDF_FRAG_WO + 2 * mt + c, lane & 32);  // row 0 of W_out in the order of h
				dot[t] = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_shufflevector(wv, wv, 0, 1, 2, 3), __builtin_shufflevector(h[c], h[c], 0, 1, 2, 3), dot[t], 0, 0, 0);
				dot[t] = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_shufflevector(wv, wv, 4, 5, 6, 7), __builtin_shufflevector(h[c], h[c], 4, 5, 6, 7), dot[t], 0, 0, 0);
			}
			__builtin_amdgcn_sched_barrier(0);
		}
	}
	// tile 0 belongs to lanes 0..31, tile 1 to the upper ones
	uint32_t s0 = __float_as_uint(dot[0][0]), s1 = __float_as_uint(dot[1][0]);
	swap_halves(s0, s1);
	return (hf)(__uint_as_float(s0) + __uint_as_float(s1)) + (hf)bias;
}

// The walk.  NM levels are interpolated here, the others come from a.features.  A row of a walked level's vertices that a run of 64
// points meets fits the wave's lanes (n2_lattice_row_levels): lane v holds vertex v of the run, the two rows of a plane are loaded
// as consecutive words and interpolated in y there, and the points pick their two neighbours through LDS.
// Three waves per SIMD (157 registers for ten levels, 22 scalars spilled to vector lanes), whose vector instructions and waits fill the time.  What took instructions away, the walk of 512^3 in ms: masks kept as they are (below) and rows'
// offsets by one product instead of five 2.06 -> 1.92, the coordinates in registers of their own 1.91, features loaded one step ahead instead of two, without twelve moves a
// step, 1.87, the second layer by small matrix products 1.81.
template <int NM>
__global__ void __launch_bounds__(LT_BLOCK, 3) lattice_walk_kernel(const LatticeArgs a) {
	__shared__ __align__(16) hf F[SDF_FRAG_COUNT * 512];
	__shared__ float2 line[LT_BLOCK / 64][NM][64];
	__shared__ uint2 place[LT_BLOCK / 64][NM][64];  // of the lane's point in a level's row: its weight, and the byte in `line` where its two vertices begin
	for (uint32_t i = threadIdx.x; i < SDF_FRAG_COUNT * 64u; i += LT_BLOCK) *reinterpret_cast<half8*>(F + i * 8u) = *reinterpret_cast<const half8*>(a.frags + i * 8u);
	__syncthreads();
	const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (LT_BLOCK / 64) + (threadIdx.x >> 6));
	uint32_t x, y, z, nz;
	if (!lattice_run(a, wave, x, y, z, nz)) return;
	const uint32_t lane = threadIdx.x & 63u, plane = a.nx * a.ny;
	const bool inside = x < a.nx;
	const float px = lattice_coord(a.lat, 0, a.x0 + min(x, a.nx - 1u)), py = lattice_coord(a.lat, 1, y);
	float2 (&mine)[NM][64] = line[threadIdx.x >> 6];
	// lane l: what depends on y and z of level l, and its lowest cell along x
	const uint32_t ll = lane & (LT_LEVELS - 1u);
	const float my_scale = a.scale[ll];
	const uint32_t my_res = a.res[ll], my_entries = a.entries[ll];
	const bool my_hashed = (a.hash_mask >> ll) & 1u;
	const uint32_t on = (1u << min(a.active_levels, (uint32_t)NM)) - 1u;  // levels in use here
	float my_wy, my_back, unused;  // my_back: from the plane above to the walk's position
	uint32_t my_cy, my_cz, my_first, my_last;
	n2_locate(py, my_scale, my_wy, my_cy);
	n2_locate(lane_f32(px, 0), my_scale, unused, my_first);
	n2_locate(lane_f32(px, 63), my_scale, unused, my_last);
	my_first = (uint32_t)min((int32_t)my_first, (int32_t)my_last);
	float unit = 1.f;  // (a product with a literal 1 would be taken out, and the operands converted one by one)
	asm("" : "+s"(unit));
	// A row of vertices (y, z) is at byte offset  y part ^ z part  on a hashed level (within its table) and  y part + z part  on a dense one: row_part, with one product a step.
	const uint32_t my_z_factor = (my_hashed ? 805459861u : my_res * my_res) << 2, my_z_most = my_hashed ? ~0u : my_res;
	const uint32_t my_bytes = my_entries << 2, my_in_table = (my_entries - 1u) << 2;
	const uint32_t my_y0 = (my_hashed ? my_cy * 2654435761u : min(my_cy, my_res) * my_res) << 2, my_y1 = (my_hashed ? (my_cy + 1u) * 2654435761u : min(my_cy + 1u, my_res) * my_res) << 2;
	auto rows_of = [&](uint32_t cz, uint32_t& r0, uint32_t& r1) __attribute__((always_inline)) {
		const uint32_t z = min(cz, my_z_most) * my_z_factor;
		r0 = my_hashed ? (my_y0 ^ z) & my_in_table : my_y0 + z;
		r1 = my_hashed ? (my_y1 ^ z) & my_in_table : my_y1 + z;
	};
	// the plane of vertices whose rows y, y + 1 are at byte offsets row0, row1; of_run: four times the vertex's number in the run
	my_first <<= 2;
	auto fetch = [&](int l, uint32_t of_run, uint32_t row0, uint32_t row1, uint32_t hash_mask, uint32_t (&raw)[2]) __attribute__((always_inline)) {
		const char* base = reinterpret_cast<const char*>(a.table + a.offset[l]);
		const uint32_t bytes = lane_u32(my_bytes, l), v = lane_u32(my_first, l) + of_run;
		if ((hash_mask >> l) & 1u) {
			const uint32_t xo = v & (bytes - 4u);
			raw[0] = *reinterpret_cast<const uint32_t*>(base + (xo ^ row0));
			raw[1] = *reinterpret_cast<const uint32_t*>(base + (xo ^ row1));
		} else {
			const uint32_t xo = min(v, lane_u32(my_res, l) << 2);
			raw[0] = *reinterpret_cast<const uint32_t*>(base + vertex(false, bytes, xo, row0));
			raw[1] = *reinterpret_cast<const uint32_t*>(base + vertex(false, bytes, xo, row1));
		}
	};
	auto blend_y = [&](int l, const uint32_t (&raw)[2]) __attribute__((always_inline)) {
		const float2 v0 = lt_h2f(raw[0]), v1 = lt_h2f(raw[1]);
		const float wy = lane_f32(my_wy, l);
		// (the differences as multiply-adds: those take half-precision operands as they are)
		mine[l][lane] = make_float2(fmaf(wy, fmaf(unit, v1.x, -v0.x), v0.x), fmaf(wy, fmaf(unit, v1.y, -v0.y), v0.y));
	};
	// What depends on x waits in LDS: kept in registers, cell and weight of every level take 20, and working them out at each plane takes 40 clocks of a
	// level's 110.
	uint2 (&places)[NM][64] = place[threadIdx.x >> 6];
#pragma unroll
	for (int l = 0; l < NM; ++l) {
		float w;
		uint32_t cx;
		n2_locate(px, lane_f32(my_scale, l), w, cx);
		places[l][lane] = make_uint2(__float_as_uint(w), ((threadIdx.x >> 6) * NM + l) * 512u + min(cx * 4u - lane_u32(my_first, l), 62u * 4u) * 2u);
	}
	auto blend_at = [&](const uint2 p, float2& to) __attribute__((always_inline)) {
		const float2* at = reinterpret_cast<const float2*>(reinterpret_cast<const char*>(line) + p.y);
		const float2 lo = at[0], hi = at[1];
		const float w = __uint_as_float(p.x);
		to = make_float2(fmaf(w, hi.x - lo.x, lo.x), fmaf(w, hi.y - lo.y, lo.y));
	};
	float2 hi[NM], rise[NM];  // the plane above, and by how much it is above the one below
	// (all levels, also those that are switched off: behind branches the loads would be waited for one by one)
	auto fetch_plane = [&](uint32_t cz, uint32_t (&raw)[NM][2]) __attribute__((always_inline)) {
		uint32_t r0, r1, v = lane * 4u;
		asm volatile("" : "+v"(v));  // (addresses formed here: kept for the next start, they take registers that a step needs)
		rows_of(cz, r0, r1);
#pragma unroll
		for (int l = 0; l < NM; ++l) fetch(l, v, lane_u32(r0, l), lane_u32(r1, l), a.hash_mask, raw[l]);
	};
	auto blend_plane = [&](const uint32_t (&raw)[NM][2], float2 (&to)[NM]) __attribute__((always_inline)) {
#pragma unroll
		for (int l = 0; l < NM; ++l) blend_y(l, raw[l]);
		__builtin_amdgcn_wave_barrier();
#pragma unroll
		for (int l = 0; l < NM; ++l) blend_at(places[l][lane], to[l]);
		__builtin_amdgcn_wave_barrier();
	};
	const uint64_t feat_at = (uint64_t)(z - a.z0) * plane + (uint64_t)(y - a.y0) * a.nx;  // (the same for the wave, like out)
	const uint32_t feat_x = min(x, a.nx - 1u) * 4u;  // in bytes
	float* out = a.out + (uint64_t)(z - a.z0) * ((uint64_t)a.lat.res[0] * a.lat.res[1]) + (uint64_t)(y - a.y0) * a.lat.res[0];
	uint32_t xc0, xc1;
	lattice_xy(px, py, lane >> 5, xc0, xc1);
	uint4v at[2] = {uint4v{xc0, 0u, 0u, 0u}, uint4v{xc1, 0u, 0u, 0u}};
	// (levels that the table does not have read the last one's row: their weights are zero)
	const uint32_t have_fine = a.n_levels > (uint32_t)NM ? ~0u : 0u;
	const uint32_t* row[LT_LEVELS - NM];
#pragma unroll
	for (uint32_t f = 0; f < LT_LEVELS - NM; ++f) row[f] = lattice_features(a, have_fine ? min(f, a.n_levels - 1u - NM) : 0u) + feat_at;
	uint32_t fine[LT_LEVELS - NM];
	auto load_fine = [&](uint32_t k, uint32_t (&to)[LT_LEVELS - NM]) __attribute__((always_inline)) {
		uint32_t at = feat_x;
		asm volatile("" : "+v"(at));  // (the lane's 32 bits beside a uniform address; their sum, formed in front of the loop, takes registers that a step needs)
#pragma unroll
		for (uint32_t f = 0; f < LT_LEVELS - NM; ++f) to[f] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(row[f] + (uint64_t)k * plane) + at));
	};
	// Steps one after the other from plane k on, until the end or to where some level's next plane is not the one above (a box upside down;
	// steps of more than a cell): there the walk starts anew.  (With that case inside the loop, where it is hardly ever met, its
	// loads cost all others their overlap: whether they are under way is then not known, and everything is waited for; 131 -> 190 us.)
	uint32_t k = 0;
	while (true) {
	n2_locate(lattice_coord(a.lat, 2, z + k), my_scale, my_back, my_cz);
	my_back -= 1.f;
	{
		// (all of a start's loads under way together)
		uint32_t below[NM][2], above[NM][2];
		fetch_plane(my_cz, below);
		fetch_plane(my_cz + 1u, above);
		load_fine(k, fine);
		blend_plane(below, rise);
		blend_plane(above, hi);
	}
#pragma unroll
	for (int l = 0; l < NM; ++l) {
		rise[l] = make_float2(hi[l].x - rise[l].x, hi[l].y - rise[l].y);
		if (!((on >> l) & 1u)) hi[l] = rise[l] = make_float2(0.f, 0.f);  // switched off
	}
	while (true) {
		const float pz = lattice_coord(a.lat, 2, z + k);
		// features of this step
		uint32_t enc[LT_LEVELS];
#pragma unroll
		for (int l = 0; l < NM; ++l) {
			const float back = lane_f32(my_back, l);
			enc[l] = lt_pack(fmaf(back, rise[l].x, hi[l].x), fmaf(back, rise[l].y, hi[l].y));
		}
#pragma unroll
		for (int f = 0; f < (int)LT_LEVELS - NM; ++f) {
			enc[NM + f] = fine[f];
			asm volatile("" : "+v"(enc[NM + f]));  // waited for here, in front of the next step's loads: behind them the wait would include those
		}
		if (!have_fine) {  // (a branch that is hardly ever taken, not a select a level)
#pragma unroll
			for (int f = 0; f < (int)LT_LEVELS - NM; ++f) {
				enc[NM + f] = 0u;
				asm volatile("" : "+v"(enc[NM + f]));
			}
		}
		// the next step: where it stands, and the loads it needs (the last step looks at its own position again: no loads)
		const uint32_t next = k + 1u < nz ? k + 1u : k;
		uint32_t cz;
		float wz;
		n2_locate(lattice_coord(a.lat, 2, z + next), my_scale, wz, cz);
		const uint32_t moved = cz - my_cz;
		const uint32_t one = (uint32_t)__ballot(moved == 1u) & on, far = (uint32_t)__ballot(moved > 1u) & on;  // lanes 0..15 speak for the levels
		uint32_t r0, r1, v = lane * 4u;
		asm volatile("" : "+v"(v));
		rows_of(cz + 1u, r0, r1);
		// (bits of a mask are looked up where they are needed: what the compiler takes for the same condition at two places it keeps as a mask of lanes, through a vector
		// register, two instructions a level and step)
		uint32_t raw[NM][2], hash_mask = a.hash_mask;
		asm("" : "+s"(hash_mask));
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((one >> l) & 1u) fetch(l, v, lane_u32(r0, l), lane_u32(r1, l), hash_mask, raw[l]);
		// Behind them the next step's fine features (they come from far away): the planes can then be waited for without waiting for these.
		load_fine(next, fine);
		float bias = a.sdf_bias;
		asm volatile("" : "+s"(bias));
		const hf sdf = lattice_network(F, lane, enc, at, pz, bias);
		uint32_t out_x = x * 4u;
		asm volatile("" : "+v"(out_x));
		if (inside) __builtin_nontemporal_store((float)sdf, reinterpret_cast<float*>(reinterpret_cast<char*>(out) + out_x));
		out += (uint64_t)a.lat.res[0] * a.lat.res[1];
		if (++k == nz) return;
		if (far) break;
		// the planes the next step has crossed into (the points' places come into the registers that held the vertices)
		uint32_t into = one;
		asm("" : "+s"(into));
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((into >> l) & 1u) {
				blend_y(l, raw[l]);
				const uint2 p = places[l][lane];
				raw[l][0] = p.x;
				raw[l][1] = p.y;
			}
		__builtin_amdgcn_wave_barrier();
		asm("" : "+s"(into));
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((into >> l) & 1u) {
				const float2 below = hi[l];
				blend_at(make_uint2(raw[l][0], raw[l][1]), hi[l]);
				rise[l] = make_float2(hi[l].x - below.x, hi[l].y - below.y);
			}
		my_cz = cz;
		my_back = wz - 1.f;
	}
	}
}

// The walk for lattices of a few dozen points along x, or with steps along z of more than a walked level's cell: every point gathers
// its own vertices, and a step meets any planes.  Masks, rows and features as in lattice_walk_kernel: 96 x 304 x 304 833 -> 802 us, 64^3 57.9 -> 56.8; with six levels it
// fits three waves per SIMD then, 256 x 256 x 64 277 -> 250 us, 512 x 64 x 64 113 -> 105.
constexpr uint32_t lattice_gather_waves(uint32_t levels) { return levels <= 6u ? 3u : 2u; }  // per SIMD
template <int NM>
__global__ void __launch_bounds__(LT_BLOCK, lattice_gather_waves(NM)) lattice_gather_walk_kernel(const LatticeArgs a) {
	__shared__ __align__(16) hf F[SDF_FRAG_COUNT * 512];
	for (uint32_t i = threadIdx.x; i < SDF_FRAG_COUNT * 64u; i += LT_BLOCK) *reinterpret_cast<half8*>(F + i * 8u) = *reinterpret_cast<const half8*>(a.frags + i * 8u);
	__syncthreads();
	const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (LT_BLOCK / 64) + (threadIdx.x >> 6));
	uint32_t x, y, z, nz;
	if (!lattice_run(a, wave, x, y, z, nz)) return;
	const uint32_t lane = threadIdx.x & 63u, rx = a.lat.res[0], plane = a.nx * a.ny;
	const bool inside = x < a.nx;
	const float px = lattice_coord(a.lat, 0, a.x0 + min(x, a.nx - 1u)), py = lattice_coord(a.lat, 1, y);
	const char* base[NM];
#pragma unroll
	for (int l = 0; l < NM; ++l) base[l] = reinterpret_cast<const char*>(a.table + a.offset[l]);
	// lane l: what depends on y and z of level l
	const uint32_t ll = lane & (LT_LEVELS - 1u);
	const float my_scale = a.scale[ll];
	const uint32_t my_res = a.res[ll], my_entries = a.entries[ll];
	const bool my_hashed = (a.hash_mask >> ll) & 1u;
	const uint32_t on = (1u << min(a.active_levels, (uint32_t)NM)) - 1u;  // levels in use here
	float my_wy, my_wz;
	uint32_t my_cy, my_cz;
	n2_locate(py, my_scale, my_wy, my_cy);
	n2_locate(lattice_coord(a.lat, 2, z), my_scale, my_wz, my_cz);
	float wy[NM];
#pragma unroll
	for (int l = 0; l < NM; ++l) wy[l] = lane_f32(my_wy, l);
	// the plane of vertices at `row0`, `row1` (byte offsets of its rows y, y + 1): four gathers, and their interpolation in x and y
	// What depends on x is worked out at each plane, from an opaque copy of the position: kept across the loop, cell and weight of
	// every level would come on top of the 168 registers of six levels, which are all that three waves per SIMD have, the 183 of eight and the 197 of ten.
	auto place = [&](int l, float& w, uint32_t& c) {
		float p = px;
		asm volatile("" : "+v"(p));
		n2_locate(p, a.scale[l], w, c);
	};
	auto fetch = [&](int l, uint32_t row0, uint32_t row1, uint32_t hash_mask, uint32_t (&raw)[4]) __attribute__((always_inline)) {
		const bool hashed = (hash_mask >> l) & 1u;
		const uint32_t bytes = a.entries[l] << 2;
		float w;
		uint32_t cx;
		place(l, w, cx);
		if (hashed) {
			const uint32_t x0 = x_part(true, a.entries[l], a.res[l], cx), x1 = x_part(true, a.entries[l], a.res[l], cx + 1u);
			raw[0] = *reinterpret_cast<const uint32_t*>(base[l] + (x0 ^ row0));
			raw[1] = *reinterpret_cast<const uint32_t*>(base[l] + (x1 ^ row0));
			raw[2] = *reinterpret_cast<const uint32_t*>(base[l] + (x0 ^ row1));
			raw[3] = *reinterpret_cast<const uint32_t*>(base[l] + (x1 ^ row1));
		} else {
			const uint32_t x0 = x_part(false, a.entries[l], a.res[l], cx), x1 = x_part(false, a.entries[l], a.res[l], cx + 1u);
			raw[0] = *reinterpret_cast<const uint32_t*>(base[l] + vertex(false, bytes, x0, row0));
			raw[1] = *reinterpret_cast<const uint32_t*>(base[l] + vertex(false, bytes, x1, row0));
			raw[2] = *reinterpret_cast<const uint32_t*>(base[l] + vertex(false, bytes, x0, row1));
			raw[3] = *reinterpret_cast<const uint32_t*>(base[l] + vertex(false, bytes, x1, row1));
		}
	};
	auto blend = [&](int l, const uint32_t (&raw)[4], float2& p) {
		const float2 v0 = lt_h2f(raw[0]), v1 = lt_h2f(raw[1]), v2 = lt_h2f(raw[2]), v3 = lt_h2f(raw[3]);
		float vx, vy = wy[l];
		uint32_t cx;
		place(l, vx, cx);
		asm volatile("" : "+v"(vy));
		const float uy = 1.f - vy, ux = 1.f - vx, w0 = ux * uy, w1 = vx * uy, w2 = ux * vy, w3 = vx * vy;
		// (the products too as multiply-adds: those take half-precision operands as they are)
		p.x = fmaf(w0, v0.x, fmaf(w1, v1.x, fmaf(w2, v2.x, fmaf(w3, v3.x, 0.f))));
		p.y = fmaf(w0, v0.y, fmaf(w1, v1.y, fmaf(w2, v2.y, fmaf(w3, v3.y, 0.f))));
	};
	const uint32_t my_z_factor = (my_hashed ? 805459861u : my_res * my_res) << 2, my_z_most = my_hashed ? ~0u : my_res, my_in_table = (my_entries - 1u) << 2;
	const uint32_t my_y0 = (my_hashed ? my_cy * 2654435761u : min(my_cy, my_res) * my_res) << 2, my_y1 = (my_hashed ? (my_cy + 1u) * 2654435761u : min(my_cy + 1u, my_res) * my_res) << 2;
	auto rows_of = [&](uint32_t cz, uint32_t& r0, uint32_t& r1) __attribute__((always_inline)) {
		const uint32_t z = min(cz, my_z_most) * my_z_factor;
		r0 = my_hashed ? (my_y0 ^ z) & my_in_table : my_y0 + z;
		r1 = my_hashed ? (my_y1 ^ z) & my_in_table : my_y1 + z;
	};
	float2 lo[NM], hi[NM], rise[NM];  // planes below and above, and their difference
	auto both_planes = [&](uint32_t which, uint32_t cz) {
		uint32_t r0, r1, q0, q1;
		rows_of(cz, r0, r1);
		rows_of(cz + 1u, q0, q1);
		uint32_t raw[NM][4], hash_mask = a.hash_mask;
		asm("" : "+s"(hash_mask));
		// (all levels' loads of a plane in flight together)
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((which >> l) & 1u) fetch(l, lane_u32(r0, l), lane_u32(r1, l), hash_mask, raw[l]);
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((which >> l) & 1u) blend(l, raw[l], lo[l]);
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((which >> l) & 1u) fetch(l, lane_u32(q0, l), lane_u32(q1, l), hash_mask, raw[l]);
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((which >> l) & 1u) {
				blend(l, raw[l], hi[l]);
				rise[l] = make_float2(hi[l].x - lo[l].x, hi[l].y - lo[l].y);
			}
	};
#pragma unroll
	for (int l = 0; l < NM; ++l) lo[l] = hi[l] = rise[l] = make_float2(0.f, 0.f);  // switched-off levels
	both_planes(on, my_cz);
	const size_t feat_at = (size_t)(z - a.z0) * plane + (size_t)(y - a.y0) * a.nx + min(x, a.nx - 1u);
	float* out = a.out + (size_t)(z - a.z0) * ((size_t)rx * a.lat.res[1]) + (size_t)(y - a.y0) * rx + x;
	uint32_t xc0, xc1;
	lattice_xy(px, py, lane >> 5, xc0, xc1);
	uint4v at[2] = {uint4v{xc0, 0u, 0u, 0u}, uint4v{xc1, 0u, 0u, 0u}};
	// (levels that the table does not have read the last one's row: their weights are zero)
	const uint32_t have_fine = a.n_levels > (uint32_t)NM ? ~0u : 0u;
	const uint32_t* row[LT_LEVELS - NM];
#pragma unroll
	for (uint32_t f = 0; f < LT_LEVELS - NM; ++f) row[f] = lattice_features(a, have_fine ? min(f, a.n_levels - 1u - NM) : 0u);
	uint32_t fine[LT_LEVELS - NM];
	auto load_fine = [&](uint32_t k, uint32_t (&to)[LT_LEVELS - NM]) {
#pragma unroll
		for (uint32_t f = 0; f < LT_LEVELS - NM; ++f) to[f] = __builtin_nontemporal_load(row[f] + feat_at + (size_t)k * plane);
	};
	load_fine(0, fine);
	for (uint32_t k = 0; k < nz; ++k) {
		const float pz = lattice_coord(a.lat, 2, z + k);
		// features of this step
		uint32_t enc[LT_LEVELS];
#pragma unroll
		for (int l = 0; l < NM; ++l) {
			const float vz = lane_f32(my_wz, l);
			enc[l] = lt_pack(fmaf(vz, rise[l].x, lo[l].x), fmaf(vz, rise[l].y, lo[l].y));
		}
#pragma unroll
		for (int f = 0; f < (int)LT_LEVELS - NM; ++f) {
			enc[NM + f] = fine[f];
			asm volatile("" : "+v"(enc[NM + f]));  // waited for here, in front of the next step's loads: behind them the wait would include those
		}
		if (!have_fine) {  // (as there)
#pragma unroll
			for (int f = 0; f < (int)LT_LEVELS - NM; ++f) {
				enc[NM + f] = 0u;
				asm volatile("" : "+v"(enc[NM + f]));
			}
		}
		// the next step: where it stands, and the loads it needs (the last step looks at its own position again: no loads)
		const uint32_t next = k + 1u < nz ? k + 1u : k;
		uint32_t cz;
		float wz;
		n2_locate(lattice_coord(a.lat, 2, z + next), my_scale, wz, cz);
		const uint32_t moved = cz - my_cz;
		const uint32_t one = (uint32_t)__ballot(moved == 1u) & on, far = (uint32_t)__ballot(moved > 1u) & on;  // lanes 0..15 speak for the levels
		uint32_t r0, r1;
		rows_of(cz + 1u, r0, r1);
		uint32_t raw[NM][4], hash_mask = a.hash_mask;
		asm("" : "+s"(hash_mask));
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((one >> l) & 1u) fetch(l, lane_u32(r0, l), lane_u32(r1, l), hash_mask, raw[l]);
		// Behind them the next step's fine features (they come from far away): the planes can then be waited for without waiting for these.
		load_fine(next, fine);
		const hf sdf = lattice_network(F, lane, enc, at, pz, a.sdf_bias);
		if (inside) __builtin_nontemporal_store((float)sdf, out);
		out += (size_t)rx * a.lat.res[1];
		// the planes the next step has crossed into
		uint32_t into = one;
		asm("" : "+s"(into));
#pragma unroll
		for (int l = 0; l < NM; ++l)
			if ((into >> l) & 1u) {
				lo[l] = hi[l];
				blend(l, raw[l], hi[l]);
				rise[l] = make_float2(hi[l].x - lo[l].x, hi[l].y - lo[l].y);
			}
		if (far) both_planes(far, cz);
		my_cz = cz;
		my_wz = wz;
	}
}

uint64_t n2_lattice_frag_bytes() { return SDF_FRAG_COUNT * 1024ull; }

// d_scratch holds LT_MAX_FINE 4-byte rows of `chunk` points, d_frags the fragment image.  The part of d_out behind a slab holds features too.
int n2_fused_lattice_sdf(const N2FusedNets& nets, hipStream_t s, const N2Lattice& lat, uint32_t chunk, void* d_scratch, void* d_frags, float* d_out) {
	const N2LevelTable& tab = *nets.tab;
	LatticeArgs a{};
	a.n_levels = tab.n_levels;
	a.active_levels = tab.active_levels < tab.n_levels ? tab.active_levels : tab.n_levels;
	for (uint32_t l = 0; l < LT_LEVELS; ++l) {
		const bool have = l < tab.n_levels;  // levels the table does not have count as switched off
		a.scale[l] = have ? tab.scale[l] : 1.f;
		a.res[l] = have ? tab.resolution[l] : 1u;
		a.entries[l] = have ? tab.entries[l] : 8u;
		a.offset[l] = have ? tab.offset[l] : 0u;
		if (have && tab.mode[l] == N2_LEVEL_HASH) a.hash_mask |= 1u << l;
	}
	a.table = nets.table;
	a.frags = reinterpret_cast<hf*>(d_frags);
	a.sdf_w = reinterpret_cast<const hf*>(nets.sdf_w);
	a.sdf_in_w = nets.sdf_in_w;
	a.sdf_bias = nets.sdf_bias;
	a.lat = lat;
	a.near = reinterpret_cast<uint32_t*>(d_scratch);
	const float step_z = lat.inv_res[2] * lat.extent[2], end_x = lat.corner[0] + lat.extent[0];
	const uint32_t rows = n2_lattice_row_levels(a.scale, lat.res[0], fabsf(lat.inv_res[0] * lat.extent[0]), fmaxf(fabsf(lat.corner[0]), fabsf(end_x)), step_z);
	const uint32_t walked = n2_lattice_walked_levels(a.scale, fabsf(step_z));
	const bool by_rows = n2_lattice_by_rows(rows, walked, (uint64_t)lat.res[0] * lat.res[1] * lat.res[2]);
	const uint32_t nm = by_rows ? rows : walked;
	a.first_fine = nm;
	const uint32_t n_fine = tab.n_levels > nm ? tab.n_levels - nm : 0u;
	void (*const kernels[7])(LatticeArgs) = {lattice_walk_kernel<4>, lattice_walk_kernel<5>, lattice_walk_kernel<6>, lattice_walk_kernel<7>, lattice_walk_kernel<8>, lattice_walk_kernel<9>,
	                                         lattice_walk_kernel<10>};
	auto* const walk_kernel = by_rows ? kernels[nm - 4u] : nm == 10u ? lattice_gather_walk_kernel<10> : nm == 8u ? lattice_gather_walk_kernel<8> : lattice_gather_walk_kernel<6>;
	if (n_fine == 0) {
		lattice_frags_kernel<<<dim3(FRAG_BLOCKS), dim3(LT_BLOCK), 0, s>>>(a);
		N2_LAUNCH_CHECK();
	}
	const uint32_t rx = lat.res[0], ry = lat.res[1], rz = lat.res[2];
	const uint64_t words = (uint64_t)LT_MAX_FINE * chunk, all = (uint64_t)rx * ry * rz;
	const bool large = n2_lattice_large_slabs(all, words, n_fine);
	uint64_t done = 0;
	auto launch = [&](uint32_t x0, uint32_t nx, uint32_t y0, uint32_t ny, uint32_t z0, uint32_t nz, uint32_t near_levels) -> int {
		a.x0 = x0; a.nx = nx; a.y0 = y0; a.ny = ny; a.z0 = z0; a.nz = nz;
		a.points = (uint64_t)nx * ny * nz;
		a.out = d_out + done;
		a.near_levels = near_levels;
		a.beyond = reinterpret_cast<uint32_t*>(a.out + a.points) - near_levels * a.points;
		a.x_runs = (nx + 63u) / 64u;
		const uint32_t runs = a.x_runs * ny;  // per plane
		auto blocks = [&]() { return (runs * ((nz + a.walk - 1u) / a.walk) + LT_BLOCK / 64 - 1) / (LT_BLOCK / 64); };
		if (n_fine) {
			a.walk = n2_lattice_fine_walk(runs, nz);
			auto* const fine_kernel = n2_lattice_fine_waves(runs, nz) == 5u ? lattice_fine_kernel<5> : lattice_fine_kernel<6>;
			fine_kernel<<<dim3(blocks() * n_fine + (done == 0 ? FRAG_BLOCKS : 0u)), dim3(LT_BLOCK), 0, s>>>(a, blocks());
			N2_LAUNCH_CHECK();
		}
		a.walk = n2_lattice_walk(runs, nz, by_rows ? 3u : lattice_gather_waves(nm));
		walk_kernel<<<dim3(blocks()), dim3(LT_BLOCK), 0, s>>>(a);
		N2_LAUNCH_CHECK();
		done += a.points;
		return N2_OK;
	};
	for (uint32_t z0 = 0; z0 < rz;) {
		uint32_t near_levels;
		const uint32_t left[3] = {rx, ry, rz - z0};
		N2LatticeSlab slab = n2_lattice_slab(left, n2_lattice_slab_points(all - done, words, n_fine, large, near_levels));
		if (slab.ny == ry) {
			if (!large || left[2] < 2u * slab.nz) slab.nz = n2_lattice_part(left[2], slab.nz);  // slabs alike (large ones: the last two)
			if (const int rc = launch(0, rx, 0, ry, z0, slab.nz, near_levels)) return rc;
			z0 += slab.nz;
			continue;
		}
		// a plane in parts: rows, or pieces of one, by what the scratch alone holds
		slab = n2_lattice_slab(left, words / (n_fine ? n_fine : 1u));
		for (uint32_t y0 = 0; y0 < ry; y0 += slab.ny)
			for (uint32_t x0 = 0; x0 < rx; x0 += slab.nx)
				if (const int rc = launch(x0, slab.nx < rx - x0 ? slab.nx : rx - x0, y0, slab.ny < ry - y0 ? slab.ny : ry - y0, z0, 1, n_fine ? n_fine : 1u)) return rc;
		++z0;
	}
	return N2_OK;
}
