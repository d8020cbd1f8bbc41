// Device-side index arithmetic of the multi-resolution hash grid, shared by the stand-alone grid kernels and the
// fused field kernels: cell location, level mask and the entry index of a grid vertex.
#pragma once
#include "n2_common.h"
#include "launch_rules.h"

// ----------------------------------------------------------------------------
// device helpers
// ----------------------------------------------------------------------------

// pos = x*scale + 0.5 as one fused multiply-add, then floor: the integer cell
// and the fractional weight.  The fused form is part of the bit-exact contract
// with the CPU oracle.
__device__ __forceinline__ void n2_locate(float x, float scale, float& w, uint32_t& cell) {
	const float p = __fmaf_rn(x, scale, 0.5f);
	const float f = floorf(p);
	cell = (uint32_t)(int32_t)f;
	w = p - f;
}

// Level mask of tcnn's grid encoding: the limit is (max_level * n_output_features) / n_features_per_level in fp32
// and a level is off when level >= limit + 1e-3; the progressive mask adds level >= valid_levels.
__device__ __forceinline__ bool n2_level_masked(const N2LevelTable& tab, uint32_t level, uint32_t i) {
	if (tab.max_level_gpu == nullptr) return level >= tab.active_levels;  // uniform: the host has applied both rules
	const float limit = (tab.max_level_gpu[i] * (float)(tab.n_levels * tab.n_features)) / (float)tab.n_features;
	return (float)level >= limit + 1e-3f || level >= tab.valid_levels;
}

template <uint32_t MODE>
__device__ __forceinline__ uint32_t n2_entry(uint32_t entries, uint32_t res, uint32_t gx, uint32_t gy, uint32_t gz) {
	if (MODE == N2_LEVEL_DENSE) {
		// Positions inside [0,1]^3 never give a coordinate above res; the clamp only keeps
		// stray inputs (padding rows of a batch) inside the table.  The host has checked
		// res^3 + res^2 + res < 2*entries, so one subtraction is the modulo.
		gx = min(gx, res); gy = min(gy, res); gz = min(gz, res);
		uint32_t i = gx + gy * res + gz * res * res;
		return i >= entries ? i - entries : i;
	} else if (MODE == N2_LEVEL_HASH) {
		return (gx ^ (gy * 2654435761u) ^ (gz * 805459861u)) & (entries - 1u);
	} else if (MODE == N2_LEVEL_DENSE_MOD) {
		return (gx + gy * res + gz * res * res) % entries;
	} else {
		return (gx ^ (gy * 2654435761u) ^ (gz * 805459861u)) % entries;
	}
}

// Byte offsets in the level's table of the four (y, z) corners k = y + 2 z of a cell at x corner gx: what n2_entry gives, times four.
// On power-of-two tables y and z come as the hash's terms (n2_hash_terms; a multiplication by a constant and one by four commute
// modulo 2^32), which two x corners share.
__device__ __forceinline__ void n2_hash_terms(uint32_t (&c)[3]) {
	c[1] *= 2654435761u * 4u;
	c[2] *= 805459861u * 4u;
}
template <uint32_t MODE>
__device__ __forceinline__ void n2_corner_bytes(uint32_t entries, uint32_t res, uint32_t gx, uint32_t cy, uint32_t cz, uint32_t (&at)[4]) {
	if (MODE == N2_LEVEL_HASH) {
		const uint32_t mask = (entries - 1u) << 2, x = gx << 2, z1 = cz + 805459861u * 4u, xy0 = x ^ cy, xy1 = x ^ (cy + 2654435761u * 4u);
		at[0] = (xy0 ^ cz) & mask;
		at[1] = (xy1 ^ cz) & mask;
		at[2] = (xy0 ^ z1) & mask;
		at[3] = (xy1 ^ z1) & mask;
	} else if (MODE == N2_LEVEL_DENSE) {
		const uint32_t bytes = entries << 2, row = res << 2, plane = row * res;
		const uint32_t x = min(gx, res) << 2, y0 = x + min(cy, res) * row, y1 = x + min(cy + 1u, res) * row, z0 = min(cz, res) * plane, z1 = min(cz + 1u, res) * plane;
		const uint32_t sum[4] = {y0 + z0, y1 + z0, y0 + z1, y1 + z1};
#pragma unroll
		for (uint32_t k = 0; k < 4; ++k) at[k] = min(sum[k], sum[k] - bytes);  // one conditional subtraction is the modulo (unsigned wrap-around)
	} else {
#pragma unroll
		for (uint32_t k = 0; k < 4; ++k) at[k] = n2_entry<MODE>(entries, res, gx, cy + (k & 1u), cz + (k >> 1)) << 2;
	}
}

// A dense level's entries in blocks: block (x, y, z) holds the four (y, z) corners, at x corner x and in the order of n2_corner_bytes, of the cell that
// starts at y - 1 and z - 1.  x runs up to the level's resolution, y and z one further: cells are bounded as there, and cell -1 is the first.
struct alignas(16) N2Block {
	uint32_t entry[4];
};
N2_HD inline uint32_t n2_block_count(uint32_t res) { return (res + 1u) * (res + 2u) * (res + 2u); }
__device__ __forceinline__ uint32_t n2_block_row(uint32_t res, uint32_t cy, uint32_t cz) { return (res + 1u) * (min(cy + 1u, res + 1u) + (res + 2u) * min(cz + 1u, res + 1u)); }
__device__ __forceinline__ N2Block n2_make_block(const char* __restrict__ table, uint32_t entries, uint32_t res, uint32_t k) {
	const uint32_t row = k / (res + 1u), x = k - row * (res + 1u), z = row / (res + 2u), y = row - z * (res + 2u);
	uint32_t at[4];
	n2_corner_bytes<N2_LEVEL_DENSE>(entries, res, x, y - 1u, z - 1u, at);
	N2Block b;
#pragma unroll
	for (int q = 0; q < 4; ++q) b.entry[q] = *reinterpret_cast<const uint32_t*>(table + at[q]);
	return b;
}

// value held by the other lane of the pair (lane ^ 1), and by the pair's lane M: quad permutes inside the VALU, no LDS crossbar
__device__ __forceinline__ uint32_t n2_pair_swap(uint32_t x) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, true); }
__device__ __forceinline__ float n2_pair_swap(float x) { return __uint_as_float(n2_pair_swap(__float_as_uint(x))); }
template <int M>
__device__ __forceinline__ uint32_t n2_pair_lane(uint32_t x) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, M ? 0xF5 : 0xA0, 0xF, 0xF, true); }
template <int M>
__device__ __forceinline__ float n2_pair_lane(float x) { return __uint_as_float(n2_pair_lane<M>(__float_as_uint(x))); }

// Which of a wave's 64 points lane l owns in n2_encode_level: point l / 2 + 32 (l % 2).  A pair's points are 32 apart, so that the loads for the
// pairs' first points and those for their second ones go to other lines where neighbouring points share theirs (along rays, in cells walked
// in sequence): a line asked for again before it has come costs another request.  Memory is read and written in the points' own order,
// lane l point l, and the values change lanes through the LDS crossbar, which has nothing else to do here.  Adjacent points -> this -> this with
// memory accessed in the lanes' order: encoding forward and backward of 250 000 points along rays 175 -> 164 -> 171 us, 2^18 uniform points
// 206 -> 206 -> 209, cells of the occupancy grid 466 -> 468 -> 485.
__device__ __forceinline__ uint32_t n2_lane_value(uint32_t x, uint32_t lane) { return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(lane << 2), (int)x); }
// the value of the point this lane owns, from the lane that has loaded it
__device__ __forceinline__ float n2_to_pairs(float x) {
	const uint32_t l = threadIdx.x & 63u;
	return __uint_as_float(n2_lane_value(__float_as_uint(x), (l >> 1) + ((l & 1u) << 5)));
}
// the value of point l for lane l, from the lane that owns it
__device__ __forceinline__ uint32_t n2_from_pairs(uint32_t x) {
	const uint32_t l = threadIdx.x & 63u;
	return n2_lane_value(x, ((l & 31u) << 1) + (l >> 5));
}
__device__ __forceinline__ float n2_from_pairs(float x) { return __uint_as_float(n2_from_pairs(__float_as_uint(x))); }

// The encoding of one level at the lane's own point: both features and, with WANT_J, their derivatives along the axes (times jscale).
// Two adjacent lanes share the work on their two points: for either point lane b gathers the four (y, z) corners of x corner b, whose
// other x corner stands beside it (dense levels: index + 1; hashed levels: x enters the hash with prime 1), nearly always in the same
// line of 128 bytes.  What bounds the gathers is lines: an L1 takes one in from the L2 every 2.3 clocks (measured with loads of 4, 8 and
// 16 bytes alike), and a wave's load of 64 words it has takes 40 clocks.  So a pair's load meets 32 lines and not 64, and because
// every lane keeps a point of its own, positions come in and results go out as whole lines (8 clocks a load), where two lanes to a point
// took 16 clocks for each of three coordinates.  Call in us, two lanes per point -> this: 2^21 cells of the occupancy grid 503 -> 467, 2^20
// uniform points 304 -> 297, the encoding forward and backward on 2^18 points 214 -> 211.  Two or four points per lane with their loads under
// way together are no faster, and neither are loads of the 8 or 16 bytes round a corner, which an L1 serves in less time when the lanes
// of a pair share them.  All lanes of the wave take part.
template <uint32_t MODE, bool WANT_J>
__device__ __forceinline__ void n2_encode_level(const char* __restrict__ base, uint32_t entries, uint32_t res, float scale, const float (&p)[3], float jscale,
                                                float (&feat)[2], float (&J)[2][3]) {
	const uint32_t b = threadIdx.x & 1u;
	float w[3];
	uint32_t c[3], at[2][4], raw[2][4];
#pragma unroll
	for (int d = 0; d < 3; ++d) n2_locate(p[d], scale, w[d], c[d]);
	if (MODE == N2_LEVEL_HASH) n2_hash_terms(c);
	n2_corner_bytes<MODE>(entries, res, n2_pair_lane<0>(c[0]) + b, n2_pair_lane<0>(c[1]), n2_pair_lane<0>(c[2]), at[0]);
	n2_corner_bytes<MODE>(entries, res, n2_pair_lane<1>(c[0]) + b, n2_pair_lane<1>(c[1]), n2_pair_lane<1>(c[2]), at[1]);
#pragma unroll
	for (int m = 0; m < 2; ++m)
#pragma unroll
		for (int k = 0; k < 4; ++k) raw[m][k] = *reinterpret_cast<const uint32_t*>(base + at[m][k]);
	const float wy[2] = {n2_pair_lane<0>(w[1]), n2_pair_lane<1>(w[1])}, wz[2] = {n2_pair_lane<0>(w[2]), n2_pair_lane<1>(w[2])};
	// of point m's x corner b: the bilinear value s, and its y and z differences ty, tz
	float s[2][2], ty[2][2], tz[2][2];  // [point][feature]
	// (differences as multiply-adds as well, by a one that the compiler does not see through: it would convert the halves first, an instruction
	// each.  With the shorter n2_slopes_pack 27 fewer of 265: gather of 2^18 samples along rays 64.1 -> 61.2 us, second order of 131 072
	// points 174.3 -> 169.7 for the call)
	float one = 1.f;
	asm("" : "+s"(one));
#pragma unroll
	for (int m = 0; m < 2; ++m) {
		float v[4][2];
#pragma unroll
		for (int k = 0; k < 4; ++k) {
			const float2 h = __half22float2(*reinterpret_cast<const __half2*>(&raw[m][k]));
			v[k][0] = h.x;
			v[k][1] = h.y;
		}
		const float uy = 1.f - wy[m], uz = 1.f - wz[m], w00 = uy * uz, w10 = wy[m] * uz, w01 = uy * wz[m], w11 = wy[m] * wz[m];
#pragma unroll
		for (int f = 0; f < 2; ++f) {
			// (the last product as a multiply-add too: those take half-precision operands as they are)
			s[m][f] = fmaf(w00, v[0][f], fmaf(w10, v[1][f], fmaf(w01, v[2][f], fmaf(w11, v[3][f], 0.f))));
			if (WANT_J) {
				const auto less = [&](int i, int j) { return fmaf(v[i][f], one, -v[j][f]); };
				ty[m][f] = fmaf(uz, less(1, 0), wz[m] * less(3, 2));
				tz[m][f] = fmaf(uy, less(2, 0), wy[m] * less(3, 1));
			}
		}
	}
	// of the lane's own point, x corner b is its own and the other one its partner's
	const float wx = w[0], ux = 1.f - wx;
	auto corners = [&](const float q0, const float q1, float& lo, float& hi) {
		const float from0 = n2_pair_swap(q0), from1 = n2_pair_swap(q1);
		lo = b ? from1 : q0;
		hi = b ? q1 : from0;
	};
#pragma unroll
	for (int f = 0; f < 2; ++f) {
		float lo, hi;
		corners(s[0][f], s[1][f], lo, hi);
		feat[f] = fmaf(ux, lo, wx * hi);
		if (WANT_J) {
			J[f][0] = (hi - lo) * jscale;
			corners(ty[0][f], ty[1][f], lo, hi);
			J[f][1] = fmaf(ux, lo, wx * hi) * jscale;
			corners(tz[0][f], tz[1][f], lo, hi);
			J[f][2] = fmaf(ux, lo, wx * hi) * jscale;
		}
	}
}

// ----------------------------------------------------------------------------
// Slopes of one (sample, level): the six values d feature_f / d x_d (before the level's scale factor) as one 16-byte
// block-float: 20-bit signed mantissas q_0..q_5 and a shared exponent e (value_i = q_i * 2^(e - 19), |value_i| < 2^e).
// The contraction of the slopes with a gradient then carries an error of 2^-20 of the largest slope, where fp16 storage
// (2^-11 of every slope) shows in the normals; fp32 storage takes 24 bytes.  A 12-byte form (15-bit mantissas, 6-bit
// exponent) is not enough: the second-order input J v of the SDF net cancels between the slopes' terms, and the weight
// gradients that follow from it then miss the oracle's by 7e-3 in relative L2.
//   word 0: q0 | q1 << 20     word 1: q1 >> 12 | q2 << 8 | q3 << 28     word 2: q3 >> 4 | q4 << 16
//   word 3: q4 >> 16 | q5 << 4 | e << 24
// ----------------------------------------------------------------------------
__device__ __forceinline__ uint4 n2_slopes_pack(const float (&slopes)[6]) {
	float v[6];
#pragma unroll
	for (int i = 0; i < 6; ++i) v[i] = slopes[i];
	float m = 0.f;  // no number where one of the slopes is none
#pragma unroll
	for (int i = 0; i < 6; ++i) m = __builtin_elementwise_maximum(m, fabsf(v[i]));
	// A slope that is no number counts as zero (the bounds below would make the lowest mantissa of it), an infinite one as the largest there is.
	if (__builtin_isnan(m)) {
		m = 0.f;
#pragma unroll
		for (int i = 0; i < 6; ++i) {
			v[i] = __builtin_isnan(v[i]) ? 0.f : v[i];
			m = fmaxf(m, fabsf(v[i]));
		}
	}
	int e = 0;
	(void)frexpf(m, &e);  // m = f * 2^e with f in [0.5, 1); 0 for m = 0
	e = min(max(e, -100), 100);
	// (added to 3 * 2^22 a mantissa is rounded to the nearest integer and stands in the sum's low bits: two instructions a value where ldexp, rint, the conversion and
	// two bounds were four)
	const float scale = ldexpf(1.f, 19 - e), base = 12582912.f;
	uint32_t q[6];
#pragma unroll
	for (int i = 0; i < 6; ++i)
		q[i] = __float_as_uint(__builtin_amdgcn_fmed3f(fmaf(v[i], scale, base), base - 524287.f, base + 524287.f)) & 0xFFFFFu;
	uint4 w;
	w.x = q[0] | (q[1] << 20);
	w.y = (q[1] >> 12) | (q[2] << 8) | (q[3] << 28);
	w.z = (q[3] >> 4) | (q[4] << 16);
	w.w = (q[4] >> 16) | (q[5] << 4) | ((uint32_t)e << 24);
	return w;
}

// mantissas as floats and the factor 2^(e - 19) they share
__device__ __forceinline__ float n2_slopes_unpack(const uint4 w, float (&q)[6]) {
	auto sext20 = [](uint32_t x) { return (float)((int32_t)(x << 12) >> 12); };
	q[0] = sext20(w.x);
	q[1] = sext20((w.x >> 20) | (w.y << 12));
	q[2] = sext20(w.y >> 8);
	q[3] = sext20((w.y >> 28) | (w.z << 4));
	q[4] = sext20((w.z >> 16) | (w.w << 16));
	q[5] = sext20(w.w >> 4);
	return ldexpf(1.f, ((int32_t)w.w >> 24) - 19);
}
