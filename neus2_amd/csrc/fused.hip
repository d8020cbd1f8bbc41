// Fused forward of the NeuS field for gfx950 (counterpart of NerfNetwork::forward_impl, nerf_network.h:132-315, and of
// NerfNetwork::sdf / density, :643-726).
//
// Training forward = two kernels.
//  * field_gather_kernel walks the grid level by level (one workgroup = one level x 256 samples; every XCD takes whole
//    levels, or all take the same one at a time: launch_gather), so that the tables being read (2 MiB at most each) stay
//    resident in the L2s; a sample-major walk touches all 24 MiB of tables at once and three of five L2 requests miss.  It
//    writes the features into the SDF net's input rows and the level's slopes (the Jacobian of the encoding without the
//    level's scale factor) as a 16-byte block-float per sample and level (n2_slopes_pack), against 24 bytes of fp32.
//  * field_fused_forward_kernel then takes 32 samples per wave through everything else without touching memory in
//    between: SDF net forward, the gradient of its first output w.r.t. its input, the normal (that gradient contracted
//    with the slopes), the direction encoding, the colour net and the 16 output rows.
// Inference (sdf / density) of points in no order is a gather of features alone and the second kernel without its second half,
// or one launch for a few thousand points; positions that arrive in lattice or near-lattice order hit cached lines whatever
// the order of the levels, and take the second kernel alone with the gather inside it.
//
// Layout of the network kernel.  Lane (n, g), n = lane % 32, g = lane / 32, works for sample b0 + n.  In the MFMA
// layouts (see mlp_device.h) lane (n, g)
// holds, of a B operand in chained order, the rows {16c + 4g + 0..3, 16c + 8 + 4g + 0..3} of chunk c, and of a D tile
// the rows {8q + 4g + 0..3}, q = 0..3.  With the encoding's features as rows 0..31 of the SDF net's input (row
// 2 l + f for feature f of level l; the three centred coordinates follow as rows 32..34) both sets are the levels
//     l(j, g) = 4 (j / 2) + 2 g + j % 2,   j = 0..7,
// so a lane loads (or gathers) exactly those eight levels of its sample: the features are its B operand registers,
// the rows of d sdf / d encoding come back to it in the D tile of the input-gradient product, and the contraction
// with the slopes it holds (normal = J^T g) is lane-local up to one exchange between the two halves of the wave.  The permutation of the input rows is folded into the weight fragments, which are built once per
// workgroup in LDS.
#include "n2_common.h"

#include "grid_device.h"
#include "mlp_device.h"
#include "sdf_frags.h"

constexpr int FF_BLOCK = 256;  // 4 waves
constexpr uint32_t FF_LEVELS = 16;  // levels the lane layout covers

// fragment numbers (64 lanes x 16 bytes each)
enum : int {
	S_W0 = SDF_FRAG_W0,  // the SDF net's forward (sdf_frags.h)
	S_WO = SDF_FRAG_WO,
	FF_SDF_COUNT = SDF_FRAG_COUNT,
	S_W0T = 10,  // [mt][c]  SDF net W_0^T, row = internal input row 32 mt + n, chained K over the neurons
	S_DH = 18,   // [c]      row 0 of W_out as a chained B operand (every column the same): d sdf / d hidden before the mask
	C_W0 = 22,   // [mt][c]  colour net W_0 rows 32 mt + n; c = 0 chained (SDF-net outputs), c = 1, 2 natural
	C_WH = 28,   // [mt][c]  colour net hidden matrix, chained K
	C_WO = 36,   // [c]      colour net W_out rows n < 16, chained K
	FF_COUNT = 40
};

// per-level constants as the kernel reads them: one 16-byte LDS entry per level
struct FusedLevels {
	float scale[FF_LEVELS];
	uint32_t res[FF_LEVELS], entries[FF_LEVELS], offset[FF_LEVELS];  // offset in entries
	uint32_t hash_mask;      // bit l: level l is hashed (power-of-two table), else dense
	uint32_t active_levels;  // levels >= this are switched off (or do not exist)
};

constexpr uint32_t FS_LEVELS = 2, FB_LEVELS = 3;  // the coarsest levels of a large query (field_staged_forward_kernel): from LDS, and from blocks
struct FusedArgs {
	FusedLevels lv;
	const __half2* table;   // grid parameters
	const hf* sdf_w;        // SDF net weights: W_0 [64][sdf_in_w], W_out [16][64]
	const hf* rgb_w;        // colour net weights: W_0 [64][48], W_1 [64][64], W_out [16][64]
	const hf* variance;
	uint32_t sdf_in_w, enc_w;
	float sdf_bias;
	uint32_t N;
	const uint32_t* live;   // or null: only samples below min(*live, N) are evaluated (N stays the column count of the matrices)
	// A listed pass (full field only; list null: off) evaluates the samples begin .. begin + counts[round] of the
	// coordinates, begin = counts[0] + ... + counts[round - 1]: sample c writes row list[c] of the output, and everything
	// the backward reads is stored at column c.
	const uint32_t* list;
	const uint32_t* counts;
	uint32_t round, n_levels;
	// full field: the weight fragments of the network kernel as one image in global memory (FF_COUNT KiB; null: every
	// workgroup builds them from the weights).  The gather launch in front of the network kernel writes it.
	hf* frags;
	const float* pos;       // coordinate d of sample i at pos[i * ps + d * ds]
	uint32_t ps, ds;
	const float* coords;    // full field: [N][7] NerfCoordinate (direction at 4..6)
	// full field: what the backward pass reads, and the output
	hf* sdf_in;             // [sdf_in_w][N]  rows 0..2 centred coordinates, 3.. features
	float* xyz_rows;        // [3][N]
	uint4* slopes;          // [n_levels][N]: d feature / d position of each level (2 x 3 values, see n2_slopes_pack), without the level's scale
	hf* dsdf_din;           // [sdf_in_w][N]
	hf* rgb_in;             // [N][N2_RGB_IN_PITCH]: sample-major
	hf* output;             // [N][16]
	// SDF only
	hf* sdf_out;            // [16][N] or null
	float* row0;            // [row0_n] fp32 copy of row 0 of the first row0_n samples, or null
	uint32_t row0_n;
	int density;            // row 0 becomes the logistic density
	uint32_t first_level;   // levels that a query's gather leaves to its network kernel
	N2Block* blocks;        // [n_blocks] of the levels FS_LEVELS .. first_level - 1, each from a multiple of 256 on; written by the gather's launch
	uint32_t n_blocks, block_first[FB_LEVELS];
};

// lane l's 16 bytes of fragment f
__device__ __forceinline__ half8 fused_frag_value(const FusedArgs& a, int f, int l) {
	const hf* W0s = a.sdf_w;
	const int ld_s = (int)a.sdf_in_w;
	const hf* W1s = W0s + MLP_WIDTH * ld_s;
	const hf* W0c = a.rgb_w;
	const hf* Whc = W0c + MLP_WIDTH * 48;
	const hf* Woc = Whc + MLP_WIDTH * MLP_WIDTH;
	{
		const int n = l & 31, g = l >> 5;
		half8 v = zero8();
		if (f < S_W0T) {
			v = sdf_forward_frag(W0s, ld_s, a.enc_w, f, l);
		} else if (f < S_DH) {
			const int q = f - S_W0T, mt = q >> 2, c = q & 3, col = sdf_col(32 * mt + n, a.enc_w);
#pragma unroll
			for (int e = 0; e < 8; ++e) v[e] = h_or_zero(W0s, col >= 0, (size_t)chained_k(c, g, e) * ld_s + (col >= 0 ? col : 0));
		} else if (f < C_W0) {
#pragma unroll
			for (int e = 0; e < 8; ++e) v[e] = W1s[chained_k(f - S_DH, g, e)];
		} else if (f < C_WH) {
			const int q = f - C_W0, mt = q / 3, c = q % 3;
			v = c == 0 ? wfrag_chained(W0c, 48, 32 * mt + n, 0, g) : wfrag_natural(W0c, 48, 32 * mt + n, c, g);
		} else if (f < C_WO) {
			const int q = f - C_WH;
			v = wfrag_chained(Whc, MLP_WIDTH, 32 * (q >> 2) + n, q & 3, g);
		} else {
			if (n < MLP_OUT) v = wfrag_chained(Woc, MLP_WIDTH, n, f - C_WO, g);
		}
		return v;
	}
}

__device__ __forceinline__ void build_fused_frags(hf* F, const FusedArgs& a, int count) {
	for (int idx = threadIdx.x; idx < count * 64; idx += FF_BLOCK) *reinterpret_cast<half8*>(F + (size_t)idx * 8) = fused_frag_value(a, idx >> 6, idx & 63);
	__syncthreads();
}
// Workgroups FRAG_BLOCKS .. of a gather launch (behind those that gather) write the image: the network kernel's fragments,
// then those of the backward's weight-gradient kernels (colour net: FragMap<3, 2>; SDF net with 48 inputs: FragMap<3, 1>).
constexpr uint32_t BWD_RGB_FRAGS = FragMap<3, 2>::SEL, BWD_SDF_FRAGS = FragMap<3, 1>::SEL;
static_assert(FF_COUNT * 1024 == N2_FUSED_FRAG_FORWARD && BWD_RGB_FRAGS * 1024 == N2_FUSED_FRAG_RGB && BWD_SDF_FRAGS * 1024 == N2_FUSED_FRAG_SDF,
              "the image's parts as n2_common.h sizes them");
constexpr uint32_t FG_BLOCK = 256;  // threads of a gather workgroup (128: the gather 1.8 us shorter, the step 5 us longer; 512: +2 / +5; 1024: +11 / +11)
constexpr uint32_t FRAG_BLOCKS = ((FF_COUNT + BWD_RGB_FRAGS + BWD_SDF_FRAGS) * 64 + FG_BLOCK - 1) / FG_BLOCK;
__device__ __forceinline__ void write_frag_image(const FusedArgs& a, uint32_t block) {
	const uint32_t idx = block * FG_BLOCK + threadIdx.x;
	half8* at = reinterpret_cast<half8*>(a.frags) + idx;
	if (idx < (uint32_t)FF_COUNT * 64u) {
		*at = fused_frag_value(a, (int)(idx >> 6), (int)(idx & 63u));
	} else if (idx < (FF_COUNT + BWD_RGB_FRAGS) * 64u) {
		const uint32_t i = idx - FF_COUNT * 64u;
		*at = mlp_frag_value<3, 2>(a.rgb_w, (int)(i >> 6), (int)(i & 63u));
	} else if (idx < (FF_COUNT + BWD_RGB_FRAGS + BWD_SDF_FRAGS) * 64u && a.sdf_in_w == 48u) {
		const uint32_t i = idx - (FF_COUNT + BWD_RGB_FRAGS) * 64u;
		*at = mlp_frag_value<3, 1>(a.sdf_w, (int)(i >> 6), (int)(i & 63u));
	}
}

// ----------------------------------------------------------------------------
// gather of one (sample, level) item
// ----------------------------------------------------------------------------
struct LaneLevel {
	float scale;
	uint32_t res, entries, offset;  // offset in entries
	bool hashed;
};

// byte offsets of the 8 corner entries in the table (corner k: +1 on dimension d iff bit d of k is set)
template <int KIND>  // 0: every lane dense, 1: every lane hashed, 2: mixed
__device__ __forceinline__ void corner_offsets(const LaneLevel& L, const uint32_t (&c)[3], uint32_t (&boff)[8]) {
	uint32_t hx[2], hyz[4], dx[2], dyz[4];
	if (KIND != 0) {
		const uint32_t mask = L.entries - 1u;
		const uint32_t y0 = c[1] * 2654435761u, y1 = y0 + 2654435761u, z0 = c[2] * 805459861u, z1 = z0 + 805459861u;
		hyz[0] = (y0 ^ z0) & mask; hyz[1] = (y1 ^ z0) & mask; hyz[2] = (y0 ^ z1) & mask; hyz[3] = (y1 ^ z1) & mask;
		hx[0] = c[0] & mask; hx[1] = (c[0] + 1u) & mask;
	}
	if (KIND != 1) {
		const uint32_t r = L.res;
		dx[0] = min(c[0], r); dx[1] = min(c[0] + 1u, r);
		const uint32_t y0 = min(c[1], r) * r, y1 = min(c[1] + 1u, r) * r, z0 = min(c[2], r) * r * r, z1 = min(c[2] + 1u, r) * r * r;
		dyz[0] = y0 + z0; dyz[1] = y1 + z0; dyz[2] = y0 + z1; dyz[3] = y1 + z1;
	}
#pragma unroll
	for (int k = 0; k < 8; ++k) {
		uint32_t ih = 0, id = 0;
		if (KIND != 0) ih = hx[k & 1] ^ hyz[k >> 1];
		if (KIND != 1) {
			id = dx[k & 1] + dyz[k >> 1];
			id = min(id, id - L.entries);  // one conditional subtraction stands in for the modulo (unsigned wrap-around)
		}
		const uint32_t i = KIND == 0 ? id : KIND == 1 ? ih : (L.hashed ? ih : id);
		boff[k] = (L.offset + i) << 2;
	}
}

struct Item {
	uint32_t raw[8];
	float w[3];
	float scale;  // 0 for a switched-off level
};

// J: the lane's step; its level is l = 4 (J / 2) + 2 g + J % 2.  LV: the level constants in LDS.
template <int J>
__device__ __forceinline__ void item_fetch(const uint4* LV, uint32_t hash_mask, uint32_t active, const __half2* __restrict__ table, int g,
                                           const float (&p)[3], Item& it) {
	constexpr int lo = 4 * (J >> 1) + (J & 1), hi = lo + 2;
	const uint4 q = LV[lo + 2 * g];
	LaneLevel L;
	L.scale = __uint_as_float(q.x); L.res = q.y; L.entries = q.z; L.offset = q.w;
	L.hashed = g ? ((hash_mask >> hi) & 1u) : ((hash_mask >> lo) & 1u);
	const bool off = (uint32_t)(lo + 2 * g) >= active;
	uint32_t c[3], boff[8];
#pragma unroll
	for (int d = 0; d < 3; ++d) n2_locate(p[d], L.scale, it.w[d], c[d]);
	it.scale = off ? 0.f : L.scale;
	const bool h_lo = (hash_mask >> lo) & 1u, h_hi = (hash_mask >> hi) & 1u;  // wave-uniform
	if (h_lo && h_hi) corner_offsets<1>(L, c, boff);
	else if (!h_lo && !h_hi) corner_offsets<0>(L, c, boff);
	else corner_offsets<2>(L, c, boff);
	const char* base = reinterpret_cast<const char*>(table);
#pragma unroll
	for (int k = 0; k < 8; ++k) {
		if (off) boff[k] = 0;  // a switched-off level reads entry 0 and ignores it
		it.raw[k] = *reinterpret_cast<const uint32_t*>(base + boff[k]);
	}
}

__device__ __forceinline__ float2 h2f(uint32_t raw) {
	const half2v h = __builtin_bit_cast(half2v, raw);
	return make_float2((float)h[0], (float)h[1]);
}

// trilinear value and (with WANT_J) Jacobian of both features of one level
__device__ __forceinline__ void item_finish(const Item& it, float (&feat)[2]) {
	float2 v[8];
#pragma unroll
	for (int k = 0; k < 8; ++k) v[k] = h2f(it.raw[k]);
	const float wx = it.w[0], wy = it.w[1], wz = it.w[2], ux = 1.f - wx, uy = 1.f - wy, uz = 1.f - wz;
	const float w00 = uy * uz, w10 = wy * uz, w01 = uy * wz, w11 = wy * wz;
	float s[2][2];  // [x plane][feature]
#pragma unroll
	for (int b = 0; b < 2; ++b) {
		const float2 a0 = v[b], a1 = v[b + 2], a2 = v[b + 4], a3 = v[b + 6];
		s[b][0] = fmaf(w00, a0.x, fmaf(w10, a1.x, fmaf(w01, a2.x, w11 * a3.x)));
		s[b][1] = fmaf(w00, a0.y, fmaf(w10, a1.y, fmaf(w01, a2.y, w11 * a3.y)));
	}
	const float on = it.scale != 0.f ? 1.f : 0.f;
#pragma unroll
	for (int f = 0; f < 2; ++f) feat[f] = fmaf(ux, s[0][f], wx * s[1][f]) * on;
}

// degree-4 real spherical harmonics of the direction 2 d - 1 (tcnn's SphericalHarmonics encoding, nerf_network.h:251-257)
__device__ __forceinline__ void sh4(float x, float y, float z, float* o) {
	const float xy = x * y, xz = x * z, yz = y * z, x2 = x * x, y2 = y * y, z2 = z * z;
	o[0] = 0.28209479177387814f;
	o[1] = -0.48860251190291987f * y;
	o[2] = 0.48860251190291987f * z;
	o[3] = -0.48860251190291987f * x;
	o[4] = 1.0925484305920792f * xy;
	o[5] = -1.0925484305920792f * yz;
	o[6] = 0.94617469575755997f * z2 - 0.31539156525251999f;
	o[7] = -1.0925484305920792f * xz;
	o[8] = 0.54627421529603959f * x2 - 0.54627421529603959f * y2;
	o[9] = 0.59004358992664352f * y * (-3.0f * x2 + y2);
	o[10] = 2.8906114426405538f * xy * z;
	o[11] = 0.45704579946446572f * y * (1.0f - 5.0f * z2);
	o[12] = 0.3731763325901154f * z * (5.0f * z2 - 3.0f);
	o[13] = 0.45704579946446572f * x * (1.0f - 5.0f * z2);
	o[14] = 1.4453057213202769f * z * (x2 - y2);
	o[15] = 0.59004358992664352f * x * (-x2 + 3.0f * y2);
}

// ----------------------------------------------------------------------------
// level-major gather: features into the SDF net's input rows, slopes as fp16
// ----------------------------------------------------------------------------

// Full field: one (sample, level) item, features and slopes; the item is column i of the matrices, and its
// coordinates are row i of the input (the [N][7] coordinates, or three rows of positions).  (2^18 samples of a training step: one lane per sample
// with eight gathers 66.0 us, lane pairs with samples 32 apart 63.8, with adjacent samples slower than either; a trained state's step 509.5 -> 504.2.)
__device__ __forceinline__ void gather_item(const FusedArgs& a, uint32_t level, uint32_t i, uint32_t end) {
	const uint32_t N = a.N, at = min(i, end - 1u);  // (lanes behind the last sample take part in its pair's exchange)
	// (full field: the positions from the coordinate rows, or from three rows of their own when the caller has them: a wave
	// then reads two lines per coordinate instead of fourteen)
	const bool rows = a.pos == nullptr;
	const float* q = rows ? a.coords + (size_t)at * 7 : a.pos + (size_t)at * a.ps;
	const size_t qs = rows ? 1 : a.ds;
	const float p[3] = {q[0], q[qs], q[2 * qs]};
	if (level == 0 && i < end) {
#pragma unroll
		for (int d = 0; d < 3; ++d) {
			a.sdf_in[(size_t)d * N + i] = (hf)p[d] - (hf)0.5f;
			a.xyz_rows[(size_t)d * N + i] = p[d];
		}
	}
	uint32_t both = 0u;
	uint4 slopes = make_uint4(0u, 0u, 0u, 0u);
	if (level < a.lv.active_levels) {  // a switched-off level: zero features, zero slopes
		float feat[2], J[2][3];
		const float own[3] = {n2_to_pairs(p[0]), n2_to_pairs(p[1]), n2_to_pairs(p[2])};
		const uint32_t entries = a.lv.entries[level], res = a.lv.res[level];
		const char* base = reinterpret_cast<const char*>(a.table + a.lv.offset[level]);
		// (slopes are stored without the level's scale factor)
		if ((a.lv.hash_mask >> level) & 1u) n2_encode_level<N2_LEVEL_HASH, true>(base, entries, res, a.lv.scale[level], own, 1.f, feat, J);
		else n2_encode_level<N2_LEVEL_DENSE, true>(base, entries, res, a.lv.scale[level], own, 1.f, feat, J);
		const half2v packed = {(hf)feat[0], (hf)feat[1]};
		both = n2_from_pairs(__builtin_bit_cast(uint32_t, packed));
		const float six[6] = {J[0][0], J[0][1], J[0][2], J[1][0], J[1][1], J[1][2]};
		const uint4 w = n2_slopes_pack(six);
		slopes = make_uint4(n2_from_pairs(w.x), n2_from_pairs(w.y), n2_from_pairs(w.z), n2_from_pairs(w.w));
	}
	if (i >= end) return;
	const half2v feat = __builtin_bit_cast(half2v, both);
	a.sdf_in[(size_t)(3 + 2 * level) * N + i] = feat[0];
	a.sdf_in[(size_t)(4 + 2 * level) * N + i] = feat[1];
	a.slopes[(size_t)level * N + i] = slopes;
}

// Small queries: one (sample, level) item by a PAIR of adjacent lanes.  Lane b gathers the four (y, z) corners of x corner b, and
// finishes feature b.
struct PairItem {
	uint32_t raw[4];
	float w[3];
};
// a level of the wave's own, all of it in scalar registers
struct WaveLevel {
	float scale;
	uint32_t res, entries, offset;
	bool hashed;
};
__device__ __forceinline__ void pair_fetch(const __half2* __restrict__ table, const WaveLevel& L, const float (&p)[3], uint32_t b, PairItem& it) {
	uint32_t c[3], at[4];
#pragma unroll
	for (int d = 0; d < 3; ++d) n2_locate(p[d], L.scale, it.w[d], c[d]);
	if (L.hashed) {  // (the same for the wave)
		n2_hash_terms(c);
		n2_corner_bytes<N2_LEVEL_HASH>(L.entries, L.res, c[0] + b, c[1], c[2], at);
	} else {
		n2_corner_bytes<N2_LEVEL_DENSE>(L.entries, L.res, c[0] + b, c[1], c[2], at);
	}
	const char* base = reinterpret_cast<const char*>(table + L.offset);
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k) it.raw[k] = *reinterpret_cast<const uint32_t*>(base + at[k]);
}
__device__ __forceinline__ float pair_finish(const PairItem& it, uint32_t b) {
	float2 v[4];
#pragma unroll
	for (int k = 0; k < 4; ++k) v[k] = h2f(it.raw[k]);
	const float wy = it.w[1], wz = it.w[2], uy = 1.f - wy, uz = 1.f - wz;
	const float w00 = uy * uz, w10 = wy * uz, w01 = uy * wz, w11 = wy * wz;
	// (the first products as multiply-adds too: those take half-precision operands as they are)
	const float s0 = fmaf(w00, v[0].x, fmaf(w10, v[1].x, fmaf(w01, v[2].x, fmaf(w11, v[3].x, 0.f))));
	const float s1 = fmaf(w00, v[0].y, fmaf(w10, v[1].y, fmaf(w01, v[2].y, fmaf(w11, v[3].y, 0.f))));
	// lane b keeps feature b of its own x plane and receives feature b of the partner's
	const float mine = b ? s1 : s0, other = n2_pair_swap(b ? s0 : s1);
	float feat = fmaf(1.f - it.w[0], b ? other : mine, it.w[0] * (b ? mine : other));
	asm volatile("" : "+v"(feat));  // rounded to fp32 before fp16, as in the gather kernels: one instruction could do both and round once
	return feat;
}
// Inference on points in no particular order: between gather and network a level's features stand side by side, a row of N words to each level.  (In the training forward's
// rows of halves, which they were, the network's loads and the gather's stores took the address units twice: queries of 2^20 uniform points 259 -> 254 us, 2^21 494 -> 484.)
__device__ __forceinline__ uint32_t* query_rows(const FusedArgs& a) { return reinterpret_cast<uint32_t*>(a.sdf_in); }
// The features of one (point, level) item per lane
__device__ __forceinline__ void gather_features(const FusedArgs& a, uint32_t level, uint32_t i, uint32_t n_live) {
	uint32_t both = 0u;
	if (level < a.lv.active_levels) {  // a switched-off level: zero features
		float feat[2], unused[2][3];
		// (lanes behind the last point take part in its pair's exchange)
		const float* q = a.pos + (size_t)min(i, n_live - 1u) * a.ps;
		const float p[3] = {n2_to_pairs(q[0]), n2_to_pairs(q[a.ds]), n2_to_pairs(q[2 * (size_t)a.ds])};
		const uint32_t entries = a.lv.entries[level], res = a.lv.res[level];
		const char* base = reinterpret_cast<const char*>(a.table + a.lv.offset[level]);
		if ((a.lv.hash_mask >> level) & 1u) n2_encode_level<N2_LEVEL_HASH, false>(base, entries, res, a.lv.scale[level], p, 1.f, feat, unused);
		else n2_encode_level<N2_LEVEL_DENSE, false>(base, entries, res, a.lv.scale[level], p, 1.f, feat, unused);
		const half2v packed = {(hf)feat[0], (hf)feat[1]};
		both = n2_from_pairs(__builtin_bit_cast(uint32_t, packed));
	}
	if (i < n_live) query_rows(a)[(size_t)level * a.N + i] = both;
}

// first column and number of samples of a listed pass
__device__ __forceinline__ void listed_range(const FusedArgs& a, uint32_t& begin, uint32_t& count) {
	uint32_t listed[N2_CHUNK_MAX_ROUNDS];
#pragma unroll
	for (uint32_t q = 0; q < N2_CHUNK_MAX_ROUNDS; ++q) listed[q] = a.counts[min(q, a.round)];  // (all of them under way together)
	begin = count = 0;
#pragma unroll
	for (uint32_t q = 0; q < N2_CHUNK_MAX_ROUNDS; ++q) {
		begin += q < a.round ? listed[q] : 0u;
		count = q == a.round ? listed[q] : count;
	}
	count = min(count, a.N - min(begin, a.N));
}

// The listed pass: the number of samples is known on the device only.  The launch has est_tiles workgroups per level, levels dealt
// to the XCDs (figures at n2_gather_grid); workgroup t of a
// level takes the tiles t, t + est_tiles, ...: any estimate gives the right result, a good one gives every workgroup one
// tile.  (A fixed number of workgroups that walk all items by a stride is 1.6 times slower beside the trainer's sample
// generator: its waves keep some of them from starting until others have finished their whole share.)
__global__ void __launch_bounds__(FG_BLOCK) field_gather_list_kernel(const FusedArgs a, uint32_t est_tiles) {
	__builtin_amdgcn_s_setprio(3);
	const uint32_t gather_blocks = n2_xcd_blocks(a.n_levels, est_tiles);
	if (blockIdx.x >= gather_blocks) {  // the network kernel's weight fragments (round 0 only)
		write_frag_image(a, blockIdx.x - gather_blocks);
		return;
	}
	uint32_t level, first_tile;
	if (!n2_xcd_level_tile(blockIdx.x, a.n_levels, est_tiles, level, first_tile)) return;
	uint32_t begin, count;
	listed_range(a, begin, count);
	const uint32_t tiles = (count + FG_BLOCK - 1) / FG_BLOCK;
	for (uint32_t tile = first_tile; tile < tiles; tile += est_tiles) {
		const uint32_t j = tile * FG_BLOCK + threadIdx.x;
		if (j - (threadIdx.x & 63u) < count) gather_item(a, level, begin + j, begin + count);  // (whole waves)
	}
}

template <bool FULL>
__global__ void __launch_bounds__(FG_BLOCK) field_gather_kernel(const FusedArgs a, uint32_t tiles, int by_xcd) {
	// Bound by the L1s (n2_encode_level): a query of 2^20 uniform points takes a line in from the L2 in every 2.7 clocks of a CU, four per
	// point on every level above the coarsest, with the address units busy in 93 % of the clocks; points in the order of the occupancy grid's
	// cells share lines on the coarse levels (35 a point, one every 3.2 clocks) and look one up in every clock.  The samples of a
	// training step share lines along their rays (one every 5.2, a lookup every 1.65, address units busy in 66 %) but also hold the vector unit
	// in 54 % of the cycles for their slopes: without its gathers the launch would still take 46 of 66 us.  Measured on the training
	// step and dropped: loads of the hashed levels that bypass the L1 (agent- or system-scope: +27 us, the x neighbour's line is then
	// requested twice and a request is no cheaper) or carry the non-temporal hint (no change), the positions read as consecutive words
	// and picked apart in LDS (+9).
	// Staging the coarse levels in LDS has nothing to win: with all caches cold, levels 0..2 together add 2 us to the launch
	// and the five dense levels 4 us, against 5 to 6 us for each of the fine hashed levels and 19 us for reading the
	// positions and writing 320 bytes of features and slopes per sample.
	// The trainer's sample generator runs beside this kernel on a second stream: where a wave of each is ready on a SIMD, this
	// one issues first (the generator has the rest of the step to finish; measured 4 us on the forward, 2 us on the step).
	__builtin_amdgcn_s_setprio(3);
	const uint32_t gather_blocks = by_xcd ? n2_xcd_blocks(a.n_levels, tiles) : a.n_levels * tiles;
	if (FULL && blockIdx.x >= gather_blocks) {  // the workgroups behind those that gather: the network kernel's weight fragments
		write_frag_image(a, blockIdx.x - gather_blocks);
		return;
	}
	uint32_t level, tile;
	if (!FULL && a.n_blocks > 0 && (by_xcd ? blockIdx.x >= gather_blocks : blockIdx.y >= a.n_levels)) {  // the workgroups behind those that gather: the coarse levels' blocks
		const uint32_t k = (by_xcd ? blockIdx.x - gather_blocks : (blockIdx.y - a.n_levels) * gridDim.x + blockIdx.x) * FG_BLOCK + threadIdx.x;
		if (k >= a.n_blocks) return;
		uint32_t q = 0;
#pragma unroll
		for (uint32_t l = 1; l < FB_LEVELS; ++l) q += k >= a.block_first[l] ? 1u : 0u;
		const uint32_t in = k - a.block_first[q], res = a.lv.res[FS_LEVELS + q];
		if (in < n2_block_count(res)) a.blocks[k] = n2_make_block(reinterpret_cast<const char*>(a.table + a.lv.offset[FS_LEVELS + q]), a.lv.entries[FS_LEVELS + q], res, in);
		return;
	}
	// (the full field's workgroups are counted along x alone)
	const uint32_t y = FULL && !by_xcd ? blockIdx.x / tiles : blockIdx.y, x = FULL ? blockIdx.x - y * tiles : blockIdx.x;
	if (!n2_gather_item(x, y, by_xcd ? 1u : a.n_levels, a.n_levels, tiles, level, tile)) return;
	if (!FULL) level += a.first_level;
	const uint32_t n_live = a.live ? min(*a.live, a.N) : a.N;
	const uint32_t i = tile * FG_BLOCK + threadIdx.x;
	if (FULL) {
		if (i - (threadIdx.x & 63u) < n_live) gather_item(a, level, i, n_live);  // (whole waves)
	} else {
		if (tile * FG_BLOCK >= n_live) return;
		gather_features(a, level, i, n_live);
	}
}

// ----------------------------------------------------------------------------
// the SDF net of 32 samples by one wave: lane (n, g) works for sample n
// ----------------------------------------------------------------------------
// h: the hidden layer; the result holds rows 4g .. 4g+3 and 8+4g .. 8+4g+3
__device__ __forceinline__ half8 sdf_net(const hf* F, int lane, const half8 (&xs)[3], half8 (&h)[4]) {
#pragma unroll
	for (int mt = 0; mt < 2; ++mt) {
		float16v acc = zero16();
#pragma unroll
		for (int c = 0; c < 3; ++c) acc = N2_MFMA(frag(F, S_W0 + mt * 3 + c, lane), xs[c], acc);
		relu_pack(acc, h[2 * mt], h[2 * mt + 1]);
	}
	float16v out = zero16();
#pragma unroll
	for (int c = 0; c < 4; ++c) out = N2_MFMA(frag(F, S_WO + c, lane), h[c], out);
	return round8(out, 0);
}

// inference: bias, density and what the caller wants stored of sample `col` (col_raw: its number before clamping)
template <bool STREAM = false, class Args>
__device__ __forceinline__ void store_sdf(const Args& a, half8 y, uint32_t col, bool valid, uint32_t col_raw, int g) {
	if (g == 0) {
		hf s = y[0] + (hf)a.sdf_bias;
		if (a.density) {
			const hf is = (hf)__expf((float)(a.variance[0] * (hf)10.0f));
			const hf x = s * is;
			const hf sig = (hf)(1.0f / (1.0f + __expf(-(float)x)));
			s = is * sig * ((hf)1.0f - sig);
		}
		y[0] = s;
		if (a.row0 && col_raw < a.row0_n) a.row0[col] = (float)s;
	}
	if (a.sdf_out && valid) {
		const size_t off4 = (size_t)4u * g * a.N + col;
#pragma unroll
		for (int e = 0; e < 4; ++e) {
			hf *const lo = a.sdf_out + (size_t)e * a.N + off4, *const hi = a.sdf_out + (size_t)(8 + e) * a.N + off4;
			if (STREAM) {
				__builtin_nontemporal_store(y[e], lo);
				__builtin_nontemporal_store(y[4 + e], hi);
			} else {
				*lo = y[e];
				*hi = y[4 + e];
			}
		}
	}
}

// A small query in one launch: a workgroup takes 32 points, wave w gathers levels w and w + 8 (a lane pair per point, as in
// PairItem), the features meet in LDS and wave 0 puts them through the net.  Latency bounds it, and the lines that the weights' loads
// ask the L1 for: the arguments, then the positions and the weights together, then the gathers of both levels, are a trip each.
// The weights come four elements a load: with one element a load every lane asked for a line of its own, eight times.  (1000 points, in us: one
// element a load and branches round those of zero elements 6.6, without the branches 7.1, so 5.6; arguments where they are used 5.8.  The launch
// alone takes 1.6, without the gathers 5.4 of the 7.1.  The call takes 7.4 and so does one of 8 points: the host's part.)
constexpr uint32_t FQ_BLOCK = 512, FQ_POINTS = 32;
constexpr uint32_t FQ_PITCH = 36;  // halves per point in LDS: an odd multiple of 8 bytes, so that the net's 8-byte reads spread over the banks
__global__ void __launch_bounds__(FQ_BLOCK) field_query_kernel(const FusedArgs a) {
	static_assert(FF_LEVELS == 2 * (FQ_BLOCK / 64), "two levels per wave");
	__shared__ __align__(16) hf F[FF_SDF_COUNT * 512];
	__shared__ __align__(16) hf X[FQ_POINTS * FQ_PITCH];
	const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), b = lane & 1u;
	const uint32_t first = blockIdx.x * FQ_POINTS, n = lane & 31u, g = lane >> 5;
	// Every argument but the variance in one trip to the scalar cache, the wave's levels among them; left to the compiler each comes where it is used.
	struct {
		const __half2* table;
		const hf *sdf_w, *variance;
		const float* pos;
		uint32_t sdf_in_w, enc_w, N, ps, ds, hash_mask, active, row0_n;
		hf* sdf_out;
		float *row0, sdf_bias;
		int density;
	} q{a.table, a.sdf_w, a.variance, a.pos, a.sdf_in_w, a.enc_w, a.N, a.ps, a.ds, a.lv.hash_mask, a.lv.active_levels, a.row0_n, a.sdf_out, a.row0, a.sdf_bias, a.density};
	// (levels that the table does not have: n2_fused_field_sdf gives them eight entries, which any table has)
	uint32_t v[2][3];
	float scale[2];
#pragma unroll
	for (uint32_t k = 0; k < 2; ++k) {
		const uint32_t l = wave + 8u * k;
		scale[k] = a.lv.scale[l];
		v[k][0] = a.lv.res[l]; v[k][1] = a.lv.entries[l]; v[k][2] = a.lv.offset[l];
	}
	asm volatile("" : "+s"(q.N), "+s"(q.row0_n), "+s"(q.sdf_bias), "+s"(q.density)
	             : "s"(q.table), "s"(q.sdf_w), "s"(q.pos), "s"(q.sdf_in_w), "s"(q.enc_w), "s"(q.ps), "s"(q.ds), "s"(q.hash_mask), "s"(q.active), "s"(q.sdf_out), "s"(q.row0),
	               "s"(v[0][0]), "s"(v[0][1]), "s"(v[0][2]), "s"(scale[0]), "s"(v[1][0]), "s"(v[1][1]), "s"(v[1][2]), "s"(scale[1]));
	auto position = [&](uint32_t k, float (&p)[3]) {
		const uint32_t i = min(first + k, q.N - 1u);
		const float* at = q.pos + (size_t)i * q.ps;
		p[0] = at[0]; p[1] = at[q.ds]; p[2] = at[2 * (size_t)q.ds];
	};
	float p[3];
	position(lane >> 1, p);
	// The wave's fragment of the weights, and for two waves a second one: what sdf_forward_frag gives, four elements a load and without a branch
	// round any.  Element e is column x + (e & 3) + step (e >> 2) + shift of its row where x + .. is below `columns`, else zero; the four columns
	// a load takes may reach past the row, but not past the weights, where W_out follows W_0.
	constexpr uint32_t WAVES = FQ_BLOCK / 64, MORE = SDF_FRAG_COUNT - WAVES;
	static_assert(FF_SDF_COUNT == SDF_FRAG_COUNT && SDF_FRAG_WO < WAVES && MORE <= WAVES, "one fragment per wave, and some of the waves a second one");
	typedef hf four __attribute__((ext_vector_type(4), aligned(2)));
	const bool out = wave >= SDF_FRAG_WO, features = !out && wave % 3u < 2u;
	const uint32_t c = out ? wave - SDF_FRAG_WO : wave % 3u, row_n = min(n, MLP_OUT - 1u);
	const hf* const W1 = q.sdf_w + MLP_WIDTH * q.sdf_in_w;
	const hf* const row = out ? W1 + row_n * MLP_WIDTH : q.sdf_w + (32u * (wave / 3u) + n) * q.sdf_in_w;
	const uint32_t x = out || features ? 16u * c + 4u * g : 8u * g, step = out || features ? 8u : 4u, shift = features ? 3u : 0u;
	const uint32_t columns = out ? (n < MLP_OUT ? (uint32_t)MLP_WIDTH : 0u) : features ? q.enc_w : 3u;
	const four f_lo = *reinterpret_cast<const four*>(row + x + shift), f_hi = *reinterpret_cast<const four*>(row + x + step + shift);
	half8 f1 = wfrag_chained(W1, MLP_WIDTH, wave < MORE ? (int)row_n : 0, (int)(WAVES - SDF_FRAG_WO + wave % MORE), (int)g);
	PairItem it[2];
#pragma unroll
	for (uint32_t k = 0; k < 2; ++k) pair_fetch(q.table, WaveLevel{scale[k], v[k][0], v[k][1], v[k][2], ((q.hash_mask >> (wave + 8u * k)) & 1u) != 0u}, p, b, it[k]);
	asm volatile("" : "+v"(f1));  // (not loaded in the branch below)
	half8 f0;
#pragma unroll
	for (uint32_t e = 0; e < 4; ++e) {
		f0[e] = x + e < columns ? f_lo[e] : (hf)0;
		f0[4 + e] = x + step + e < columns ? f_hi[e] : (hf)0;
	}
	reinterpret_cast<half8*>(F)[threadIdx.x] = f0;
	if (n >= MLP_OUT) f1 = zero8();
	if (wave < MORE) reinterpret_cast<half8*>(F)[FQ_BLOCK + threadIdx.x] = f1;
#pragma unroll
	for (uint32_t k = 0; k < 2; ++k) {
		const float feat = pair_finish(it[k], b);
		X[(lane >> 1) * FQ_PITCH + 2u * (wave + 8u * k) + b] = wave + 8u * k < q.active ? (hf)feat : (hf)0.f;  // (switched off or not there: zero)
	}
	__syncthreads();
	if (wave != 0) return;
	half8 xs[3], h[4];
#pragma unroll
	for (int c = 0; c < 2; ++c) {
		const hf* at = X + n * FQ_PITCH + 16 * c + 4u * g;
		const half4v lo = *reinterpret_cast<const half4v*>(at), hi = *reinterpret_cast<const half4v*>(at + 8);
		xs[c] = half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
	}
	xs[2] = zero8();
#pragma unroll
	for (int d = 0; d < 3; ++d) {
		const float at = __shfl(p[d], 2 * (int)n);  // the point's position, from the pair that gathered for it
		xs[2][d] = g == 0 ? (hf)at - (hf)0.5f : (hf)0.f;
	}
	const half8 y = sdf_net(F, (int)lane, xs, h);
	const bool valid = first + n < q.N;
	store_sdf(q, y, valid ? first + n : q.N - 1u, valid, first + n, (int)g);
}

// The network of a large query, which takes the coarsest levels itself: gathered from memory they cost a query nearly what fine ones do, four lookups and lines a
// point and level, here they are issue beside a chain of loads, and their rows are neither written nor read.
//  * The two coarsest from tables of its own in LDS (of the default grid 16^3 and 24^3 entries, with the weights' fragments 80 KiB): one workgroup per CU stages
//    them, half a wave works on each level's feature of the tile's 32 samples.  Level 2 of the default grid takes 157 KB and a launch of its own, beside which
//    levels 0 to 2 were no cheaper than gathered (staged by 256 workgroups 17.6 us for 2^20 points; points along rays 187 -> 192.5).
//  * BLOCKS: the three dense levels behind them from blocks (N2Block), a line a point instead of four.  The gather's launch writes them, in workgroups behind those that
//    gather (in front 2 us more, in a launch of their own 4); nothing is kept for another call.  Lower lanes take level 4, upper ones level 2, where the network's
//    operands want them, and of level 3 either half an x corner.  Held by the blocks' lines and latency: 2^20 uniform points 47 us against 32 without, of the gather's
//    260 it takes 45.  With 64 samples to a wave and tile points in order and small batches took up to 4 % more; with the next tile's blocks under way meanwhile
//    ordered points 1.5 % more; tables that an index can run past, which spares the modulo: no change.
constexpr int FS_BLOCK = 1024;
constexpr uint32_t FS_GRID = 256, FS_LDS_MAX = 160 * 1024;
// a level's features at one x corner of a sample's cell from the four entries there, and in between: summed up as in n2_encode_level
__device__ __forceinline__ float2 staged_corner(const float (&w)[3], const uint32_t (&raw)[4]) {
	const float uy = 1.f - w[1], uz = 1.f - w[2], w00 = uy * uz, w10 = w[1] * uz, w01 = uy * w[2], w11 = w[1] * w[2];
	float2 v[4];
#pragma unroll
	for (int k = 0; k < 4; ++k) v[k] = __half22float2(*reinterpret_cast<const __half2*>(&raw[k]));
	return make_float2(fmaf(w00, v[0].x, fmaf(w10, v[1].x, fmaf(w01, v[2].x, fmaf(w11, v[3].x, 0.f)))), fmaf(w00, v[0].y, fmaf(w10, v[1].y, fmaf(w01, v[2].y, fmaf(w11, v[3].y, 0.f)))));
}
__device__ __forceinline__ uint32_t staged_feature(float wx, const float2 lo, const float2 hi) {
	const float ux = 1.f - wx;
	const half2v feat = {(hf)fmaf(ux, lo.x, wx * hi.x), (hf)fmaf(ux, lo.y, wx * hi.y)};
	return __builtin_bit_cast(uint32_t, feat);
}
// what lanes n and n + 32 hold, for both of them
__device__ __forceinline__ void staged_halves(float own, float& lower, float& upper) {
	const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(own), __float_as_uint(own), false, false);
	lower = __uint_as_float(r[0]);
	upper = __uint_as_float(r[1]);
}
// STREAM (with BLOCKS): rows are read and outputs written past the caches, each of which is met once, so that the blocks stay there (QUERY_STREAM_MIN).
template <bool BLOCKS, bool STREAM>
__global__ void __launch_bounds__(FS_BLOCK) field_staged_forward_kernel(const FusedArgs a) {
	extern __shared__ __align__(16) unsigned char smem[];
	hf* F = reinterpret_cast<hf*>(smem);
	unsigned char* const tables = smem + FF_SDF_COUNT * 1024;
	const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
	const uint32_t N = a.N, n_tiles = (N + 31u) / 32u, wave = blockIdx.x * (FS_BLOCK / 64) + (threadIdx.x >> 6), n_waves = gridDim.x * (FS_BLOCK / 64);
	auto position = [&](uint32_t tile, float (&p)[3]) __attribute__((always_inline)) {
		const float* q = a.pos + (size_t)min(tile * 32u + n, N - 1u) * a.ps;
#pragma unroll
		for (int d = 0; d < 3; ++d) p[d] = q[(size_t)d * a.ds];
	};
	float next[3];
	position(min(wave, n_tiles - 1u), next);
	const uint32_t second = 4u * a.lv.entries[0], bytes = second + 4u * a.lv.entries[1];
	{
		// (the parameters are 16-byte aligned, and weights and levels come in multiples of that)
		const uint4 *const from0 = reinterpret_cast<const uint4*>(a.table + a.lv.offset[0]), *const from1 = reinterpret_cast<const uint4*>(a.table + a.lv.offset[1]);
		const uint32_t all = bytes / 16u, firsts = second / 16u;
		constexpr uint32_t AHEAD = 5;
		for (uint32_t k0 = threadIdx.x; k0 < all; k0 += AHEAD * FS_BLOCK) {
			uint4 v[AHEAD];
#pragma unroll
			for (uint32_t q = 0; q < AHEAD; ++q) {
				const uint32_t k = min(k0 + q * FS_BLOCK, all - 1u);
				v[q] = k < firsts ? from0[k] : from1[k - firsts];
			}
#pragma unroll
			for (uint32_t q = 0; q < AHEAD; ++q)
				if (k0 + q * FS_BLOCK < all) reinterpret_cast<uint4*>(tables)[k0 + q * FS_BLOCK] = v[q];
		}
	}
	for (int idx = threadIdx.x; idx < FF_SDF_COUNT * 64; idx += FS_BLOCK) *reinterpret_cast<half8*>(F + (size_t)idx * 8) = fused_frag_value(a, idx >> 6, idx & 63);
	const float scale = a.lv.scale[g];
	const uint32_t entries = a.lv.entries[g], res = a.lv.res[g];
	const unsigned char* const table = tables + (g ? second : 0u);
	const bool on = (uint32_t)g < a.lv.active_levels;  // a switched-off level: zero features
	// the levels from blocks: lower lanes have 4, upper ones 2, where the network's operands want them; of level 3 either half of the wave takes an x corner
	const uint32_t blevel = g ? 2u : 4u, bres = a.lv.res[blevel], cres = a.lv.res[3];
	const float bscale = a.lv.scale[blevel], cscale = a.lv.scale[3];
	const N2Block *const bfrom = a.blocks + a.block_first[blevel - FS_LEVELS], *const cfrom = a.blocks + a.block_first[3 - FS_LEVELS];
	const bool bon = blevel < a.lv.active_levels, con = 3u < a.lv.active_levels;
	// (the next tile's rows are fetched ahead where waves take several tiles)
	uint32_t ahead[8];
	auto fetch_rows = [&](uint32_t tile) __attribute__((always_inline)) {
		const uint32_t col = min(tile * 32u + n, N - 1u);
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const uint32_t level = 4u * (j >> 1) + 2u * g + (j & 1);
			// (levels that have no row read that of the first level that does and are replaced, or meet weights of zero)
			const uint32_t lr = level < a.first_level || 2u * level >= a.enc_w ? a.first_level : level;
			const uint32_t* const at = query_rows(a) + (size_t)lr * N + col;
			ahead[j] = STREAM ? __builtin_nontemporal_load(at) : *at;
		}
	};
	if constexpr (BLOCKS) fetch_rows(min(wave, n_tiles - 1u));
	__syncthreads();
	for (uint32_t tile = wave; tile < n_tiles; tile += n_waves) {
		const uint32_t col_raw = tile * 32u + n;
		const bool valid = col_raw < N;
		const uint32_t col = valid ? col_raw : N - 1u;
		const float p[3] = {next[0], next[1], next[2]};
		half8 xs[3];
		if constexpr (!BLOCKS) fetch_rows(tile);
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const half2v f = __builtin_bit_cast(half2v, ahead[j]);
			xs[j >> 2][2 * (j & 3)] = f[0];
			xs[j >> 2][2 * (j & 3) + 1] = f[1];
		}
		float bw[3], cw[3];
		uint32_t braw[2][4], craw[4];
		if constexpr (BLOCKS) {
			uint32_t c[3];
#pragma unroll
			for (int d = 0; d < 3; ++d) n2_locate(p[d], bscale, bw[d], c[d]);
			const N2Block* const row = bfrom + n2_block_row(bres, c[1], c[2]);
			const N2Block v0 = row[min(c[0], bres)], v1 = row[min(c[0] + 1u, bres)];
#pragma unroll
			for (int d = 0; d < 3; ++d) n2_locate(p[d], cscale, cw[d], c[d]);
			const N2Block v2 = (cfrom + n2_block_row(cres, c[1], c[2]))[min(c[0] + (uint32_t)g, cres)];
#pragma unroll
			for (int q = 0; q < 4; ++q) { braw[0][q] = v0.entry[q]; braw[1][q] = v1.entry[q]; craw[q] = v2.entry[q]; }
		}
		position(tile + n_waves < n_tiles ? tile + n_waves : tile, next);
		if constexpr (BLOCKS) fetch_rows(tile + n_waves < n_tiles ? tile + n_waves : tile);
		xs[2] = zero8();
		if (g == 0) {
#pragma unroll
			for (int d = 0; d < 3; ++d) xs[2][d] = (hf)p[d] - (hf)0.5f;
		}
		// sample n's feature of level g
		float w[3];
		uint32_t c[3], raw[2][4];
#pragma unroll
		for (int d = 0; d < 3; ++d) n2_locate(p[d], scale, w[d], c[d]);
#pragma unroll
		for (uint32_t b = 0; b < 2; ++b) {
			uint32_t at[4];
			n2_corner_bytes<N2_LEVEL_DENSE>(entries, res, c[0] + b, c[1], c[2], at);
#pragma unroll
			for (int k = 0; k < 4; ++k) raw[b][k] = *reinterpret_cast<const uint32_t*>(table + at[k]);
		}
		const uint32_t own = on ? staged_feature(w[0], staged_corner(w, raw[0]), staged_corner(w, raw[1])) : 0u, other = (uint32_t)__shfl_xor((int)own, 32);
		uint32_t x4[4] = {0u, 0u, 0u, 0u};
		*reinterpret_cast<half8*>(x4) = xs[0];
		if constexpr (BLOCKS) {
			const uint32_t b0 = bon ? staged_feature(bw[0], staged_corner(bw, braw[0]), staged_corner(bw, braw[1])) : 0u;
			const float2 mine = staged_corner(cw, craw);
			float2 lo, hi;
			staged_halves(mine.x, lo.x, hi.x);
			staged_halves(mine.y, lo.y, hi.y);
			const uint32_t b1 = con ? staged_feature(cw[0], lo, hi) : 0u;
			x4[0] = g ? b0 : own;
			x4[1] = g ? b1 : other;
			x4[2] = g ? x4[2] : b0;
		} else if (g == 0) {
			x4[0] = own;
			x4[1] = other;
		}
		xs[0] = *reinterpret_cast<half8*>(x4);
		half8 h[4];
		const half8 y = sdf_net(F, lane, xs, h);
		store_sdf<STREAM>(a, y, col, valid, col_raw, g);
		tile_fence();
	}
}


// ----------------------------------------------------------------------------
// the network kernel: a wave takes 32 samples per pass, lane (n, g) works for sample b0 + n on the levels l(j, g).
// GATHER: the features come from the table (inference on points in lattice order); else from the rows the gather kernel wrote.
// ----------------------------------------------------------------------------
template <bool FULL, bool GATHER>
__global__ void __launch_bounds__(FF_BLOCK, 2) field_fused_forward_kernel(const FusedArgs a) {
	static_assert(!(FULL && GATHER), "the full forward reads the gather kernel's rows");
	extern __shared__ __align__(16) unsigned char smem[];
	hf* F = reinterpret_cast<hf*>(smem);
	uint4* LV = reinterpret_cast<uint4*>(smem + (size_t)(FULL ? FF_COUNT : FF_SDF_COUNT) * 1024);
	// FULL: each wave's staging area for the colour net's input (32 samples)
	unsigned char* const stage = smem + (size_t)(FULL ? FF_COUNT : FF_SDF_COUNT) * 1024 + FF_LEVELS * sizeof(uint4) + (threadIdx.x >> 6) * (32 * 2 * N2_RGB_IN_PITCH);
	const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
	const uint32_t N = a.N, hash_mask = a.lv.hash_mask, active = a.lv.active_levels;
	uint32_t n_live = a.live ? min(*a.live, N) : N, col0 = 0;
	if (FULL && a.list) listed_range(a, col0, n_live);  // a listed pass: columns col0 .. col0 + n_live
	const uint32_t n_tiles = (n_live + 31u) / 32u;
	const uint32_t wave_gid = blockIdx.x * (FF_BLOCK / 64) + (threadIdx.x >> 6), n_waves = gridDim.x * (FF_BLOCK / 64);
	// FULL: what a tile starts with (features, coordinates, place in the output); the next tile's is under way while the current one is computed, the
	// first one's beside the weights.  (2^18 samples 37.1 -> 33.0 us, the weights' copies included, a depth round 16.0 -> 13.4: two waves a SIMD hide little, and the loads of a tile also waited for the
	// stores of the last one.  Three workgroups per CU at 168 registers spill.)
	struct Start {
		hf feat[16];
		float p[3], dir[3];
		uint32_t dst;
	};
	const uint32_t* const places = a.list ? a.list : reinterpret_cast<const uint32_t*>(a.coords);  // (no branch round the load; without a list its value is not used)
	auto start = [&](uint32_t tile) __attribute__((always_inline)) {
		Start t;
		const uint32_t col = col0 + min(tile * 32u + n, n_live - 1u);
		const float* q = a.coords + (size_t)col * 7;
#pragma unroll
		for (int d = 0; d < 3; ++d) { t.p[d] = q[d]; t.dir[d] = q[4 + d]; }
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const uint32_t level = 4u * (j >> 1) + 2u * g + (j & 1);
			// levels the grid does not have read level 0's rows and are ignored (their weights are zero)
			const uint32_t lr = 2u * level < a.enc_w ? level : 0u;
			t.feat[2 * j] = a.sdf_in[(size_t)(3 + 2 * lr) * N + col];
			t.feat[2 * j + 1] = a.sdf_in[(size_t)(4 + 2 * lr) * N + col];
		}
		t.dst = places[col];
		return t;
	};
	Start next;
	hf variance = (hf)0;
	if constexpr (FULL) {
		if (n_tiles > 0) next = start(min(wave_gid, n_tiles - 1u));
		variance = a.variance[0];
	}
	if (threadIdx.x < FF_LEVELS)
		LV[threadIdx.x] = make_uint4(__float_as_uint(a.lv.scale[threadIdx.x]), a.lv.res[threadIdx.x], a.lv.entries[threadIdx.x], a.lv.offset[threadIdx.x]);
	// (a.frags: copied from the image a gather launch left in global memory, instead of two-byte picks all over the weight matrices: 5 to 7 us of a launch)
	if (FULL && a.frags) load_frags<FF_COUNT, FF_BLOCK>(F, a.frags);
	else build_fused_frags(F, a, FULL ? FF_COUNT : FF_SDF_COUNT);
	for (uint32_t tile = wave_gid; tile < n_tiles; tile += n_waves) {
		const uint32_t col_raw = tile * 32u + n;
		const bool valid = col_raw < n_live;
		const uint32_t col = col0 + (valid ? col_raw : n_live - 1u);
		uint32_t dst = col;  // the sample's row in the output
		half8 xs[3];               // SDF net input, B operands
		float p[3], dir[3] = {0.f, 0.f, 0.f};
		uint4 slope[8];            // FULL: the slopes of the lane's 8 levels as stored
		if (GATHER) {
			const float* q = a.pos + (size_t)col * a.ps;
#pragma unroll
			for (int d = 0; d < 3; ++d) p[d] = q[(size_t)d * a.ds];
			// the lane's 8 levels, the next level's loads in flight while one is finished
			Item cur, nxt;
			item_fetch<0>(LV, hash_mask, active, a.table, g, p, cur);
#define FF_STEP(J)                                                                           \
			if (J < 7) item_fetch<(J < 7 ? J + 1 : 0)>(LV, hash_mask, active, a.table, g, p, nxt); \
			{                                                                                \
				float feat[2];                                                               \
				item_finish(cur, feat);                                                      \
				xs[J >> 2][2 * (J & 3)] = (hf)feat[0];                                       \
				xs[J >> 2][2 * (J & 3) + 1] = (hf)feat[1];                                   \
			}                                                                                \
			cur = nxt;                                                                       \
			__builtin_amdgcn_sched_barrier(0);
			FF_STEP(0) FF_STEP(1) FF_STEP(2) FF_STEP(3) FF_STEP(4) FF_STEP(5) FF_STEP(6) FF_STEP(7)
#undef FF_STEP
		} else {
			if (FULL) {
				if (a.list) dst = next.dst;
#pragma unroll
				for (int d = 0; d < 3; ++d) { p[d] = next.p[d]; dir[d] = next.dir[d]; }
			} else {
				const float* q = a.pos + (size_t)col * a.ps;
#pragma unroll
				for (int d = 0; d < 3; ++d) p[d] = q[(size_t)d * a.ds];
			}
#pragma unroll
			for (int j = 0; j < 8; ++j) {
				const uint32_t level = 4u * (j >> 1) + 2u * g + (j & 1);
				// levels the grid does not have read level 0's rows and are ignored (their weights are zero)
				const uint32_t lr = 2u * level < a.enc_w ? level : 0u;
				half2v f;
				if (FULL) f = half2v{next.feat[2 * j], next.feat[2 * j + 1]};
				else f = __builtin_bit_cast(half2v, query_rows(a)[(size_t)lr * N + col]);
				xs[j >> 2][2 * (j & 3)] = f[0];
				xs[j >> 2][2 * (j & 3) + 1] = f[1];
				if (FULL) slope[j] = a.slopes[(size_t)lr * N + col];
			}
		}
		xs[2] = zero8();
		if (g == 0) {
#pragma unroll
			for (int d = 0; d < 3; ++d) xs[2][d] = (hf)p[d] - (hf)0.5f;
		}
		// ---- SDF net ----
		half8 h[4];
		half8 y = sdf_net(F, lane, xs, h);
		if (!FULL) {
			store_sdf(a, y, col, valid, col_raw, g);
			tile_fence();
			continue;
		}
		const uint32_t next_tile = tile + n_waves;
		if constexpr (FULL) next = start(next_tile < n_tiles ? next_tile : tile);
		// ---- d sdf / d input: dh = mask * W_out[0, :], dX = W_0^T dh ----
		half8 dh[4];
#pragma unroll
		for (int c = 0; c < 4; ++c) dh[c] = mask8(frag(F, S_DH + c, lane), h[c]);
		float16v dx0 = zero16(), dx1 = zero16();
#pragma unroll
		for (int c = 0; c < 4; ++c) dx0 = N2_MFMA(frag(F, S_W0T + c, lane), dh[c], dx0);
#pragma unroll
		for (int c = 0; c < 4; ++c) dx1 = N2_MFMA(frag(F, S_W0T + 4 + c, lane), dh[c], dx1);
		// register r of dx0 is feature r % 2 of the lane's level step r / 2; registers 0..2 of dx1 (g = 0) the coordinates
		const half8 g_lo = round8(dx0, 0), g_hi = round8(dx0, 8);
		const hf gx[3] = {(hf)dx1[0], (hf)dx1[1], (hf)dx1[2]};
		float nrm[3];
#pragma unroll
		for (int d = 0; d < 3; ++d) nrm[d] = g == 0 ? (float)gx[d] : 0.f;
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const uint32_t level = 4u * (j >> 1) + 2u * g + (j & 1);
			const float sc = 2u * level < a.enc_w ? __uint_as_float(LV[level].x) : 0.f;
			float q[6];
			const float unit = n2_slopes_unpack(slope[j], q) * sc;
			const float g0 = (float)(j < 4 ? g_lo[2 * j] : g_hi[2 * j - 8]) * unit, g1 = (float)(j < 4 ? g_lo[2 * j + 1] : g_hi[2 * j - 7]) * unit;
#pragma unroll
			for (int d = 0; d < 3; ++d) nrm[d] = fmaf(g0, q[d], fmaf(g1, q[3 + d], nrm[d]));
		}
#pragma unroll
		for (int d = 0; d < 3; ++d) nrm[d] += __shfl_xor(nrm[d], 32);
		const hf hn[3] = {(hf)nrm[0], (hf)nrm[1], (hf)nrm[2]};
		// ---- colour net input: SDF-net outputs | SH of the direction | position, normal ----
		float sh[16];
		sh4(dir[0] * 2.f - 1.f, dir[1] * 2.f - 1.f, dir[2] * 2.f - 1.f, sh);
		half8 xc[3];
		xc[0] = y;
		{
			// both halves are formed and one is picked value by value: picking between sh[e] and sh[8 + e] inside the
			// conversion turns into an index that depends on the lane, and the array then lives in scratch memory
			half8 lo8, hi8;
#pragma unroll
			for (int e = 0; e < 8; ++e) { lo8[e] = (hf)sh[e]; hi8[e] = (hf)sh[8 + e]; }
			const uint4 lo = __builtin_bit_cast(uint4, lo8), hi = __builtin_bit_cast(uint4, hi8);
			xc[1] = __builtin_bit_cast(half8, make_uint4(g ? hi.x : lo.x, g ? hi.y : lo.y, g ? hi.z : lo.z, g ? hi.w : lo.w));
		}
		xc[2] = zero8();
		if (g == 0) {
#pragma unroll
			for (int d = 0; d < 3; ++d) { xc[2][d] = (hf)p[d]; xc[2][3 + d] = hn[d]; }
		}
		{
			// The colour net's input goes out sample-major for the backward pass (N2_RGB_IN_PITCH = 40 values per sample: rows
			// 38, 39 zero, rows 40..47 of the padded input left out): the wave's 32 samples are 2560 consecutive bytes.  A
			// lane's registers are runs of 4 and 8 rows of its sample; stored from there, every 16 bytes would be a write
			// request of their own.  Through LDS (80 bytes per sample: the 16-byte writes of 16 lanes fall on different
			// banks) the wave writes whole lines.
			unsigned char* sp = stage + n * (2 * N2_RGB_IN_PITCH);
			*reinterpret_cast<half4v*>(sp + 8 * g) = half4v{y[0], y[1], y[2], y[3]};
			*reinterpret_cast<half4v*>(sp + 16 + 8 * g) = half4v{y[4], y[5], y[6], y[7]};
			*reinterpret_cast<half8*>(sp + 32 + 16 * g) = xc[1];
			if (g == 0) *reinterpret_cast<half8*>(sp + 64) = xc[2];
			__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
			__builtin_amdgcn_wave_barrier();
			__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
			// (The next tile's start has arrived before this one's stores are issued: a load behind a store in a branch is awaited
			// with the store.)
#pragma unroll
			for (int k = 0; k < 16; ++k) asm volatile("" : "+v"(next.feat[k]));
#pragma unroll
			for (int d = 0; d < 3; ++d) asm volatile("" : "+v"(next.p[d]), "+v"(next.dir[d]));
			asm volatile("" : "+v"(next.dst));
			const uint32_t chunks = 5u * min(32u, n_live - tile * 32u);  // 16-byte chunks of the tile's samples
			unsigned char* out = reinterpret_cast<unsigned char*>(a.rgb_in) + ((size_t)col0 + (size_t)tile * 32u) * (2u * N2_RGB_IN_PITCH);
#pragma unroll
			for (int i = 0; i < 3; ++i) {
				const uint32_t k = (uint32_t)lane + 64u * i;
				if (k < chunks) *reinterpret_cast<uint4*>(out + (size_t)k * 16u) = *reinterpret_cast<const uint4*>(stage + k * 16u);
			}
		}
		if (valid) {
			// (rows 0..2 of d sdf / d input, gx, have no reader behind this kernel)
#pragma unroll
			for (int r = 0; r < 16; ++r) {
				const uint32_t level = 4u * (r >> 2) + 2u * g + ((r >> 1) & 1);
				if (2u * level < a.enc_w) a.dsdf_din[(size_t)(3 + 2 * level + (r & 1)) * N + col] = r < 8 ? g_lo[r] : g_hi[r - 8];
			}
		}
		half8 h0[4], h1[4];
#pragma unroll
		for (int mt = 0; mt < 2; ++mt) {
			float16v acc = zero16();
#pragma unroll
			for (int c = 0; c < 3; ++c) acc = N2_MFMA(frag(F, C_W0 + mt * 3 + c, lane), xc[c], acc);
			relu_pack(acc, h0[2 * mt], h0[2 * mt + 1]);
		}
#pragma unroll
		for (int mt = 0; mt < 2; ++mt) {
			float16v acc = zero16();
#pragma unroll
			for (int c = 0; c < 4; ++c) acc = N2_MFMA(frag(F, C_WH + mt * 4 + c, lane), h0[c], acc);
			relu_pack(acc, h1[2 * mt], h1[2 * mt + 1]);
		}
		float16v co = zero16();
#pragma unroll
		for (int c = 0; c < 4; ++c) co = N2_MFMA(frag(F, C_WO + c, lane), h1[c], co);
		// ---- output rows: r g b | sdf + bias | normal | variance | direction | colour-net rows 11..15 ----
		half4 lo = half4{(hf)co[0], (hf)co[1], (hf)co[2], (hf)co[3]}, hi = half4{(hf)co[4], (hf)co[5], (hf)co[6], (hf)co[7]};
		if (g == 0) {
			lo[3] = y[0] + (hf)a.sdf_bias;
			hi[0] = (hf)dir[0]; hi[1] = (hf)dir[1]; hi[2] = (hf)dir[2];
		} else {
			lo[0] = hn[0]; lo[1] = hn[1]; lo[2] = hn[2]; lo[3] = variance;
		}
		if (valid) {
			hf* o = a.output + (size_t)dst * MLP_OUT;
			*reinterpret_cast<half4*>(o + 4 * g) = lo;
			*reinterpret_cast<half4*>(o + 8 + 4 * g) = hi;
		}
		tile_fence();
	}
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------
bool n2_fused_supported(const N2LevelTable& tab, uint32_t sdf_hidden_layers, uint32_t rgb_hidden_layers) {
	if (tab.n_levels > FF_LEVELS || tab.n_features != 2 || sdf_hidden_layers != 1 || rgb_hidden_layers != 2) return false;
	if (tab.max_level_gpu != nullptr) return false;  // per-point level masks take the unfused path
	for (uint32_t l = 0; l < tab.n_levels; ++l)
		if (tab.mode[l] != N2_LEVEL_DENSE && tab.mode[l] != N2_LEVEL_HASH) return false;
	return true;
}

template <bool FULL>
static void launch_gather(const FusedArgs& a, hipStream_t s) {
	const uint32_t tiles = (a.N + FG_BLOCK - 1) / FG_BLOCK;
	const N2GatherGrid g = n2_gather_grid(FULL ? N2_FIELD_XCD_MAX : N2_QUERY_XCD_MAX, a.N, a.n_levels, FG_BLOCK);
	const uint32_t more = (a.n_blocks + FG_BLOCK - 1) / FG_BLOCK;
	const dim3 grid = FULL ? dim3(g.x * g.y + (a.frags ? FRAG_BLOCKS : 0u)) : g.y == 1u ? dim3(g.x + more) : dim3(g.x, g.y + (more + g.x - 1) / g.x);
	field_gather_kernel<FULL><<<grid, dim3(FG_BLOCK), 0, s>>>(a, tiles, g.y == 1u ? 1 : 0);
}

// Up to here a query is one launch: 256 workgroups of FQ_POINTS, one for each CU.  Beyond, some CUs run two, and the fragments that every 32 points
// rebuild from the weights weigh more than the second launch and its wait.  (Device time in a graph, two launches | one: 64 points 6.3 | 3.5 us, 1000 8.1 | 5.0,
// 4096 10.3 | 6.9, 6144 11.5 | 8.4, 8192 11.7 | 9.7, 10 240 12.85 | 12.7, 12 288 12.8 | 13.4, 16 384 14.1 | 16.3; a call from Python, bound by the host below
// 5000 points: 1000 9.4 | 7.2, 8192 11.7 | 9.7.)
constexpr uint32_t QUERY_ONE_LAUNCH_MAX = 256 * FQ_POINTS;
// From here on the two coarsest levels are the network kernel's (field_staged_forward_kernel): its start, two tables to every CU, costs smaller queries more than their
// two levels.  (Call in us, gathered | staged, uniform points: 32 768 18.3 | 20.5, 65 536 28.7 | 28.7, 98 304 39.1 | 36.4, 2^17 49.1 | 44.2, 2^18 87.2 | 77.7, 2^20 292 | 278,
// 2^21 566 | 531; along rays 65 536 20.3 | 21.2, 98 304 26.5 | 26.8, 2^17 33.7 | 32.1, 2^20 184 | 182; on a lattice 65 536 19.6 | 20.0, 98 304 26.1 | 25.7, 2^20 142 | 141.  Updates of
// the occupancy grid: 2^17 samples 67.5 | 64.0, 700 000 264 | 250, 2^20 252 | 245, 2^21 421 | 415.)
constexpr uint32_t QUERY_STAGED_MIN = 3u << 15;
// ... and from here on three more come from blocks: making these costs smaller queries what they save.  The line is that of points in no order; points that come in one share lines
// without blocks, and those between here and 2^19 lose two to three per cent to them.  (Call in us, staged | with blocks, uniform points: 98 304 36.4 | 37.3, 2^17
// 44.2 | 43.9, 2^18 77.7 | 73.3, 2^19 148 | 136, 2^20 278 | 250, 2^21 531 | 480; along rays 2^17 32.1 | 35.2, 2^18 56.1 | 57.8, 2^19 99.0 | 98.2, 2^20 182 | 177; on a lattice 2^17
// 31.4 | 34.4, 2^18 55.1 | 56.5, 2^19 77.2 | 77.6, 2^20 141 | 136.  Updates of the occupancy grid: 2^19 samples 160.4 | 157.2, 700 000 250 | 231, 2^20 245 | 236, 2^21 415 | 400.)
constexpr uint32_t QUERY_BLOCKS_MIN = 1u << 18;
// ... and from here on rows and outputs are streams, which smaller queries find in the caches.  (Call in us, cached | streamed, uniform points: 2^18 71.9 | 73.6, 2^19 135.6 | 137,
// 655 360 163.3 | 164.3, 786 432 193.7 | 193.1, 2^20 254.6 | 249.7, 1 572 864 371.5 | 363.5, 2^21 490.7 | 476.5; update of the occupancy grid, which keeps one row, 2^21 398.3 | 398.1.)
// Only where every row of features starts a line: of a line that two tiles share, the first one's streamed load takes it from the second (800 008 points 206.4 | 208.4, 1 000 008
// 251.7 | 253.6, 2 000 008 485.4 | 487.6).
constexpr uint32_t QUERY_STREAM_MIN = 3u << 18;

// ----------------------------------------------------------------------------
// The SDF network on its own (48 inputs: coordinates, 32 features, padding) with the eikonal loss: network, d sdf / d input, normals from the
// encoding's fp32 Jacobian, the loss's terms and everything the backward takes, in one pass over the input rows and the Jacobian.
// ----------------------------------------------------------------------------
struct SdfEikonalArgs {
	const hf* weights;
	uint32_t N;
	const hf* input;       // [48][N]
	const float* dy_dx;    // [32][N][3]
	hf* output;            // [16][N]
	hf* dsdf;              // [48][N]
	float* normal;         // [3][N]
	float ek_weight, scale;
	hf* dL_dy;             // [16][N], row 0
	float* v;              // [3][N]
	hf* v_in;              // [48][N], rows 0 .. 34
	float* parts;          // a workgroup's part of the loss's sum
};
constexpr int SE_FRAGS = C_W0;  // the SDF net's fragments come first

// d sdf / d input's rows behind the features: tile row t < 3 is a coordinate, the others are the padding inputs (whose weights count like any)
__device__ __forceinline__ int sdf_tail_col(int t) { return t < 3 ? t : 32 + t; }
// Bound by memory: 678 bytes a point, of which the Jacobian's rows are 384; at 2^18 points 38.7 us, 4.6 TB/s (network and normals in two launches 17.7 + 30.0),
// at 2^14 7.0 (6.1 + 6.0).  No store stands in a branch (lanes behind the last point repeat it), so that a tile waits for its own loads alone, and matrices are
// addressed by a scalar row and a 32-bit offset: with 64-bit addresses per lane and the next tile's Jacobian under way too the registers spill (56 us).
template <bool STREAM>
__global__ void __launch_bounds__(FF_BLOCK, 2) sdf_eikonal_forward_kernel(const SdfEikonalArgs a) {
	constexpr int RAW = mlp_n_params<3, 1>();
	__shared__ __align__(16) hf F[SE_FRAGS * 512], raw[RAW];
	__shared__ float part[FF_BLOCK / 64];
	const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
	const uint32_t N = a.N, n_tiles = (N + 31u) / 32u;
	const uint32_t wave_gid = blockIdx.x * (FF_BLOCK / 64) + (threadIdx.x >> 6), n_waves = gridDim.x * (FF_BLOCK / 64);
	// Of a matrix [rows][N], row u + 4 g of the lane's point: the row u stands in a scalar address, the rest in a 32-bit lane offset (n2_sdf_one_pass: 60 N - 12 bytes at most).
	auto at = [&](auto* matrix, uint32_t u, uint32_t lane_at, uint32_t width) __attribute__((always_inline)) {
		typedef typename std::conditional<std::is_const<std::remove_pointer_t<decltype(matrix)>>::value, const char, char>::type bytes;
		typedef std::remove_pointer_t<decltype(matrix)> value;
		return reinterpret_cast<value*>(reinterpret_cast<bytes*>(matrix + (size_t)u * N * width) + lane_at * (uint32_t)(sizeof(value) * width));
	};
	auto row_of = [](int r) { return 8u * (uint32_t)(r >> 2) + (uint32_t)(r & 3); };  // of D register r, without 4 g
	struct Start {
		hf feat[16], p[3];
	};
	auto start = [&](uint32_t tile) __attribute__((always_inline)) {
		Start t;
		const uint32_t col = min(tile * 32u + n, N - 1u), mine = 4u * g * N + col;
#pragma unroll
		for (int d = 0; d < 3; ++d) t.p[d] = *at(a.input, d, col, 1u);
#pragma unroll
		for (int r = 0; r < 16; ++r) t.feat[r] = *at(a.input, 3u + row_of(r), mine, 1u);
		return t;
	};
	Start next = start(min(wave_gid, n_tiles - 1u));
	copy_to_lds<FF_BLOCK, RAW / 8>(raw, a.weights);
	__syncthreads();
	for (int idx = threadIdx.x; idx < SE_FRAGS * 64; idx += FF_BLOCK) {
		const int f = idx >> 6, l = idx & 63, m = l & 31, lg = l >> 5;
		half8 w = zero8();
		if (f < S_W0T) {
			w = sdf_forward_frag(raw, 48, 32u, f, l);
		} else if (f < S_DH) {
			const int q = f - S_W0T, t = 32 * (q >> 2) + m, col = t < 32 ? 3 + t : sdf_tail_col(t - 32);
#pragma unroll
			for (int e = 0; e < 8; ++e) w[e] = col < 48 ? raw[chained_k(q & 3, lg, e) * 48 + col] : (hf)0;
		} else {
#pragma unroll
			for (int e = 0; e < 8; ++e) w[e] = raw[MLP_WIDTH * 48 + chained_k(f - S_DH, lg, e)];
		}
		*reinterpret_cast<half8*>(F + (size_t)idx * 8) = w;
	}
	__syncthreads();
	float term = 0.f;
	for (uint32_t tile = wave_gid; tile < n_tiles; tile += n_waves) {
		const uint32_t col_raw = tile * 32u + n, col = min(col_raw, N - 1u), next_tile = tile + n_waves;
		const uint32_t mine = 4u * g * N + col;
		const Start cur = next;
		n2_float3 j[16];
#pragma unroll
		for (int r = 0; r < 16; ++r) j[r] = n2_load3<STREAM>(at(a.dy_dx, row_of(r), mine, 3u));
		next = start(next_tile < n_tiles ? next_tile : tile);
		half8 xs[3], h[4], dh[4];
#pragma unroll
		for (int r = 0; r < 16; ++r) xs[r >> 3][r & 7] = cur.feat[r];
		xs[2] = zero8();
#pragma unroll
		for (int d = 0; d < 3; ++d) xs[2][d] = g == 0 ? cur.p[d] : (hf)0;
		const half8 y = sdf_net(F, lane, xs, h);
		// d sdf / d input: dh = mask * W_out[0, :], dX = W_0^T dh
#pragma unroll
		for (int c = 0; c < 4; ++c) dh[c] = mask8(frag(F, S_DH + c, lane), h[c]);
		float16v dx0 = zero16(), dx1 = zero16();
#pragma unroll
		for (int c = 0; c < 4; ++c) dx0 = N2_MFMA(frag(F, S_W0T + c, lane), dh[c], dx0);
#pragma unroll
		for (int c = 0; c < 4; ++c) dx1 = N2_MFMA(frag(F, S_W0T + 4 + c, lane), dh[c], dx1);
		const half8 lo = round8(dx0, 0), hi = round8(dx0, 8), tail = round8(dx1, 0);
		float nrm[3];
#pragma unroll
		for (int d = 0; d < 3; ++d) nrm[d] = 0.f;
#pragma unroll
		for (int r = 0; r < 16; ++r) {
			const float f = (float)(r < 8 ? lo[r & 7] : hi[r & 7]);
			nrm[0] = fmaf(f, j[r].x, nrm[0]);
			nrm[1] = fmaf(f, j[r].y, nrm[1]);
			nrm[2] = fmaf(f, j[r].z, nrm[2]);
		}
		float len2 = 0.f, x[3];
#pragma unroll
		for (int d = 0; d < 3; ++d) {
			const float gx = g == 0 ? (float)tail[d] : 0.f;  // the direct rows: the first half of the wave holds them
			nrm[d] += __shfl_xor(nrm[d], 32);
			nrm[d] += gx + __shfl_xor(gx, 32);
			len2 = fmaf(nrm[d], nrm[d], len2);
		}
		const float len = fmaxf(sqrtf(len2), 1e-12f), k = 2.f * a.ek_weight * (len - 1.f) / len * a.scale, sdf = (float)y[0];
		if (col_raw < N && g == 0) term += fabsf(sdf) + a.ek_weight * (len - 1.f) * (len - 1.f);
#pragma unroll
		for (int d = 0; d < 3; ++d) x[d] = nrm[d] * k;
		// (the next tile's start has arrived before this one's stores are issued: where it is used the compiler would wait for those, too)
#pragma unroll
		for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(next.feat[r]));
#pragma unroll
		for (int d = 0; d < 3; ++d) asm volatile("" : "+v"(next.p[d]));
#pragma unroll
		for (int r = 0; r < 8; ++r) {
			*at(a.output, row_of(r), mine, 1u) = y[r];
			// (the second half's tail rows 4.. are columns 36..; of the first half's rows the coordinates are columns 0..2)
			if (r < 3) *(at(a.dsdf, r, col, 1u) + (g ? (size_t)36 * N : 0)) = tail[r];
			else *at(a.dsdf, 32u + row_of(r), mine, 1u) = tail[r];
		}
#pragma unroll
		for (int r = 0; r < 16; ++r) {
			*at(a.dsdf, 3u + row_of(r), mine, 1u) = r < 8 ? lo[r & 7] : hi[r & 7];
			*at(a.v_in, 3u + row_of(r), mine, 1u) = (hf)fmaf(j[r].x, x[0], fmaf(j[r].y, x[1], j[r].z * x[2]));
		}
		float* const out3 = g ? a.v : a.normal;
#pragma unroll
		for (int d = 0; d < 3; ++d) out3[(size_t)d * N + col] = g ? x[d] : nrm[d];
		// row 0 of dL_dy and row 0 of v_in by the first half, rows 1 and 2 by the second
		const hf sign = (hf)((sdf > 0.f ? 1.f : sdf < 0.f ? -1.f : 0.f) * a.scale);
		*(g ? a.v_in + (size_t)N + col : a.dL_dy + col) = g ? (hf)x[1] : sign;
		a.v_in[(g ? (size_t)2 * N : 0) + col] = g ? (hf)x[2] : (hf)x[0];
		tile_fence();
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) term += __shfl_xor(term, o);
	if (lane == 0) part[threadIdx.x >> 6] = term;
	__syncthreads();
	if (threadIdx.x == 0) a.parts[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
}

static uint32_t fused_grid(uint32_t n, uint32_t most = 512u) {
	const uint32_t tiles = (n + 31u) / 32u, blocks = (tiles + 3u) / 4u;
	return blocks < most ? blocks : most;
}
static size_t fused_lds(int n_frags, bool staged = false) {
	return (size_t)n_frags * 1024 + FF_LEVELS * sizeof(uint4) + (staged ? (size_t)(FF_BLOCK / 64) * 32 * 2 * N2_RGB_IN_PITCH : 0);
}

static FusedArgs fused_base(const N2FusedNets& nets, uint32_t n) {
	FusedArgs a{};
	const N2LevelTable& tab = *nets.tab;
	const uint32_t active = tab.active_levels < tab.n_levels ? tab.active_levels : tab.n_levels;
	for (uint32_t l = 0; l < FF_LEVELS; ++l) {
		const bool have = l < tab.n_levels;  // levels the table does not have read as switched off
		a.lv.scale[l] = have ? tab.scale[l] : 1.f;
		a.lv.res[l] = have ? tab.resolution[l] : 1u;
		a.lv.entries[l] = have ? tab.entries[l] : 8u;
		a.lv.offset[l] = have ? tab.offset[l] : 0u;
		if (have && tab.mode[l] == N2_LEVEL_HASH) a.lv.hash_mask |= 1u << l;
	}
	a.lv.active_levels = active;
	a.table = nets.table;
	a.sdf_w = reinterpret_cast<const hf*>(nets.sdf_w);
	a.rgb_w = reinterpret_cast<const hf*>(nets.rgb_w);
	a.variance = reinterpret_cast<const hf*>(nets.variance);
	a.sdf_in_w = nets.sdf_in_w;
	a.enc_w = tab.n_levels * 2;
	a.n_levels = tab.n_levels;
	a.sdf_bias = nets.sdf_bias;
	a.N = n;
	a.live = nullptr;
	a.list = nullptr;
	a.counts = nullptr;
	a.round = 0;
	a.frags = nullptr;
	return a;
}

int n2_fused_field_forward(const N2FusedNets& nets, hipStream_t s, const float* d_coords, uint32_t n, n2_half* sdf_in, float* xyz_rows,
                           void* slopes, n2_half* dsdf_din, n2_half* rgb_in, n2_half* d_output, const uint32_t* d_live, const uint32_t* d_list,
                           const uint32_t* d_counts, uint32_t round, uint32_t est_samples, const float* d_xyz_soa) {
	FusedArgs a = fused_base(nets, n);
	if (d_xyz_soa) { a.pos = d_xyz_soa; a.ps = 1; a.ds = n; }
	a.live = d_live;
	a.list = d_list;
	a.counts = d_counts;
	a.round = round;
	a.frags = reinterpret_cast<hf*>(nets.frag_image);
	a.coords = d_coords;
	a.sdf_in = reinterpret_cast<hf*>(sdf_in);
	a.xyz_rows = xyz_rows;
	a.slopes = reinterpret_cast<uint4*>(slopes);
	a.dsdf_din = reinterpret_cast<hf*>(dsdf_din);
	a.rgb_in = reinterpret_cast<hf*>(rgb_in);
	a.output = reinterpret_cast<hf*>(d_output);
	if (d_list) {
		// est_samples: the caller's estimate of this round's sample count (it only sizes the launches)
		const uint32_t est = est_samples < 1u ? 1u : (est_samples > n ? n : est_samples);
		const uint32_t est_tiles = (est + FG_BLOCK - 1) / FG_BLOCK;
		field_gather_list_kernel<<<dim3(n2_xcd_blocks(a.n_levels, est_tiles) + (a.frags && round == 0 ? FRAG_BLOCKS : 0u)), dim3(FG_BLOCK), 0, s>>>(a, est_tiles);
		N2_LAUNCH_CHECK();
		// (two workgroups per CU, as many as run at a time: a workgroup's start copies 40 KiB of fragments.  Up to 2048 of one tile per
		// wave: the first round of a trained step 47 us instead of 38, the step 544 instead of 533; 768 and 1024: 541)
		field_fused_forward_kernel<true, false><<<dim3(fused_grid(est)), dim3(FF_BLOCK), fused_lds(FF_COUNT, true), s>>>(a);
		N2_LAUNCH_CHECK();
		return N2_OK;
	}
	{
		N2ProfScope prof(N2_PROF_FIELD_GATHER, s);
		launch_gather<true>(a, s);
	}
	N2_LAUNCH_CHECK();
	field_fused_forward_kernel<true, false><<<dim3(fused_grid(n)), dim3(FF_BLOCK), fused_lds(FF_COUNT, true), s>>>(a);
	N2_LAUNCH_CHECK();
	return N2_OK;
}

int n2_fused_field_sdf(const N2FusedNets& nets, hipStream_t s, const float* d_xyz, uint32_t ps, uint32_t ds, uint32_t n, n2_half* d_out_soa,
                       float* d_row0, bool density, n2_half* sdf_in, uint32_t row0_n, void* scratch, uint64_t scratch_bytes) {
	FusedArgs a = fused_base(nets, n);
	a.pos = d_xyz; a.ps = ps; a.ds = ds;
	a.sdf_out = reinterpret_cast<hf*>(d_out_soa);
	a.row0 = d_row0;
	a.row0_n = row0_n < n ? row0_n : n;
	a.density = density ? 1 : 0;
	if (sdf_in == nullptr) {
		field_fused_forward_kernel<false, true><<<dim3(fused_grid(n)), dim3(FF_BLOCK), fused_lds(FF_SDF_COUNT), s>>>(a);
		N2_LAUNCH_CHECK();
		return N2_OK;
	}
	// points in no particular order: a sample-major walk would touch all tables at once, so the features are gathered level
	// by level into the network's input rows first
	if (n <= QUERY_ONE_LAUNCH_MAX) {
		field_query_kernel<<<dim3((n + FQ_POINTS - 1) / FQ_POINTS), dim3(FQ_BLOCK), 0, s>>>(a);
		N2_LAUNCH_CHECK();
		return N2_OK;
	}
	a.sdf_in = reinterpret_cast<hf*>(sdf_in);
	const N2LevelTable& tab = *nets.tab;
	const bool dense = tab.n_levels > FS_LEVELS &&  // (one level at least is gathered)
	                    tab.mode[0] == N2_LEVEL_DENSE && tab.mode[1] == N2_LEVEL_DENSE;
	const uint64_t lds = FF_SDF_COUNT * 1024ull + 4ull * ((uint64_t)tab.entries[0] + tab.entries[1]);
	if (n >= QUERY_STAGED_MIN && dense && lds <= FS_LDS_MAX) {
		a.first_level = FS_LEVELS;
		uint32_t blocks = 0;
		bool blocked = a.n_levels > FS_LEVELS + FB_LEVELS && n >= QUERY_BLOCKS_MIN;
		for (uint32_t l = 0; l < FB_LEVELS && blocked; ++l) {
			blocked = tab.mode[FS_LEVELS + l] == N2_LEVEL_DENSE;
			a.block_first[l] = blocks;
			blocks += (n2_block_count(tab.resolution[FS_LEVELS + l]) + FG_BLOCK - 1) / FG_BLOCK * FG_BLOCK;
		}
		blocked = blocked && sizeof(N2Block) * (uint64_t)blocks <= scratch_bytes;
		if (blocked) {
			a.first_level += FB_LEVELS;
			a.blocks = reinterpret_cast<N2Block*>(scratch);
			a.n_blocks = blocks;
		}
		FusedArgs others = a;
		others.n_levels -= a.first_level;
		launch_gather<false>(others, s);
		N2_LAUNCH_CHECK();
		auto* const kernel = !blocked ? field_staged_forward_kernel<false, false> : n >= QUERY_STREAM_MIN && n2_rows_of_whole_lines(n, 4u) ? field_staged_forward_kernel<true, true> : field_staged_forward_kernel<true, false>;
		N2_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)FS_LDS_MAX));
		kernel<<<dim3(FS_GRID), dim3(FS_BLOCK), lds, s>>>(a);
		N2_LAUNCH_CHECK();
		return N2_OK;
	}
	launch_gather<false>(a, s);
	N2_LAUNCH_CHECK();
	// (bound by the latency of its loads at few registers: four workgroups per CU for large batches, where 512 | 1024 | 2048 of them
	// take 28.8 | 26.8 | 31 us for 2^20 points and 45.8 | 38.2 | 41.6 for 2^21; every workgroup builds the fragments, which
	// costs smaller batches more than it gains: 2^17 to 2^19 points 0.5 to 1.4 us)
	field_fused_forward_kernel<false, false><<<dim3(fused_grid(n, n >= (1u << 20) ? 1024u : 512u)), dim3(FF_BLOCK), fused_lds(FF_SDF_COUNT), s>>>(a);
	N2_LAUNCH_CHECK();
	return N2_OK;
}

uint32_t n2_fused_sdf_eikonal_parts(uint32_t n) { return fused_grid(n); }
int n2_fused_sdf_eikonal(hipStream_t s, const n2_half* weights, uint32_t n, const n2_half* input, const float* dy_dx, n2_half* output, n2_half* dsdf, float* normal,
                         float ek_weight, float scale, n2_half* dL_dy, float* v, n2_half* v_in, float* parts) {
	N2_REQUIRE(n2_sdf_one_pass(n), "n2_fused_sdf_eikonal: %u points are beyond the lanes' 32-bit offsets", n);
	SdfEikonalArgs a{};
	a.weights = reinterpret_cast<const hf*>(weights);
	a.N = n;
	a.input = reinterpret_cast<const hf*>(input);
	a.dy_dx = dy_dx;
	a.output = reinterpret_cast<hf*>(output);
	a.dsdf = reinterpret_cast<hf*>(dsdf);
	a.normal = normal;
	a.ek_weight = ek_weight;
	a.scale = scale;
	a.dL_dy = reinterpret_cast<hf*>(dL_dy);
	a.v = v;
	a.v_in = reinterpret_cast<hf*>(v_in);
	a.parts = parts;
	if (n2_step_jacobian_loads_stream(n, 32u)) sdf_eikonal_forward_kernel<true><<<dim3(fused_grid(n)), dim3(FF_BLOCK), 0, s>>>(a);
	else sdf_eikonal_forward_kernel<false><<<dim3(fused_grid(n)), dim3(FF_BLOCK), 0, s>>>(a);
	N2_LAUNCH_CHECK();
	return N2_OK;
}
