// Backward pass of the fully fused 64-wide MLP WITH weight gradients (and, for one hidden layer, the second-order pass
// riding along): every wave runs the forward and the data-gradient chain for tiles of 32 samples of its own and adds the
// tile's part of the batch reductions dW = dh h^T to accumulators of its own; the waves meet once, at the end, to add up.
//
// The chain produces matrices in sample-lane form (lane = sample, registers = rows); a product over samples needs
// them in row-lane form (lane = row, registers = 8 samples), for both operands.  They change form through a staging
// buffer of the wave's own in LDS, laid out as quads, S[quad q][sample s] = rows 4q .. 4q+3 of sample s (8 bytes): a lane
// writes the rows it holds with 8-byte stores, and ds_read_b64_tr_b16 hands a row-lane its samples: in every group of 16
// lanes, lane i receives as element j the (i % 4)-th 16-bit value of what lane i / 4 + 4 j of the group addressed.  With
// lane a + 4 j' of a group addressing quad qb + a of sample k + j', lane i gets row 4 qb + i for the samples k .. k+3: two
// such reads are one operand of v_mfma_f32_16x16x32_f16 (16 rows x 32 samples).  Which samples a lane holds where does not
// matter as long as both operands agree: group G takes samples 16 (G & 1) + 4 (G >> 1) + {0..3, 8..11}, so that with quad
// rows of 32 x 8 + 32 bytes the four quads of two groups fall on different banks.
//
// Stages (a stage = write, read back, products; the LDS runs a wave's accesses in their order, so no barrier and no second
// buffer), two hidden layers:  {dy, h1} -> dW_out, {dh1, h0} -> dW_1, {dh0, x} -> dW_0; one hidden layer with the second-order
// pass:  {dy, h} -> dW_out, {g, a} -> dW_out, {dh, x} -> dW_0, {b, v} -> dW_0.
// A wave holds all tiles of the weight gradients: 16 x 16 tiles have no padding, 128 accumulator registers for 48 -> 64 -> 64 -> 16,
// which leaves the chain 128 at two waves per SIMD.  (The tiles dealt to the four waves of a workgroup, 48 accumulator
// registers, takes eight barriers for every 128 samples: at 2^18 samples 36.5 us for that network and 32.8 for 48 -> 64 -> 16 with the
// second-order pass, now 35.4 and 27.5; a trained step's 44.5 and 36.6, now 40.7 and 32.7; both at 52344 samples 28 -> 25.5, and at 16 384, with the
// weights' copies under way together, 22 -> 18.)
#pragma once
#include "grid_device.h"
#include "mlp_device.h"

#include <type_traits>

constexpr int WG_QP = 32 * 8 + 32;      // bytes per quad row of a wave's staging buffer
constexpr int WG_STAGE = 32 * WG_QP;    // a wave's staging buffer: two matrices of 64 rows

typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

// staging writes: v holds 8 rows of the lane's sample; `at` = S + quad offset of the rows' block + the lane's part
// natural row order (rows 8 g + e of a 16-row chunk):  lane part = s * 8 + 2 g * WG_QP, quads q, q + 1
__device__ __forceinline__ void stage_natural(unsigned char* at, const half8& v) {
	const uint4v w = __builtin_bit_cast(uint4v, v);
	*reinterpret_cast<uint2*>(at) = make_uint2(w[0], w[1]);
	*reinterpret_cast<uint2*>(at + WG_QP) = make_uint2(w[2], w[3]);
}
// chained row order (rows 4 g + 0..3 and 8 + 4 g + 0..3 of a 16-row chunk):  lane part = s * 8 + g * WG_QP, quads q, q + 2
__device__ __forceinline__ void stage_chained(unsigned char* at, const half8& v) {
	const uint4v w = __builtin_bit_cast(uint4v, v);
	*reinterpret_cast<uint2*>(at) = make_uint2(w[0], w[1]);
	*reinterpret_cast<uint2*>(at + 2 * WG_QP) = make_uint2(w[2], w[3]);
}
// row-lane MFMA operand: rows 16 c .. 16 c + 15, the 32 samples; tr = S + the lane's part
// (l & 3) * WG_QP + (16 (G & 1) + 4 (G >> 1) + ((l & 15) >> 2)) * 8, G = l / 16
__device__ __forceinline__ half8 row_operand(const unsigned char* tr, int c) {
	const unsigned char* p = tr + 4 * c * WG_QP;
	const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(p));
	const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(p + 64));
	const short8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
	return __builtin_bit_cast(half8, v);
}
// Between a wave's writes to its staging buffer and its reads, and the reads and the next writes: the LDS keeps them in
// order, this keeps the compiler from changing it.
__device__ __forceinline__ void stage_order() {
	asm volatile("" ::: "memory");
	__builtin_amdgcn_sched_barrier(0);
}
// acc[AT + i * NB + j] += A_i B_j^T: A = the 16 NA rows from chunk ca of the staging buffer, B = the 16 NB rows from chunk cb
template <int AT, int NA, int NB, int T>
__device__ __forceinline__ void wgrad_tiles(const unsigned char* tr, int ca, int cb, float4v (&acc)[T]) {
	static_assert(AT + NA * NB <= T, "tiles of the network");
	half8 b[NB];
#pragma unroll
	for (int j = 0; j < NB; ++j) b[j] = row_operand(tr, cb + j);
#pragma unroll
	for (int i = 0; i < NA; ++i) {
		const half8 a = row_operand(tr, ca + i);
#pragma unroll
		for (int j = 0; j < NB; ++j) acc[AT + i * NB + j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[j], acc[AT + i * NB + j], 0, 0, 0);
	}
}

// input operands (natural K order) of one 32-sample tile; column `col` of a matrix with n_cols columns
template <int IC>
__device__ __forceinline__ void load_tile_rows(const hf* __restrict__ X, uint32_t n_cols, uint32_t col, int g, half8 (&x)[IC]) {
	const uint32_t b = (8u * g * n_cols + col) * 2u;
#pragma unroll
	for (int c = 0; c < IC; ++c)
#pragma unroll
		for (int e = 0; e < 8; ++e) x[c][e] = *reinterpret_cast<const hf*>(reinterpret_cast<const char*>(X + (size_t)(16 * c + e) * n_cols) + b);
}

// Which rows of dL/dinput a launch stores: all of them, or only those its caller reads (rows that differ between the two
// halves of a wave turn into a predicate on the half, rows nobody reads cost no instruction)
enum : int {
	WG_DX_NONE = 0,
	WG_DX_ALL = 1,
	WG_DX_OUT_AND_NORMAL = 2,  // rows 0..15 and 35..37: the field's colour net (gradient of the SDF net's output and of the normal)
	WG_DX_ENCODING = 3         // rows 3..34: the field's SDF net over up to 16 levels (gradient of the encoding; positions are not optimised)
};
__device__ __forceinline__ constexpr bool wg_dx_row(int mode, int row, int in_w) {
	return row < in_w && (mode == WG_DX_ALL || (mode == WG_DX_OUT_AND_NORMAL && (row < 16 || (row >= 35 && row < 38))) ||
	                      (mode == WG_DX_ENCODING && row >= 3 && row < 35));
}

// A tail: work on the same samples that rides along with a launch.  The field hangs the preparation of its SDF net's
// backward on the colour net's kernel (N2FieldPrepTail, n2_common.h): that work streams 256 bytes of slopes per sample, and
// inside this kernel, whose waves wait for barriers and matrix results half of their time, it costs less than as a launch
// of its own between the two networks' kernels.
struct WgNoTail {
	static constexpr bool active = false;
};
// With the tail, the launch also takes the field's layouts: X holds a column's first N2_RGB_IN_PITCH values side by side
// (column c at X + N2_RGB_IN_PITCH c), and rows 0..15 of dL/dinput are written the same way (16 values per column, dX + 16 c); nothing else of
// dL/dinput is stored.
struct WgFieldPrepTail {
	static constexpr bool active = true;
	N2FieldPrepTail a;
};

// the 16 x 16 tiles of the weight gradients: W_0 (4 x IC), W_1 (4 x 4, two hidden layers), W_out (1 x 4), row by row
template <int IC, int NH>
struct WgTiles {
	static constexpr int WH = 4 * IC, WO = WH + (NH - 1) * 16, COUNT = WO + 4;
};
// dynamic LDS of the kernel: fragments, then the waves' staging buffers
template <int WAVES, int IC, int NH>
constexpr size_t mlp_wgrad_lds() {
	return (size_t)FragMap<IC, NH>::SEL * 1024 + (size_t)WAVES * WG_STAGE;
}
// At the end the waves exchange their tiles through LDS in columns of four (a column of 16 of W_0 or W_1, the whole of W_out), as many at a
// time as fit it (a column of every wave: WAVES * 4 KiB), and wave w adds up tile w % 4 of every column (of every second one, where there are eight).
template <int WAVES, int IC, int NH>
struct WgFold {
	static constexpr int COLS = WgTiles<IC, NH>::COUNT / 4, FIT = (int)(mlp_wgrad_lds<WAVES, IC, NH>() - 64) / (WAVES * 4096);
	static constexpr int PASSES = (COLS + FIT - 1) / FIT, PER = (COLS + PASSES - 1) / PASSES;
	static_assert(FIT >= 1 && WAVES * PER * 4096 + 64 <= mlp_wgrad_lds<WAVES, IC, NH>(), "a pass, and a value of every wave behind it, fit");
	// place of tile t of column c among the accumulators
	static constexpr int tile(int c, int t) {
		using T = WgTiles<IC, NH>;
		return c < IC ? t * IC + c : c < COLS - 1 ? T::WH + t * 4 + (c - IC) : T::WO + t;
	}
};

template <int WAVES, int IC, int NH, int WANT_DX, bool SECOND, bool DY_AOS, class Tail = WgNoTail>
__global__ void __launch_bounds__(64 * WAVES, 8 / WAVES) mlp_wgrad_kernel(const hf* __restrict__ W, const hf* __restrict__ X, uint32_t N, const hf* __restrict__ dY,
                                                                 int dy_rows, hf* __restrict__ dX, float* __restrict__ partials,
                                                                 const hf* __restrict__ V, const hf* __restrict__ G2, int unit_row2,
                                                                 const uint32_t* __restrict__ x_index, uint32_t x_cols, float dy_gain, float dy_gain_inv,
                                                                 const hf* __restrict__ frag_image, const Tail tail = Tail()) {
	static_assert(!SECOND || NH == 1, "the second-order pass needs one hidden layer");
	static_assert(!Tail::active || (IC == 3 && NH == 2 && WANT_DX == WG_DX_OUT_AND_NORMAL && DY_AOS), "the field's tail goes with the colour net");
	// dy_gain = 2^k, dy_gain_inv = 2^-k (first-order launches only).  The output gradient is multiplied by 2^k when it is
	// loaded and everything the launch hands on (dL/dinput, the weight-gradient slab) by 2^-k in fp32, so the chain between
	// them, whose matrices are rounded to fp16 for the matrix cores, works on values 2^k larger: an output gradient in the
	// subnormal range of fp16 (a loss scale of 128 over thousands of rays puts the colour rows there: steps of 6e-8 on values
	// near 2e-6) then loses nothing, the products with a power of two being exact.  2^0 leaves every value as it is.
	const float gain_inv = SECOND ? 1.f : dy_gain_inv;
	using M = FragMap<IC, NH>;
	using T = WgTiles<IC, NH>;
	using Fold = WgFold<WAVES, IC, NH>;
	constexpr uint32_t ROUND = 32 * WAVES;  // samples of a workgroup's round
	constexpr int IN_W = 16 * IC, IN_MT = M::IN_MT;
	constexpr int N_PARAMS = mlp_n_params<IC, NH>();
	static_assert(2 * N_PARAMS <= WAVES * WG_STAGE, "the weights fit where the staging buffers are");
	extern __shared__ __align__(16) unsigned char smem[];
	hf* F = reinterpret_cast<hf*>(smem);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 31;
	const uint32_t s_local = 32u * wave + n;
	unsigned char* const S = smem + (size_t)M::SEL * 1024 + wave * WG_STAGE;  // the wave's staging buffer behind the fragments
	unsigned char* const st_nat = S + n * 8 + 2 * (lane >> 5) * WG_QP;
	unsigned char* const st_ch = S + n * 8 + (lane >> 5) * WG_QP;
	const int G = lane >> 4;
	const unsigned char* const tr = S + (lane & 3) * WG_QP + (16 * (G & 1) + 4 * (G >> 1) + ((lane & 15) >> 2)) * 8;
	float4v acc[T::COUNT];
#pragma unroll
	for (auto& t : acc) t = float4v{0.f, 0.f, 0.f, 0.f};
	float var_acc = 0.f;  // tail: this lane's part of the variance gradient
	const uint32_t n_rounds = (N + ROUND - 1) / ROUND;
	// A round's operands are loaded while the round before it works: x and dy once its own are staged, the index they go by (a
	// sample's column in X) before that.  A round has the arithmetic of 6 k cycles and two waves share a SIMD: waiting for
	// three loads one behind the other, it took 21 k.
	// (Nothing here may sit in a branch: its join would wait for all loads.  Without an index its load takes a word of X, which has one for each column.)
	const uint32_t* const index = x_index ? x_index : reinterpret_cast<const uint32_t*>(X);
	auto column = [&](uint32_t round) { return min(round * ROUND + s_local, N - 1u); };
	half8 x[IC], dy;
	auto load = [&](uint32_t col, uint32_t src, int g) __attribute__((always_inline)) {
		const uint32_t col_src = x_index ? min(src, x_cols - 1u) : col;
		if constexpr (Tail::active) {
			// the field keeps the colour net's input sample-major (N2_RGB_IN_PITCH values per column, the rows behind them
			// are the padding's zeros): an operand is one 16-byte load
			const hf* const at = X + (size_t)col_src * N2_RGB_IN_PITCH;
#pragma unroll
			for (int c = 0; c < IC; ++c) x[c] = *reinterpret_cast<const half8*>(at + (16 * c + 8 * g < (int)N2_RGB_IN_PITCH ? 16 * c + 8 * g : 0));
		} else {
			load_tile_rows<IC>(X, x_index ? x_cols : N, col_src, g, x);
		}
		if constexpr (DY_AOS) {
			dy = *reinterpret_cast<const half8*>(dY + (size_t)col * MLP_OUT + 8 * g);
		} else {
#pragma unroll
			for (int e = 0; e < 8; ++e) dy[e] = dY[(size_t)(8 * g + e) * N + col];
		}
		return col_src;
	};
	// Awaits the next round's operands (and all loads before them) in front of a round's stores: behind a branch round a store,
	// a wait for a load becomes one for the store as well.
	auto arrived = [&]() __attribute__((always_inline)) {
#pragma unroll
		for (int c = 0; c < IC; ++c) asm volatile("" : "+v"(x[c]));
		asm volatile("" : "+v"(dy));
	};
	const uint32_t col0 = column(blockIdx.x);
	uint32_t col_src = load(col0, index[col0], lane >> 5);
	// (frag_image: the fragments as a launch in front of this one has left them in global memory, M::SEL KiB; null: built here)
	if (frag_image) load_frags<M::SEL, 64 * WAVES>(F, frag_image);
	else build_frags_staged<IC, NH, 64 * WAVES>(F, F + M::SEL * 512, W, M::SEL);
	for (uint32_t round = blockIdx.x; round < n_rounds; round += gridDim.x) {
		int g = lane >> 5;
		asm volatile("" : "+v"(g));  // addresses that depend on it are formed anew in every round: kept, they take 40 registers
		const bool valid = round * ROUND + s_local < N, more = round + gridDim.x < n_rounds;
		const uint32_t col = column(round), next_col = column(min(round + gridDim.x, n_rounds - 1u));
		const uint32_t off4 = (4u * g * N + col) * 2u;  // of the column's value in row 4 g (N <= 2^28)
		const uint32_t next_src = index[next_col];
		half8 v[SECOND ? IC : 1];
		if constexpr (SECOND) load_tile_rows<IC>(V, N, col, g, v);
		// ---- the chain of this wave's 32 samples ----
		half8 h[NH][4];
		if constexpr (Tail::active) {
#pragma unroll
			for (int c = 0; c < IC; ++c)
				if (16 * c + 8 * g >= (int)N2_RGB_IN_PITCH) x[c] = zero8();
		}
		const half8 dy_all = dy;  // tail: all 16 rows of the output gradient
#pragma unroll
		for (int e = 0; e < 8; ++e)
			if (!valid || 8 * g + e >= dy_rows) dy[e] = (hf)0;
		if constexpr (!SECOND) {
			const hf gain = (hf)dy_gain;
#pragma unroll
			for (int e = 0; e < 8; ++e) dy[e] = dy[e] * gain;
		}
		hidden_S<IC, NH>(F, lane, x, h);
		// ---- dW_out = dy h_last^T: chunks dy 0 | h_last 1..4 ----
		stage_order();
		stage_natural(st_nat, dy);
#pragma unroll
		for (int c = 0; c < 4; ++c) stage_chained(st_ch + 4 * (1 + c) * WG_QP, h[NH - 1][c]);
		stage_order();
		wgrad_tiles<T::WO, 1, 4>(tr, 0, 1, acc);
		half8 dh[NH][4];
#pragma unroll
		for (int t = 0; t < 2; ++t)
			mask_pack(N2_MFMA(frag(F, M::WOT + t, lane), dy, zero16()), h[NH - 1][2 * t], h[NH - 1][2 * t + 1], dh[NH - 1][2 * t], dh[NH - 1][2 * t + 1]);
		// ---- hidden matrix: dW_1 = dh_1 h_0^T: chunks dh_1 0..3 | h_0 4..7 ----
		if constexpr (NH > 1) {
			static_assert(NH <= 2, "one hidden matrix");
			stage_order();
#pragma unroll
			for (int c = 0; c < 4; ++c) {
				stage_chained(st_ch + 4 * c * WG_QP, dh[1][c]);
				stage_chained(st_ch + 4 * (4 + c) * WG_QP, h[0][c]);
			}
			stage_order();
			wgrad_tiles<T::WH, 4, 4>(tr, 0, 4, acc);
#pragma unroll
			for (int t = 0; t < 2; ++t) {
				float16v a = zero16();
#pragma unroll
				for (int c = 0; c < 4; ++c) a = N2_MFMA(frag(F, M::WHT + t * 4 + c, lane), dh[1][c], a);
				mask_pack(a, h[0][2 * t], h[0][2 * t + 1], dh[0][2 * t], dh[0][2 * t + 1]);
			}
		}
		// ---- first matrix: dW_0 = dh_0 x^T: chunks dh_0 0..3 | x 4.. ----
		stage_order();
#pragma unroll
		for (int c = 0; c < 4; ++c) stage_chained(st_ch + 4 * c * WG_QP, dh[0][c]);
#pragma unroll
		for (int c = 0; c < IC; ++c) stage_natural(st_nat + 4 * (4 + c) * WG_QP, x[c]);
		stage_order();
		uint4 sl[Tail::active ? 8 : 1];
		if constexpr (Tail::active) {
			// the slopes of this lane's 8 levels (level 4 (j / 2) + 2 g + j % 2): their last use, past the caches.  At any size: a row of a batch, which is a multiple of 8 samples of 16
			// bytes, starts a line, and so does a tile's part of it; where a selection picks the columns two tiles may meet a line, which shows in no time.  In us, cached | streamed: the field's
			// forward and backward 2^18 245.4 | 239.2, 262 136 245.3 | 243.6, 150 008 165.2 | 164.8, 100 008 125.3 | 125.4, 52 344 88.9 | 87.7; training step 2^18 339.3 | 336.5, 100 096 216.0 | 216.4;
			// with columns picked (trained) 2^18 494.2 | 491.8, 100 096 289.3 | 289.5, 59 904 225.3 | 224.5, 29 952 170.6 | 170.1.
			const uint4* const at = reinterpret_cast<const uint4*>(tail.a.slopes) + (size_t)(4u * g < tail.a.enc_w ? 2u * g : 0u) * tail.a.n_src + col_src;
#pragma unroll
			for (int j = 0; j < 8; ++j) {
				const uint32_t level = 4u * (j >> 1) + (j & 1);  // + 2 g
				sl[j] = n2_stream_load(at + (size_t)(2u * (level + 2u * g) < tail.a.enc_w ? level : 0u) * tail.a.n_src);
			}
		}
		const uint32_t next_col_src = load(next_col, next_src, g);
		wgrad_tiles<0, 4, IC>(tr, 0, 4, acc);
		if constexpr (SECOND) {
			if (!valid) {
#pragma unroll
				for (int c = 0; c < IC; ++c) v[c] = zero8();
			}
			// a = m * (W_0 v),  b = m * (W_out^T g); m = the sign of the hidden layer.  dW_out += g a^T, dW_0 += b v^T
			half8 s2[4];
#pragma unroll
			for (int t = 0; t < 2; ++t) {
				float16v a = zero16();
#pragma unroll
				for (int c = 0; c < IC; ++c) a = N2_MFMA(frag(F, M::W0 + t * IC + c, lane), v[c], a);
				mask_pack(a, h[0][2 * t], h[0][2 * t + 1], s2[2 * t], s2[2 * t + 1]);
			}
			half8 gg;
			if (unit_row2 >= 0) {
#pragma unroll
				for (int e = 0; e < 8; ++e) gg[e] = (8 * g + e == unit_row2) ? (hf)1 : (hf)0;
			} else {
#pragma unroll
				for (int e = 0; e < 8; ++e) gg[e] = G2[(size_t)(8 * g + e) * N + col];
			}
			if (!valid) gg = zero8();
			stage_order();
			stage_natural(st_nat, gg);
#pragma unroll
			for (int c = 0; c < 4; ++c) stage_chained(st_ch + 4 * (1 + c) * WG_QP, s2[c]);
			stage_order();
			wgrad_tiles<T::WO, 1, 4>(tr, 0, 1, acc);
#pragma unroll
			for (int t = 0; t < 2; ++t)
				mask_pack(N2_MFMA(frag(F, M::WOT + t, lane), gg, zero16()), h[0][2 * t], h[0][2 * t + 1], s2[2 * t], s2[2 * t + 1]);
			stage_order();
#pragma unroll
			for (int c = 0; c < 4; ++c) stage_chained(st_ch + 4 * c * WG_QP, s2[c]);
#pragma unroll
			for (int c = 0; c < IC; ++c) stage_natural(st_nat + 4 * (4 + c) * WG_QP, v[c]);
			stage_order();
			wgrad_tiles<0, 4, IC>(tr, 0, 4, acc);
		}
		stage_order();
		half4v out_lo, out_hi;
		hf dn[2] = {(hf)0, (hf)0};  // tail: g = 0: row 35; g = 1: rows 36, 37 of dL/dinput
		if (WANT_DX != WG_DX_NONE) {
#pragma unroll
			for (int t = 0; t < IN_MT; ++t) {
				float16v d = zero16();
#pragma unroll
				for (int c = 0; c < 4; ++c) d = N2_MFMA(frag(F, M::W0T + t * 4 + c, lane), dh[0][c], d);
#pragma unroll
				for (int r = 0; r < 16; ++r) d[r] *= gain_inv;
				if constexpr (Tail::active) {
					// row 0 also takes the direct gradient of the SDF output (row 3 of dL/doutput); rows 35..37 are dL/dnormal
					if (t == 0 && g == 0) d[0] = (float)((hf)d[0] + dy_all[3]);
					if (t == 1) { dn[0] = (hf)(g == 0 ? d[3] : d[0]); dn[1] = (hf)d[1]; }
					// rows 0..15 go out sample-major (16 values per column, the SDF net's output gradient): the lane holds
					// rows 4 g .. 4 g + 3 and 8 + 4 g .. 8 + 4 g + 3; rows 35..37 stay in registers (dn)
					if (t == 0) {
						out_lo = half4v{(hf)d[0], (hf)d[1], (hf)d[2], (hf)d[3]};
						out_hi = half4v{(hf)d[4], (hf)d[5], (hf)d[6], (hf)d[7]};
					}
				}
				if (t == 0 && !Tail::active && more) arrived();
				if (!Tail::active && valid) {
#pragma unroll
					for (int r = 0; r < 16; ++r) {
						const int row = 32 * t + 8 * (r >> 2) + (r & 3);  // + 4 g
						const bool lo = wg_dx_row(WANT_DX, row, IN_W), hi = wg_dx_row(WANT_DX, row + 4, IN_W);
						// (row + 4 g; a uniform base and the lane's offset, whose 64-bit sums would be kept for all rows from round to round)
						hf* const o = reinterpret_cast<hf*>(reinterpret_cast<char*>(dX + (size_t)row * N) + off4);
						if (lo && hi) *o = (hf)d[r];
						else if (lo) { if (g == 0) *o = (hf)d[r]; }
						else if (hi) { if (g == 1) *o = (hf)d[r]; }
					}
				}
			}
		}
		if constexpr (Tail::active) {
			// dL/dnormal = row 35..37 of dL/dinput + rows 4..6 of dL/doutput / ek_batch + rows 8..10 of dL/doutput; its pieces
			// sit in the two halves of the wave: g = 0 holds dn[0] and rows 4..6, g = 1 holds dn[0..1] (rows 36, 37) and rows 8..10
			auto pk = [](hf a, hf b) { return (uint32_t)__builtin_bit_cast(unsigned short, a) | ((uint32_t)__builtin_bit_cast(unsigned short, b) << 16); };
			auto lo16 = [](uint32_t w) { return (float)__builtin_bit_cast(hf, (unsigned short)(w & 0xFFFFu)); };
			auto hi16 = [](uint32_t w) { return (float)__builtin_bit_cast(hf, (unsigned short)(w >> 16)); };
			const uint32_t m0 = g == 0 ? pk(dn[0], dy_all[4]) : pk(dn[0], dn[1]);
			const uint32_t m1 = g == 0 ? pk(dy_all[5], dy_all[6]) : pk(dy_all[0], dy_all[1]);
			const uint32_t m2 = g == 0 ? 0u : pk(dy_all[2], (hf)0);
			const uint32_t o0 = (uint32_t)__shfl_xor((int)m0, 32), o1 = (uint32_t)__shfl_xor((int)m1, 32), o2 = (uint32_t)__shfl_xor((int)m2, 32);
			const uint32_t a0 = g == 0 ? m0 : o0, a1 = g == 0 ? m1 : o1;             // what the lower half holds
			const uint32_t b0 = g == 0 ? o0 : m0, b1 = g == 0 ? o1 : m1, b2 = g == 0 ? o2 : m2;  // what the upper half holds
#pragma unroll
			for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(sl[j].x), "+v"(sl[j].y), "+v"(sl[j].z), "+v"(sl[j].w));
			if (more) arrived();
			float vv[3] = {lo16(a0), lo16(b0), hi16(b0)};
			const float r4[3] = {hi16(a0), lo16(a1), hi16(a1)}, r8[3] = {lo16(b1), hi16(b1), lo16(b2)};
#pragma unroll
			for (int d = 0; d < 3; ++d) {
				vv[d] += r4[d] / tail.a.ek_batch;
				vv[d] += r8[d];
			}
			if (valid) {
				hf* const o = dX + (size_t)col * MLP_OUT + 4 * g;
				*reinterpret_cast<half4v*>(o) = out_lo;
				*reinterpret_cast<half4v*>(o + 8) = out_hi;
				if (g == 0) {
					var_acc += (float)dy_all[7];
#pragma unroll
					for (int d = 0; d < 3; ++d) {
						tail.a.v[(size_t)d * N + col] = vv[d];
						reinterpret_cast<hf*>(tail.a.d_density_in)[(size_t)d * N + col] = (hf)vv[d];
					}
				}
				// rows 3.. of the SDF net's second-order input: the encoding's dL_ddLdoutput = J v
#pragma unroll
				for (int j = 0; j < 8; ++j) {
					const uint32_t level = 4u * (j >> 1) + (j & 1);  // + 2 g
					float m[6];
					float scale0 = tail.a.scale[level], scale2 = tail.a.scale[level + 2u];
					asm("" : "+s"(scale0), "+s"(scale2));  // (the compiler would choose the address and load per lane)
					const float unit = n2_slopes_unpack(sl[j], m) * (g == 0 ? scale0 : scale2);
					hf f0 = (hf)((m[0] * vv[0] + m[1] * vv[1] + m[2] * vv[2]) * unit), f1 = (hf)((m[3] * vv[0] + m[4] * vv[1] + m[5] * vv[2]) * unit);
					asm volatile("" : "+v"(f0), "+v"(f1));  // (formed outside the condition, which then takes no branch)
					char* const rows = reinterpret_cast<char*>(reinterpret_cast<hf*>(tail.a.d_density_in) + (size_t)(3 + 2 * level) * N);
					if (2u * (level + 2u * g) < tail.a.enc_w) {
						*reinterpret_cast<hf*>(rows + off4) = f0;
						*reinterpret_cast<hf*>(rows + 2 * (size_t)N + off4) = f1;
					}
				}
			}
		}
		col_src = next_col_src;
	}
	// ---- the workgroup's slab: the sum over its waves, a share of the tiles by each ----
	constexpr int OFF_H = MLP_WIDTH * IN_W, OFF_O = OFF_H + (NH - 1) * MLP_WIDTH * MLP_WIDTH;
	float4v* const Wl = reinterpret_cast<float4v*>(smem);
	float* const slab = partials + (size_t)blockIdx.x * N_PARAMS;
	const int w_fold = __builtin_amdgcn_readfirstlane(wave), t_fold = w_fold & 3, row = 4 * (lane >> 4), col = lane & 15;
	float* const at_0 = slab + (16 * t_fold + row) * IN_W + col;
	float* const at_h = slab + OFF_H + (16 * t_fold + row) * MLP_WIDTH + col;
	float* const at_o = slab + OFF_O + row * MLP_WIDTH + 16 * t_fold + col;
	float* const var = reinterpret_cast<float*>(smem + WAVES * Fold::PER * 4096);
	if constexpr (Tail::active) {
		// the workgroup's part of the variance gradient (row 7 of dL/doutput), summed in a fixed order
#pragma unroll
		for (int o = 32; o > 0; o >>= 1) var_acc += __shfl_xor(var_acc, o);
	}
#pragma unroll
	for (int c0 = 0; c0 < Fold::COLS; c0 += Fold::PER) {
		__syncthreads();  // every wave is done with the fragments and staging buffers, or the tiles, that these overlay
#pragma unroll
		for (int c = c0; c < c0 + Fold::PER && c < Fold::COLS; ++c)
#pragma unroll
			for (int t = 0; t < 4; ++t) Wl[((wave * Fold::PER + c - c0) * 4 + t) * 64 + lane] = acc[Fold::tile(c, t)];
		if (Tail::active && c0 == 0 && lane == 0) var[wave] = var_acc;
		__syncthreads();
#pragma unroll
		for (int c = c0; c < c0 + Fold::PER && c < Fold::COLS; ++c) {
			if (WAVES == 8 && (c & 1) != (w_fold >> 2)) continue;
			const float4v* const tiles = Wl + ((c - c0) * 4 + t_fold) * 64 + lane;
			float4v s = tiles[0];
#pragma unroll
			for (int w = 1; w < WAVES; ++w) s += tiles[w * Fold::PER * 256];
			float* const o = c < IC ? at_0 + 16 * c : c < Fold::COLS - 1 ? at_h + 16 * (c - IC) : at_o;
#pragma unroll
			for (int r = 0; r < 4; ++r) o[r * (c < IC ? IN_W : MLP_WIDTH)] = s[r] * gain_inv;
		}
		if constexpr (Tail::active) if (c0 == 0 && threadIdx.x == 0) {
			float sum = var[0];
#pragma unroll
			for (int w = 1; w < WAVES; ++w) sum += var[w];
			tail.a.var_part[blockIdx.x] = sum;
		}
	}
}
