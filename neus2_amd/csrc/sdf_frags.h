// Weight fragments of the SDF network's forward for kernels that form its input themselves: the encoding's features as rows
// 0..31 (row 2 l + f for feature f of level l), the three centred coordinates as rows 32..34.
#pragma once
#include "mlp_device.h"

enum : int {
	SDF_FRAG_W0 = 0,  // [mt][c]  W_0 rows 32 mt + n; c = 0, 1: feature rows in chained order, c = 2: centred coordinates
	SDF_FRAG_WO = 6,  // [c]      W_out rows n < 16, chained K
	SDF_FRAG_COUNT = 10
};

// internal input row of the SDF net -> column of W_0 (or -1): rows 0..31 are features, 32..34 the coordinates
__device__ __forceinline__ int sdf_col(int row, uint32_t enc_w) {
	if (row < 32) return (uint32_t)row < enc_w ? 3 + row : -1;
	return row < 35 ? row - 32 : -1;
}
__device__ __forceinline__ int chained_k(int c, int g, int e) { return 16 * c + 4 * g + (e & 3) + ((e >> 2) << 3); }
__device__ __forceinline__ hf h_or_zero(const hf* W, bool ok, size_t at) { return ok ? W[at] : (hf)0; }

// lane l's 16 bytes of fragment f < SDF_FRAG_COUNT; ld: columns of W_0
__device__ __forceinline__ half8 sdf_forward_frag(const hf* W, int ld, uint32_t enc_w, int f, int l) {
	const int n = l & 31, g = l >> 5;
	half8 v = zero8();
	if (f < SDF_FRAG_WO) {
		const int mt = f / 3, c = f % 3, row = 32 * mt + n;
#pragma unroll
		for (int e = 0; e < 8; ++e) {
			const int col = c < 2 ? sdf_col(chained_k(c, g, e), enc_w) : sdf_col(32 + 8 * g + e, enc_w);
			v[e] = h_or_zero(W, col >= 0, (size_t)row * ld + (col >= 0 ? col : 0));
		}
	} else if (n < MLP_OUT) {
		v = wfrag_chained(W + MLP_WIDTH * ld, MLP_WIDTH, n, f - SDF_FRAG_WO, g);
	}
	return v;
}
