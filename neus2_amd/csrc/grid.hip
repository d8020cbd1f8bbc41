// Multi-resolution hash grid encoding for gfx950: forward, backward
// (parameter scatter + input gradient) and the second-order
// backward_backward_input, behind the n2_grid_* C ABI.
//
// Work decomposition: one workgroup handles a tile of points for ONE level.
// The gather kernels deal whole levels to the XCDs (n2_gather_item), each of
// which then streams all points through about two levels and fetches only those
// levels' tables (<= 2 MiB each at T = 2^19) into its private 4 MiB L2 instead of
// all 24 MiB; with costs from n2_grid_set_level_costs they cut the level-major
// list of items into 8 contiguous pieces of equal estimated cost.
#include "n2_common.h"
#include "grid_device.h"
#include "slab_reduce.h"

#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>

struct n2_grid {
	N2LevelTable tab;
	uint32_t n_features;
	uint32_t n_params;
	const __half2* params;
	__half2* grads;
	// relative cost of one tile of each level (balances the levels over the XCDs)
	float level_cost[N2_MAX_LEVELS];
	bool costs_set;  // by n2_grid_set_level_costs
	// progressive training (base_training_step 0: off)
	float base_valid_level_scale, valid_level_scale;
	uint32_t base_training_step;
	uint32_t training_step;  // as last told by n2_grid_set_training_step
	// optional scratch of the bucketed scatter
	unsigned char* ws;
	uint64_t ws_bytes;
	uint32_t ws_max_points;
	uint64_t ws_partials;  // where the images of split buckets stand in it
	bool lattice_order;  // points of the next forwards come in lattice order (n2_grid_set_point_order)
};

struct N2Point {
	float w[3];
	uint32_t c[3];
};

__device__ __forceinline__ N2Point n2_load_point(const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                                 uint32_t i, float scale) {
	N2Point p;
	const float* q = xyz + (size_t)i * point_stride;
#pragma unroll
	for (int d = 0; d < 3; ++d) n2_locate(q[(size_t)d * dim_stride], scale, p.w[d], p.c[d]);
	return p;
}

template <uint32_t MODE>
__device__ __forceinline__ void n2_corner_entries(const N2Point& p, uint32_t entries, uint32_t res, uint32_t e[8]) {
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) {
		e[k] = n2_entry<MODE>(entries, res, p.c[0] + (k & 1u), p.c[1] + ((k >> 1) & 1u), p.c[2] + ((k >> 2) & 1u));
	}
}

__device__ __forceinline__ float n2_corner_weight(const N2Point& p, uint32_t k) {
	float wt = (k & 1u) ? p.w[0] : 1.f - p.w[0];
	wt *= (k & 2u) ? p.w[1] : 1.f - p.w[1];
	wt *= (k & 4u) ? p.w[2] : 1.f - p.w[2];
	return wt;
}

#define N2_DISPATCH_MODE(mode, CALL)                        \
	switch (mode) {                                         \
		case N2_LEVEL_DENSE: { CALL(N2_LEVEL_DENSE); } break;       \
		case N2_LEVEL_HASH: { CALL(N2_LEVEL_HASH); } break;         \
		case N2_LEVEL_DENSE_MOD: { CALL(N2_LEVEL_DENSE_MOD); } break; \
		default: { CALL(N2_LEVEL_HASH_MOD); } break;                \
	}

constexpr uint32_t GRID_BLOCK = 256;
constexpr uint32_t N_XCD = N2_XCDS;

// Piece x of the level-major item list [begin[x], begin[x + 1]) belongs to XCD x; begin[N_XCD] = 0: no plan, n2_gather_item deals
// the items (2^18 points with dy_dx, plain stores: 84 us uniform, 60 in ray order; with the plan of the default costs 101 and 74.  Streamed
// stores lengthen the uniform launch to 91 and shorten what follows it: n2_jacobian_streams).
struct N2XcdPlan {
	uint32_t begin[N_XCD + 1];
	uint32_t height;  // of a launch without a plan: its workgroups in y
};

// The (level, tile) item of this workgroup, or false if its XCD's piece is shorter than the longest one.
__device__ __forceinline__ bool n2_xcd_item(const N2XcdPlan& plan, uint32_t tiles, uint32_t& level, uint32_t& tile) {
	const uint32_t xcd = blockIdx.x % N_XCD, item = plan.begin[xcd] + blockIdx.x / N_XCD;
	if (item >= plan.begin[xcd + 1]) return false;
	level = item / tiles;
	tile = item - level * tiles;
	return true;
}

// ----------------------------------------------------------------------------
// forward
// ----------------------------------------------------------------------------
constexpr uint32_t FWD_POINTS = GRID_BLOCK;  // points per workgroup and level

template <uint32_t MODE, bool WANT_DYDX, bool STREAM>
__device__ __forceinline__ void grid_forward_item(const N2LevelTable& tab, uint32_t level, uint32_t i, uint32_t N,
                                                  const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                                  const __half2* __restrict__ params, __half* __restrict__ out,
                                                  float* __restrict__ dy_dx, __half* __restrict__ centred) {
	if (centred != nullptr && level == 0 && i < N) {
		const float* q = xyz + (size_t)i * point_stride;
#pragma unroll
		for (uint32_t d = 0; d < 3; ++d) centred[(size_t)d * N + i] = __float2half_rn(q[(size_t)d * dim_stride]) - __float2half_rn(0.5f);
	}
	const bool off = n2_level_masked(tab, level, min(i, N - 1u));
	float feat[2] = {0.f, 0.f}, J[2][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
	if (!__all(off)) {
		// (lanes behind the last point take part in its pair's exchange)
		const float* q = xyz + (size_t)min(i, N - 1u) * point_stride;
		const float p[3] = {n2_to_pairs(q[0]), n2_to_pairs(q[dim_stride]), n2_to_pairs(q[2 * (size_t)dim_stride])}, scale = tab.scale[level];
		n2_encode_level<MODE, WANT_DYDX>(reinterpret_cast<const char*>(params + tab.offset[level]), tab.entries[level], tab.resolution[level], scale, p, scale, feat, J);
#pragma unroll
		for (uint32_t f = 0; f < 2; ++f) {
			feat[f] = n2_from_pairs(feat[f]);
#pragma unroll
			for (uint32_t d = 0; d < 3; ++d)
				if (WANT_DYDX) J[f][d] = n2_from_pairs(J[f][d]);
		}
	}
	if (i >= N) return;
#pragma unroll
	for (uint32_t f = 0; f < 2; ++f) {
		const size_t row = (size_t)level * 2 + f;
		out[row * N + i] = __float2half_rn(off ? 0.f : feat[f]);
		if (WANT_DYDX) n2_store3<STREAM>(dy_dx + (row * N + i) * 3, off ? n2_float3{0.f, 0.f, 0.f} : n2_float3{J[f][0], J[f][1], J[f][2]});
	}
}

// STREAM: dy_dx is written past the last-level cache (n2_jacobian_streams).  centred (or null): three rows for the positions minus 0.5, the SDF network's first inputs
template <bool WANT_DYDX, bool STREAM>
__global__ void __launch_bounds__(GRID_BLOCK) grid_forward_kernel(N2LevelTable tab, N2XcdPlan plan, uint32_t N, uint32_t tiles,
                                                                  const float* __restrict__ xyz, uint32_t point_stride,
                                                                  uint32_t dim_stride, const __half2* __restrict__ params,
                                                                  __half* __restrict__ out, float* __restrict__ dy_dx,
                                                                  __half* __restrict__ centred) {
	uint32_t level, tile;
	if (!(plan.begin[N_XCD] ? n2_xcd_item(plan, tiles, level, tile) : n2_gather_item(blockIdx.x, blockIdx.y, plan.height, tab.n_levels, tiles, level, tile))) return;
	const uint32_t i = tile * FWD_POINTS + threadIdx.x;
#define CALL(M) grid_forward_item<M, WANT_DYDX, STREAM>(tab, level, i, N, xyz, point_stride, dim_stride, params, out, dy_dx, centred)
	N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
}

// One lane per (point, level): eight gathers and one fused multiply-add chain per feature.  For points that arrive
// in lattice order (neighbouring lanes in neighbouring cells) the gathers hit lines the wave has just fetched and
// the kernel is bound by instruction issue, where the lane pairs of the kernel above cost twice the lanes.
template <uint32_t MODE>
__device__ __forceinline__ void grid_forward_point(const N2LevelTable& tab, uint32_t level, uint32_t i, uint32_t N,
                                                   const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                                   const __half2* __restrict__ params, __half* __restrict__ out) {
	const size_t row = (size_t)level * 2;
	if (n2_level_masked(tab, level, i)) {
		out[row * N + i] = __float2half_rn(0.f);
		out[(row + 1) * N + i] = __float2half_rn(0.f);
		return;
	}
	const __half2* P = params + tab.offset[level];
	const N2Point p = n2_load_point(xyz, point_stride, dim_stride, i, tab.scale[level]);
	uint32_t e[8];
	n2_corner_entries<MODE>(p, tab.entries[level], tab.resolution[level], e);
	float2 v[8];
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) v[k] = __half22float2(P[e[k]]);
	float a0 = 0.f, a1 = 0.f;
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) {
		const float wt = n2_corner_weight(p, k);
		a0 = fmaf(wt, v[k].x, a0);
		a1 = fmaf(wt, v[k].y, a1);
	}
	out[row * N + i] = __float2half_rn(a0);
	out[(row + 1) * N + i] = __float2half_rn(a1);
}

__global__ void __launch_bounds__(GRID_BLOCK) grid_forward_point_kernel(N2LevelTable tab, uint32_t N, uint32_t tiles,
                                                                        const float* __restrict__ xyz, uint32_t point_stride,
                                                                        uint32_t dim_stride, const __half2* __restrict__ params,
                                                                        __half* __restrict__ out) {
	// level-major workgroup ids, dealt round-robin over the XCDs: every XCD sees an eighth of the tiles of every level.
	// (Giving whole levels to an XCD, as the scattered-point kernel does, makes every XCD stream all positions and
	// nearly doubles the time of a lattice chunk: with coherent points the tables' hot lines fit every L2 anyway.)
	const uint32_t level = blockIdx.x / tiles, tile = blockIdx.x - level * tiles;
	const uint32_t i = tile * GRID_BLOCK + threadIdx.x;
	if (i >= N) return;
#define CALL(M) grid_forward_point<M>(tab, level, i, N, xyz, point_stride, dim_stride, params, out)
	N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
}

// ----------------------------------------------------------------------------
// corner indices (test hook of the bit-exact contract)
// ----------------------------------------------------------------------------
__global__ void __launch_bounds__(GRID_BLOCK) grid_indices_kernel(N2LevelTable tab, uint32_t N, uint32_t tiles,
                                                                  const float* __restrict__ xyz, uint32_t point_stride,
                                                                  uint32_t dim_stride, uint32_t* __restrict__ idx) {
	const uint32_t level = blockIdx.x / tiles;
	const uint32_t i = (blockIdx.x - level * tiles) * GRID_BLOCK + threadIdx.x;
	if (i >= N) return;
	const N2Point p = n2_load_point(xyz, point_stride, dim_stride, i, tab.scale[level]);
	uint32_t e[8];
#define CALL(M) n2_corner_entries<M>(p, tab.entries[level], tab.resolution[level], e)
	N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) idx[((size_t)level * 8 + k) * N + i] = e[k];
}

// ----------------------------------------------------------------------------
// backward: parameter scatter (packed fp16 atomics), first and second order in
// one pass.
//
// Atomics retire at a fixed rate per REQUEST, and lanes of one instruction that
// hit the same 8 bytes travel as one request.  Corners that differ only in x
// are neighbours in the table (dense levels: index + 1; hashed levels: the x
// term enters the hash with prime 1, so even x and x+1 differ in bit 0 only).
// A point is therefore handled by a PAIR of adjacent lanes: lane bit 0 selects
// the x corner, each lane issues the four (y, z) corners.  That halves the
// number of atomic requests against one lane per point.
//
// Per corner c of level l the two contributions are
//   first order   dL_dy[l,f] * weight_c
//   second order  g[l,f] * scale_l * sum_d v_d * s_{c,d} * prod_{d' != d} w_{c,d'}
// and they leave as ONE packed fp16 atomic (one rounding instead of two).
// ----------------------------------------------------------------------------
constexpr uint32_t PAIR_POINTS = GRID_BLOCK / 2;  // points per workgroup and level

template <uint32_t MODE, bool FIRST, bool SECOND, bool WANT_OUT>
__device__ __forceinline__ void grid_scatter_pair(const N2LevelTable& tab, uint32_t level, uint32_t i, uint32_t b, uint32_t N,
                                                  const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                                  const __half* __restrict__ dL_dy, const float* __restrict__ v,
                                                  const __half* __restrict__ g2, const __half2* __restrict__ params,
                                                  __half2* __restrict__ grads, __half* __restrict__ dL_ddLdy, uint32_t xi, uint32_t Ng) {
	// xi: where this point's position and g2 column stand (i itself unless the call reads them through an index); Ng: columns of g2
	const float scale = tab.scale[level];
	const uint32_t entries = tab.entries[level], res = tab.resolution[level];
	const size_t row = (size_t)level * 2;
	if (n2_level_masked(tab, level, i)) {  // both lanes of a pair share i
		if (SECOND && WANT_OUT) dL_ddLdy[(row + b) * N + i] = __float2half_rn(0.f);
		return;
	}
	const N2Point p = n2_load_point(xyz, point_stride, dim_stride, xi, scale);
	float a0 = 0.f, a1 = 0.f, c0 = 0.f, c1 = 0.f, v0 = 0.f, v1 = 0.f, v2 = 0.f;
	if (FIRST) {
		a0 = __half2float(dL_dy[row * N + i]);
		a1 = __half2float(dL_dy[(row + 1) * N + i]);
	}
	if (SECOND) {
		c0 = __half2float(g2[row * Ng + xi]);
		c1 = __half2float(g2[(row + 1) * Ng + xi]);
		v0 = v[i] * scale; v1 = v[(size_t)N + i] * scale; v2 = v[(size_t)2 * N + i] * scale;
	}
	const bool skip = !SECOND && a0 == 0.f && a1 == 0.f;  // nothing to add (both lanes of a pair agree)
	const float wx = b ? p.w[0] : 1.f - p.w[0];
	const float sx = b ? 1.f : -1.f;
	const uint32_t gx = p.c[0] + b;
	const __half2* P = params + tab.offset[level];
	__half2* G = grads ? grads + tab.offset[level] : nullptr;
	float o0 = 0.f, o1 = 0.f;
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k) {
		const uint32_t y = k & 1u, z = k >> 1;
		const uint32_t e = n2_entry<MODE>(entries, res, gx, p.c[1] + y, p.c[2] + z);
		const float wy = y ? p.w[1] : 1.f - p.w[1], wz = z ? p.w[2] : 1.f - p.w[2];
		float r0 = 0.f, r1 = 0.f;
		if (FIRST) {
			const float wt = wx * wy * wz;
			r0 = a0 * wt;
			r1 = a1 * wt;
		}
		if (SECOND) {
			const float sy = y ? 1.f : -1.f, sz = z ? 1.f : -1.f;
			const float coef = v0 * sx * wy * wz + v1 * sy * wx * wz + v2 * sz * wx * wy;
			r0 = fmaf(c0, coef, r0);
			r1 = fmaf(c1, coef, r1);
			if (WANT_OUT) {
				const float2 val = __half22float2(P[e]);
				o0 = fmaf(coef, val.x, o0);
				o1 = fmaf(coef, val.y, o1);
			}
		}
		if (G && !skip) unsafeAtomicAdd(&G[e], __floats2half2_rn(r0, r1));
	}
	if (SECOND && WANT_OUT) {
		// lane b finishes feature b: it needs the partner's partial sum of that feature
		const float mine = b ? o1 : o0, theirs = n2_pair_swap(b ? o0 : o1);
		dL_ddLdy[(row + b) * N + i] = __float2half_rn(mine + theirs);
	}
}

template <bool FIRST, bool SECOND, bool WANT_OUT>
__global__ void __launch_bounds__(GRID_BLOCK) grid_scatter_kernel(N2LevelTable tab, uint32_t N, uint32_t tiles,
                                                                  const float* __restrict__ xyz, uint32_t point_stride,
                                                                  uint32_t dim_stride, const __half* __restrict__ dL_dy,
                                                                  const float* __restrict__ v, const __half* __restrict__ g2,
                                                                  const __half2* __restrict__ params, __half2* __restrict__ grads,
                                                                  __half* __restrict__ dL_ddLdy, const uint32_t* __restrict__ index, uint32_t n_cols) {
	const uint32_t level = blockIdx.x / tiles;
	const uint32_t i = (blockIdx.x - level * tiles) * PAIR_POINTS + (threadIdx.x >> 1);
	const uint32_t b = threadIdx.x & 1u;
	if (i >= N) return;  // both lanes of a pair share i, so pairs leave together
	const uint32_t xi = index ? min(index[i], n_cols - 1u) : i, Ng = index ? n_cols : N;
#define CALL(M) grid_scatter_pair<M, FIRST, SECOND, WANT_OUT>(tab, level, i, b, N, xyz, point_stride, dim_stride, dL_dy, v, g2, params, grads, dL_ddLdy, xi, Ng)
	N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
}

// ... and input gradient dL_dx[d][i] = sum_k dL_dy[k][i] * dy_dx[k][i][d].  Bound by HBM on large batches and by latency on small
// ones: eight rows' loads are under way together (one row at a time: 10.5 us for 5003 points, 23.5 for 2^18; now 4.4 and 20.3).
constexpr uint32_t BWD_IN_ROWS = 8;
template <bool STREAM>
__device__ __forceinline__ void grid_backward_input_point(uint32_t i, uint32_t N, uint32_t n_out, const __half* __restrict__ dL_dy, const float* __restrict__ dy_dx,
                                                          float* __restrict__ dL_dx) {
	if (i >= N) return;
	float r0 = 0.f, r1 = 0.f, r2 = 0.f;
	for (uint32_t k0 = 0; k0 < n_out; k0 += BWD_IN_ROWS) {
		__half g[BWD_IN_ROWS];
		n2_float3 j[BWD_IN_ROWS];
#pragma unroll
		for (uint32_t u = 0; u < BWD_IN_ROWS; ++u) {
			const size_t at = (size_t)min(k0 + u, n_out - 1u) * N + i;
			g[u] = dL_dy[at];
			j[u] = n2_load3<STREAM>(dy_dx + at * 3);
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (uint32_t u = 0; u < BWD_IN_ROWS; ++u) {
			if (k0 + u < n_out) {
				const float f = __half2float(g[u]);
				r0 = fmaf(f, j[u].x, r0);
				r1 = fmaf(f, j[u].y, r1);
				r2 = fmaf(f, j[u].z, r2);
			}
		}
	}
	dL_dx[i] = r0;
	dL_dx[(size_t)N + i] = r1;
	dL_dx[(size_t)2 * N + i] = r2;
}
template <bool STREAM>
__global__ void __launch_bounds__(GRID_BLOCK) grid_backward_input_kernel(uint32_t N, uint32_t n_out,
                                                                         const __half* __restrict__ dL_dy,
                                                                         const float* __restrict__ dy_dx,
                                                                         float* __restrict__ dL_dx) {
	grid_backward_input_point<STREAM>(blockIdx.x * GRID_BLOCK + threadIdx.x, N, n_out, dL_dy, dy_dx, dL_dx);
}

// ----------------------------------------------------------------------------
// second order: gradient of <v, dL_dx> w.r.t. the table, dL_dy and x
// ----------------------------------------------------------------------------
template <uint32_t MODE>
__device__ __forceinline__ void grid_bbi_point(const N2LevelTable& tab, uint32_t level, uint32_t i, uint32_t N,
                                               const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                               const float* __restrict__ v, const __half* __restrict__ dL_dy,
                                               const __half2* __restrict__ params, __half2* __restrict__ grads,
                                               __half* __restrict__ dL_ddLdy, float* __restrict__ dL_dx) {
	const float scale = tab.scale[level];
	const size_t row = (size_t)level * 2;
	if (n2_level_masked(tab, level, i)) {
		if (dL_ddLdy) {
			dL_ddLdy[row * N + i] = __float2half_rn(0.f);
			dL_ddLdy[(row + 1) * N + i] = __float2half_rn(0.f);
		}
		return;
	}
	const N2Point p = n2_load_point(xyz, point_stride, dim_stride, i, scale);
	uint32_t e[8];
	n2_corner_entries<MODE>(p, tab.entries[level], tab.resolution[level], e);
	const float v0 = v[i] * scale, v1 = v[(size_t)N + i] * scale, v2 = v[(size_t)2 * N + i] * scale;
	const float g0 = __half2float(dL_dy[row * N + i]);
	const float g1 = __half2float(dL_dy[(row + 1) * N + i]);
	const bool need_vals = dL_ddLdy != nullptr || dL_dx != nullptr;
	const __half2* P = params + tab.offset[level];
	__half2* G = grads ? grads + tab.offset[level] : nullptr;
	float o0 = 0.f, o1 = 0.f, dx0 = 0.f, dx1 = 0.f, dx2 = 0.f;
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) {
		const float w0 = (k & 1u) ? p.w[0] : 1.f - p.w[0];
		const float w1 = (k & 2u) ? p.w[1] : 1.f - p.w[1];
		const float w2 = (k & 4u) ? p.w[2] : 1.f - p.w[2];
		const float s0 = (k & 1u) ? 1.f : -1.f, s1 = (k & 2u) ? 1.f : -1.f, s2 = (k & 4u) ? 1.f : -1.f;
		// sum_d v_d * d(weight_k)/dx_d   (v already carries one factor of scale)
		const float coef = v0 * s0 * w1 * w2 + v1 * s1 * w0 * w2 + v2 * s2 * w0 * w1;
		if (G) unsafeAtomicAdd(&G[e[k]], __floats2half2_rn(g0 * coef, g1 * coef));
		if (need_vals) {
			const float2 val = __half22float2(P[e[k]]);
			o0 = fmaf(coef, val.x, o0);
			o1 = fmaf(coef, val.y, o1);
			if (dL_dx) {
				const float gp = (g0 * val.x + g1 * val.y) * scale;  // second factor of scale
				const float h01 = s0 * s1 * w2, h02 = s0 * s2 * w1, h12 = s1 * s2 * w0;
				dx0 = fmaf(gp, v1 * h01 + v2 * h02, dx0);
				dx1 = fmaf(gp, v0 * h01 + v2 * h12, dx1);
				dx2 = fmaf(gp, v0 * h02 + v1 * h12, dx2);
			}
		}
	}
	if (dL_ddLdy) {
		dL_ddLdy[row * N + i] = __float2half_rn(o0);
		dL_ddLdy[(row + 1) * N + i] = __float2half_rn(o1);
	}
	if (dL_dx) {
		unsafeAtomicAdd(&dL_dx[i], dx0);
		unsafeAtomicAdd(&dL_dx[(size_t)N + i], dx1);
		unsafeAtomicAdd(&dL_dx[(size_t)2 * N + i], dx2);
	}
}

__global__ void __launch_bounds__(GRID_BLOCK) grid_bbi_kernel(N2LevelTable tab, uint32_t N, uint32_t tiles,
                                                              const float* __restrict__ xyz, uint32_t point_stride,
                                                              uint32_t dim_stride, const float* __restrict__ v,
                                                              const __half* __restrict__ dL_dy, const __half2* __restrict__ params,
                                                              __half2* __restrict__ grads, __half* __restrict__ dL_ddLdy,
                                                              float* __restrict__ dL_dx) {
	const uint32_t level = blockIdx.x / tiles;
	const uint32_t i = (blockIdx.x - level * tiles) * GRID_BLOCK + threadIdx.x;
	if (i >= N) return;
#define CALL(M) grid_bbi_point<M>(tab, level, i, N, xyz, point_stride, dim_stride, v, dL_dy, params, grads, dL_ddLdy, dL_dx)
	N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
}

// ----------------------------------------------------------------------------
// bucketed scatter: parameter gradients WITHOUT global atomics
//
// Global atomics retire at ~2e10 requests/s on this part however they are
// issued, which caps the scatter above at ~55 us per level.  Loads, stores and
// LDS atomics are two orders of magnitude faster, so the scatter is turned
// into a two-kernel counting sort on entry ranges:
//
//  bin     one workgroup per (level, tile of up to 1024 points): computes the tile's records (an entry, or a pair of neighbouring ones, and what is added
//          there), sorts them in LDS by bucket (up to 4096 entries, at most 128 to a level) and writes the sorted tile, fully coalesced, plus its bucket offsets.
//  reduce  a workgroup per (level, bucket[, group of tiles]) at a time: walks the bucket's run in every tile, accumulates in an LDS
//          image of 64-bit integers with LDS atomics, and writes the bucket's entries with plain stores.
// The sums are exact until their one rounding at the store, which also removes the rounding drift of chained fp16 atomics.
// ----------------------------------------------------------------------------
#ifndef N2_BKT_SHIFT
#define N2_BKT_SHIFT 12
#endif
constexpr uint32_t BKT_SHIFT = N2_BKT_SHIFT;           // 4096 entries per bucket: a 64 KiB accumulator image, two reduce workgroups per CU
constexpr uint32_t BKT_ENTRIES = 1u << BKT_SHIFT;
constexpr uint32_t BKT_MAX = (1u << 19) >> BKT_SHIFT;  // buckets per level (entries <= 2^19)
constexpr uint32_t BKT_MIN_SHIFT = 5;                  // smallest bucket of a level that chooses its own size (N2LevelTable::bucket_shift)
constexpr uint32_t PAIR_MAX_CELL = BKT_ENTRIES - 2u;  // pair records (grid_bin_kernel): x + 1 <= BKT_ENTRIES - 1
static_assert(BKT_SHIFT <= 12, "a pair record's 16-bit key holds the entry within the bucket and four bits of carry length");
constexpr uint32_t BIN_BLOCK = 512;       // 8 waves: three workgroups (3 x 49 KiB of LDS) keep 6 waves on every SIMD, at 80 registers (with 96 or 128: pair +10 us)
// Points per thread of a bin workgroup (a tile: BIN_BLOCK * per points, eight records each): n2_bin_points_per_thread.
__host__ __device__ constexpr uint32_t bin_points(uint32_t per) { return BIN_BLOCK * per; }
__host__ __device__ constexpr uint32_t bin_records(uint32_t per) { return bin_points(per) * 8u; }

// (see n2_queue_draw)
constexpr uint32_t QUEUE_STRIDE = 32, QUEUE_WORDS = N_XCD * QUEUE_STRIDE;

// The items of a reduce launch, a (bucket, group of tiles) each, by level: levels of one kind of records, single ones or pairs, then those of the other.
struct N2BucketPlan {
	uint32_t begin[N2_MAX_LEVELS + 1];  // first item of each place in that order
	struct Level {
		uint32_t level, n_buckets;
		uint32_t groups;          // tile groups per bucket
		uint32_t part_begin;      // of split buckets (groups > 1): where the level's partial images start (bucket-major, then group)
		uint32_t bucket_entries;  // split buckets always have BKT_ENTRIES
		uint32_t entries, offset; // the level's table
		uint32_t pair;
	} at[N2_MAX_LEVELS];
	uint32_t second_from;  // first item of the second kind
};

// what a point brings along: its position, dL/dy of the level's two features, g2 of them and v
struct N2BinInput {
	float p[3], v[3];
	__half dy[2], g2[2];
};
template <bool FIRST, bool SECOND, bool STREAM>
__device__ __forceinline__ N2BinInput grid_bin_load(uint32_t level, uint32_t i, uint32_t N, const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                                    const __half* __restrict__ dL_dy, const float* __restrict__ v, const __half* __restrict__ g2, uint32_t xi, uint32_t Ng) {
	N2BinInput in;
	const float* q = xyz + (size_t)xi * point_stride;
	const size_t row = (size_t)level * 2;
#pragma unroll
	for (int d = 0; d < 3; ++d) in.p[d] = q[(size_t)d * dim_stride];
#pragma unroll
	for (int f = 0; f < 2; ++f) {
		if (FIRST) in.dy[f] = n2_load_half<STREAM>(dL_dy + (row + f) * N + i);
		if (SECOND) in.g2[f] = n2_load_half<STREAM>(g2 + (row + f) * Ng + xi);
	}
#pragma unroll
	for (int d = 0; d < 3; ++d)
		if (SECOND) in.v[d] = v[(size_t)d * N + i];
	return in;
}

template <uint32_t MODE, bool FIRST, bool SECOND, bool CLAMP_X>
__device__ __forceinline__ void grid_bin_point(const N2LevelTable& tab, uint32_t level, const N2BinInput& in, uint32_t* e_out, float* r0_out, float* r1_out,
                                               uint32_t* cell) {
	const float scale = tab.scale[level];
	N2Point p;
#pragma unroll
	for (int d = 0; d < 3; ++d) n2_locate(in.p[d], scale, p.w[d], p.c[d]);
	if (CLAMP_X) p.c[0] = min(p.c[0], PAIR_MAX_CELL);  // pair records: x + 1 stays inside the bucket's index bits
	cell[0] = p.c[0]; cell[1] = p.c[1]; cell[2] = p.c[2];
	uint32_t e[8];
	n2_corner_entries<MODE>(p, tab.entries[level], tab.resolution[level], e);
	float a0 = 0.f, a1 = 0.f, c0 = 0.f, c1 = 0.f, v0 = 0.f, v1 = 0.f, v2 = 0.f;
	if (FIRST) {
		a0 = __half2float(in.dy[0]);
		a1 = __half2float(in.dy[1]);
	}
	if (SECOND) {
		c0 = __half2float(in.g2[0]);
		c1 = __half2float(in.g2[1]);
		v0 = in.v[0] * scale; v1 = in.v[1] * scale; v2 = in.v[2] * scale;
	}
	// Corner k = i + 2 j + 4 l has weight X_i Y_j Z_l and signs (sx_i, sy_j, sz_l).  Its record is
	//   a X Y Z + c (v0 sx Y Z + v1 sy X Z + v2 sz X Y)  =  (Y Z) (a X + c v0 sx) + (c X) (v1 sy Z + v2 sz Y),
	// so the eight corners share two x terms per feature and four (y, z) terms.
	const float X[2] = {1.f - p.w[0], p.w[0]}, Y[2] = {1.f - p.w[1], p.w[1]}, Z[2] = {1.f - p.w[2], p.w[2]};
	float Pyz[4], Qyz[4], A0[2], A1[2], B0[2] = {0.f, 0.f}, B1[2] = {0.f, 0.f};
#pragma unroll
	for (uint32_t jl = 0; jl < 4; ++jl) {
		const uint32_t j = jl & 1u, l = jl >> 1;
		Pyz[jl] = Y[j] * Z[l];
		Qyz[jl] = SECOND ? (j ? v1 : -v1) * Z[l] + (l ? v2 : -v2) * Y[j] : 0.f;
	}
#pragma unroll
	for (uint32_t ix = 0; ix < 2; ++ix) {
		const float sv = ix ? v0 : -v0;
		A0[ix] = FIRST ? fmaf(a0, X[ix], c0 * sv) : c0 * sv;
		A1[ix] = FIRST ? fmaf(a1, X[ix], c1 * sv) : c1 * sv;
		if (SECOND) { B0[ix] = c0 * X[ix]; B1[ix] = c1 * X[ix]; }
	}
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) {
		const uint32_t ix = k & 1u, jl = k >> 1;
		float r0 = Pyz[jl] * A0[ix], r1 = Pyz[jl] * A1[ix];
		if (SECOND) {
			r0 = fmaf(B0[ix], Qyz[jl], r0);
			r1 = fmaf(B1[ix], Qyz[jl], r1);
		}
		e_out[k] = e[k];
		r0_out[k] = r0;
		r1_out[k] = r1;
	}
}

// Samples arrive in ray order, so on the coarser levels consecutive samples (= consecutive lanes)
// fall into the same cell and would hit the same eight entries.  When runs of equal cells are long
// enough (at most MERGE_MAX_HEADS runs in a wave), they are summed across lanes in fp32 and only the
// last lane of a run emits records: fewer records, and no pile-up on a few hot entries in the sort's
// counters or the reduce's accumulators.  The sums are segmented scans inside rows of 16 lanes, which
// the data-parallel-primitive lane shifts do at full ALU rate without touching LDS; a run that
// crosses a row boundary simply emits one record per row.
constexpr uint32_t MERGE_MAX_HEADS = 52;  // measured on the training step: 16: +16 us for the scatter pair, 24: +6, 32: +1, 40: +2 against 48 .. 58
constexpr unsigned long long ROW_HEADS = 0x0001000100010001ull;  // first lane of each 16-lane row

// r += take * (r of the lane D places below in the same 16-lane row; 0 if that leaves the row), for the sixteen values of a point.
// (Written out: the compiler makes a move with the lane shift, a wait state and a multiply-add of each.  s_nop: a lane shift must not
// read what one of the two instructions before it wrote.  &: `take` is read after the first values are written, so no value may share its register.)
// A value that is not finite makes no numbers of the sums above it in its row that do not take it, either: those count as zero.
template <int D>
__device__ __forceinline__ void n2_row_add(float (&a)[8], float (&b)[8], const float take) {
#define N2_ROW_ADD(K) "v_fmac_f32_dpp %" #K ", %" #K ", %16 row_shr:%17 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
	asm("s_nop 1\n\t" N2_ROW_ADD(0) N2_ROW_ADD(1) N2_ROW_ADD(2) N2_ROW_ADD(3) N2_ROW_ADD(4) N2_ROW_ADD(5) N2_ROW_ADD(6) N2_ROW_ADD(7)
	    N2_ROW_ADD(8) N2_ROW_ADD(9) N2_ROW_ADD(10) N2_ROW_ADD(11) N2_ROW_ADD(12) N2_ROW_ADD(13) N2_ROW_ADD(14) N2_ROW_ADD(15) "s_nop 0"
	    : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7]),
	      "+&v"(b[0]), "+&v"(b[1]), "+&v"(b[2]), "+&v"(b[3]), "+&v"(b[4]), "+&v"(b[5]), "+&v"(b[6]), "+&v"(b[7]) : "v"(take), "n"(D));
#undef N2_ROW_ADD
}
constexpr uint32_t REC_SKIP = 0xFFFFFFFFu;

// Pair records.  On a hashed level the entry of corner (x, y, z) is (x ^ y P1 ^ z P2) & (T - 1); while x + 1 stays below
// the bucket size, x only reaches the bits below BKT_SHIFT: the two x-neighbours of a (y, z) corner pair always share a
// bucket, and their places in it differ by x ^ (x + 1) = 2^(t+1) - 1, t = number of trailing one bits of x.  Such levels
// (pair_levels in the level table) sort and store ONE record per pair: both packed values (8 bytes) and a 16-bit key,
// entry of the x corner within the bucket | t << BKT_SHIFT.  Half the counter updates, prefix look-ups and staging
// stores here, half the key traffic and decoding in the reduce kernel.  Points outside the unit cube could carry an x
// beyond that range: their cell is clamped for the records (the dense levels clamp such points too).

// What a workgroup takes is its chain of waits (three share a CU, and the vector units are busy two thirds of the time): loads, counter
// updates and prefix look-ups are therefore issued together, and nothing waits in a branch.  With each of them awaited where it was used,
// and the second point's loads behind the first one's counters: training step at 2^18 samples 69 us, now 59 (57 and 47 on another card); trained 58, now 51; 2^18 uniform points
// 51.5, now 47.8; 52344 samples 15.1, now 12.7.
template <uint32_t PER, bool FIRST, bool SECOND, bool PAIR, bool STREAM>
__device__ __forceinline__ void grid_bin_tile(const N2LevelTable& tab, const uint32_t level, const uint32_t tile, uint32_t N, uint32_t tiles,
                                              const float* __restrict__ xyz, uint32_t point_stride, uint32_t dim_stride,
                                              const __half* __restrict__ dL_dy, const float* __restrict__ v, const __half* __restrict__ g2,
                                              uint32_t* __restrict__ rec_vals, uint16_t* __restrict__ rec_keys, uint16_t* __restrict__ offsets,
                                              uint32_t* hist, uint32_t* prefix, uint32_t* stage_val, uint16_t* stage_key,
                                              const uint32_t* __restrict__ index, uint32_t n_cols) {
	constexpr uint32_t R = PAIR ? 4 : 8;  // sorted records per point
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t shift = PAIR ? BKT_SHIFT : (uint32_t)tab.bucket_shift[level], in_bucket = (1u << shift) - 1u;
	// records of this thread: entry | rank << 19 after the counting step (REC_SKIP: merged into a later lane)
	uint32_t re[PER * R], rv[PER * 8], tcode[PER];
	// The second point's inputs are under way while the first one's records are merged and counted, the index it reads some of them by before
	// that.  (The
	// position and g2's columns may be read through an index: n2_grid_backward_fused_indexed.)
	const uint32_t Ng = index ? n_cols : N;
	uint32_t src[PER];
#pragma unroll
	for (uint32_t j = 0; j < PER; ++j) src[j] = min(tile * bin_points(PER) + j * BIN_BLOCK + threadIdx.x, N - 1u);
	if (index) {
#pragma unroll
		for (uint32_t j = 0; j < PER; ++j) src[j] = index[src[j]];
#pragma unroll
		for (uint32_t j = 0; j < PER; ++j) src[j] = min(src[j], n_cols - 1u);
	}
	auto load = [&](uint32_t j) __attribute__((always_inline)) {
		const uint32_t i = min(tile * bin_points(PER) + j * BIN_BLOCK + threadIdx.x, N - 1u);
		return grid_bin_load<FIRST, SECOND, STREAM>(level, i, N, xyz, point_stride, dim_stride, dL_dy, v, g2, src[j], Ng);
	};
	N2BinInput next = load(0);
#pragma unroll
	for (uint32_t j = 0; j < PER; ++j) {
		const uint32_t i = tile * bin_points(PER) + j * BIN_BLOCK + threadIdx.x;
		bool valid = i < N;
		if (valid && n2_level_masked(tab, level, i)) valid = false;  // a switched-off level: no records
		// Points that have no record go through all of this with the others, as points without a gradient.  (With the whole of it in a branch, and zeros in front for
		// those that it leaves out, and the runs found through the LDS crossbar: 2^18 uniform points 58.2 -> 56.5 us beside the input gradient, the SDF network's 48.6 -> 46.6.)
		N2BinInput in = next;
		const unsigned long long valids = __ballot(valid);
		if (valids != ~0ull) {  // (few waves; all of what they read may be no number)
#pragma unroll
			for (int d = 0; d < 3; ++d) {
				in.p[d] = valid ? in.p[d] : 0.f;
				if (SECOND) in.v[d] = valid ? in.v[d] : 0.f;
			}
#pragma unroll
			for (int f = 0; f < 2; ++f) {
				if (FIRST) in.dy[f] = valid ? in.dy[f] : __half(0.f);
				if (SECOND) in.g2[f] = valid ? in.g2[f] : __half(0.f);
			}
		}
		uint32_t e[8], cell[3];
		float r0[8], r1[8];
		if (PAIR) {
			grid_bin_point<N2_LEVEL_HASH, FIRST, SECOND, true>(tab, level, in, e, r0, r1, cell);
		} else {
#define CALL(M) grid_bin_point<M, FIRST, SECOND, false>(tab, level, in, e, r0, r1, cell)
			N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
		}
		if (j + 1 < PER) next = load(j + 1);
		// runs of equal cells among the wave's 64 consecutive points: where one begins (lane shifts inside the rows, whose first lanes begin one anyway)
		uint32_t other = 0u;
#pragma unroll
		for (int d = 0; d < 3; ++d) other |= cell[d] ^ (uint32_t)__builtin_amdgcn_update_dpp(0, (int)cell[d], 0x111, 0xf, 0xf, true);
		const unsigned long long heads = __ballot(other != 0u) | ~valids | ~(valids << 1) | ROW_HEADS;
		bool emit = valid;
		if (__popcll(heads) <= MERGE_MAX_HEADS) {
			// first lane of this lane's run (same row), and whether the next lane starts a new one
			const uint32_t start = 63u - (uint32_t)__clzll(heads & (~0ull >> (63u - lane)));
			emit = valid && (lane == 63u || ((heads >> (lane + 1u)) & 1ull));
			const uint32_t depth = lane - start;  // lanes of the run below this one
			// (a step that no run of the wave is long enough for adds nothing)
			n2_row_add<1>(r0, r1, depth >= 1u ? 1.f : 0.f);
			if (__ballot(depth >= 2u)) n2_row_add<2>(r0, r1, depth >= 2u ? 1.f : 0.f);
			if (__ballot(depth >= 4u)) n2_row_add<4>(r0, r1, depth >= 4u ? 1.f : 0.f);
			if (__ballot(depth >= 8u)) n2_row_add<8>(r0, r1, depth >= 8u ? 1.f : 0.f);
		}
		if (PAIR) tcode[j] = ((uint32_t)__popc((e[0] ^ e[1]) & (BKT_ENTRIES - 1u)) - 1u) << BKT_SHIFT;
#pragma unroll
		for (uint32_t k = 0; k < 8; ++k) {
			const __half2 h = __floats2half2_rn(r0[k], r1[k]);
			rv[8 * j + k] = *reinterpret_cast<const uint32_t*>(&h);
		}
#pragma unroll
		for (uint32_t q = 0; q < R; ++q) re[R * j + q] = REC_SKIP;
		if (emit) {
			uint32_t rank[R];
#pragma unroll
			for (uint32_t q = 0; q < R; ++q) rank[q] = atomicAdd(&hist[e[PAIR ? 2 * q : q] >> shift], 1u);
#pragma unroll
			for (uint32_t q = 0; q < R; ++q) re[R * j + q] = e[PAIR ? 2 * q : q] | (rank[q] << 19);
		}
	}
	__syncthreads();
	if (threadIdx.x < 64) {  // one wave scans the counters, BKT_MAX / 64 consecutive ones per lane
		constexpr uint32_t EACH = BKT_MAX / 64;
		uint32_t c[EACH], s = 0;
#pragma unroll
		for (uint32_t q = 0; q < EACH; ++q) { c[q] = hist[threadIdx.x * EACH + q]; s += c[q]; }
		const uint32_t own = s;
		s = n2_wave_prefix(s);
		uint32_t run = s - own;
#pragma unroll
		for (uint32_t q = 0; q < EACH; ++q) { prefix[threadIdx.x * EACH + q] = run; run += c[q]; }
		if (threadIdx.x == 63) prefix[BKT_MAX] = s;
	}
	__syncthreads();
#pragma unroll
	for (uint32_t j = 0; j < PER; ++j) {
		if (re[R * j] == REC_SKIP) continue;  // (a point's records go in together or not at all)
		uint32_t pos[R];
#pragma unroll
		for (uint32_t k = 0; k < R; ++k) pos[k] = prefix[(re[R * j + k] & 0x7FFFFu) >> shift] + (re[R * j + k] >> 19);
#pragma unroll
		for (uint32_t k = 0; k < R; ++k) {
			const uint32_t e = re[R * j + k] & 0x7FFFFu;
			if (PAIR) {
				reinterpret_cast<uint2*>(stage_val)[pos[k]] = make_uint2(rv[8 * j + 2 * k], rv[8 * j + 2 * k + 1]);
				stage_key[pos[k]] = (uint16_t)((e & (BKT_ENTRIES - 1u)) | tcode[j]);
			} else {
				stage_val[pos[k]] = rv[8 * j + k];
				stage_key[pos[k]] = (uint16_t)(e & in_bucket);
			}
		}
	}
	__syncthreads();
	const uint32_t total = prefix[BKT_MAX];
	// 16 bytes per lane; the last store of each array may run past `total` inside the tile's own slot, which nobody reads
	const size_t slot = ((size_t)level * tiles + tile) * bin_records(PER);
	uint4* out_val = reinterpret_cast<uint4*>(rec_vals + slot);
	uint4* out_key = reinterpret_cast<uint4*>(rec_keys + (size_t)level * tiles * bin_records(PER) + (size_t)tile * (bin_records(PER) / (PAIR ? 2u : 1u)));
	const uint4* sv = reinterpret_cast<const uint4*>(stage_val);
	const uint4* sk = reinterpret_cast<const uint4*>(stage_key);
	for (uint32_t t = threadIdx.x; (PAIR ? 2 : 4) * t < total; t += BIN_BLOCK) out_val[t] = sv[t];
	for (uint32_t t = threadIdx.x; 8 * t < total; t += BIN_BLOCK) out_key[t] = sk[t];
	if (threadIdx.x <= BKT_MAX) offsets[((size_t)level * tiles + tile) * (BKT_MAX + 1) + threadIdx.x] = (uint16_t)prefix[threadIdx.x];
}

// What else a sorting launch does, in workgroups of its own: work that needs nothing of the scatter's and would be a launch behind it.
// The input gradient streams the Jacobian while the others sort, its workgroups spread evenly among theirs (one behind each `every`): forward and
// backward of 2^18 uniform points 206.7 -> 196.1 us, along rays 168.1 -> 159.3; 65 536 uniform 77.4 -> 72.7; 20 000 along rays 37.9 -> 34.0.
struct N2RideNone {};
template <bool STREAM>
struct N2RideInput {
	const float* dy_dx;
	float* dL_dx;
	uint32_t n_out, every;
};
// The networks' weight-gradient slabs, two units to a workgroup, in the first workgroups: the field's forward and backward on 2^18 samples
// 251.0 -> 247.9 us, on 52 344 94.8 -> 91.6, on 2048 47.6 -> 41.3.
struct N2RideSums {
	N2SlabReduce sums;
	uint32_t blocks;
};
// The second order's dL_ddLdy = J v, gathered like the forward's Jacobian and contracted where it is formed: a group of eight workgroups that sort (an XCD each)
// follows `every` groups that gather, in the order of n2_gather_item.  Inside the sorting itself, where a lane took the eight corners of its point and any
// XCD's L2 came to hold every level, the gather took longer than all else: 2^18 second-order points (uniform) 154 -> 121 us for the launch (of which the
// sorting is 59), 131 072 along rays 61 -> 51, 5003 9.4 -> 7.0; the calls 400 -> 363 (forward and first order included), 189 -> 173 and 39.2 -> 36.9.
struct N2RideSecond {
	__half* dL_ddLdy;
	uint32_t blocks, every;  // workgroups that gather, and groups of them per group that sorts
	uint32_t tiles, height;  // as n2_gather_item takes them
};
template <class Ride> constexpr bool RIDES_INPUT = false;
template <bool STREAM> constexpr bool RIDES_INPUT<N2RideInput<STREAM>> = true;

template <uint32_t MODE>
__device__ __forceinline__ void grid_second_item(const N2LevelTable& tab, uint32_t level, uint32_t i, uint32_t N, const float* __restrict__ xyz, uint32_t point_stride,
                                                 uint32_t dim_stride, const __half2* __restrict__ params, const float* __restrict__ v, __half* __restrict__ dL_ddLdy) {
	const uint32_t at = min(i, N - 1u);  // (lanes behind the last point take part in its pair's exchange)
	const bool off = n2_level_masked(tab, level, at);
	uint32_t both = 0u;
	if (!__all(off)) {
		const float* q = xyz + (size_t)at * point_stride;
		const float p[3] = {n2_to_pairs(q[0]), n2_to_pairs(q[dim_stride]), n2_to_pairs(q[2 * (size_t)dim_stride])}, scale = tab.scale[level];
		const float along[3] = {n2_to_pairs(v[at]), n2_to_pairs(v[(size_t)N + at]), n2_to_pairs(v[2 * (size_t)N + at])};
		float feat[2], J[2][3];
		n2_encode_level<MODE, true>(reinterpret_cast<const char*>(params + tab.offset[level]), tab.entries[level], tab.resolution[level], scale, p, scale, feat, J);
		const __half2 h = __floats2half2_rn(fmaf(J[0][0], along[0], fmaf(J[0][1], along[1], J[0][2] * along[2])),
		                                    fmaf(J[1][0], along[0], fmaf(J[1][1], along[1], J[1][2] * along[2])));
		both = n2_from_pairs(*reinterpret_cast<const uint32_t*>(&h));
	}
	if (i >= N) return;
	if (off) both = 0u;
	const __half2 h = *reinterpret_cast<const __half2*>(&both);
	dL_ddLdy[(size_t)level * 2 * N + i] = __low2half(h);
	dL_ddLdy[((size_t)level * 2 + 1) * N + i] = __high2half(h);
}

template <uint32_t PER, bool FIRST, bool SECOND, bool STREAM, class Ride>
__global__ void __launch_bounds__(BIN_BLOCK, 6) grid_bin_kernel(N2LevelTable tab, uint32_t first_level, uint32_t N, uint32_t tiles,
                                                              const float* __restrict__ xyz, uint32_t point_stride,
                                                              uint32_t dim_stride, const __half* __restrict__ dL_dy,
                                                              const float* __restrict__ v, const __half* __restrict__ g2,
                                                              const __half2* __restrict__ params,
                                                              uint32_t* __restrict__ rec_vals, uint16_t* __restrict__ rec_keys,
                                                              uint16_t* __restrict__ offsets, uint32_t* __restrict__ queue,
                                                              const uint32_t* __restrict__ index, uint32_t n_cols, Ride ride) {
	__shared__ uint32_t hist[BKT_MAX];
	__shared__ uint32_t prefix[BKT_MAX + 1];
	__shared__ __align__(16) uint32_t stage_val[bin_records(PER)];  // sorted records: packed half2 value (a pair of them on pair levels) ...
	__shared__ __align__(16) uint16_t stage_key[bin_records(PER)];  // ... and entry within its bucket
	uint32_t block = blockIdx.x;
	if (blockIdx.x == 0u && blockIdx.y == 0u && threadIdx.x < N_XCD) queue[threadIdx.x * QUEUE_STRIDE] = 0u;
	if constexpr (RIDES_INPUT<Ride>) {
		bool rides;
		block = n2_turn(block, ride.every, 1u, rides);
		if (rides) {
			const auto point = [&](auto stream) {
				grid_backward_input_point<decltype(stream)::value>(block * BIN_BLOCK + threadIdx.x, N, ride.n_out, dL_dy, ride.dy_dx, ride.dL_dx);
			};
			point(std::bool_constant<std::is_same<Ride, N2RideInput<true>>::value>());
			return;
		}
		if (block >= tiles * tab.n_levels) return;
	} else if constexpr (std::is_same<Ride, N2RideSecond>::value) {
		bool sorts;
		block = n2_turn(block + blockIdx.y * gridDim.x, ride.every, N_XCD, sorts);
		if (!sorts) {
			const uint32_t y = ride.height == 1u ? 0u : block / ride.tiles;
			uint32_t level, tile;
			if (block >= ride.blocks || !n2_gather_item(block - y * ride.tiles, y, ride.height, tab.n_levels, ride.tiles, level, tile)) return;
			const uint32_t i = tile * BIN_BLOCK + threadIdx.x;
#define CALL(M) grid_second_item<M>(tab, level, i, N, xyz, point_stride, dim_stride, params, v, ride.dL_ddLdy)
			N2_DISPATCH_MODE(tab.mode[level], CALL)
#undef CALL
			return;
		}
		if (block >= tiles * tab.n_levels) return;
	} else if constexpr (std::is_same<Ride, N2RideSums>::value) {
		if (block < ride.blocks) {
			constexpr uint32_t UNITS = BIN_BLOCK / 256;
			static_assert(sizeof(float) * 32 * 33 * UNITS <= sizeof(stage_val), "the units' folds");
			float(*fold)[33] = reinterpret_cast<float(*)[33]>(stage_val) + (threadIdx.x >> 8) * 32;
			n2_slab_reduce_unit(ride.sums, block * UNITS + (threadIdx.x >> 8), fold, [](const _Float16*, _Float16) {}, threadIdx.x & 255u);
			return;
		}
		block -= ride.blocks;
	}
	const uint32_t level = first_level + block / tiles, tile = block % tiles;
	if (threadIdx.x < BKT_MAX) hist[threadIdx.x] = 0;
	__syncthreads();
	if ((tab.pair_levels >> level) & 1u)
		grid_bin_tile<PER, FIRST, SECOND, true, STREAM>(tab, level, tile, N, tiles, xyz, point_stride, dim_stride, dL_dy, v, g2, rec_vals,
		                                        rec_keys, offsets, hist, prefix, stage_val, stage_key, index, n_cols);
	else
		grid_bin_tile<PER, FIRST, SECOND, false, STREAM>(tab, level, tile, N, tiles, xyz, point_stride, dim_stride, dL_dy, v, g2, rec_vals,
		                                         rec_keys, offsets, hist, prefix, stage_val, stage_key, index, n_cols);
}

// LDS float atomics retire about one lane every three clocks on this part, integer ones at ~9 (32-bit) and
// ~5.5 (64-bit) lanes per clock.  The reduce therefore accumulates in 64-bit fixed point: a record holds
// fp16 values, i.e. multiples of 2^-24 below 2^16, so value * 2^24 is an exact integer below 2^40 and the
// sum of a whole bucket stays far inside 64 bits.  The accumulation is exact and independent of order.
constexpr uint32_t RED_BLOCK = 512;               // 8 waves; two workgroups share a CU
constexpr uint32_t RED_FLIGHT = 6, RED_FLIGHT_PAIRS = 3;  // single records, and pairs, that a lane has under way at a time
constexpr uint32_t RED_AT_A_TIME = 512;           // workgroups of a launch: what runs at one time (a multiple of the XCDs)
constexpr float FIX_SCALE = 16777216.0f;          // 2^24

// x * 2^24 as a two's complement 64-bit integer, given that product (of an fp16 value, so it is a whole number).  For |x| < 128 it has 32 bits: two instructions.
__device__ __forceinline__ unsigned long long fixed_small(float scaled) { return (unsigned long long)(long long)(int32_t)scaled; }
__device__ __forceinline__ bool is_fixed_small(float scaled) { return fabsf(scaled) < 2147483648.f; }
// Up to 2^51: added to 3 * 2^51 it stands in the sum's low bits.
__device__ __forceinline__ unsigned long long fixed_large(float scaled) {
	return __builtin_bit_cast(unsigned long long, (double)scaled + 6755399441055744.0) - 0x4338000000000000ull;
}
// What is not finite adds nothing to a sum: no number counts as zero, and an infinite value leaves a mark beside it, two bits for each feature (one for either sign), four for an
// entry.  (A large whole number in its place is brought back by enough finite values of the other sign, or wraps round with others like it: both gave finite gradients.)
__device__ __forceinline__ float finite_or_zero(float x) { return fabsf(x) < __builtin_inff() ? x : 0.f; }
__device__ __forceinline__ uint32_t infinite_mark(float x) { return fabsf(x) == __builtin_inff() ? 1u + (__builtin_bit_cast(uint32_t, x) >> 31) : 0u; }
__device__ __forceinline__ uint32_t infinite_mark(float x, float y) { return infinite_mark(x) | infinite_mark(y) << 2; }
__device__ __forceinline__ float marked_sum(float sum, uint32_t bits) {  // infinite, or no number where there were both signs
	return bits == 0u ? sum : __builtin_bit_cast(float, 0x7F800000u | (bits & 2u) << 30 | (bits & bits >> 1) << 22);
}
__device__ __forceinline__ float2 marked_sums(float2 sums, uint32_t bits) { return make_float2(marked_sum(sums.x, bits & 3u), marked_sum(sums.y, bits >> 2 & 3u)); }
constexpr uint32_t MARKS_PER_WORD = 8;  // entries' marks in 32 bits
__device__ __forceinline__ float from_fixed(unsigned long long q) {
	return (float)fma((double)(int32_t)(q >> 32), 4294967296.0, (double)(uint32_t)q) * (1.f / FIX_SCALE);
}

// A sum in fp32 and the gradient that it is added to, in fp32, so that all ways to the sum round alike, to fp32 and then to fp16.  (Left to the compiler, the sum's factor,
// the addition and the conversion are one instruction in some kernels, which rounds once.)
__device__ __forceinline__ float2 added_to(float2 sum, float2 old) {
#pragma clang fp contract(off)
	return make_float2(sum.x + old.x, sum.y + old.y);
}

// Which (level, bucket, group of tiles) is an item?  (Lane l asks about place l: sixteen scalar loads one after the other were a microsecond.)
struct N2ReduceItem {
	uint32_t bucket, group;
	N2BucketPlan::Level l;
};
__device__ __forceinline__ uint32_t n2_lane_end(const N2BucketPlan& plan) {  // end of place `lane`
	const uint32_t lane = threadIdx.x & 63u;
	return lane < N2_MAX_LEVELS ? plan.begin[lane + 1u] : 0xFFFFFFFFu;
}
__device__ __forceinline__ N2ReduceItem n2_reduce_item(const N2BucketPlan& plan, uint32_t lane_end, uint32_t item) {
	N2ReduceItem it;
	const uint32_t place = __popcll(__ballot(item >= lane_end)), local = item - plan.begin[place];
	it.l = plan.at[place];
	it.bucket = local;
	it.group = 0u;
	if (it.l.groups > 1u) {
		it.bucket = __builtin_amdgcn_readfirstlane(local / it.l.groups);
		it.group = local - it.bucket * it.l.groups;
	} else if (it.l.n_buckets % N_XCD == 0u) {
		// A tile's runs for neighbouring buckets meet inside a 128-byte line, which both buckets' workgroups fetch.  Workgroup
		// ids are dealt round-robin over the XCDs (and an item's number is its workgroup's but for whole rounds of them): XCD x takes the x-th eighth
		// of the level's buckets, in order, so that both fetches of such a line go through the same L2 at about the same time.
		it.bucket = (item % N_XCD) * (it.l.n_buckets / N_XCD) + local / N_XCD;
	}
	return it;
}

// The gradients of a bucket that a lane writes, four entries (16 bytes) at a time: a level's table is whole multiples of eight entries and a bucket of 32.  An
// accumulating launch has their old values under way before the last records are added.  (Loaded where they are added they were a trip to memory each, of four in
// a workgroup's life: forward, backward and second order of 180 000 points 214 -> 245 us.)
constexpr uint32_t RED_WRITES = BKT_ENTRIES / (RED_BLOCK * 4u);
static_assert(RED_WRITES * RED_BLOCK * 4u == BKT_ENTRIES, "a bucket is whole rounds of a workgroup");
typedef uint32_t n2_four_entries __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void grid_reduce_old(const N2ReduceItem& it, const __half2* __restrict__ grads, n2_four_entries (&old)[RED_WRITES]) {
#pragma unroll
	for (uint32_t k = 0; k < RED_WRITES; ++k)
		old[k] = *reinterpret_cast<const n2_four_entries*>(grads + it.l.offset + min(it.bucket * it.l.bucket_entries + (k * RED_BLOCK + threadIdx.x) * 4u, it.l.entries - 4u));
}
// The sums of a bucket's records: out to the gradients, or as they are where the bucket is split, and back to zero.
template <bool ACCUMULATE>
__device__ __forceinline__ void grid_reduce_out(const N2ReduceItem& it, unsigned long long* acc, __half2* __restrict__ grads, const n2_four_entries (&old)[RED_WRITES],
                                                float2* __restrict__ partials) {
	ulonglong2* const wide_acc = reinterpret_cast<ulonglong2*>(acc);
	const ulonglong2 none = make_ulonglong2(0ull, 0ull);
	if (it.l.groups > 1u) {
		// Several workgroups hold parts of this bucket's sums (coarse levels of large batches).  Each leaves its image as
		// fp32 and grid_combine_kernel adds the G images up in the order of the groups: every entry is the same sum of the
		// same terms in the same order however the workgroups were scheduled (the images themselves are exact integer sums).
		float2* mine = partials + ((size_t)it.l.part_begin + (size_t)it.bucket * it.l.groups + it.group) * BKT_ENTRIES;
		for (uint32_t e = threadIdx.x; e < BKT_ENTRIES; e += RED_BLOCK) {
			mine[e] = make_float2(from_fixed(acc[e]), from_fixed(acc[BKT_ENTRIES + e]));
			acc[e] = acc[BKT_ENTRIES + e] = 0ull;
		}
		return;
	}
	__half2* Gd = grads + it.l.offset;
#pragma unroll
	for (uint32_t k = 0; k < RED_WRITES; ++k) {
		const uint32_t e = (k * RED_BLOCK + threadIdx.x) * 4u, idx = it.bucket * it.l.bucket_entries + e;
		if (e >= it.l.bucket_entries || idx >= it.l.entries) break;
		n2_four_entries out;
#pragma unroll
		for (uint32_t q = 0; q < 4; q += 2) {
			const ulonglong2 x = wide_acc[(e + q) / 2u], y = wide_acc[(BKT_ENTRIES + e + q) / 2u];
			wide_acc[(e + q) / 2u] = wide_acc[(BKT_ENTRIES + e + q) / 2u] = none;
#pragma unroll
			for (uint32_t p = 0; p < 2; ++p) {
				float2 f = make_float2(from_fixed(p ? x.y : x.x), from_fixed(p ? y.y : y.x));
				if (ACCUMULATE) {
					const uint32_t o = old[k][q + p];
					const float2 g = __half22float2(*reinterpret_cast<const __half2*>(&o));
					f = added_to(f, g);
				}
				const __half2 h = __floats2half2_rn(f.x, f.y);
				out[q + p] = *reinterpret_cast<const uint32_t*>(&h);
			}
		}
		*reinterpret_cast<n2_four_entries*>(Gd + idx) = out;
	}
}

// What is infinite of them, over those sums: the marks of four entries at a time, and back to zero.
template <bool ACCUMULATE>
__device__ __forceinline__ void grid_reduce_marked(const N2ReduceItem& it, uint16_t* marks, __half2* __restrict__ grads, float2* __restrict__ partials) {
	__syncthreads();  // (the sums may be other threads')
	float* const image = reinterpret_cast<float*>(partials + ((size_t)it.l.part_begin + (size_t)it.bucket * it.l.groups + it.group) * BKT_ENTRIES);
	__half* const grad = reinterpret_cast<__half*>(grads + it.l.offset + it.bucket * it.l.bucket_entries);
	for (uint32_t at = threadIdx.x; at < BKT_ENTRIES / 4u; at += RED_BLOCK) {
		const uint32_t m = marks[at];
		if (m == 0u) continue;
		marks[at] = 0u;
		for (uint32_t v = 0; v < 8; ++v) {  // two values of four entries
			const uint32_t bits = m >> (2u * v) & 3u, place = at * 8u + v;
			if (bits == 0u) continue;
			if (it.l.groups > 1u) image[place] = marked_sum(0.f, bits);
			else grad[place] = __float2half(marked_sum(0.f, bits) + (ACCUMULATE ? __half2float(grad[place]) : 0.f));
		}
	}
}

// A reduce launch's queue: a workgroup begins with the item of its own number and goes on with what it draws, for items differ by a factor of three in what
// they take (dealt out by numbers alone, a training step's launch had its median workgroup end at 32 us and its last one at 46.9; drawn two ahead 34.2 and 43.6).  It draws when
// it has asked for the last records of what it is at: drawn when it began, an item waited for a workgroup that a full bucket kept, and the launch for that item (52 344 points
// in a box of a fifth of the cube's side: backward 94.4 us, now 90.7; 2^18 points 331 and 324, uniform 89.3 and 88.6).
// One counter for each XCD, in a line of its own; the sorting launch in front clears them.
__device__ __forceinline__ uint32_t n2_queue_draw(uint32_t* queue) { return atomicAdd(queue + blockIdx.x % N_XCD * QUEUE_STRIDE, 1u); }
__device__ __forceinline__ uint32_t n2_queue_item(uint32_t drawn) { return blockIdx.x % N_XCD + N_XCD * ((gridDim.x + N_XCD - 1u) / N_XCD + drawn); }  // (behind all first ones)

// What a workgroup works on, as long as it is below `end` (all of one kind of records): `item`, then what it draws.  `acc` is all zeros before and after.
//
// Lane j of wave w takes run w + WAVES j of the bucket's (a tile's run, or one of the 2^part_shift parts of it, so that a batch of few
// tiles keeps all waves busy), and the wave walks through the records of its up to 64 runs as if they stood one behind the other, 64 at a time: which
// runs the next 64 meet is the same question for the whole wave, so a run costs it two lane reads and three vector instructions, and every lane has a
// record until the last.  FLIGHT times 64 records are being added while the next are on their way, the next item's first ones while this item's sums are written
// (its bounds before that).
template <bool PAIR, uint32_t FLIGHT, bool ACCUMULATE>
__device__ __forceinline__ void grid_reduce_items(const N2BucketPlan& plan, const uint32_t lane_end, uint32_t& item, const uint32_t end, const uint32_t tiles, const uint32_t slot_records,
                                                  const uint32_t part_shift, const uint32_t* __restrict__ rec_vals, const uint16_t* __restrict__ rec_keys,
                                                  const uint16_t* __restrict__ offsets, __half2* __restrict__ grads, float2* __restrict__ partials,
                                                  unsigned long long* acc, uint32_t* marks, uint32_t* queue, uint2* drawn) {
	typedef typename std::conditional<PAIR, uint2, uint32_t>::type value;
	constexpr uint32_t WAVES = RED_BLOCK / 64, STEP = 64u * FLIGHT;
	if (item >= end) return;
	const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	N2ReduceItem it = n2_reduce_item(plan, lane_end, item);
	// Of the wave's 64 runs at hand, lane j: the records up to the end of run j, and what takes a record's number among them to its place behind `vals` and `keys`.
	uint32_t upto, place, total;
	uint32_t at, k, k_upto, k_place;  // the next records begin at number `at`, in run k
	const value* vals;
	const uint16_t* keys;
	auto tile_of = [&](const N2ReduceItem& i, uint32_t run) { return n2_run_tile(i.group, i.l.groups, run, part_shift, tiles); };
	auto bounds = [&](const N2ReduceItem& i, uint32_t first) __attribute__((always_inline)) {  // of the lane's run
		uint32_t two;
		__builtin_memcpy(&two, offsets + ((size_t)i.l.level * tiles + tile_of(i, first + WAVES * lane)) * (BKT_MAX + 1) + i.bucket, sizeof(two));
		return two;
	};
	auto runs_of = [&](const N2ReduceItem& i) { return (i.l.groups == 1u ? tiles : (tiles - i.group + i.l.groups - 1u) / i.l.groups) << part_shift; };
	auto take = [&](const N2ReduceItem& i, uint32_t first, uint32_t two) __attribute__((always_inline)) {
		const uint32_t run = first + WAVES * lane, part = run & ((1u << part_shift) - 1u);
		const uint32_t all = (two >> 16) - (two & 0xFFFFu), begin = all * part >> part_shift, stop = all * (part + 1u) >> part_shift;
		const uint32_t n = run < runs_of(i) ? stop - begin : 0u;
		upto = n2_wave_prefix(n);
		const uint32_t tile_records = PAIR ? slot_records / 2u : slot_records, first_tile = tile_of(i, first);
		place = n2_run_place(first_tile, tile_of(i, run), tile_records) + (two & 0xFFFFu) + begin - (upto - n);
		total = (uint32_t)__builtin_amdgcn_readlane((int)upto, 63);
		const size_t level0 = (size_t)i.l.level * tiles * slot_records, base = n2_run_base(first_tile, tile_records);
		vals = reinterpret_cast<const value*>(rec_vals + level0) + base;
		keys = rec_keys + level0 + base;
		at = k = 0u;
		k_upto = (uint32_t)__builtin_amdgcn_readlane((int)upto, 0);
		k_place = (uint32_t)__builtin_amdgcn_readlane((int)place, 0);
	};
	struct Record {
		value v;
		uint32_t key;
	};
	auto load = [&](Record& q) __attribute__((always_inline)) {  // (behind the last record the last one is read again: all loads are issued, so a wait can be for one step's)
		const uint32_t last = min(at + 63u, total - 1u), r = min(at + lane, total - 1u);
		uint32_t p = k_place;
		while (k_upto <= last) {  // (the last run ends at `total`)
			const uint32_t below = k_upto;
			++k;
			k_upto = (uint32_t)__builtin_amdgcn_readlane((int)upto, (int)k);
			k_place = (uint32_t)__builtin_amdgcn_readlane((int)place, (int)k);
			p = r >= below ? k_place : p;
		}
		q.key = keys[r + p];
		q.v = vals[r + p];
		at += 64u;
	};
	auto load_step = [&](Record (&q)[FLIGHT]) __attribute__((always_inline)) {
#pragma unroll
		for (uint32_t u = 0; u < FLIGHT; ++u) load(q[u]);
	};
	constexpr uint32_t EACH = PAIR ? 2u : 1u;  // entries of a record
	bool not_finite = false;  // a value of the wave's records of this item is not
	auto add_step = [&](const Record (&q)[FLIGHT], uint32_t from) __attribute__((always_inline)) {
		float f[FLIGHT][2 * EACH], most = 0.f;  // (of lanes behind the last record those of the last one)
#pragma unroll
		for (uint32_t u = 0; u < FLIGHT; ++u)
#pragma unroll
			for (uint32_t e = 0; e < EACH; ++e) {
				uint32_t raw;
				if constexpr (PAIR) raw = e ? q[u].v.y : q[u].v.x;
				else raw = q[u].v;
				const __half2 h = *reinterpret_cast<const __half2*>(&raw);
				f[u][2 * e] = fmaf(__low2float(h), FIX_SCALE, 0.f);
				f[u][2 * e + 1] = fmaf(__high2float(h), FIX_SCALE, 0.f);
				most = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(f[u][2 * e]), fabsf(f[u][2 * e + 1])), most);  // (no number where one is none)
			}
		auto add = [&](auto fixed) __attribute__((always_inline)) {
#pragma unroll
			for (uint32_t u = 0; u < FLIGHT; ++u) {
				if (from + 64u * u + lane >= total) break;
				const uint32_t a = q[u].key << 3;  // (bytes into a plane of sums)
				auto sum_at = [&](uint32_t bytes) { return reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(acc) + bytes); };
				unsigned long long* to[EACH];
				to[0] = sum_at(PAIR ? a & (BKT_ENTRIES - 1u) << 3 : a);
				if constexpr (PAIR) to[1] = sum_at((a ^ ((16u << (q[u].key >> BKT_SHIFT)) - 8u)) & (BKT_ENTRIES - 1u) << 3);  // x ^ (x + 1) = 2^(t+1) - 1
#pragma unroll
				for (uint32_t e = 0; e < EACH; ++e) {
					atomicAdd(to[e], fixed(f[u][2 * e]));
					atomicAdd(to[e] + BKT_ENTRIES, fixed(f[u][2 * e + 1]));
				}
			}
		};
		if (__any(!is_fixed_small(most))) {
			if (__any(!(most < FIX_SCALE * 65536.f))) {
#pragma unroll
				for (uint32_t u = 0; u < FLIGHT; ++u)
#pragma unroll
					for (uint32_t e = 0; e < 2 * EACH; ++e) f[u][e] = finite_or_zero(f[u][e]);
				not_finite = true;
			}
			add([](float x) { return fixed_large(x); });
		} else add([](float x) { return fixed_small(x); });
	};
	Record qa[FLIGHT], qb[FLIGHT];
	take(it, wave, bounds(it, wave));
	if (total > 0u) load_step(qa);
	__syncthreads();  // the sums are zero
	while (true) {
		uint32_t draw = 0u;
		for (uint32_t first = wave;;) {
			auto draw_behind_the_last = [&]() __attribute__((always_inline)) {
				if (wave == 0u && first + WAVES * 64u >= runs_of(it) && lane == 0u) draw = n2_queue_draw(queue);
			};
			if (total == 0u) draw_behind_the_last();
			while (total > 0u) {
				if (at >= total) {
					draw_behind_the_last();
					add_step(qa, at - STEP);
					break;
				}
				load_step(qb);
				add_step(qa, at - 2u * STEP);
				if (at >= total) {
					draw_behind_the_last();
					add_step(qb, at - STEP);
					break;
				}
				load_step(qa);
				add_step(qb, at - 2u * STEP);
			}
			first += WAVES * 64u;
			if (first >= runs_of(it)) break;
			take(it, first, bounds(it, first));
			if (total > 0u) load_step(qa);
		}
		if (not_finite) {  // (once more through them, for the marks: with those left on the way, 2^18 uniform points lose 4 % of the launch)
			not_finite = false;
			for (uint32_t first = wave; first < runs_of(it); first += WAVES * 64u) {
				take(it, first, bounds(it, first));
				while (at < total) {
					Record q;
					load(q);
					if (at - 64u + lane >= total) continue;
					for (uint32_t e = 0; e < EACH; ++e) {
						uint32_t raw, entry = q.key & (BKT_ENTRIES - 1u);
						if constexpr (PAIR) {
							raw = e ? q.v.y : q.v.x;
							if (e) entry ^= (2u << (q.key >> BKT_SHIFT)) - 1u;
						} else raw = q.v;
						const float2 v = __half22float2(*reinterpret_cast<const __half2*>(&raw));
						const uint32_t mark = infinite_mark(v.x, v.y);
						if (mark == 0u) continue;
						atomicOr(&marks[entry / MARKS_PER_WORD], mark << (entry % MARKS_PER_WORD * 4u));
						drawn->y = 1u;
					}
				}
			}
		}
		n2_four_entries old[RED_WRITES];
		if (ACCUMULATE) grid_reduce_old(it, grads, old);
		if (threadIdx.x == 0u) drawn->x = draw;
		__syncthreads();
		const uint2 now = *drawn;
		const bool any_marks = __builtin_amdgcn_readfirstlane(now.y) != 0u;
		item = n2_queue_item(__builtin_amdgcn_readfirstlane(now.x));
		const N2ReduceItem next = n2_reduce_item(plan, lane_end, min(item, end - 1u));
		const uint32_t two = bounds(next, wave);
		grid_reduce_out<ACCUMULATE>(it, acc, grads, old, partials);
		if (any_marks) grid_reduce_marked<ACCUMULATE>(it, reinterpret_cast<uint16_t*>(marks), grads, partials);
		if (item < end) {
			take(next, wave, two);
			if (total > 0u) load_step(qa);
		}
		__syncthreads();
		if (item >= end) return;
		it = next;
	}
}

// What bounds it is the LDS (busy in 67 % of a CU's clocks on 2^18 uniform points, two thirds of that bank conflicts), vector instructions (69 %) and the records' way through memory;
// of 50.4 us it took without the LDS additions 45.6, with records out of the L1 46.8, with neither 39.6, without writing the sums 44.9 (buckets drawn early then).  Before, one
// workgroup of 1024 threads to a bucket, groups of 8 or 16 lanes to a tile's run, values in 2^32 fixed point by five instructions each, | now, launch in us: a training
// step's 54.6 | 43.1, trained 44.5 | 40.2, the SDF network's 65.2 | 54.8, 52 344 samples 20.0 | 18.3, 2^18 uniform points 51.8 | 48.0 (vector instructions 24.9 | 15.3 M).  Other shapes, of 50.7
// uniform: 256 threads 59.8, 768 50.6 (registers spill: an accumulating backward of 52 344 points 40 -> 47), 1024 66.0; items dealt out by number 53.2, training step 51.0.  Records under
// way, single ones and pairs, 6 and 3: 4 and 2, and 4 and 3, take the same within 1 %, 6 and 4 1 to 2 % longer, 8 and 3 spill and take 3 to 6.
// Values from 128 on (a second order's, whose J holds the level's scale) take an instruction more, chosen for a wave's step as a whole: second order and both others on 60 000
// points along rays 100.0 -> 95.7.  Points packed into a fifth of the cube's side, which meet a few full buckets, lose 2 per cent of a backward: 52 344 88.4 | 90.7, 2^18 319 | 325.
template <bool ACCUMULATE, bool PAIRS_FIRST>
__global__ void __launch_bounds__(RED_BLOCK, 4) grid_reduce_kernel(N2BucketPlan plan, uint32_t tiles, uint32_t slot_records, uint32_t part_shift,
                                                                   const uint32_t* __restrict__ rec_vals, const uint16_t* __restrict__ rec_keys,
                                                                   const uint16_t* __restrict__ offsets,
                                                                   __half2* __restrict__ grads, float2* __restrict__ partials, uint32_t* __restrict__ queue) {
	// one plane per feature: lanes of a wave's atomic then spread over all bank pairs (entry-major pairs of features would
	// leave every other pair unused)
	__shared__ __align__(16) unsigned long long acc[2 * BKT_ENTRIES];
	__shared__ uint32_t marks[BKT_ENTRIES / MARKS_PER_WORD];
	__shared__ uint2 drawn;  // x: the item drawn, y: whether there were marks since the workgroup began
	const uint32_t lane_end = n2_lane_end(plan), items = plan.begin[N2_MAX_LEVELS];
	for (uint32_t e = threadIdx.x; e < BKT_ENTRIES; e += RED_BLOCK) reinterpret_cast<ulonglong2*>(acc)[e] = make_ulonglong2(0ull, 0ull);
	for (uint32_t e = threadIdx.x; e < BKT_ENTRIES / MARKS_PER_WORD; e += RED_BLOCK) marks[e] = 0u;
	if (threadIdx.x == 0u) drawn.y = 0u;
	uint32_t item = blockIdx.x;
#define ITEMS(P, FLIGHT, END) grid_reduce_items<P, FLIGHT, ACCUMULATE>(plan, lane_end, item, END, tiles, slot_records, part_shift, rec_vals, rec_keys, offsets, grads, partials, acc, marks, queue, &drawn)
	if (PAIRS_FIRST) {
		ITEMS(true, RED_FLIGHT_PAIRS, plan.second_from);
		ITEMS(false, RED_FLIGHT, items);
	} else {
		ITEMS(false, RED_FLIGHT, plan.second_from);
		ITEMS(true, RED_FLIGHT_PAIRS, items);
	}
#undef ITEMS
}

// Small batches: the gradient of a bucket with few records.
// grid_reduce_kernel keeps a sum for each of a bucket's 4096 entries: 64 KiB of LDS to clear and to read again, at two workgroups per CU, for a bucket that
// holds 160 records when the batch has 5000 points.  Here a record claims a sum: every record writes its own number to the 16-bit place of its entry, and
// whichever number stands there afterwards is the entry's sum (64-bit fixed point as above, so the result is the same whoever wins).  Nothing is cleared but
// the sums that exist; the other entries' zeros go out while the first loads are under way (an accumulating launch leaves them alone), and a workgroup's
// 40 KiB let four of 512 threads share a CU.  Every thread finds its records by their number among the bucket's, so no lane has to
// match a tile's run.  Levels of few entries keep an image, as does (range by range) a bucket with more records than
// there are sums to claim.  What bounds it is the chain level -> bounds -> records -> sums and the 25 MB the gradient's zeros take.
// Launch in us, image -> claims: 600 uniform points 15 -> 10.1, 5003 along rays 15.1 -> 10.6 (accumulating 15.6 -> 9.5), training step of 2^14 samples 17.5 -> 14.8.
// (256 threads: the same up to 5000 points, 16 384 uniform +4; 1024: +4; 128: +0.5.  In 32 KiB there are 1536 sums instead of 2048,
// and batches beyond 16 384 points took grid_reduce_kernel: 20 000 along rays 34.0 against 29.5.)
// With the next item's bounds on their way meanwhile (its level and tiles looked up behind the last item's stores before): forward, backward and second order, 1000
// points along rays 32.4 -> 30.3, 2000 33.7 -> 31.3, 5003 36.2 -> 35.2, uniform 42.7 -> 41.4; points packed into a fifth or a twentieth of the cube's side lose the time of an
// item, 5003 backward 33.5 -> 35.2 and 55.2 -> 56.1: a workgroup with a full bucket has another one to do.  (Drawn from the queue, late where an item is long, those take 33.0 and
// 57.4, but 5003 along rays 19.2 -> 21.4, the way to the counter and to the bounds behind it; full buckets' kinds a workgroup each, the others in turn: 21.1.)  Half the sums and threads, seven
// workgroups to a CU: 5003 along rays 32.6, but 6000 points of a cube's fifth 17.7 -> 31.9, whose buckets hold more records than there are sums then.
constexpr uint32_t FEW_BLOCK = 512, FEW_WORDS = 5120;
constexpr uint32_t FEW_AT_A_TIME = 1024;                            // workgroups of a launch: what runs at one time (a multiple of the XCDs)
constexpr uint32_t FEW_TILES = 64;                                  // a lane of every wave looks up one tile's run
constexpr uint32_t FEW_CLAIMS = (FEW_WORDS - BKT_ENTRIES / 4) / 2;  // sums of both features, beside the table of 16-bit claims
constexpr uint32_t FEW_RANGE = FEW_WORDS * 16 / 33 / 8 * 8;          // entries of an image: two sums and four bits of marks each
constexpr uint32_t FEW_PAIRS = 768;                                 // pair records of a bucket, on average, in a batch that takes the kernel (batch_buckets)

// Here x * 2^32 as a two's complement 64-bit integer, for any finite fp16 value x: the high word is floor(x), the low word the rest, both exact; zero for what is no number.  (Five instructions and no
// branch, whatever the value: a few records a thread, whose latency counts.)
__device__ __forceinline__ unsigned long long few_to_fixed(float x) {
	const float fl = floorf(x);
	const uint32_t hi = (uint32_t)(int32_t)fl, lo = (uint32_t)((x - fl) * 4294967296.f);
	return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ float few_from_fixed(unsigned long long q) { return from_fixed(q) * (FIX_SCALE / 4294967296.f); }

// A bucket's records, numbered through its tiles' runs.
struct N2FewRuns {
	uint32_t first, upto, total;  // lane t: where tile t's run starts in its slot, records in the tiles up to t; all records
	// the tile of record r < total and its place in the tile's slot (by all lanes of the wave)
	__device__ __forceinline__ void find(uint32_t r, uint32_t& tile, uint32_t& at) const {
		uint32_t t = 0;
#pragma unroll
		for (uint32_t s = FEW_TILES / 2; s > 0; s >>= 1) t += r >= n2_lane_value(upto, t + s - 1u) ? s : 0u;
		// (every lane takes part in the exchanges: a lane that a branch had left out would pass nothing on)
		const uint32_t begin = n2_lane_value(first, t), below = n2_lane_value(upto, t - 1u);
		tile = t;
		at = begin + r - (t > 0u ? below : 0u);
	}
};

template <bool PAIR>
__device__ __forceinline__ void grid_reduce_few_bucket(const uint32_t slot_records, const uint32_t tiles, const N2ReduceItem& it,
                                                       const uint32_t* __restrict__ rec_vals, const uint16_t* __restrict__ rec_keys,
                                                       const uint32_t two, __half2* __restrict__ grads, const bool accumulate, unsigned long long* mem) {
	typedef typename std::conditional<PAIR, uint2, uint32_t>::type value;
	constexpr uint32_t EACH = PAIR ? 2u : 1u;                                               // entries of a record
	constexpr uint32_t K = (FEW_CLAIMS / EACH + FEW_BLOCK - 1u) / FEW_BLOCK;  // records of a thread that may claim
	const size_t level_tile0 = (size_t)it.l.level * tiles;
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t left = min(it.l.bucket_entries, it.l.entries - it.bucket * it.l.bucket_entries);  // entries of the bucket (a level's are a multiple of eight)
	__half2* G = grads + it.l.offset + it.bucket * it.l.bucket_entries;
	const bool claims = it.l.bucket_entries > FEW_RANGE;
	typedef uint32_t wide __attribute__((ext_vector_type(4)));
	if (claims && !accumulate)
		for (uint32_t e = threadIdx.x * 4u; e < left; e += FEW_BLOCK * 4u) *reinterpret_cast<wide*>(G + e) = wide(0u);
	N2FewRuns runs;
	runs.first = two & 0xFFFFu;
	const uint32_t own = lane < tiles ? (two >> 16) - runs.first : 0u;
	runs.upto = n2_wave_prefix(own);
	runs.total = __builtin_amdgcn_readlane(runs.upto, 63);
	auto load = [&](uint32_t r, uint32_t& key, value& v) {
		uint32_t tile, at;
		runs.find(r, tile, at);
		const size_t slot = level_tile0 * slot_records;
		const uint32_t record = tile * (slot_records / EACH) + at;
		key = rec_keys[slot + record];
		v = reinterpret_cast<const value*>(rec_vals + slot)[record];
	};
	auto places = [&](uint32_t key, uint32_t (&e)[EACH]) {
		if constexpr (PAIR) {
			e[0] = key & (BKT_ENTRIES - 1u);
			e[1] = e[0] ^ ((2u << (key >> BKT_SHIFT)) - 1u);  // x ^ (x + 1) = 2^(t+1) - 1
		} else e[0] = key;
	};
	auto word = [](const value& v, uint32_t q) {
		if constexpr (sizeof(value) == 8) return q ? v.y : v.x;
		else return v;
	};
	auto sum_of = [&](uint32_t old, unsigned long long a, unsigned long long b, uint32_t marks) {
		const float2 f = accumulate ? __half22float2(*reinterpret_cast<const __half2*>(&old)) : make_float2(0.f, 0.f);
		float2 sum = make_float2(few_from_fixed(a), few_from_fixed(b));
		if (marks != 0u) sum = marked_sums(sum, marks);
		const float2 all = added_to(sum, f);
		return __floats2half2_rn(all.x, all.y);
	};
	// adds a record's two values; `mark` leaves the marks of infinite ones
	auto add = [&](unsigned long long* x, unsigned long long* y, uint32_t raw, auto mark) __attribute__((always_inline)) {
		const float2 f = __half22float2(*reinterpret_cast<const __half2*>(&raw));
		if (fabsf(f.x) == __builtin_inff() || fabsf(f.y) == __builtin_inff()) mark(infinite_mark(f.x, f.y));  // (whatever it adds to its sum, the mark stands for it)
		atomicAdd(x, few_to_fixed(f.x));
		atomicAdd(y, few_to_fixed(f.y));
	};
	if (claims && runs.total * EACH <= FEW_CLAIMS) {
		uint16_t* claim = reinterpret_cast<uint16_t*>(mem);  // a record's number, and from 2^12 on the entry's marks
		constexpr uint32_t NUMBERS = (1u << 12) - 1u;
		static_assert(FEW_CLAIMS <= NUMBERS, "the numbers of records leave room for the marks");
		unsigned long long* acc = mem + BKT_ENTRIES / 4;
		uint32_t key[K], e[K][EACH], old[K][EACH];
		value v[K];
#pragma unroll
		for (uint32_t k = 0; k < K; ++k) {
			const uint32_t r = threadIdx.x + k * FEW_BLOCK;
			if (k * FEW_BLOCK < runs.total) load(min(r, runs.total - 1u), key[k], v[k]);
		}
#pragma unroll
		for (uint32_t k = 0; k < K; ++k) {
			const uint32_t r = threadIdx.x + k * FEW_BLOCK;
			if (r >= runs.total) break;
			places(key[k], e[k]);
#pragma unroll
			for (uint32_t q = 0; q < EACH; ++q) {
				claim[e[k][q]] = (uint16_t)(r * EACH + q);
				acc[r * EACH + q] = 0ull;
				acc[FEW_CLAIMS + r * EACH + q] = 0ull;
			}
		}
		__syncthreads();
#pragma unroll
		for (uint32_t k = 0; k < K; ++k) {
			if (threadIdx.x + k * FEW_BLOCK >= runs.total) break;
#pragma unroll
			for (uint32_t q = 0; q < EACH; ++q) {
				const uint32_t by = claim[e[k][q]] & NUMBERS;
				add(&acc[by], &acc[FEW_CLAIMS + by], word(v[k], q), [&](uint32_t m) { atomicOr(reinterpret_cast<uint32_t*>(mem) + e[k][q] / 2u, m << (e[k][q] % 2u * 16u + 12u)); });
				old[k][q] = accumulate && by == (threadIdx.x + k * FEW_BLOCK) * EACH + q && e[k][q] < left ? *reinterpret_cast<const uint32_t*>(G + e[k][q]) : 0u;
			}
		}
		__syncthreads();
#pragma unroll
		for (uint32_t k = 0; k < K; ++k) {
			const uint32_t r = threadIdx.x + k * FEW_BLOCK;
			if (r >= runs.total) break;
#pragma unroll
			for (uint32_t q = 0; q < EACH; ++q) {
				const uint32_t id = r * EACH + q, by = claim[e[k][q]];
				const unsigned long long x = acc[id], y = acc[FEW_CLAIMS + id];
				if ((by & NUMBERS) != id || e[k][q] >= left) continue;
				G[e[k][q]] = sum_of(old[k][q], x, y, by >> 12);
			}
		}
		return;
	}
	uint32_t* const marks = reinterpret_cast<uint32_t*>(mem + 2u * FEW_RANGE);
	static_assert(2u * FEW_RANGE * sizeof(*mem) + FEW_RANGE / MARKS_PER_WORD * sizeof(*marks) <= FEW_WORDS * sizeof(*mem), "an image and its marks");
	for (uint32_t from = 0; from < left; from += FEW_RANGE) {
		const uint32_t n = min(FEW_RANGE, left - from);
		for (uint32_t e = threadIdx.x; e < n; e += FEW_BLOCK) { mem[e] = 0ull; mem[FEW_RANGE + e] = 0ull; }
		if (threadIdx.x < FEW_RANGE / MARKS_PER_WORD) marks[threadIdx.x] = 0u;
		static_assert(FEW_RANGE / MARKS_PER_WORD <= FEW_BLOCK, "a word of marks to a thread");
		__syncthreads();
		for (uint32_t r = threadIdx.x; __any(r < runs.total); r += FEW_BLOCK) {
			uint32_t key, e[EACH];
			value v;
			load(min(r, runs.total - 1u), key, v);
			places(key, e);
#pragma unroll
			for (uint32_t q = 0; q < EACH; ++q) {
				const uint32_t at = e[q] - from;
				if (r >= runs.total || at >= n) continue;
				add(&mem[at], &mem[FEW_RANGE + at], word(v, q), [&](uint32_t m) { atomicOr(&marks[at / MARKS_PER_WORD], m << (at % MARKS_PER_WORD * 4u)); });
			}
		}
		__syncthreads();
		for (uint32_t e = threadIdx.x * 4u; e < n; e += FEW_BLOCK * 4u) {
			wide* at = reinterpret_cast<wide*>(G + from + e);
			const wide old = accumulate ? *at : wide(0u);
			wide out;
			const uint32_t four_marks = marks[e / MARKS_PER_WORD] >> (e % MARKS_PER_WORD * 4u);
#pragma unroll
			for (uint32_t q = 0; q < 4; ++q) {
				const __half2 h = sum_of(old[q], mem[e + q], mem[FEW_RANGE + e + q], four_marks >> (q * 4u) & 15u);
				out[q] = *reinterpret_cast<const uint32_t*>(&h);
			}
			*at = out;
		}
		__syncthreads();
	}
}

// A workgroup takes the items of its number, that and a round of workgroups further, ... (if the launch has fewer workgroups than items); where the next one's runs lie is on
// its way meanwhile.
__global__ void __launch_bounds__(FEW_BLOCK, 8) grid_reduce_few_kernel(N2BucketPlan plan, uint32_t tiles, uint32_t slot_records,
                                                                    const uint32_t* __restrict__ rec_vals, const uint16_t* __restrict__ rec_keys,
                                                                    const uint16_t* __restrict__ offsets, __half2* __restrict__ grads, int accumulate) {
	__shared__ __align__(16) unsigned long long mem[FEW_WORDS];
	const uint32_t lane_end = n2_lane_end(plan), items = plan.begin[N2_MAX_LEVELS], lane = threadIdx.x & 63u;
	auto bounds = [&](const N2ReduceItem& it) __attribute__((always_inline)) {  // of the bucket's run in tile `lane`
		uint32_t two;
		__builtin_memcpy(&two, offsets + ((size_t)it.l.level * tiles + min(lane, tiles - 1u)) * (BKT_MAX + 1) + it.bucket, sizeof(two));
		return two;
	};
	N2ReduceItem it = n2_reduce_item(plan, lane_end, blockIdx.x);
	uint32_t two = bounds(it);
	for (uint32_t item = blockIdx.x;;) {
		const uint32_t next = item + gridDim.x;
		const N2ReduceItem next_it = n2_reduce_item(plan, lane_end, min(next, items - 1u));
		const uint32_t next_two = bounds(next_it);
		if (it.l.pair) grid_reduce_few_bucket<true>(slot_records, tiles, it, rec_vals, rec_keys, two, grads, accumulate != 0, mem);
		else grid_reduce_few_bucket<false>(slot_records, tiles, it, rec_vals, rec_keys, two, grads, accumulate != 0, mem);
		if (next >= items) return;
		__syncthreads();  // the sums have been read
		item = next;
		it = next_it;
		two = next_two;
	}
}

// Split buckets: the sum of a bucket's G partial images in a fixed order (n2_image_combine_unit, slab_reduce.h: with the
// images added one after the other by one thread the launch was a chain of memory round trips, 9 us for 5 MB).  Run as units
// of the optimiser's kernel instead of a launch of its own it shortens the training step by 0.9 us (measured): not built.
// (Doing this in the reduce kernel, by the workgroup of a bucket that finishes last, needs two device-scope fences per
// workgroup, which write back and invalidate the L2s: the scatter took 150 us longer.  Packed fp16 atomics into the
// gradient buffer cost nothing extra but add in arrival order.)
static_assert(BKT_ENTRIES % N2_CMB_ENTRIES == 0, "whole units per bucket");
__global__ void __launch_bounds__(256) grid_combine_kernel(N2ImageCombine plan) {
	__shared__ float2 part[N2_CMB_SLICES][N2_CMB_ENTRIES];
	n2_image_combine_unit(plan, blockIdx.x, part, [](const _Float16*, _Float16) {});
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------
static uint32_t level_mode(uint32_t res, uint32_t entries) {
	// Mirror of the reference index rule: add dimensions while the running
	// stride still fits into the level; hashed iff the final stride exceeds it.
	uint64_t stride = 1;
	for (int d = 0; d < 3 && stride <= entries; ++d) stride *= res;
	const bool hashed = entries < stride;
	const bool pow2 = (entries & (entries - 1u)) == 0;
	if (hashed) return pow2 ? N2_LEVEL_HASH : N2_LEVEL_HASH_MOD;
	const uint64_t r = res;
	const uint64_t max_index = r + r * r + r * r * r;  // every coordinate at most res
	return (max_index < 2ull * entries) ? N2_LEVEL_DENSE : N2_LEVEL_DENSE_MOD;
}

N2_API int n2_grid_create(uint32_t n_levels, uint32_t n_features_per_level, uint32_t log2_hashmap_size,
                          uint32_t base_resolution, float per_level_scale, n2_grid_t** out) {
	N2_REQUIRE(out != nullptr, "n2_grid_create: out is null");
	*out = nullptr;
	N2_REQUIRE(n_levels >= 1 && n_levels <= N2_MAX_LEVELS, "n2_grid_create: n_levels %u outside [1, %u]", n_levels, N2_MAX_LEVELS);
	if (n_features_per_level != 2) {
		n2_set_error("n2_grid_create: only n_features_per_level = 2 is implemented (got %u)", n_features_per_level);
		return N2_ERR_UNSUPPORTED;
	}
	N2_REQUIRE(log2_hashmap_size >= 3 && log2_hashmap_size <= 28, "n2_grid_create: log2_hashmap_size %u outside [3, 28]", log2_hashmap_size);
	N2_REQUIRE(base_resolution >= 1 && per_level_scale >= 1.0f, "n2_grid_create: base_resolution >= 1 and per_level_scale >= 1 required");
	n2_grid* g = new (std::nothrow) n2_grid();
	N2_REQUIRE(g != nullptr, "n2_grid_create: out of host memory");
	g->n_features = n_features_per_level;
	g->tab.n_levels = n_levels;
	g->tab.n_features = n_features_per_level;
	g->tab.max_level = 1.0f;
	g->tab.max_level_gpu = nullptr;
	g->tab.valid_levels = n_levels;
	g->tab.active_levels = n_levels;
	g->tab.pair_levels = 0;
	g->base_valid_level_scale = 1.0f;
	g->valid_level_scale = 0.0f;
	g->base_training_step = 0;
	g->training_step = 0;
	uint64_t off = 0;
	const float log2_b = std::log2(per_level_scale);
	for (uint32_t l = 0; l < n_levels; ++l) {
		const float s = exp2f((float)l * log2_b) * (float)base_resolution - 1.0f;
		const uint32_t res = (uint32_t)ceilf(s) + 1u;
		const uint32_t max_params = 0xFFFFFFFFu / 2u;
		const double cube = (double)res * (double)res * (double)res;
		uint32_t n = cube > (double)max_params ? max_params : res * res * res;
		n = (n + 7u) / 8u * 8u;
		const uint32_t cap = 1u << log2_hashmap_size;
		if (n > cap) n = cap;
		g->tab.scale[l] = s;
		g->tab.resolution[l] = res;
		g->tab.entries[l] = n;
		g->tab.offset[l] = (uint32_t)off;
		g->tab.mode[l] = level_mode(res, n);
		// hashed levels gather from all over their table; the dense ones mostly hit lines their neighbours fetched
		g->level_cost[l] = (g->tab.mode[l] == N2_LEVEL_HASH || g->tab.mode[l] == N2_LEVEL_HASH_MOD) ? 1.0f : 0.6f;
		// pair records in the bucketed scatter: x and x + 1 must stay below the bucket size (see grid_bin_kernel)
		if (g->tab.mode[l] == N2_LEVEL_HASH && res <= PAIR_MAX_CELL + 1u && n >= BKT_ENTRIES) g->tab.pair_levels |= 1u << l;
		off += n;
	}
	if (off * n_features_per_level > 0x7FFFFFFFull) {
		delete g;
		n2_set_error("n2_grid_create: %llu parameters exceed the 2^31 limit", (unsigned long long)(off * n_features_per_level));
		return N2_ERR_UNSUPPORTED;
	}
	g->tab.offset[n_levels] = (uint32_t)off;
	g->n_params = (uint32_t)off * n_features_per_level;
	g->params = nullptr;
	g->grads = nullptr;
	g->ws = nullptr;
	g->ws_bytes = 0;
	g->ws_max_points = 0;
	g->ws_partials = 0;
	g->lattice_order = false;
	g->costs_set = false;
	*out = g;
	return N2_OK;
}

N2_API void n2_grid_destroy(n2_grid_t* grid) { delete grid; }
const N2LevelTable* n2_grid_table(const n2_grid_t* grid) { return &grid->tab; }
const __half2* n2_grid_params(const n2_grid_t* grid) { return grid->params; }
bool n2_grid_lattice_order(const n2_grid_t* grid) { return grid->lattice_order; }
N2_API uint32_t n2_grid_n_params(const n2_grid_t* grid) { return grid ? grid->n_params : 0; }
N2_API uint32_t n2_grid_output_width(const n2_grid_t* grid) { return grid ? grid->tab.n_levels * grid->n_features : 0; }
N2_API uint32_t n2_grid_n_levels(const n2_grid_t* grid) { return grid ? grid->tab.n_levels : 0; }

N2_API int n2_grid_level_table(const n2_grid_t* grid, float* scale, uint32_t* resolution, uint32_t* entries, uint32_t* offset) {
	N2_REQUIRE(grid != nullptr, "n2_grid_level_table: grid is null");
	for (uint32_t l = 0; l < grid->tab.n_levels; ++l) {
		if (scale) scale[l] = grid->tab.scale[l];
		if (resolution) resolution[l] = grid->tab.resolution[l];
		if (entries) entries[l] = grid->tab.entries[l];
		if (offset) offset[l] = grid->tab.offset[l];
	}
	if (offset) offset[grid->tab.n_levels] = grid->tab.offset[grid->tab.n_levels];
	return N2_OK;
}

N2_API int n2_grid_set_level_costs(n2_grid_t* grid, const float* costs) {
	N2_REQUIRE(grid != nullptr && costs != nullptr, "n2_grid_set_level_costs: null argument");
	for (uint32_t l = 0; l < grid->tab.n_levels; ++l) {
		N2_REQUIRE(costs[l] > 0.f && costs[l] <= 1e6f, "n2_grid_set_level_costs: cost of level %u must be in (0, 1e6]", l);
	}
	for (uint32_t l = 0; l < grid->tab.n_levels; ++l) grid->level_cost[l] = costs[l];
	grid->costs_set = true;
	return N2_OK;
}

// levels in use under the global settings, with the device predicate's arithmetic
static uint32_t count_active_levels(const N2LevelTable& tab) {
	const float limit = (tab.max_level * (float)(tab.n_levels * tab.n_features)) / (float)tab.n_features;
	uint32_t n = 0;
	while (n < tab.n_levels && n < tab.valid_levels && !((float)n >= limit + 1e-3f)) ++n;  // both rules cut a suffix of the levels
	return n;
}

N2_API int n2_grid_set_max_level(n2_grid_t* grid, float max_level) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_max_level: grid is null");
	N2_REQUIRE(max_level >= 0.f && max_level <= 1000.f, "n2_grid_set_max_level: max_level %g outside [0, 1000]", (double)max_level);
	grid->tab.max_level = max_level;
	grid->tab.active_levels = count_active_levels(grid->tab);
	return N2_OK;
}

N2_API int n2_grid_set_max_level_gpu(n2_grid_t* grid, const float* d_max_level) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_max_level_gpu: grid is null");
	grid->tab.max_level_gpu = d_max_level;
	return N2_OK;
}

N2_API int n2_grid_set_progressive(n2_grid_t* grid, float base_valid_level_scale, float valid_level_scale, uint32_t base_training_step) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_progressive: grid is null");
	N2_REQUIRE(base_valid_level_scale >= 0.f && valid_level_scale >= 0.f, "n2_grid_set_progressive: scales must be >= 0");
	grid->base_valid_level_scale = base_valid_level_scale;
	grid->valid_level_scale = valid_level_scale;
	grid->base_training_step = base_training_step;
	// the levels in use follow from the keys and the training step last set
	return n2_grid_set_training_step(grid, grid->training_step);
}

// levels in use at a training step: the fraction base + scale * (step / base_training_step), whole periods only,
// of all levels, rounded down (after + 1e-3, so that a fraction that reaches 1 up to rounding gives every level),
// at least one level and at most all of them
N2_API int n2_grid_set_training_step(n2_grid_t* grid, uint32_t training_step) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_training_step: grid is null");
	grid->training_step = training_step;
	if (grid->base_training_step == 0) {
		grid->tab.valid_levels = grid->tab.n_levels;
		grid->tab.active_levels = count_active_levels(grid->tab);
		return N2_OK;
	}
	const float fraction = grid->base_valid_level_scale + grid->valid_level_scale * (float)(training_step / grid->base_training_step);
	const float levels = fraction * (float)grid->tab.n_levels + 1e-3f;
	uint32_t n = levels >= (float)grid->tab.n_levels ? grid->tab.n_levels : (uint32_t)levels;
	if (n < 1) n = 1;
	grid->tab.valid_levels = n;
	grid->tab.active_levels = count_active_levels(grid->tab);
	return N2_OK;
}

N2_API uint32_t n2_grid_active_levels(const n2_grid_t* grid) { return grid ? grid->tab.active_levels : 0; }

N2_API int n2_grid_set_point_order(n2_grid_t* grid, int lattice_order) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_point_order: grid is null");
	grid->lattice_order = lattice_order != 0;
	return N2_OK;
}

N2_API int n2_grid_set_params(n2_grid_t* grid, const n2_half* d_params, n2_half* d_gradients) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_params: grid is null");
	N2_REQUIRE(d_params != nullptr, "n2_grid_set_params: d_params is null");
	N2_REQUIRE(reinterpret_cast<uintptr_t>(d_params) % 16 == 0, "n2_grid_set_params: d_params must be 16-byte aligned");
	N2_REQUIRE(reinterpret_cast<uintptr_t>(d_gradients) % 16 == 0, "n2_grid_set_params: d_gradients must be 16-byte aligned");
	grid->params = reinterpret_cast<const __half2*>(d_params);
	grid->grads = reinterpret_cast<__half2*>(d_gradients);
	return N2_OK;
}

// Shared argument checks.  Row offsets are computed in 64 bits on the device;
// the point index itself is 32 bits.
static int check_batch(const n2_grid_t* grid, const char* fn, const float* d_xyz, uint32_t point_stride, uint32_t dim_stride,
                       uint32_t n_points) {
	N2_REQUIRE(grid != nullptr, "%s: grid is null", fn);
	N2_REQUIRE(grid->params != nullptr, "%s: n2_grid_set_params has not been called", fn);
	N2_REQUIRE(d_xyz != nullptr || n_points == 0, "%s: d_xyz is null", fn);
	N2_REQUIRE(point_stride >= 1 && dim_stride >= 1, "%s: strides must be >= 1", fn);
	N2_REQUIRE(n_points <= (1u << 30), "%s: n_points %u exceeds 2^30", fn, n_points);
	return N2_OK;
}

static inline uint32_t n_tiles(uint32_t n_points) { return (n_points + GRID_BLOCK - 1) / GRID_BLOCK; }

// Cuts the level-major list of n_levels x tiles items into N_XCD contiguous pieces of equal estimated cost.
// Returns the length of the longest piece (the launch needs N_XCD times that many workgroups).
static uint32_t make_xcd_plan(const n2_grid_t* grid, uint32_t tiles, N2XcdPlan& plan) {
	const uint32_t L = grid->tab.n_levels;
	double total = 0.0;
	for (uint32_t l = 0; l < L; ++l) total += (double)grid->level_cost[l] * tiles;
	plan.begin[0] = 0;
	uint32_t level = 0, longest = 0;
	double before = 0.0;  // cost of the levels below `level`
	for (uint32_t x = 1; x < N_XCD; ++x) {
		const double target = total * x / N_XCD;
		while (level + 1 < L && before + (double)grid->level_cost[level] * tiles <= target) {
			before += (double)grid->level_cost[level] * tiles;
			++level;
		}
		double in_level = (target - before) / grid->level_cost[level];
		if (in_level < 0.0) in_level = 0.0;
		if (in_level > tiles) in_level = tiles;
		uint32_t b = level * tiles + (uint32_t)(in_level + 0.5);
		if (b < plan.begin[x - 1]) b = plan.begin[x - 1];
		plan.begin[x] = b;
	}
	plan.begin[N_XCD] = L * tiles;
	for (uint32_t x = 0; x < N_XCD; ++x) {
		const uint32_t len = plan.begin[x + 1] - plan.begin[x];
		if (len > longest) longest = len;
	}
	return longest;
}

static int grid_forward(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride,
                        uint32_t dim_stride, uint32_t n_points, n2_half* d_out, float* d_dy_dx, n2_half* d_centred, bool one_reader) {
	if (int rc = check_batch(grid, "n2_grid_forward", d_xyz, point_stride, dim_stride, n_points)) return rc;
	if (n_points == 0) return N2_OK;
	N2_REQUIRE(d_out != nullptr, "n2_grid_forward: d_out is null");
	N2XcdPlan plan;
	N2ProfScope prof(N2_PROF_GRID_FORWARD, n2_stream(stream));
	if (grid->lattice_order && !d_dy_dx && !d_centred) {
		const uint32_t tiles = n_tiles(n_points);
		const dim3 grid_dim(tiles * grid->tab.n_levels);
		grid_forward_point_kernel<<<grid_dim, dim3(GRID_BLOCK), 0, n2_stream(stream)>>>(grid->tab, n_points, tiles, d_xyz, point_stride, dim_stride,
			grid->params, reinterpret_cast<__half*>(d_out));
		N2_LAUNCH_CHECK();
		return N2_OK;
	}
	const uint32_t tiles = (n_points + FWD_POINTS - 1) / FWD_POINTS;
	const N2GatherGrid dealt = n2_gather_grid(N2_ENCODING_XCD_MAX, n_points, grid->tab.n_levels, FWD_POINTS);
	plan.begin[N_XCD] = 0;
	plan.height = dealt.y;
	const dim3 grid_dim = grid->costs_set ? dim3(make_xcd_plan(grid, tiles, plan) * N_XCD) : dim3(dealt.x, dealt.y), block(GRID_BLOCK);
	const uint32_t rows = grid->tab.n_levels * grid->n_features;
	const bool streams = one_reader ? n2_step_jacobian_stores_stream(n_points, rows) : n2_jacobian_streams(n_points, rows);
	auto* const kernel = !d_dy_dx ? grid_forward_kernel<false, false> : streams ? grid_forward_kernel<true, true> : grid_forward_kernel<true, false>;
	kernel<<<grid_dim, block, 0, n2_stream(stream)>>>(grid->tab, plan, n_points, tiles, d_xyz, point_stride, dim_stride, grid->params,
	                                                  reinterpret_cast<__half*>(d_out), d_dy_dx, reinterpret_cast<__half*>(d_centred));
	N2_LAUNCH_CHECK();
	return N2_OK;
}
N2_API int n2_grid_forward(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride,
                           uint32_t dim_stride, uint32_t n_points, n2_half* d_out, float* d_dy_dx) {
	return grid_forward(grid, stream, d_xyz, point_stride, dim_stride, n_points, d_out, d_dy_dx, nullptr, false);
}
int n2_grid_forward_sdf_input(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride, uint32_t dim_stride, uint32_t n_points, n2_half* d_input,
                              float* d_dy_dx, bool one_reader) {
	return grid_forward(grid, stream, d_xyz, point_stride, dim_stride, n_points, d_input ? d_input + (size_t)3 * n_points : nullptr, d_dy_dx, d_input, one_reader);
}

N2_API int n2_grid_corner_indices(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride,
                                  uint32_t dim_stride, uint32_t n_points, uint32_t* d_indices) {
	if (int rc = check_batch(grid, "n2_grid_corner_indices", d_xyz, point_stride, dim_stride, n_points)) return rc;
	if (n_points == 0) return N2_OK;
	N2_REQUIRE(d_indices != nullptr, "n2_grid_corner_indices: d_indices is null");
	const uint32_t tiles = n_tiles(n_points);
	grid_indices_kernel<<<dim3(tiles * grid->tab.n_levels), dim3(GRID_BLOCK), 0, n2_stream(stream)>>>(
		grid->tab, n_points, tiles, d_xyz, point_stride, dim_stride, d_indices);
	N2_LAUNCH_CHECK();
	return N2_OK;
}

static bool uses_bucketed(const n2_grid_t* grid, uint32_t n_points);

// OVERWRITE: the gradient buffer starts from zero.  The bucketed scatter writes every entry itself (with plain stores),
// so only the scatter with atomics needs the buffer cleared beforehand.
static int prepare_grads(n2_grid_t* grid, const char* fn, hipStream_t stream, n2_grad_mode mode, uint32_t n_points) {
	N2_REQUIRE(mode == N2_GRAD_IGNORE || mode == N2_GRAD_OVERWRITE || mode == N2_GRAD_ACCUMULATE, "%s: bad gradient mode %d", fn, (int)mode);
	if (mode == N2_GRAD_IGNORE) return N2_OK;
	N2_REQUIRE(grid->grads != nullptr, "%s: gradient mode %d needs a gradient buffer (n2_grid_set_params)", fn, (int)mode);
	if (mode != N2_GRAD_OVERWRITE) return N2_OK;
	if (!uses_bucketed(grid, n_points)) return n2_fill_zero_u32(stream, grid->grads, (size_t)grid->n_params * sizeof(__half));
	return N2_OK;
}

bool n2_grid_has_gradients(const n2_grid_t* grid) { return grid->params != nullptr && grid->grads != nullptr; }

static inline uint32_t n_pair_tiles(uint32_t n_points) { return (n_points + PAIR_POINTS - 1) / PAIR_POINTS; }
static inline uint32_t bin_per_thread(const n2_grid_t* grid, uint32_t n_points) { return n2_bin_points_per_thread(grid->tab.n_levels, n_points, BIN_BLOCK); }
static inline uint32_t n_bin_tiles(const n2_grid_t* grid, uint32_t n_points) {
	const uint32_t points = bin_points(bin_per_thread(grid, n_points));
	return (n_points + points - 1) / points;
}

static bool bucket_supported(const n2_grid_t* grid) {
	for (uint32_t l = 0; l < grid->tab.n_levels; ++l)
		if (grid->tab.entries[l] > BKT_ENTRIES * BKT_MAX) return false;
	return true;
}
// workspace: the reduce launch's queue, the records' values, their keys, the tiles' bucket offsets, then one fp32 image per (bucket, group) of the
// split buckets
struct BucketCarve {
	uint64_t queue, vals, keys, offsets, partials, total;
};
static BucketCarve bucket_carve(const n2_grid_t* grid, uint32_t max_points, uint32_t images) {
	const uint64_t tiles = n_bin_tiles(grid, max_points), L = grid->tab.n_levels;
	const uint64_t n_rec = L * tiles * bin_records(bin_per_thread(grid, max_points));
	auto up = [](uint64_t x) { return (x + 255) / 256 * 256; };
	BucketCarve c{};
	c.queue = 0;
	c.vals = QUEUE_WORDS * sizeof(uint32_t);
	c.keys = c.vals + n_rec * sizeof(uint32_t);
	c.offsets = c.keys + n_rec * sizeof(uint16_t);
	c.partials = up(c.offsets + L * tiles * (BKT_MAX + 1) * sizeof(uint16_t));
	// (a batch of half as many points per tile has twice the tiles and bucket offsets: the images of a larger one stand behind those, too)
	const uint32_t largest = n2_bin_single_points(grid->tab.n_levels, BIN_BLOCK);
	if (max_points > largest) c.partials = std::max(c.partials, bucket_carve(grid, largest, 0u).partials);
	c.total = up(c.partials + (uint64_t)images * BKT_ENTRIES * sizeof(float2));
	return c;
}

// With a workspace every batch size takes the bucketed scatter, whose result does not depend on the order in which
// workgroups run; the scatter with atomics (no workspace, or more points than it was sized for) sums in arrival order.
static bool uses_bucketed(const n2_grid_t* grid, uint32_t n_points) {
	return grid->grads != nullptr && grid->ws != nullptr && n_points <= grid->ws_max_points && n_points >= 1;
}
// Entries per bucket of a level (log2).  Levels that sort pair records keep 4096-entry buckets (a pair's second entry is
// encoded against that size); the others take the largest size (a power of two, at most 4096 entries and at most BKT_MAX
// buckets) under which a bucket holds at most `target` of the level's 8 records per point, or the smallest there is: small
// dense levels get many small buckets instead of few that outlast the others.  When even the smallest buckets hold more than
// 65536, they stay large and are split.
// The target is 16384 for grid_reduce_kernel (8192 and 32768: the same within 2 %, 65536: 49 us against 36 at 1.2e5 points, where a dense
// level's few workgroups outlast the others) and 512, a record per thread, for grid_reduce_few_kernel.
static uint32_t bucket_shift(const n2_grid_t* grid, uint32_t level, uint32_t n_points, uint32_t target) {
	if ((grid->tab.pair_levels >> level) & 1u) return BKT_SHIFT;
	const uint32_t entries = grid->tab.entries[level];
	const uint64_t records = (uint64_t)n_points * 8;
	for (uint32_t shift = BKT_SHIFT; shift >= BKT_MIN_SHIFT; --shift) {
		const uint32_t nb = (entries + (1u << shift) - 1u) >> shift, finer = (entries + (1u << (shift - 1u)) - 1u) >> (shift - 1u);
		if (nb > BKT_MAX) break;
		if (records < (target + 1ull) * nb || (records < 65537ull * nb && (shift == BKT_MIN_SHIFT || finer > BKT_MAX))) return shift;
	}
	return BKT_SHIFT;
}
static inline uint32_t bucket_count(uint32_t entries, uint32_t shift) { return (entries + (1u << shift) - 1u) >> shift; }

// A batch's buckets.  few: it takes grid_reduce_few_kernel.  That is where on average its buckets hold no more records than three quarters of the claims there
// are on levels of pair records, and four times as many on the others, whose buckets are the smallest there can be: with the default table up to 24 576
// points.  Encoding forward and backward in us, grid_reduce_kernel (before it drew its buckets) | grid_reduce_few_kernel: uniform 600 30.1 | 25.5, 5003 32.6 | 27.5,
// 8192 33.5 | 29.1, 12 288 35.5 | 32.7, 16 384 37.7 | 37.0, 20 000 37.5 | 36.4, 24 576 40.4 | 40.5; along rays 3000 28.7 | 25.2, 16 384 34.9 | 31.1, 20 000 34.0 | 29.5,
// 24 576 36.0 | 32.0, 32 768 41.8 | 43.2.
// groups: workgroups a bucket is split over; images: fp32 images of all split buckets (never more for a smaller batch: the groups per bucket grow with it).
struct BatchBuckets {
	bool few;
	uint8_t shift[N2_MAX_LEVELS];
	uint32_t count[N2_MAX_LEVELS], groups[N2_MAX_LEVELS], images;
};
static BatchBuckets batch_buckets(const n2_grid_t* grid, uint32_t n_points) {
	BatchBuckets b;
	const uint32_t tiles = n_bin_tiles(grid, n_points), L = grid->tab.n_levels;
	b.few = tiles <= FEW_TILES;
	for (uint32_t l = 0; l < L && b.few; ++l) {
		const bool pair = (grid->tab.pair_levels >> l) & 1u;
		b.shift[l] = (uint8_t)bucket_shift(grid, l, n_points, FEW_BLOCK);
		b.few = (uint64_t)n_points * (pair ? 4u : 8u) <= (uint64_t)bucket_count(grid->tab.entries[l], b.shift[l]) * (pair ? FEW_PAIRS : 4u * FEW_PAIRS);
	}
	b.images = 0;
	for (uint32_t l = 0; l < L; ++l) {
		if (!b.few) b.shift[l] = (uint8_t)bucket_shift(grid, l, n_points, 16384u);
		b.count[l] = bucket_count(grid->tab.entries[l], b.shift[l]);
		const uint64_t per_bucket = (uint64_t)n_points * 8 / b.count[l];
		b.groups[l] = std::max<uint32_t>(1u, std::min<uint64_t>((per_bucket + 65535) / 65536, std::min(N2_CMB_MAX_GROUPS, tiles)));
		if (b.groups[l] > 1) b.images += b.count[l] * b.groups[l];
	}
	return b;
}

N2_API uint64_t n2_grid_workspace_bytes(const n2_grid_t* grid, uint32_t max_points) {
	if (!grid || !bucket_supported(grid)) return 0;
	return bucket_carve(grid, max_points, batch_buckets(grid, max_points).images).total;
}

N2_API int n2_grid_set_workspace(n2_grid_t* grid, void* d_workspace, uint64_t n_bytes, uint32_t max_points) {
	N2_REQUIRE(grid != nullptr, "n2_grid_set_workspace: grid is null");
	if (d_workspace == nullptr) {
		grid->ws = nullptr; grid->ws_bytes = 0; grid->ws_max_points = 0;
		return N2_OK;
	}
	N2_REQUIRE(reinterpret_cast<uintptr_t>(d_workspace) % 256 == 0, "n2_grid_set_workspace: workspace must be 256-byte aligned");
	N2_REQUIRE(n_bytes >= n2_grid_workspace_bytes(grid, max_points), "n2_grid_set_workspace: %llu bytes given, %llu needed for %u points",
	           (unsigned long long)n_bytes, (unsigned long long)n2_grid_workspace_bytes(grid, max_points), max_points);
	grid->ws = reinterpret_cast<unsigned char*>(d_workspace);
	grid->ws_bytes = n_bytes;
	grid->ws_max_points = bucket_supported(grid) ? max_points : 0;
	grid->ws_partials = bucket_carve(grid, max_points, 0u).partials;
	return N2_OK;
}

// What a scatter is asked to do beside it: the input gradient (first order alone: dL_dx set), or a slab summation (first and second order together
// and no dL_ddLdy).
struct N2ScatterRider {
	const float* dy_dx = nullptr;
	float* dL_dx = nullptr;
	N2SlabReduce sums = {};
};

// Parameter gradients through the bin + reduce kernels.  The gradient buffer has been zeroed for OVERWRITE.
static int launch_bucketed(n2_grid_t* grid, hipStream_t s, const float* d_xyz, uint32_t point_stride, uint32_t dim_stride, uint32_t n_points,
                           const __half* dL_dy, const float* v, const __half* g2, __half* dL_ddLdy, bool accumulate,
                           const uint32_t* index, uint32_t n_cols, const N2ScatterRider& rider) {
	const uint32_t tiles = n_bin_tiles(grid, n_points), per = bin_per_thread(grid, n_points), L = grid->tab.n_levels;
	const bool first = dL_dy != nullptr, second = v != nullptr, out = dL_ddLdy != nullptr;
	N2_REQUIRE(rider.dL_dx == nullptr || (first && !second), "n2_grid: the input gradient goes with a first-order scatter");
	N2_REQUIRE(rider.sums.units == 0 || (first && second && !out), "n2_grid: a slab summation goes with a scatter of both orders and no dL_ddLdy");
	const dim3 bd(BIN_BLOCK);
	// The records of this batch are packed as for a workspace of exactly this size (values, keys, offsets one behind the
	// other); the images of split buckets stand where the workspace's own size put them.
	const BucketCarve now = bucket_carve(grid, n_points, 0u);
	uint32_t* queue = reinterpret_cast<uint32_t*>(grid->ws + now.queue);
	uint32_t* rec_vals = reinterpret_cast<uint32_t*>(grid->ws + now.vals);
	uint16_t* rec_keys = reinterpret_cast<uint16_t*>(grid->ws + now.keys);
	uint16_t* offsets = reinterpret_cast<uint16_t*>(grid->ws + now.offsets);
	float2* partials = reinterpret_cast<float2*>(grid->ws + grid->ws_partials);
	N2BucketPlan plan{};
	uint32_t wg = 0, images = 0, split = 0;
	N2LevelTable tab = grid->tab;  // with this launch's bucket sizes
	// At least four runs, or parts of them, for a wave of a reduce workgroup.  One | two | four | eight, backward in us: 30 000 points uniform 35.6 | 35.3 | 35.9 | 36.9, in a box of a fifth
	// of the cube's side 71.9 | 72.0 | 70.4 | 70.0, 52 344 uniform 40.9 | 40.9 | 40.9 | 41.6, with tables of 2^14 entries a level 42.3 | 42.2 | 42.3 | 41.3.
	uint32_t part_shift = 0;
	while (part_shift < 6u && tiles << part_shift < RED_BLOCK / 64u * 4u) ++part_shift;
	const BatchBuckets buckets = batch_buckets(grid, n_points);
	uint32_t split_begin[N2_MAX_LEVELS], part_begin[N2_MAX_LEVELS];
	for (uint32_t l = 0; l < L; ++l) {
		tab.bucket_shift[l] = buckets.shift[l];
		part_begin[l] = images;
		split_begin[l] = split;
		if (buckets.groups[l] > 1) { images += buckets.count[l] * buckets.groups[l]; split += buckets.count[l]; }
	}
	// The kind whose largest items, on average, have more additions comes first, or a launch ends with one of them that has just begun.  Levels of pairs have those where
	// their buckets are full (tables of 2^14 and 2^16 entries a level, whose pairs' items have 65 536 additions of 2^18 points, the others' 16 384 to 27 000): single ones
	// first | pairs first, the launch in us, 2^18 points along rays 48.3 | 30.8 and 52.8 | 36.1, uniform 52.3 | 48.6 (2^16).  With the default table they have as many or fewer:
	// 2^18 uniform points 52.6 | 56.1, along rays 45.4 | 46.5, 52 344 18.9 | 19.9.
	uint64_t largest[2] = {0, 0};
	for (uint32_t l = 0; l < L; ++l) {
		uint64_t& most = largest[(tab.pair_levels >> l) & 1u];
		most = std::max(most, (uint64_t)n_points * 8u / (buckets.count[l] * buckets.groups[l]));
	}
	const bool pairs_first = !buckets.few && largest[1] > largest[0];  // (the kernel for few records has them behind the others always: its items are small)
	uint32_t place = 0;
	for (uint32_t kind = 0; kind < 2; ++kind) {
		const uint32_t pair = pairs_first == (kind == 0u);
		if (kind) plan.second_from = wg;
		for (uint32_t l = 0; l < L; ++l) {
			if (((tab.pair_levels >> l) & 1u) != pair) continue;
			plan.begin[place] = wg;
			plan.at[place++] = {l, buckets.count[l], buckets.groups[l], part_begin[l], 1u << buckets.shift[l], tab.entries[l], tab.offset[l], pair};
			wg += buckets.count[l] * buckets.groups[l];
		}
	}
	for (uint32_t end = place; end <= N2_MAX_LEVELS; ++end) plan.begin[end] = wg;
	auto bin = [&](auto per_thread) {
		constexpr uint32_t PER = decltype(per_thread)::value;
		// (the other launches' records exceed the card's memory before their threads exceed 32 bits: 8 and 9 threads a point of sixteen levels)
		const auto launch_dim = [](auto ride, uint32_t blocks) {
			if (!std::is_same<decltype(ride), N2RideSecond>::value) return dim3(blocks);
			const N2GatherGrid g = n2_rows_of_blocks(blocks, BIN_BLOCK);
			return dim3(g.x, g.y);
		};
#define LAUNCH(F, S, STREAM, RIDE, BLOCKS) grid_bin_kernel<PER, F, S, STREAM><<<launch_dim(RIDE, BLOCKS), bd, 0, s>>>(tab, 0u, n_points, tiles, d_xyz, point_stride, dim_stride, dL_dy, v, g2, \
                                                                                                    grid->params, rec_vals, rec_keys, offsets, queue, index, n_cols, RIDE)
		const uint32_t blocks = tiles * L;
		const N2RideNone none;
		// The rows of a fused backward are the step's own, and this is their last use: past the caches, where each wave of 64 points takes whole lines of them.  In us, cached | streamed: the
		// field's forward and backward 2^18 240.9 | 237.4, SDF network's step 2^18 253.4 | 250.4, training step 2^18 338.4 | 336.5, trained 492.0 | 492.3, 2^16 184.1 | 183.6; of lines
		// that two waves share, field 200 008 198.8 | 202.0, SDF network 100 008 131.3 | 133.3.  (The encoding's own backward reads a caller's rows, beside others that do.)
		const bool rows_stream = n2_rows_of_whole_lines(n_points, 2u) && (!index || n2_rows_of_whole_lines(n_cols, 2u));
		if (rider.dL_dx != nullptr) {  // (first order alone)
			const N2Turns turns = n2_turns(blocks, (n_points + BIN_BLOCK - 1) / BIN_BLOCK, 1u);
			const uint32_t rows = L * grid->n_features;
			if (n2_jacobian_streams(n_points, rows)) LAUNCH(true, false, false, (N2RideInput<true>{rider.dy_dx, rider.dL_dx, rows, turns.every}), turns.blocks);
			else LAUNCH(true, false, false, (N2RideInput<false>{rider.dy_dx, rider.dL_dx, rows, turns.every}), turns.blocks);
		} else if (rider.sums.units > 0) {  // (both orders)
			const uint32_t riders = (rider.sums.units + BIN_BLOCK / 256 - 1) / (BIN_BLOCK / 256);
			if (rows_stream) LAUNCH(true, true, true, (N2RideSums{rider.sums, riders}), riders + blocks);
			else LAUNCH(true, true, false, (N2RideSums{rider.sums, riders}), riders + blocks);
		} else if (out) {
			const N2GatherGrid g = n2_gather_grid(N2_ENCODING_XCD_MAX, n_points, L, BIN_BLOCK);
			const N2Turns turns = n2_turns(g.x * g.y, blocks, N_XCD);
			const N2RideSecond ride{dL_ddLdy, g.x * g.y, turns.every, (n_points + BIN_BLOCK - 1) / BIN_BLOCK, g.y};
			if (first) LAUNCH(true, true, false, ride, turns.blocks);
			else LAUNCH(false, true, false, ride, turns.blocks);
		} else if (first && second && rows_stream) LAUNCH(true, true, true, none, blocks);
		else if (first && second) LAUNCH(true, true, false, none, blocks);
		else if (second) LAUNCH(false, true, false, none, blocks);
		else LAUNCH(true, false, false, none, blocks);
#undef LAUNCH
	};
	if (per == 1u) bin(std::integral_constant<uint32_t, 1>());
	else bin(std::integral_constant<uint32_t, 2>());
	N2_LAUNCH_CHECK();
	if (buckets.few) {
		// In turn, unless a workgroup with more than three records a thread of a claimed bucket would have another item to do.  Default table (its fifth level, from 16 897 points on),
		// backward in us, a workgroup an item | in turn: uniform 12 000 points 26.2 | 25.2, 16 384 29.9 | 29.6, 18 000 31.9 | 34.2, 20 000 32.4 | 35.0, 24 000 35.5 | 38.1, along rays
		// 12 000 22.2 | 21.8, 16 384 24.6 | 23.7, 18 000 25.3 | 24.9, 24 000 28.4 | 28.0, accumulating 16 384 24.6 | 23.6, 18 000 25.8 | 24.8, 24 000 28.4 | 27.3; with twelve of its
		// levels, few enough that those workgroups have one item, uniform 18 000 28.8 | 28.5, 24 000 32.4 | 32.5, along rays 21.0 | 20.4, 23.4 | 22.4.
		bool in_turn = true;
		for (uint32_t l = 0; l < place; ++l) {
			const N2BucketPlan::Level& at = plan.at[l];
			if (!at.pair && at.bucket_entries > FEW_RANGE && (uint64_t)n_points * 8u > 3ull * FEW_BLOCK * at.n_buckets && plan.begin[l] + FEW_AT_A_TIME < wg) in_turn = false;
		}
		grid_reduce_few_kernel<<<dim3(in_turn && wg > FEW_AT_A_TIME ? FEW_AT_A_TIME : wg), dim3(FEW_BLOCK), 0, s>>>(plan, tiles, bin_records(per), rec_vals, rec_keys, offsets, grid->grads, accumulate ? 1 : 0);
	} else {
		auto* const kernel = pairs_first ? (accumulate ? grid_reduce_kernel<true, true> : grid_reduce_kernel<false, true>) : accumulate ? grid_reduce_kernel<true, false> : grid_reduce_kernel<false, false>;
		kernel<<<dim3(wg < RED_AT_A_TIME ? wg : RED_AT_A_TIME), dim3(RED_BLOCK), 0, s>>>(plan, tiles, bin_records(per), part_shift, rec_vals, rec_keys, offsets, grid->grads, partials, queue);
	}
	N2_LAUNCH_CHECK();
	if (split > 0) {
		N2ImageCombine cmb{};
		cmb.images = partials;
		cmb.grads = reinterpret_cast<_Float16*>(grid->grads);
		cmb.bucket_entries = BKT_ENTRIES;
		cmb.accumulate = accumulate ? 1 : 0;
		uint32_t k = 0;  // the split levels, in order
		for (uint32_t l = 0; l < L; ++l) {
			if (buckets.groups[l] <= 1) continue;
			N2_REQUIRE(tab.bucket_shift[l] == BKT_SHIFT, "grid scatter: level %u splits buckets of %u entries", l, 1u << tab.bucket_shift[l]);
			cmb.split_begin[k] = split_begin[l]; cmb.groups[k] = buckets.groups[l]; cmb.part_begin[k] = part_begin[l];
			cmb.entries[k] = grid->tab.entries[l]; cmb.offset[k] = grid->tab.offset[l];
			++k;
		}
		cmb.n_levels = k;
		for (uint32_t l = k; l <= N2_CMB_LEVELS; ++l) cmb.split_begin[l] = split;
		cmb.units = split * (BKT_ENTRIES / N2_CMB_ENTRIES);
		grid_combine_kernel<<<dim3(cmb.units), dim3(256), 0, s>>>(cmb);
		N2_LAUNCH_CHECK();
	}
	return N2_OK;
}

static int launch_input_gradient(const n2_grid_t* grid, hipStream_t s, uint32_t n_points, const __half* dL_dy, const float* dy_dx, float* dL_dx) {
	const uint32_t rows = grid->tab.n_levels * grid->n_features;
	auto* const kernel = n2_jacobian_streams(n_points, rows) ? grid_backward_input_kernel<true> : grid_backward_input_kernel<false>;
	kernel<<<dim3(n_tiles(n_points)), dim3(GRID_BLOCK), 0, s>>>(n_points, rows, dL_dy, dy_dx, dL_dx);
	N2_LAUNCH_CHECK();
	return N2_OK;
}

// One scatter pass with any combination of first-order (dL_dy) and second-order (v, g2) terms.
static int launch_scatter(n2_grid_t* grid, hipStream_t s, const float* d_xyz, uint32_t point_stride, uint32_t dim_stride, uint32_t n_points,
                          const __half* dL_dy, const float* v, const __half* g2, __half2* grads, __half* dL_ddLdy, bool accumulate,
                          const uint32_t* index = nullptr, uint32_t n_cols = 0, const N2ScatterRider& rider = N2ScatterRider()) {
	if (grads != nullptr && uses_bucketed(grid, n_points))
		return launch_bucketed(grid, s, d_xyz, point_stride, dim_stride, n_points, dL_dy, v, g2, dL_ddLdy, accumulate, index, n_cols, rider);
	const uint32_t tiles = n_pair_tiles(n_points);
	const dim3 gd(tiles * grid->tab.n_levels), bd(GRID_BLOCK);
	const bool first = dL_dy != nullptr, second = v != nullptr, out = dL_ddLdy != nullptr;
#define LAUNCH(F, S, O) grid_scatter_kernel<F, S, O><<<gd, bd, 0, s>>>(grid->tab, n_points, tiles, d_xyz, point_stride, dim_stride, dL_dy, v, g2, \
                                                                       grid->params, grads, dL_ddLdy, index, n_cols)
	if (first && second && out) LAUNCH(true, true, true);
	else if (first && second) LAUNCH(true, true, false);
	else if (second && out) LAUNCH(false, true, true);
	else if (second) LAUNCH(false, true, false);
	else LAUNCH(true, false, false);
#undef LAUNCH
	N2_LAUNCH_CHECK();
	if (rider.dL_dx != nullptr) {
		if (int rc = launch_input_gradient(grid, s, n_points, dL_dy, rider.dy_dx, rider.dL_dx)) return rc;
	}
	return n2_slab_reduce_launch(reinterpret_cast<n2_stream_t>(s), rider.sums);
}

N2_API int n2_grid_backward(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride,
                            uint32_t dim_stride, uint32_t n_points, const n2_half* d_dL_dy, const float* d_dy_dx,
                            float* d_dL_dx, n2_grad_mode mode) {
	if (int rc = check_batch(grid, "n2_grid_backward", d_xyz, point_stride, dim_stride, n_points)) return rc;
	N2_REQUIRE(d_dL_dy != nullptr || n_points == 0, "n2_grid_backward: d_dL_dy is null");
	N2_REQUIRE(d_dL_dx == nullptr || d_dy_dx != nullptr, "n2_grid_backward: d_dL_dx needs the d_dy_dx context of the forward");
	hipStream_t s = n2_stream(stream);
	if (int rc = prepare_grads(grid, "n2_grid_backward", s, mode, n_points)) return rc;
	if (n_points == 0) return N2_OK;
	if (mode == N2_GRAD_IGNORE) return d_dL_dx ? launch_input_gradient(grid, s, n_points, reinterpret_cast<const __half*>(d_dL_dy), d_dy_dx, d_dL_dx) : N2_OK;
	N2ScatterRider rider;
	rider.dy_dx = d_dy_dx;
	rider.dL_dx = d_dL_dx;
	N2ProfScope prof(N2_PROF_GRID_BACKWARD_PARAMS, s);
	return launch_scatter(grid, s, d_xyz, point_stride, dim_stride, n_points, reinterpret_cast<const __half*>(d_dL_dy), nullptr, nullptr, grid->grads, nullptr,
	                      mode == N2_GRAD_ACCUMULATE, nullptr, 0, rider);
}

static int backward_fused(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride, uint32_t dim_stride, uint32_t n_points,
                          const n2_half* d_dL_dy, const float* d_dL_ddLdx, const n2_half* d_dL_dy_second, n2_half* d_dL_ddLdy, n2_grad_mode mode,
                          const N2SlabReduce* sums, const uint32_t* d_index, uint32_t n_cols) {
	if (int rc = check_batch(grid, "n2_grid_backward_fused", d_xyz, point_stride, dim_stride, n_points)) return rc;
	N2_REQUIRE((d_dL_dy && d_dL_ddLdx && d_dL_dy_second) || n_points == 0, "n2_grid_backward_fused: d_dL_dy, d_dL_ddLdx and d_dL_dy_second are required");
	N2_REQUIRE(mode == N2_GRAD_OVERWRITE || mode == N2_GRAD_ACCUMULATE, "n2_grid_backward_fused: mode must be OVERWRITE or ACCUMULATE");
	N2_REQUIRE(d_index == nullptr || n_cols >= 1, "n2_grid_backward_fused: an indexed input needs at least one column");
	hipStream_t s = n2_stream(stream);
	if (int rc = prepare_grads(grid, "n2_grid_backward_fused", s, mode, n_points)) return rc;
	if (n_points == 0) return sums ? n2_slab_reduce_launch(stream, *sums) : N2_OK;
	N2ScatterRider rider;
	if (sums) rider.sums = *sums;
	N2ProfScope prof(N2_PROF_GRID_BACKWARD_PARAMS, s);
	return launch_scatter(grid, s, d_xyz, point_stride, dim_stride, n_points, reinterpret_cast<const __half*>(d_dL_dy), d_dL_ddLdx,
	                      reinterpret_cast<const __half*>(d_dL_dy_second), grid->grads, reinterpret_cast<__half*>(d_dL_ddLdy),
	                      mode == N2_GRAD_ACCUMULATE, d_index, n_cols, rider);
}
// (a launch has workgroups for one of the two beside its own: a slab summation, or dL_ddLdy)
int n2_grid_backward_fused_and_sums(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride, uint32_t dim_stride, uint32_t n_points,
                                    const n2_half* d_dL_dy, const float* d_dL_ddLdx, const n2_half* d_dL_dy_second, n2_grad_mode mode, const N2SlabReduce* sums) {
	return backward_fused(grid, stream, d_xyz, point_stride, dim_stride, n_points, d_dL_dy, d_dL_ddLdx, d_dL_dy_second, nullptr, mode, sums, nullptr, 0);
}
N2_API int n2_grid_backward_fused(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz, uint32_t point_stride,
                                  uint32_t dim_stride, uint32_t n_points, const n2_half* d_dL_dy,
                                  const float* d_dL_ddLdx, const n2_half* d_dL_dy_second, n2_half* d_dL_ddLdy,
                                  n2_grad_mode mode) {
	return backward_fused(grid, stream, d_xyz, point_stride, dim_stride, n_points, d_dL_dy, d_dL_ddLdx, d_dL_dy_second, d_dL_ddLdy, mode, nullptr, nullptr, 0);
}
int n2_grid_backward_fused_indexed(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz_rows, uint32_t n_cols, const uint32_t* d_index,
                                   uint32_t n_points, const n2_half* d_dL_dy, const float* d_dL_ddLdx, const n2_half* d_dL_dy_second,
                                   n2_grad_mode mode, const N2SlabReduce* sums) {
	if (d_index == nullptr) n_cols = n_points;  // the rows hold the batch itself
	return backward_fused(grid, stream, d_xyz_rows, 1, n_cols, n_points, d_dL_dy, d_dL_ddLdx, d_dL_dy_second, nullptr, mode, sums, d_index, n_cols);
}

N2_API int n2_grid_backward_backward_input(n2_grid_t* grid, n2_stream_t stream, const float* d_xyz,
                                           uint32_t point_stride, uint32_t dim_stride, uint32_t n_points,
                                           const float* d_dL_ddLdx, const n2_half* d_dL_dy, n2_half* d_dL_ddLdy,
                                           float* d_dL_dx, n2_grad_mode mode) {
	if (int rc = check_batch(grid, "n2_grid_backward_backward_input", d_xyz, point_stride, dim_stride, n_points)) return rc;
	N2_REQUIRE((d_dL_ddLdx != nullptr && d_dL_dy != nullptr) || n_points == 0, "n2_grid_backward_backward_input: d_dL_ddLdx and d_dL_dy are required");
	hipStream_t s = n2_stream(stream);
	if (int rc = prepare_grads(grid, "n2_grid_backward_backward_input", s, mode, d_dL_dx ? 0u : n_points)) return rc;
	if (n_points == 0) return N2_OK;
	if (mode == N2_GRAD_IGNORE && !d_dL_ddLdy && !d_dL_dx) return N2_OK;
	if (d_dL_dx) {
		if (int rc = n2_fill_zero_u32(s, d_dL_dx, sizeof(float) * 3 * (size_t)n_points)) return rc;
	}
	N2ProfScope prof(N2_PROF_GRID_SECOND_ORDER, s);
	if (!d_dL_dx) {
		return launch_scatter(grid, s, d_xyz, point_stride, dim_stride, n_points, nullptr, d_dL_ddLdx, reinterpret_cast<const __half*>(d_dL_dy),
		                      mode == N2_GRAD_IGNORE ? nullptr : grid->grads, reinterpret_cast<__half*>(d_dL_ddLdy), mode == N2_GRAD_ACCUMULATE);
	}
	const uint32_t tiles = n_tiles(n_points);
	grid_bbi_kernel<<<dim3(tiles * grid->tab.n_levels), dim3(GRID_BLOCK), 0, s>>>(
		grid->tab, n_points, tiles, d_xyz, point_stride, dim_stride, d_dL_ddLdx, reinterpret_cast<const __half*>(d_dL_dy),
		grid->params, mode == N2_GRAD_IGNORE ? nullptr : grid->grads, reinterpret_cast<__half*>(d_dL_ddLdy), d_dL_dx);
	N2_LAUNCH_CHECK();
	return N2_OK;
}
