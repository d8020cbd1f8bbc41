// Mesh extraction from a density lattice: marching cubes with shared vertices
// (marching_cubes_gpu, src/marching_cubes.cu:794-822, with gen_vertices :276-329
// and gen_faces :377-718) and the area-weighted vertex normals of
// accumulate_1ring (:331-366).
//
// Same geometry as the reference: lattice value at (x, y, z) is
// density[x + y*rx + z*rx*ry], a point is inside when density > thresh, one
// vertex per lattice edge whose ends differ, at dt = (thresh - f0) / (f1 - f0)
// along the edge, scaled by (aabb.max - aabb.min) / res and shifted by
// aabb.min; cube corner bits and edge numbers as in gen_faces.
//
// Two things are done differently.  The reference numbers vertices and
// triangles with atomicAdd, which is a race; here a lattice point's vertices
// (x, y, z edge in that order) and a cube's triangles get their slots from
// exclusive prefix sums in lattice order, so the mesh is reproducible.  And the
// 256-case table is derived by the compiler instead of being typed in: the cut
// edges on every cube face are joined into directed segments (an ambiguous face
// always separates its two inside corners), the segments chain into closed
// loops, every loop is cut into a fan of triangles from its lowest edge.
// The reference's table has the same segments on every face in all 256 cases,
// i.e. the same surface with the same orientation; only the diagonals inside
// polygons of more than three corners differ in some cases.
//
// Vertex positions are part of the bit-exact contract with the CPU oracle:
// floating-point contraction is off for this file.
#include "n2_common.h"
#include "bounded_wait.h"
#include "launch_rules.h"

#include <cstring>

#pragma clang fp contract(off)

constexpr uint32_t MC_BLOCK = 256;

struct McTable {
	alignas(16) int8_t tri[256][16];  // a case's row is read as one uint4
	uint8_t ntri[256];  // triangles of each case
};
static_assert(alignof(McTable) >= alignof(uint4) && sizeof(McTable::tri[0]) == sizeof(uint4), "rows can be read as uint4");

// ---------------------------------------------------------------------------
// case table: evaluated by the compiler, part of the library's device image
// ---------------------------------------------------------------------------
namespace {

constexpr int MC_EDGE_CORNERS[12][2] = {{0, 1}, {1, 2}, {2, 3}, {3, 0}, {4, 5}, {5, 6}, {6, 7}, {7, 4}, {0, 4}, {1, 5}, {2, 6}, {3, 7}};
// the six faces as corner cycles, counter-clockwise seen from outside: x = 0, x = 1, y = 0, y = 1, z = 0, z = 1
constexpr int MC_FACES[6][4] = {{4, 7, 3, 0}, {1, 2, 6, 5}, {1, 5, 4, 0}, {3, 7, 6, 2}, {3, 2, 1, 0}, {4, 5, 6, 7}};

constexpr int mc_edge_between(int a, int b) {
	for (int e = 0; e < 12; ++e)
		if ((MC_EDGE_CORNERS[e][0] == a && MC_EDGE_CORNERS[e][1] == b) || (MC_EDGE_CORNERS[e][0] == b && MC_EDGE_CORNERS[e][1] == a)) return e;
	return -1;
}

constexpr McTable mc_build_table() {
	McTable t{};
	for (int mask = 0; mask < 256; ++mask) {
		int next[12] = {};
		for (int e = 0; e < 12; ++e) next[e] = -1;
		for (int k = 0; k < 16; ++k) t.tri[mask][k] = -1;
		for (const auto& cyc : MC_FACES) {
			int in[4] = {}, n_in = 0;
			for (int k = 0; k < 4; ++k) { in[k] = (mask >> cyc[k]) & 1; n_in += in[k]; }
			if (n_in == 0 || n_in == 4) continue;
			// every maximal run of inside corners is cut off by one segment, directed from the edge after the run to the
			// edge before it (the surface normal then points to the inside)
			for (int k = 0; k < 4; ++k) {
				if (!in[k] || in[(k + 3) % 4]) continue;
				int j = k;
				while (in[(j + 1) % 4]) ++j;
				const int before = mc_edge_between(cyc[(k + 3) % 4], cyc[k]);
				const int after = mc_edge_between(cyc[j % 4], cyc[(j + 1) % 4]);
				next[after] = before;
			}
		}
		bool seen[12] = {};
		int n = 0;
		for (int e = 0; e < 12; ++e) {
			if (next[e] < 0 || seen[e]) continue;
			int loop[12] = {}, len = 0;
			for (int c = e; !seen[c]; c = next[c]) { seen[c] = true; loop[len++] = c; }
			for (int k = 1; k + 1 < len; ++k) {
				t.tri[mask][n++] = (int8_t)loop[0];
				t.tri[mask][n++] = (int8_t)loop[k];
				t.tri[mask][n++] = (int8_t)loop[k + 1];
			}
		}
		t.ntri[mask] = (uint8_t)(n / 3);
	}
	return t;
}

constexpr McTable MC_TABLE_HOST = mc_build_table();

// The triangles round a cut edge, as mc_normals_kernel wants them.  `axis` is the edge's; along, fast and slow are the axis and the two across
// it (mc_ring_axes); cube q of the four round the edge starts one step back along slow for q < 2 and along fast for even q.  In the
// frame (along, fast, slow) an edge of a cube is its first corner, one bit per axis, and its direction << 3.  A triangle that the edge is part of
// takes twelve bits: the other two edges in the triangle's order, and << 10 the edge's place in it; their number stands in bits 60..62.
struct McRing {
	uint64_t fan[3][4][256];  // [axis][cube][corner bits in the frame]
};
constexpr int MC_RING_AXES[3][3] = {{0, 1, 2}, {1, 0, 2}, {2, 0, 1}};
constexpr McRing mc_build_ring() {
	McRing r{};
	for (int axis = 0; axis < 3; ++axis) {
		int corner[8] = {}, local[8] = {}, edge[12] = {};  // corner of the frame -> of the cube and back; the cube's edges in the frame
		for (int c = 0; c < 8; ++c) {
			int d[3] = {};
			for (int k = 0; k < 3; ++k) d[MC_RING_AXES[axis][k]] = (c >> k) & 1;
			corner[c] = (d[1] ? (d[0] ? 2 : 3) : (d[0] ? 1 : 0)) + 4 * d[2];
			local[corner[c]] = c;
		}
		for (int e = 0; e < 12; ++e) {
			const int p = local[MC_EDGE_CORNERS[e][0]], q = local[MC_EDGE_CORNERS[e][1]], diff = p ^ q;
			edge[e] = (p & q) | (diff == 1 ? 0 : diff == 2 ? 8 : 16);
		}
		for (int mask = 0; mask < 256; ++mask) {
			int cube = 0;
			for (int c = 0; c < 8; ++c) cube |= ((mask >> c) & 1) << corner[c];
			for (int q = 0; q < 4; ++q) {
				const int self = ((q & 1) ? 0 : 2) | (q < 2 ? 4 : 0);
				uint64_t fan = 0, n = 0;
				for (int t = 0; t < MC_TABLE_HOST.ntri[cube]; ++t) {
					int at = -1;
					uint64_t others = 0;
					for (int k = 2; k >= 0; --k) {
						const int e = edge[MC_TABLE_HOST.tri[cube][3 * t + k]];
						if (e == self) at = k;
						else others = others << 5 | (uint64_t)e;
					}
					if (at >= 0) fan |= (others | (uint64_t)at << 10) << (12 * n++);
				}
				r.fan[axis][q][mask] = fan | n << 60;
			}
		}
	}
	return r;
}

}  // namespace

__device__ const McTable MC_TABLE = mc_build_table();
__device__ const McRing MC_RING = mc_build_ring();

// ---------------------------------------------------------------------------
// kernels
//
// The density is read once, for one bit per lattice point (inside or not); everything up to the vertex positions is then
// worked out from the bits, 64 points of a row at a time:
//   mc_bits     density -> bits                                                   (bound by HBM: 4 bytes per point)
//   mc_count    four words per lane: their edge vertices and triangles as bit masks, prefix sums within a block of 256 words
//   mc_scan     one workgroup: prefix sums over the blocks, the list of the blocks that own something, the totals
//   mc_emit     a workgroup per listed block: its vertices and triangles
//   mc_normals  one lane per vertex: the sum over the triangles of the four cubes round its edge
// Rows are padded to whole words, so a word's neighbours in y and z are words too and no mask crosses a row.
// Lattices whose rows have fewer than 16 points (SHORT) put several rows of a plane into the lower half of a word, each padded to
// a power of two, the pitch: a word's neighbours in y are then its own bits and the next word's, shifted by the pitch.  (With a
// word to each row, rows of two points need 36 bytes of workspace per point; so 2.3.  All 64 bits need 1.1, but leave
// twice as much behind one another in a workgroup: 2 x 512 x 512 points 69, 73 and 102 us.)
// 512^3 lattice of a bumpy sphere (1.2 M triangles), in us: bits 82 (6.6 TB/s), count 14.6, scan 4.7, emit 27.7, normals 24, with
// the host's wait for the totals 162 in all (168 while that was for the stream; 64^3 48 -> 43, 256^3 60 -> 55).  Deciding every point from the four rows of the density itself took 242 for the
// count alone and read the rows again for each output: 868 in all.
// ---------------------------------------------------------------------------
struct McGrid {
	uint32_t rx, ry, rz;
	float thresh;
	float scale[3], offset[3];
	uint32_t row_words;  // words per row
	uint32_t n_words;
	// SHORT: log2 of the pitch and of the rows of a word; words per plane; a full word's points, and those with a neighbour in x
	uint32_t pitch_log, rows_log, plane_words, here, xok;
};
constexpr uint32_t MC_SHORT_ROW = 16, MC_SHORT_BITS_LOG = 5;

typedef unsigned long long mc_word;

// where a word's bit is in the lattice
struct McPlace {
	uint32_t x, y, z;
};
template <bool SHORT>
__device__ __forceinline__ McPlace mc_place(const McGrid& g, uint32_t w, uint32_t bit) {
	if constexpr (SHORT) {
		const uint32_t z = w / g.plane_words, yw = w - z * g.plane_words;
		return {bit & ((1u << g.pitch_log) - 1u), (yw << g.rows_log) + (bit >> g.pitch_log), z};
	} else {
		const uint32_t row = w / g.row_words, col = w - row * g.row_words;
		return {col * 64u + bit, row % g.ry, row / g.ry};
	}
}

// What a word of points owns; written for the words that own something, which the `active` bits tell.
struct alignas(64) McRecord {
	mc_word edge[3];       // point has a vertex on its edge towards +axis
	uint32_t first_v, first_t;  // vertices and triangles of the words before this one in its block of 256
	mc_word tri[3];        // bits 0, 1, 2 of the number of triangles of the point's cube
	uint32_t pad[2];
};
// Which words of a block own something: four words of bits per block.
template <bool SHORT>
__device__ __forceinline__ bool mc_owns(const mc_word* __restrict__ active, uint32_t block, uint32_t word) {
	// (mc_count_kernel has four consecutive words per lane, mc_count_short_kernel one)
	return SHORT ? (active[block * 4u + (word >> 6)] >> (word & 63u)) & 1ull : (active[block * 4u + (word & 3u)] >> (word >> 2)) & 1ull;
}

constexpr uint32_t MC_BITS_WORDS = 16;  // words a wave forms at a time: 16 loads in flight per lane

// STREAM: the density is read past the last-level cache; the lattice is larger than that and would only push itself out (512^3,
// 512 MiB: 92 -> 80 us; 384^3, 216 MiB, which stays there for the emitting kernel: 32 -> 34).
constexpr uint64_t MC_STREAM_BYTES = 256ull << 20;
template <bool STREAM, bool SHORT>
__global__ void __launch_bounds__(MC_BLOCK) mc_bits_kernel(McGrid g, const float* __restrict__ density, mc_word* __restrict__ bits) {
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (MC_BLOCK / 64) + (threadIdx.x >> 6));
	const uint32_t w0 = wave * MC_BITS_WORDS;
	if (w0 >= g.n_words) return;
	uint32_t row = w0 / g.row_words, col = w0 - row * g.row_words;
	float v[MC_BITS_WORDS];
#pragma unroll
	for (uint32_t k = 0; k < MC_BITS_WORDS; ++k) {
		const uint32_t x = col * 64u + lane;
		const float* at = density + (uint64_t)row * g.rx + x;
		bool inside = x < g.rx;
		if (SHORT) {
			const McPlace p = mc_place<true>(g, w0 + k, lane);
			at = density + ((uint64_t)p.z * g.ry + p.y) * g.rx + p.x;
			inside = lane >> MC_SHORT_BITS_LOG == 0u && p.x < g.rx && p.y < g.ry;
		}
		v[k] = (w0 + k < g.n_words && inside) ? (STREAM ? __builtin_nontemporal_load(at) : *at) : -INFINITY;
		if (++col == g.row_words) { col = 0; ++row; }
	}
	mc_word mine = 0;
#pragma unroll
	for (uint32_t k = 0; k < MC_BITS_WORDS; ++k) {
		const mc_word b = __ballot(v[k] > g.thresh);
		if (lane == k) mine = b;
	}
	if (lane < MC_BITS_WORDS && w0 + lane < g.n_words) bits[w0 + lane] = mine;
}

// The bits of a word and of its neighbours, in the order of the offsets (y, z) = (0, 0), (1, 0), (0, 1), (1, 1): b the word
// itself, s the word one point further along x.  here: the word's points; xok, yok: those that have a neighbour in x, in y; zok: the
// plane at z + 1 exists (words of rows and planes that do not are zero).
struct McBits {
	mc_word b[4], s[4], here, xok, yok;
	bool zok;
};
// SHORT: the points of the first n rows of a word
__device__ __forceinline__ mc_word mc_first_rows(const McGrid& g, uint32_t n) {
	return n >> g.rows_log ? (1ull << (1u << MC_SHORT_BITS_LOG)) - 1ull : (1ull << (n << g.pitch_log)) - 1ull;
}
template <bool SHORT>
__device__ __forceinline__ McBits mc_load_bits(const McGrid& g, const mc_word* __restrict__ bits, uint32_t w) {
	McBits B;
	if constexpr (SHORT) {
		const McPlace first = mc_place<true>(g, w, 0u);
		const uint32_t rows = g.ry - first.y, pitch = 1u << g.pitch_log;  // rows from the word's first on
		B.here = g.here & mc_first_rows(g, rows);
		B.xok = g.xok & mc_first_rows(g, rows);
		B.yok = mc_first_rows(g, rows - 1u);
		B.zok = first.z + 1u < g.rz;
#pragma unroll
		for (uint32_t j = 0; j < 4; j += 2) {
			const uint32_t at = w + (j ? g.plane_words : 0u);
			const bool ok = j == 0u || B.zok;
			B.b[j] = ok ? bits[at] : 0ull;
			const mc_word next = ok && (rows - 1u) >> g.rows_log ? bits[at + 1u] : 0ull;  // the plane has rows behind the word's
			// (what the last points of a row get as their neighbours in x, and what stands above the lower half, is not used: xok, here)
			B.b[j + 1] = (B.b[j] >> pitch) | (next << ((1u << MC_SHORT_BITS_LOG) - pitch));
			B.s[j] = B.b[j] >> 1;
			B.s[j + 1] = B.b[j + 1] >> 1;
		}
		return B;
	}
	const uint32_t row = w / g.row_words, col = w - row * g.row_words;
	const uint32_t z = row / g.ry, y = row - z * g.ry;
	const bool yok = y + 1u < g.ry;
	B.yok = yok ? ~0ull : 0ull;
	B.zok = z + 1u < g.rz;
	const uint32_t left = g.rx - col * 64u;  // points from the word's first to the end of the row
	B.here = left >= 64u ? ~0ull : (1ull << left) - 1ull;
	B.xok = left > 64u ? ~0ull : (1ull << (left - 1u)) - 1ull;
#pragma unroll
	for (uint32_t j = 0; j < 4; ++j) {
		const bool ok = (!(j & 1u) || yok) && (!(j & 2u) || B.zok);
		const uint32_t at = w + ((j & 1u) ? g.row_words : 0u) + ((j & 2u) ? g.row_words * g.ry : 0u);
		B.b[j] = ok ? bits[at] : 0ull;
		const mc_word next = ok && left > 64u ? bits[at + 1u] : 0ull;
		B.s[j] = (B.b[j] >> 1) | (next << 63);
	}
	return B;
}
// corner k of the cubes, as in gen_faces: round the bottom face from the point itself, then the top face
__device__ __forceinline__ mc_word mc_corner(const McBits& B, uint32_t k) {
	const mc_word corner[8] = {B.b[0], B.s[0], B.s[1], B.b[1], B.b[2], B.s[2], B.s[3], B.b[3]};
	return corner[k];
}
// corner bits of point `lane`'s cube
__device__ __forceinline__ uint32_t mc_case(const McBits& B, uint32_t lane) {
	uint32_t m = 0;
#pragma unroll
	for (uint32_t k = 0; k < 8; ++k) m |= (uint32_t)((mc_corner(B, k) >> lane) & 1ull) << k;
	return m;
}

// The number of triangles of 64 cubes at a time.  A cube that the surface crosses in one piece has two triangles fewer than cut edges; bits
// 0, 1, 2 of that number follow from a carry-save addition of the twelve edges' words.  `several`: the cubes that it may cross in several
// pieces, namely those with a face whose four edges are cut, and those with two opposite corners (inside or outside) alone; their numbers
// come from the table.
struct McTriBits {
	mc_word tri[3], several;
};
template <class Word>
constexpr __host__ __device__ __forceinline__ void mc_add(Word a, Word b, Word c, Word& sum, Word& carry) {
	sum = a ^ b ^ c;
	carry = (a & b) | (c & (a | b));
}
template <class Word, class Bits>
constexpr __host__ __device__ __forceinline__ void mc_triangle_bits(const Word (&c)[8], Bits& out) {
	const Word x[4] = {(Word)(c[0] ^ c[1]), (Word)(c[3] ^ c[2]), (Word)(c[4] ^ c[5]), (Word)(c[7] ^ c[6])};  // edges along x: (y, z) = (0, 0), (1, 0), (0, 1), (1, 1)
	const Word y[4] = {(Word)(c[0] ^ c[3]), (Word)(c[1] ^ c[2]), (Word)(c[4] ^ c[7]), (Word)(c[5] ^ c[6])};  // along y: (x, z)
	const Word z[4] = {(Word)(c[0] ^ c[4]), (Word)(c[1] ^ c[5]), (Word)(c[3] ^ c[7]), (Word)(c[2] ^ c[6])};  // along z: (x, y)
	Word s0 = 0, s1 = 0, s2 = 0, s3 = 0, c0 = 0, c1 = 0, c2 = 0, c3 = 0, c4 = 0, c5 = 0, t0 = 0, t1 = 0, d0 = 0, d1 = 0, d2 = 0, e0 = 0, e1 = 0, e2 = 0, unused = 0;
	mc_add(x[0], x[1], x[2], s0, c0);
	mc_add(x[3], y[0], y[1], s1, c1);
	mc_add(y[2], y[3], z[0], s2, c2);
	mc_add(z[1], z[2], z[3], s3, c3);
	mc_add(s0, s1, s2, t0, c4);
	mc_add(t0, s3, (Word)0, e0, c5);
	mc_add(c0, c1, c2, t0, d0);
	mc_add(c3, c4, c5, t1, d1);
	mc_add(t0, t1, (Word)0, e1, d2);
	mc_add(d0, d1, d2, e2, unused);
	const Word faces = (x[0] & x[1] & y[0]) | (x[2] & x[3] & y[2]) | (x[0] & x[2] & z[0]) | (x[1] & x[3] & z[2]) | (y[0] & y[2] & z[0]) | (y[1] & y[3] & z[1]);
	const Word odd_z = x[0] ^ c[2] ^ c[3] ^ (Word)0, odd_y = x[0] ^ c[4] ^ c[5], odd_x = y[0] ^ c[4] ^ c[7], all = odd_z ^ c[4] ^ c[5] ^ c[6] ^ c[7];
	out.several = faces | (odd_x & odd_y & odd_z & ~all);
	out.tri[0] = e0;
	out.tri[1] = ~e1;
	out.tri[2] = e2 & e1;
}
struct McCaseBits {
	uint32_t tri[3], several;
};
constexpr bool mc_triangle_bits_hold() {
	for (uint32_t mask = 1; mask < 255; ++mask) {
		uint32_t c[8] = {};
		for (uint32_t k = 0; k < 8; ++k) c[k] = (mask >> k) & 1u;
		McCaseBits b{};
		mc_triangle_bits(c, b);
		if (!(b.several & 1u) && (b.tri[0] & 1u) + 2u * (b.tri[1] & 1u) + 4u * (b.tri[2] & 1u) != MC_TABLE_HOST.ntri[mask]) return false;
	}
	return true;
}
static_assert(mc_triangle_bits_hold(), "the cubes left to the formula have as many triangles as the table says");

// edges, triangles and their numbers of one word (B: its bits and its neighbours')
__device__ __forceinline__ void mc_own(const McBits& B, McRecord& r, uint32_t& nv, uint32_t& nt) {
	r.edge[0] = (B.b[0] ^ B.s[0]) & B.xok;
	r.edge[1] = (B.b[0] ^ B.b[1]) & B.here & B.yok;
	r.edge[2] = B.zok ? (B.b[0] ^ B.b[2]) & B.here : 0ull;
	const mc_word corner[8] = {B.b[0], B.s[0], B.s[1], B.b[1], B.b[2], B.s[2], B.s[3], B.b[3]};
	mc_word any = corner[0], all = corner[0];
#pragma unroll
	for (uint32_t k = 1; k < 8; ++k) { any |= corner[k]; all &= corner[k]; }
	const mc_word cut = B.zok ? any & ~all & B.xok & B.yok : 0ull;
	r.tri[0] = r.tri[1] = r.tri[2] = 0ull;
	if (__any(cut != 0ull)) {
		McTriBits t;
		mc_triangle_bits(corner, t);
		const mc_word simple = cut & ~t.several;
#pragma unroll
		for (int a = 0; a < 3; ++a) r.tri[a] = t.tri[a] & simple;
		for (mc_word rest = cut & t.several; rest; rest &= rest - 1ull) {
			const uint32_t p = (uint32_t)__ffsll(rest) - 1u, n = MC_TABLE.ntri[mc_case(B, p)];
#pragma unroll
			for (int a = 0; a < 3; ++a) r.tri[a] |= (mc_word)((n >> a) & 1u) << p;
		}
	}
	nv = (uint32_t)(__popcll(r.edge[0]) + __popcll(r.edge[1]) + __popcll(r.edge[2]));
	nt = (uint32_t)(__popcll(r.tri[0]) + 2 * __popcll(r.tri[1]) + 4 * __popcll(r.tri[2]));
}

// One wave per block of 256 words, four consecutive words per lane: with their neighbours in y and z four loads of 32 bytes, and nothing to
// wait for but these.  (A lane per word in workgroups of four waves, with a table of triangle numbers in LDS: four rounds of workgroups that
// each waited for the table, the bits and each other, 28 us for 512^3, of which walking through the cut cubes took 3; then 16, and 14.5 where blocks
// away from the surface, two of three, stop at their bits.)
constexpr uint32_t MC_EACH = 4;
static_assert(MC_BLOCK == 64u * MC_EACH, "a wave takes a block");
__global__ void __launch_bounds__(64) mc_count_kernel(McGrid g, const mc_word* __restrict__ bits, McRecord* __restrict__ records,
                                                      mc_word* __restrict__ active, uint2* __restrict__ blocks) {
	typedef mc_word two __attribute__((ext_vector_type(2), aligned(8)));
	const uint32_t lane = threadIdx.x, w0 = blockIdx.x * MC_BLOCK + lane * MC_EACH;
	const uint32_t plane = g.row_words * g.ry;
	// (the same for the wave: all of its loads, and the word behind its last one, are inside the array)
	const bool inner = (uint64_t)blockIdx.x * MC_BLOCK + MC_BLOCK + 1u + plane + g.row_words <= g.n_words;
	mc_word b[4][MC_EACH + 1];
	if (inner) {
#pragma unroll
		for (uint32_t j = 0; j < 4; ++j) {
			const mc_word* at = bits + w0 + ((j & 1u) ? g.row_words : 0u) + ((j & 2u) ? plane : 0u);
#pragma unroll
			for (uint32_t q = 0; q < MC_EACH; q += 2u) {
				const two v = *reinterpret_cast<const two*>(at + q);
				b[j][q] = v.x;
				b[j][q + 1u] = v.y;
			}
			b[j][MC_EACH] = lane == 63u ? at[MC_EACH] : 0ull;
		}
		// Most blocks lie away from the surface: all their bits and their neighbours' are the same.
		mc_word any = 0ull, all = ~0ull;
#pragma unroll
		for (uint32_t j = 0; j < 4; ++j) {
#pragma unroll
			for (uint32_t q = 0; q < MC_EACH; ++q) { any |= b[j][q]; all &= b[j][q]; }
			any |= b[j][MC_EACH];
			all &= lane == 63u ? b[j][MC_EACH] : ~0ull;
		}
		if (!__any(any != 0ull) || !__any(all != ~0ull)) {
			if (lane < MC_EACH) active[blockIdx.x * MC_EACH + lane] = 0ull;
			if (lane == 0) blocks[blockIdx.x] = make_uint2(0u, 0u);
			return;
		}
#pragma unroll
		for (uint32_t j = 0; j < 4; ++j) {
			const mc_word next = __shfl_down(b[j][0], 1);
			if (lane != 63u) b[j][MC_EACH] = next;
		}
	}
	McRecord r[MC_EACH];
	uint32_t nv[MC_EACH], nt[MC_EACH], sum_v = 0, sum_t = 0;
	const uint32_t row0 = w0 / g.row_words, col0 = w0 - row0 * g.row_words, z0 = row0 / g.ry;
	uint32_t col = col0, y = row0 - z0 * g.ry;
#pragma unroll
	for (uint32_t q = 0; q < MC_EACH; ++q) {
		nv[q] = nt[q] = 0;
		McBits B;
		if (inner) {
			const uint32_t left = g.rx - col * 64u;  // points from the word's first to the end of the row
			B.here = left >= 64u ? ~0ull : (1ull << left) - 1ull;
			B.xok = left > 64u ? ~0ull : (1ull << (left - 1u)) - 1ull;
			B.yok = y + 1u < g.ry ? ~0ull : 0ull;
			B.zok = true;  // (a plane lies behind all that the wave loads)
#pragma unroll
			for (uint32_t j = 0; j < 4; ++j) {
				// (rows that are not there meet yok)
				B.b[j] = b[j][q];
				B.s[j] = (B.b[j] >> 1) | (left > 64u ? b[j][q + 1u] << 63 : 0ull);
			}
			if (++col == g.row_words) {
				col = 0;
				if (++y == g.ry) y = 0;
			}
		} else if (w0 + q < g.n_words) {
			B = mc_load_bits<false>(g, bits, w0 + q);
		}
		if (inner || w0 + q < g.n_words) mc_own(B, r[q], nv[q], nt[q]);
		sum_v += nv[q];
		sum_t += nt[q];
		const mc_word mask = __ballot(nv[q] + nt[q] > 0u);
		if (lane == 0) active[blockIdx.x * MC_EACH + q] = mask;
	}
	const uint32_t iv = n2_wave_prefix(sum_v), it = n2_wave_prefix(sum_t);
	uint32_t first_v = iv - sum_v, first_t = it - sum_t;
#pragma unroll
	for (uint32_t q = 0; q < MC_EACH; ++q) {
		if (nv[q] + nt[q] > 0u) {
			r[q].first_v = first_v;
			r[q].first_t = first_t;
			records[w0 + q] = r[q];
		}
		first_v += nv[q];
		first_t += nt[q];
	}
	if (lane == 63) blocks[blockIdx.x] = make_uint2(iv, it);
}

// Short rows: one lane per word; a lane walks through the cubes of its word that the surface cuts.
__global__ void __launch_bounds__(MC_BLOCK) mc_count_short_kernel(McGrid g, const mc_word* __restrict__ bits, McRecord* __restrict__ records,
                                                            mc_word* __restrict__ active, uint2* __restrict__ blocks) {
	__shared__ uint8_t ntri[256];
	__shared__ uint32_t sum_v[MC_BLOCK / 64], sum_t[MC_BLOCK / 64];
	const uint32_t w = blockIdx.x * MC_BLOCK + threadIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	ntri[threadIdx.x] = MC_TABLE.ntri[threadIdx.x];
	__syncthreads();
	McRecord r{};
	uint32_t nv = 0, nt = 0;
	mc_word cut = 0;
	const McBits B = mc_load_bits<true>(g, bits, min(w, g.n_words - 1u));
	if (w < g.n_words) {
		r.edge[0] = (B.b[0] ^ B.s[0]) & B.xok;
		r.edge[1] = (B.b[0] ^ B.b[1]) & B.here & B.yok;
		r.edge[2] = B.zok ? (B.b[0] ^ B.b[2]) & B.here : 0ull;
#pragma unroll
		for (int a = 0; a < 3; ++a) nv += (uint32_t)__popcll(r.edge[a]);
		if (B.yok && B.zok) {
			const mc_word any = B.b[0] | B.b[1] | B.b[2] | B.b[3] | B.s[0] | B.s[1] | B.s[2] | B.s[3];
			const mc_word all = B.b[0] & B.b[1] & B.b[2] & B.b[3] & B.s[0] & B.s[1] & B.s[2] & B.s[3];
			cut = any & ~all & B.xok & B.yok;
		}
		for (; cut; cut &= cut - 1ull) {
			const uint32_t p = (uint32_t)__ffsll(cut) - 1u;
			const uint32_t t = ntri[mc_case(B, p)];
			nt += t;
#pragma unroll
			for (int a = 0; a < 3; ++a) r.tri[a] |= (mc_word)((t >> a) & 1u) << p;
		}
	}
	const bool owns = nv + nt > 0;
	const mc_word mask = __ballot(owns);
	if (lane == 0) active[w >> 6] = mask;
	if (!__syncthreads_or(owns)) {
		if (threadIdx.x == 0) blocks[blockIdx.x] = make_uint2(0, 0);
		return;
	}
	const uint32_t iv = n2_wave_prefix(nv), it = n2_wave_prefix(nt);
	if (lane == 63) { sum_v[wave] = iv; sum_t[wave] = it; }
	__syncthreads();
	uint32_t before_v = 0, before_t = 0, all_v = 0, all_t = 0;
#pragma unroll
	for (uint32_t k = 0; k < MC_BLOCK / 64; ++k) {
		if (k < wave) { before_v += sum_v[k]; before_t += sum_t[k]; }
		all_v += sum_v[k];
		all_t += sum_t[k];
	}
	if (owns) {
		r.first_v = before_v + iv - nv;
		r.first_t = before_t + it - nt;
		records[w] = r;
	}
	if (threadIdx.x == 0) blocks[blockIdx.x] = make_uint2(all_v, all_t);
}

// Exclusive prefix sums of the blocks' counts in place; element n_blocks receives the totals.  The blocks that own something are listed, their
// number goes behind the totals.
// 8192 blocks a round, consecutive lanes on consecutive ones: a group of 64 blocks is summed by a wave, the 128 groups by one wave.  (With eight consecutive blocks to
// a lane every load and store was 64 lines apart, for one CU's L1: 8 us for 512^3, now 4.6.)
constexpr uint32_t MC_SCAN_EACH = 8, MC_SCAN_GROUPS = 16 * MC_SCAN_EACH;
__global__ void __launch_bounds__(1024) mc_scan_kernel(uint32_t n_blocks, uint2* __restrict__ blocks, uint32_t* __restrict__ listed,
                                                       uint32_t* to_v, uint32_t* to_t) {
	__shared__ uint32_t group[3][MC_SCAN_GROUPS + 1];
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	uint32_t carry[3] = {0u, 0u, 0u};
	for (uint32_t c0 = 0; c0 < n_blocks; c0 += 1024u * MC_SCAN_EACH) {
		uint2 v[MC_SCAN_EACH];
		uint32_t upto[MC_SCAN_EACH][3];
#pragma unroll
		for (uint32_t k = 0; k < MC_SCAN_EACH; ++k) {
			const uint32_t i = c0 + k * 1024u + threadIdx.x;
			v[k] = i < n_blocks ? blocks[i] : make_uint2(0u, 0u);
		}
#pragma unroll
		for (uint32_t k = 0; k < MC_SCAN_EACH; ++k) {
			upto[k][0] = n2_wave_prefix(v[k].x);
			upto[k][1] = n2_wave_prefix(v[k].y);
			upto[k][2] = n2_wave_prefix((v[k].x | v[k].y) ? 1u : 0u);
			if (lane == 63u) {
#pragma unroll
				for (uint32_t q = 0; q < 3; ++q) group[q][k * 16u + wave] = upto[k][q];
			}
		}
		__syncthreads();
		if (wave < 3u) {  // sum q by wave q, two groups to a lane
			const uint32_t a = group[wave][2u * lane], b = group[wave][2u * lane + 1u], both = n2_wave_prefix(a + b);
			group[wave][2u * lane] = both - a - b;
			group[wave][2u * lane + 1u] = both - b;
			if (lane == 63u) group[wave][MC_SCAN_GROUPS] = both;
		}
		__syncthreads();
		if (threadIdx.x == 0 && to_v && c0 + 1024u * MC_SCAN_EACH >= n_blocks) {  // (in front of the stores: the host waits for these)
			__hip_atomic_store(to_v, carry[0] + group[0][MC_SCAN_GROUPS], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
			__hip_atomic_store(to_t, carry[1] + group[1][MC_SCAN_GROUPS], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
		}
#pragma unroll
		for (uint32_t k = 0; k < MC_SCAN_EACH; ++k) {
			const uint32_t i = c0 + k * 1024u + threadIdx.x, g = k * 16u + wave;
			if (i < n_blocks) blocks[i] = make_uint2(carry[0] + group[0][g] + upto[k][0] - v[k].x, carry[1] + group[1][g] + upto[k][1] - v[k].y);
			if (v[k].x | v[k].y) listed[carry[2] + group[2][g] + upto[k][2] - 1u] = i;
		}
#pragma unroll
		for (uint32_t q = 0; q < 3; ++q) carry[q] += group[q][MC_SCAN_GROUPS];
		__syncthreads();  // the sums have been read
	}
	if (threadIdx.x == 0) {
		blocks[n_blocks] = make_uint2(carry[0], carry[1]);
		blocks[n_blocks + 1u] = make_uint2(carry[2], 0u);
	}
}

// number of set bits of `b` below this lane
__device__ __forceinline__ uint32_t mc_below(mc_word b, uint32_t lane) { return (uint32_t)__popcll(b & ((1ull << lane) - 1ull)); }

// edge masks of a word and its first vertex
struct McOwned {
	mc_word e[3];
	uint32_t first;
};
// first vertex of the word's point `lane` | its edge flags << 29
__device__ __forceinline__ uint32_t mc_vertex_slot(const McOwned& o, uint32_t lane) {
	uint32_t slot = o.first, flags = 0;
#pragma unroll
	for (uint32_t a = 0; a < 3; ++a) {
		slot += mc_below(o.e[a], lane);
		flags |= (uint32_t)((o.e[a] >> lane) & 1ull) << a;
	}
	return slot | (flags << 29);
}

constexpr uint32_t MC_LIST = 2048;

// Lists the set bits of every lane's `points` in lane order, as (lane of the workgroup) << 6 | bit, and calls visit(entry)
// with one entry per lane at a time; all lanes of the workgroup take part.
template <class Visit>
__device__ __forceinline__ void mc_for_points(mc_word points, uint16_t* list, uint32_t* wave_sum, Visit visit) {
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	const uint32_t n = (uint32_t)__popcll(points), incl = n2_wave_prefix(n);
	if (lane == 63) wave_sum[wave] = incl;
	__syncthreads();
	uint32_t first = incl - n, total = 0;
#pragma unroll
	for (uint32_t k = 0; k < MC_BLOCK / 64; ++k) {
		if (k < wave) first += wave_sum[k];
		total += wave_sum[k];
	}
	for (uint32_t from = 0; from < total; from += MC_LIST) {
		for (; points && first < from + MC_LIST; points &= points - 1ull, ++first) list[first - from] = (uint16_t)(threadIdx.x << 6 | ((uint32_t)__ffsll(points) - 1u));
		__syncthreads();
		const uint32_t count = min(total - from, MC_LIST);
		for (uint32_t i = threadIdx.x; i < count; i += MC_BLOCK) visit((uint32_t)list[i]);
		__syncthreads();  // the list has been read
	}
}

// A workgroup emits what the words of a listed block own, and goes on to another one.  Only one point in ten of such a word owns anything, so the points that do
// are listed and dealt to the lanes: with a wave per word the launch was a chain of memory round trips at a tenth of the
// lanes, 240 us.  The vertices that a cube uses belong to its own point and to those one further along x, y and z: their
// slots come from the records of the (at most eight) words those points are in, and stand in LDS, where a triangle's
// corners pick theirs.  What bounds the launch is the chain of round trips: which words own something, their records (they stay in LDS, for
// their neighbours in y too), then all that a point needs at once.  A cube's case comes from the bits, as its number of triangles did: whatever
// the density is by now, a triangle's corners are vertices that this pass writes.
// (With the records read again for each point, then the bits and then the case's row: 47 us for 512^3, then 34; with the case from the density 33; with the neighbours'
// records one behind the other, each in a branch of its own, 31.8, now 27.7.)
// Vertices that normals are asked for leave their word and place in the normal's slot, for mc_normals_kernel.
// 1280 run at a time, five per CU, by their registers, and the rest begin as those end.  What the number is hardly matters: the call with 1280 | 1536 | 1792 | 2304 | 4096 in us, 512^3
// with 0.9 M triangles 170.1 | 167.8 | 166.7 | 168.9 | 169.6, with 1.6 M 191.4 | 197.0 | 190.2 | 189.8 | 191.4, 448^3 1.2 M 152.0 | 149.1 | 149.3 | 150.0 | 150.4, 384^3 0.9 M 113.7 | 112.0 |
// 112.0 | 112.2 | 112.1; the same within 1 % for 320^3, 256^3, 192^3, 128^3, 64^3 and lattices of 512 x 512 x 64 points on any side.  (Six per CU, with four registers spilled: 29.4 us for 27.5.)
constexpr uint32_t MC_EMIT_GRID = 2304;
typedef uint32_t mc_words2 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t mc_words3 __attribute__((ext_vector_type(3), aligned(4)));
typedef float mc_float2 __attribute__((ext_vector_type(2), aligned(4)));
template <bool SHORT>
__global__ void __launch_bounds__(MC_BLOCK) mc_emit_kernel(McGrid g, const float* __restrict__ density, const mc_word* __restrict__ bits,
                                                           const McRecord* __restrict__ records, const mc_word* __restrict__ active,
                                                           const uint2* __restrict__ blocks, uint32_t n_blocks, const uint32_t* __restrict__ listed,
                                                           float* __restrict__ verts, uint32_t* __restrict__ indices, uint32_t* __restrict__ origin) {
	__shared__ uint16_t list[MC_LIST];
	__shared__ uint32_t slot_of[8][MC_BLOCK];
	__shared__ uint32_t wave_sum[MC_BLOCK / 64];
	__shared__ mc_word edges[3][MC_BLOCK], tri[3][MC_BLOCK];
	__shared__ uint2 first[MC_BLOCK];
	const uint32_t n_listed = blocks[n_blocks + 1u].x;
	for (uint32_t at_block = blockIdx.x; at_block < n_listed; at_block += gridDim.x) {
		const uint32_t block = listed[at_block], block0 = block * MC_BLOCK;
		const bool owns = mc_owns<SHORT>(active, block, threadIdx.x);
		const uint2 before = blocks[block];
		mc_word points = 0;
		if (owns) {
			const McRecord& r = records[block0 + threadIdx.x];
#pragma unroll
			for (uint32_t a = 0; a < 3; ++a) {
				edges[a][threadIdx.x] = r.edge[a];
				tri[a][threadIdx.x] = r.tri[a];
				points |= r.edge[a] | r.tri[a];
			}
			first[threadIdx.x] = make_uint2(before.x + r.first_v, before.y + r.first_t);
		}
		// (mc_for_points' first barrier stands between these stores and their readers)
		auto from_memory = [&](uint32_t w) {
			const McRecord& r = records[w];
			return McOwned{{r.edge[0], r.edge[1], r.edge[2]}, blocks[w / MC_BLOCK].x + r.first_v};
		};
		mc_for_points(points, list, wave_sum, [&](uint32_t entry) {
			const uint32_t at0 = entry >> 6, w = block0 + at0, p = entry & 63u;
			const McOwned own{{edges[0][at0], edges[1][at0], edges[2][at0]}, first[at0].x};
			const mc_word t0 = tri[0][at0], t1 = tri[1][at0], t2 = tri[2][at0];
			const McPlace place = mc_place<SHORT>(g, w, p);
			const uint32_t tris = (uint32_t)((t0 >> p) & 1ull) | (uint32_t)((t1 >> p) & 1ull) << 1 | (uint32_t)((t2 >> p) & 1ull) << 2;
			// The point's density and its neighbours' (where there is none, another one), and the bits of the point and of the next along x in the
			// four rows of its cube (the cubes of the last column, row and plane have no triangles: any bits).
			const uint32_t x0 = min(place.x, g.rx - 2u), y1 = min(place.y + 1u, g.ry - 1u), z1 = min(place.z + 1u, g.rz - 1u);
			const mc_float2 along = *reinterpret_cast<const mc_float2*>(density + ((uint64_t)place.z * g.ry + place.y) * g.rx + x0);
			const float f0 = place.x == x0 ? along.x : along.y;
			const float f1[3] = {along.y, density[((uint64_t)place.z * g.ry + y1) * g.rx + place.x], density[((uint64_t)z1 * g.ry + place.y) * g.rx + place.x]};
			uint32_t at[4], bit[4], pair[4];
#pragma unroll
			for (uint32_t j = 0; j < 4; ++j) {
				at[j] = w + ((j & 1u) ? g.row_words : 0u) + ((j & 2u) ? g.row_words * g.ry : 0u);
				bit[j] = p;
				if (SHORT) {
					bit[j] = (j & 1u) ? p + (1u << g.pitch_log) : p;
					at[j] = w + (bit[j] >> MC_SHORT_BITS_LOG) + ((j & 2u) ? g.plane_words : 0u);
					bit[j] &= (1u << MC_SHORT_BITS_LOG) - 1u;
				}
				// (eight bytes from the 32 bits that the point is in; behind the last word the records follow)
				const mc_words2 two = *reinterpret_cast<const mc_words2*>(reinterpret_cast<const uint32_t*>(bits) + 2u * min(at[j], g.n_words - 1u) + (bit[j] >> 5));
				pair[j] = (uint32_t)(((uint64_t)two.y << 32 | two.x) >> (bit[j] & 31u)) & 3u;
			}
			// (corners run round a face)
			auto turned = [](uint32_t two) { return two >> 1 | (two & 1u) << 1; };
			const uint32_t mask = pair[0] | turned(pair[1]) << 2 | pair[2] << 4 | turned(pair[3]) << 6;
			uint4 row4 = make_uint4(0u, 0u, 0u, 0u);
			if (tris) {  // (the points one further along x, y and z exist)
				// The words of the plane at z + 1, most often of another block, are under way together; the one at y + 1 most often stands in LDS.
				McOwned o[4];
				o[0] = own;
				o[2] = from_memory(at[2]);
				o[3] = from_memory(at[3]);
				row4 = *reinterpret_cast<const uint4*>(MC_TABLE.tri[mask]);
				const uint32_t at1 = at[1] - block0;
				if (at1 < MC_BLOCK) o[1] = McOwned{{edges[0][at1], edges[1][at1], edges[2][at1]}, first[at1].x};
				else o[1] = from_memory(at[1]);
#pragma unroll
				for (uint32_t j = 0; j < 4; ++j) {
					const uint32_t slot = mc_vertex_slot(o[j], bit[j]), up = bit[j] + 1u;
					slot_of[2 * j][threadIdx.x] = slot;
					uint32_t next = (slot & 0x1FFFFFFFu) + (uint32_t)__popc(slot >> 29);
#pragma unroll
					for (uint32_t a = 0; a < 3; ++a) next |= (uint32_t)((o[j].e[a] >> (up & 63u)) & 1ull) << (29u + a);
					slot_of[2 * j + 1][threadIdx.x] = next;
				}
				if (!SHORT && p == 63u) {
#pragma unroll
					for (uint32_t j = 0; j < 4; ++j) o[j] = from_memory(at[j] + 1u);
#pragma unroll
					for (uint32_t j = 0; j < 4; ++j) slot_of[2 * j + 1][threadIdx.x] = mc_vertex_slot(o[j], 0u);
				}
			}
			const uint32_t slot0 = mc_vertex_slot(own, p), flags = slot0 >> 29;
			if (flags) {
				const float pos[3] = {(float)place.x, (float)place.y, (float)place.z};
				uint32_t slot = slot0 & 0x1FFFFFFFu;
#pragma unroll
				for (uint32_t a = 0; a < 3; ++a) {
					if (!((flags >> a) & 1u)) continue;
					const float dt = (g.thresh - f0) / (f1[a] - f0);
					n2_float3 v;
#pragma unroll
					for (uint32_t d = 0; d < 3; ++d) v[d] = (d == a ? pos[d] + dt : pos[d]) * g.scale[d] + g.offset[d];
					n2_store3<false>(verts + (size_t)slot * 3, v);
					if (origin) *reinterpret_cast<mc_words2*>(origin + (size_t)slot * 3) = mc_words2{w, p | a << 6};
					++slot;
				}
			}
			if (tris == 0) return;
			const uint32_t first_t = first[at0].y + mc_below(t0, p) + 2u * mc_below(t1, p) + 4u * mc_below(t2, p);
			// Lattice point and direction that own each cube edge (src/marching_cubes.cu:690-706), five bits per edge:
			// the owner's offset from this point in x, y, z and the edge's axis.
			constexpr uint64_t OWNER = 0ull | 9ull << 5 | 2ull << 10 | 8ull << 15 | 4ull << 20 | 13ull << 25 | 6ull << 30 | 12ull << 35 |
			                           16ull << 40 | 17ull << 45 | 19ull << 50 | 18ull << 55;
			const uint32_t trow[4] = {row4.x, row4.y, row4.z, row4.w};
			uint32_t* out = indices + (size_t)first_t * 3;
#pragma unroll
			for (uint32_t t = 0; t < 5; ++t) {
				if (t < tris) {
					mc_words3 v;
#pragma unroll
					for (uint32_t c = 0; c < 3; ++c) {
						const uint32_t k = 3 * t + c, e = (trow[k >> 2] >> (8u * (k & 3u))) & 0xFu;
						const uint32_t code = (uint32_t)(OWNER >> (5u * e)) & 31u;
						const uint32_t at = slot_of[code & 7u][threadIdx.x];
						// the owner's first slot plus the number of its edges before this one
						v[c] = (at & 0x1FFFFFFFu) + (uint32_t)__popc((at >> 29) & ((1u << (code >> 3)) - 1u));
					}
					*reinterpret_cast<mc_words3*>(out + 3 * t) = v;
				}
			}
		});
	}
}

// accumulate_1ring's normals: a vertex's is the sum of (pb - pa) x (pa - pc) over the triangles it is a corner of.  They lie in
// the four cubes round the vertex's edge; the cubes are visited in lattice order and their triangles in theirs, so the sum
// does not depend on how the work is scheduled.  (Adding every triangle to its corners with float atomics took 276 us for
// the 512^3 sphere's 1.2 M triangles: 11 M atomics at the part's 40 G/s.)
// The triangles' other corners are worked out again from the density, by the arithmetic that placed them: the eighteen values of the four
// cubes tell which triangles there are (MC_RING) and where their corners lie.  That is 18 loads a vertex and vector instructions; going
// through the words' records to the triangles and from those to the vertices was some 45 loads, most of them lines of their own, one a
// clock and CU: 32.5 us for 512^3, then 25.8, and 23.9 where an XCD takes consecutive vertices and finds the rows and planes next to one's own in its
// L2.  What bounds it is the vector unit, some 140 instructions for a triangle; rows loaded as three values at a time, and all triangles of a vertex in
// one loop instead of one per cube, changed nothing (24.1).
template <bool SHORT>
__global__ void __launch_bounds__(MC_BLOCK) mc_normals_kernel(McGrid g, uint32_t n_verts, const float* __restrict__ density, float* __restrict__ normals) {
	__shared__ float values[18][MC_BLOCK];  // [slow -1 .. 1][fast -1 .. 1][along 0, 1]
	// (workgroups go to the XCDs in turn: each XCD takes consecutive vertices)
	const uint32_t xcd = blockIdx.x % N2_XCDS, item = xcd * (gridDim.x / N2_XCDS) + min(xcd, gridDim.x % N2_XCDS) + blockIdx.x / N2_XCDS;
	const uint32_t i = item * MC_BLOCK + threadIdx.x;
	if (i >= n_verts) return;
	float* mine = normals + (size_t)i * 3;
	const uint32_t w = __float_as_uint(mine[0]), place = __float_as_uint(mine[1]);
	const uint32_t axis = place >> 6;
	const McPlace p = mc_place<SHORT>(g, w, place & 63u);
	// in the frame (along, fast, slow): the point, the lattice and its strides
	const uint64_t row = g.rx, plane = (uint64_t)g.rx * g.ry;
	const uint32_t at[3] = {axis == 0u ? p.x : axis == 1u ? p.y : p.z, axis == 0u ? p.y : p.x, axis == 2u ? p.y : p.z};
	const uint32_t size[3] = {0u, axis == 0u ? g.ry : g.rx, axis == 2u ? g.ry : g.rz};
	const uint64_t step[3] = {axis == 0u ? 1u : axis == 1u ? row : plane, axis == 0u ? row : 1u, axis == 2u ? row : plane};
	const float scale[3] = {axis == 0u ? g.scale[0] : axis == 1u ? g.scale[1] : g.scale[2], axis == 0u ? g.scale[1] : g.scale[0], axis == 2u ? g.scale[1] : g.scale[2]};
	const float offset[3] = {axis == 0u ? g.offset[0] : axis == 1u ? g.offset[1] : g.offset[2], axis == 0u ? g.offset[1] : g.offset[0], axis == 2u ? g.offset[1] : g.offset[2]};
	const bool below[3] = {false, at[1] > 0u, at[2] > 0u}, above[3] = {false, at[1] + 1u < size[1], at[2] + 1u < size[2]};
	const float* here = density + (p.z * plane + p.y * row + p.x);
	uint32_t inside = 0;
#pragma unroll
	for (uint32_t k = 0; k < 3; ++k) {
		// (where there is nothing beyond the point, its own row or plane again: the cubes that would use it are left out)
		const float* in_k = k == 0u ? (below[2] ? here - step[2] : here) : k == 2u ? (above[2] ? here + step[2] : here) : here;
#pragma unroll
		for (uint32_t j = 0; j < 3; ++j) {
			const float* in_j = j == 0u ? (below[1] ? in_k - step[1] : in_k) : j == 2u ? (above[1] ? in_k + step[1] : in_k) : in_k;
#pragma unroll
			for (uint32_t o = 0; o < 2; ++o) {
				const float v = in_j[o ? step[0] : 0u];
				values[6 * k + 2 * j + o][threadIdx.x] = v;
				inside |= v > g.thresh ? 1u << (6 * k + 2 * j + o) : 0u;
			}
		}
	}
	// position of the vertex on the edge that starts at `corner` of the cube whose first corner is (0, j, k) - 1 of the values, as mc_emit_kernel gives it
	auto vertex = [&](uint32_t j, uint32_t k, uint32_t edge, float (&to)[3]) {
		const uint32_t dir = edge >> 3, n = (edge & 1u) + 2u * (j + ((edge >> 1) & 1u)) + 6u * (k + ((edge >> 2) & 1u)), next = n + (dir == 0u ? 1u : dir == 1u ? 2u : 6u);
		const float f0 = values[n][threadIdx.x], f1 = values[next][threadIdx.x], dt = (g.thresh - f0) / (f1 - f0);
		const float from[3] = {(float)(at[0] + (edge & 1u)), (float)(at[1] + j - 1u + ((edge >> 1) & 1u)), (float)(at[2] + k - 1u + ((edge >> 2) & 1u))};
#pragma unroll
		for (uint32_t d = 0; d < 3; ++d) to[d] = (from[d] + (dir == d ? dt : 0.f)) * scale[d] + offset[d];
	};
	float self[3], sum[3] = {0.f, 0.f, 0.f};
	vertex(1u, 1u, 0u, self);
#pragma unroll
	for (uint32_t q = 0; q < 4; ++q) {
		const uint32_t j = q & 1u, k = q >> 1;  // the cube's first corner among the values
		if (!(j ? above[1] : below[1]) || !(k ? above[2] : below[2])) continue;
		const uint32_t corners = ((inside >> (6u * k + 2u * j)) & 15u) | ((inside >> (6u * k + 6u + 2u * j)) & 15u) << 4;
		uint64_t fan = MC_RING.fan[axis][q][corners];
		for (uint32_t n = (uint32_t)(fan >> 60); n; --n, fan >>= 12) {
			float p1[3], p2[3];
			vertex(j, k, (uint32_t)fan & 31u, p1);
			vertex(j, k, (uint32_t)(fan >> 5) & 31u, p2);
			const uint32_t me = (uint32_t)(fan >> 10) & 3u;
			float u[3], v[3];
#pragma unroll
			for (uint32_t d = 0; d < 3; ++d) {
				const float pa = me == 0u ? self[d] : p1[d], pb = me == 0u ? p1[d] : me == 1u ? self[d] : p2[d], pc = me == 2u ? self[d] : p2[d];
				u[d] = pb - pa;
				v[d] = pa - pc;
			}
			sum[0] += u[1] * v[2] - u[2] * v[1];
			sum[1] += u[2] * v[0] - u[0] * v[2];
			sum[2] += u[0] * v[1] - u[1] * v[0];
		}
	}
	// (along y the frame is left-handed)
	mine[0] = axis == 0u ? sum[0] : axis == 1u ? 0.f - sum[1] : sum[1];
	mine[1] = axis == 0u ? sum[1] : axis == 1u ? 0.f - sum[0] : sum[2];
	mine[2] = axis == 0u ? sum[2] : axis == 1u ? 0.f - sum[2] : sum[0];
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
static inline dim3 mgrid(uint64_t n) { return dim3((uint32_t)((n + MC_BLOCK - 1) / MC_BLOCK)); }
static inline uint64_t m256(uint64_t x) { return (x + 255) / 256 * 256; }

N2_API int n2_marching_cubes_table(int8_t* out_256x16) {
	N2_REQUIRE(out_256x16 != nullptr, "n2_marching_cubes_table: out is null");
	memcpy(out_256x16, MC_TABLE_HOST.tri, sizeof(MC_TABLE_HOST.tri));
	return N2_OK;
}

static int mc_check(const char* fn, const uint32_t res[3], uint64_t& n) {
	N2_REQUIRE(res != nullptr, "%s: res is null", fn);
	N2_REQUIRE(res[0] >= 2 && res[1] >= 2 && res[2] >= 2, "%s: every resolution must be at least 2 (got %u x %u x %u)", fn, res[0], res[1], res[2]);
	n = (uint64_t)res[0] * res[1] * res[2];
	N2_REQUIRE(n <= (1ull << 31), "%s: %llu lattice points exceed 2^31", fn, (unsigned long long)n);
	return N2_OK;
}

// Workspace: the points' bits, one record per word (written only where a word owns something), which words do, and the
// prefix sums over blocks of 256 words (behind them the totals and the number of blocks that own something), and a list of those blocks.
struct McCarve {
	uint32_t row_words, pitch_log, rows_log, plane_words, n_words, n_blocks;
	bool short_rows;
	uint64_t bits, records, active, blocks, listed, total;
};
static McCarve mc_carve(const uint32_t res[3]) {
	McCarve c;
	c.row_words = (res[0] + 63u) / 64u;
	c.short_rows = res[0] < MC_SHORT_ROW;
	c.pitch_log = 1;
	while ((1u << c.pitch_log) < res[0] && c.short_rows) ++c.pitch_log;
	c.rows_log = MC_SHORT_BITS_LOG - c.pitch_log;
	c.plane_words = c.short_rows ? (res[1] + (1u << c.rows_log) - 1u) >> c.rows_log : c.row_words * res[1];
	c.n_words = c.plane_words * res[2];  // at most 2^29: planes have at least four points
	c.n_blocks = (c.n_words + MC_BLOCK - 1) / MC_BLOCK;
	uint64_t o = 0;
	auto take = [&](uint64_t bytes) { const uint64_t at = o; o += m256(bytes); return at; };
	c.bits = take(sizeof(mc_word) * (uint64_t)c.n_words);
	c.records = take(sizeof(McRecord) * (uint64_t)c.n_words);
	c.active = take(sizeof(mc_word) * (uint64_t)c.n_blocks * (MC_BLOCK / 64));
	c.blocks = take(sizeof(uint2) * ((uint64_t)c.n_blocks + 2));
	c.listed = take(sizeof(uint32_t) * (uint64_t)c.n_blocks);
	c.total = o;
	return c;
}

N2_API uint64_t n2_marching_cubes_workspace_bytes(const uint32_t res[3]) {
	uint64_t n;
	if (mc_check("n2_marching_cubes_workspace_bytes", res, n) != N2_OK) return 0;
	return mc_carve(res).total;
}

static McGrid mc_grid(const uint32_t res[3], const float aabb_min[3], const float aabb_max[3], float thresh) {
	McGrid g;
	g.rx = res[0]; g.ry = res[1]; g.rz = res[2]; g.thresh = thresh;
	for (int d = 0; d < 3; ++d) { g.scale[d] = (aabb_max[d] - aabb_min[d]) / (float)res[d]; g.offset[d] = aabb_min[d]; }
	const McCarve c = mc_carve(res);
	g.row_words = c.row_words;
	g.n_words = c.n_words;
	g.pitch_log = c.pitch_log;
	g.rows_log = c.rows_log;
	g.plane_words = c.plane_words;
	g.here = g.xok = 0;
	for (uint32_t at = 0; c.short_rows && at < 1u << MC_SHORT_BITS_LOG; at += 1u << c.pitch_log) {
		g.here |= ((1u << res[0]) - 1u) << at;
		g.xok |= ((1u << (res[0] - 1u)) - 1u) << at;
	}
	return g;
}

// Where the scan can leave the totals by itself: the addresses that a kernel of this device has for the caller's variables when both lie in pinned
// host memory, else null.
static void mc_totals_of(uint32_t* n_vertices, uint32_t* n_triangles, uint32_t*& to_v, uint32_t*& to_t) {
	int device = -1;
	auto mapped = [&](uint32_t* p) -> uint32_t* {
		hipPointerAttribute_t attr{};
		if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
			(void)hipGetLastError();  // (memory that HIP does not know)
			return nullptr;
		}
		const bool ours = attr.type == hipMemoryTypeHost && attr.device == device && !(attr.allocationFlags & hipHostRegisterReadOnly);
		return ours ? static_cast<uint32_t*>(attr.devicePointer) : nullptr;
	};
	to_v = to_t = nullptr;
	if (hipGetDevice(&device) != hipSuccess) return;
	uint32_t* const v = mapped(n_vertices);
	uint32_t* const t = v ? mapped(n_triangles) : nullptr;
	if (t) { to_v = v; to_t = t; }
}

// Waits for the totals that the scan leaves in pinned memory (MC_NO_TOTAL before): for them alone, not for the end of the launch and what the runtime does about it.
// Where the work in front takes longer than MC_TOTALS_WAIT, fails, or is being captured, for the stream.
constexpr uint32_t MC_NO_TOTAL = 0xFFFFFFFFu;
constexpr std::chrono::milliseconds MC_TOTALS_WAIT(1);
static hipError_t mc_await_totals(hipStream_t s, const uint32_t* n_vertices, const uint32_t* n_triangles) {
	hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
	if (hipStreamIsCapturing(s, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone) {
		auto there = [&]() { return __atomic_load_n(n_vertices, __ATOMIC_ACQUIRE) != MC_NO_TOTAL && __atomic_load_n(n_triangles, __ATOMIC_ACQUIRE) != MC_NO_TOTAL; };
		if (n2_poll(there, MC_TOTALS_WAIT)) return hipSuccess;
	}
	return hipStreamSynchronize(s);
}

static int mc_count(const char* name, n2_stream_t stream, const uint32_t res[3], const float aabb_min[3], const float aabb_max[3], float thresh, const float* d_density, void* d_workspace,
                    uint64_t workspace_bytes, uint32_t* n_vertices, uint32_t* n_triangles, bool totals_only) {
	uint64_t n;
	if (int rc = mc_check(name, res, n)) return rc;
	N2_REQUIRE(d_density && d_workspace && n_vertices && n_triangles && aabb_min && aabb_max, "%s: null argument", name);
	N2_REQUIRE(reinterpret_cast<uintptr_t>(d_workspace) % 256 == 0, "%s: workspace must be 256-byte aligned", name);
	const McCarve c = mc_carve(res);
	N2_REQUIRE(workspace_bytes >= c.total, "%s: %llu bytes of workspace given, %llu needed", name,
	           (unsigned long long)workspace_bytes, (unsigned long long)c.total);
	hipStream_t s = n2_stream(stream);
	unsigned char* b = reinterpret_cast<unsigned char*>(d_workspace);
	mc_word* bits = reinterpret_cast<mc_word*>(b + c.bits);
	uint2* blocks = reinterpret_cast<uint2*>(b + c.blocks);
	const McGrid g = mc_grid(res, aabb_min, aabb_max, thresh);
	const bool stream_density = 4 * n >= MC_STREAM_BYTES;
	auto* const bits_kernel = c.short_rows ? (stream_density ? mc_bits_kernel<true, true> : mc_bits_kernel<false, true>)
	                                       : (stream_density ? mc_bits_kernel<true, false> : mc_bits_kernel<false, false>);
	bits_kernel<<<mgrid(((uint64_t)c.n_words + MC_BITS_WORDS - 1) / MC_BITS_WORDS * 64u), dim3(MC_BLOCK), 0, s>>>(g, d_density, bits);
	N2_LAUNCH_CHECK();
	auto* const count_kernel = c.short_rows ? mc_count_short_kernel : mc_count_kernel;
	count_kernel<<<dim3(c.n_blocks), dim3(c.short_rows ? MC_BLOCK : 64u), 0, s>>>(g, bits, reinterpret_cast<McRecord*>(b + c.records), reinterpret_cast<mc_word*>(b + c.active), blocks);
	N2_LAUNCH_CHECK();
	// (left there by the scan: 512^3 182 us, 64^3 53; copied, with a copy kernel and its staging, 191 and 61)
	uint32_t *to_v, *to_t;
	mc_totals_of(n_vertices, n_triangles, to_v, to_t);
	if (to_v && totals_only) {
		__atomic_store_n(n_vertices, MC_NO_TOTAL, __ATOMIC_RELEASE);
		__atomic_store_n(n_triangles, MC_NO_TOTAL, __ATOMIC_RELEASE);
	}
	mc_scan_kernel<<<dim3(1), dim3(1024), 0, s>>>(c.n_blocks, blocks, reinterpret_cast<uint32_t*>(b + c.listed), to_v, to_t);
	N2_LAUNCH_CHECK();
	uint32_t host[2] = {0, 0};
	if (to_v) {
		N2_HIP(totals_only ? mc_await_totals(s, n_vertices, n_triangles) : hipStreamSynchronize(s));
		host[0] = *n_vertices;
		host[1] = *n_triangles;
	} else {
		N2_HIP(hipMemcpyAsync(host, blocks + c.n_blocks, sizeof(host), hipMemcpyDeviceToHost, s));
		N2_HIP(hipStreamSynchronize(s));
	}
	if (host[0] >= (1u << 29) && totals_only) N2_HIP(hipStreamSynchronize(s));  // (no second pass will follow: nothing may be under way in a workspace that the caller frees or reuses)
	N2_REQUIRE(host[0] < (1u << 29), "%s: %u vertices exceed the 2^29 limit", name, host[0]);
	*n_vertices = host[0];
	*n_triangles = host[1];
	return N2_OK;
}

N2_API int n2_marching_cubes_count(n2_stream_t stream, const uint32_t res[3], const float aabb_min[3], const float aabb_max[3], float thresh,
                                   const float* d_density, void* d_workspace, uint64_t workspace_bytes, uint32_t* n_vertices,
                                   uint32_t* n_triangles) {
	return mc_count("n2_marching_cubes_count", stream, res, aabb_min, aabb_max, thresh, d_density, d_workspace, workspace_bytes, n_vertices, n_triangles, false);
}

N2_API int n2_marching_cubes_count_totals(n2_stream_t stream, const uint32_t res[3], const float aabb_min[3], const float aabb_max[3], float thresh,
                                          const float* d_density, void* d_workspace, uint64_t workspace_bytes, uint32_t* n_vertices,
                                          uint32_t* n_triangles) {
	return mc_count("n2_marching_cubes_count_totals", stream, res, aabb_min, aabb_max, thresh, d_density, d_workspace, workspace_bytes, n_vertices, n_triangles, true);
}

N2_API int n2_marching_cubes_emit(n2_stream_t stream, const uint32_t res[3], const float aabb_min[3], const float aabb_max[3], float thresh,
                                  const float* d_density, void* d_workspace, float* d_vertices, uint32_t* d_indices, float* d_normals,
                                  uint32_t n_vertices, uint32_t n_triangles) {
	uint64_t n;
	if (int rc = mc_check("n2_marching_cubes_emit", res, n)) return rc;
	N2_REQUIRE(d_density && d_workspace && aabb_min && aabb_max, "n2_marching_cubes_emit: null argument");
	N2_REQUIRE((d_vertices || n_vertices == 0) && (d_indices || n_triangles == 0), "n2_marching_cubes_emit: null output");
	N2_REQUIRE(d_normals == nullptr || reinterpret_cast<uintptr_t>(d_normals) % 16 == 0, "n2_marching_cubes_emit: d_normals must be 16-byte aligned");
	if (n_vertices == 0) return N2_OK;  // no cut edge: no triangles either
	hipStream_t s = n2_stream(stream);
	const McCarve c = mc_carve(res);
	unsigned char* b = reinterpret_cast<unsigned char*>(d_workspace);
	const McRecord* records = reinterpret_cast<const McRecord*>(b + c.records);
	const mc_word* active = reinterpret_cast<const mc_word*>(b + c.active);
	const uint2* blocks = reinterpret_cast<const uint2*>(b + c.blocks);
	const McGrid g = mc_grid(res, aabb_min, aabb_max, thresh);
	auto* const emit_kernel = c.short_rows ? mc_emit_kernel<true> : mc_emit_kernel<false>;
	emit_kernel<<<dim3(c.n_blocks < MC_EMIT_GRID ? c.n_blocks : MC_EMIT_GRID), dim3(MC_BLOCK), 0, s>>>(g, d_density, reinterpret_cast<const mc_word*>(b + c.bits), records, active, blocks, c.n_blocks, reinterpret_cast<const uint32_t*>(b + c.listed), d_vertices, d_indices,
	                                                        reinterpret_cast<uint32_t*>(d_normals));
	N2_LAUNCH_CHECK();
	if (d_normals) {
		auto* const normals_kernel = c.short_rows ? mc_normals_kernel<true> : mc_normals_kernel<false>;
		normals_kernel<<<mgrid(n_vertices), dim3(MC_BLOCK), 0, s>>>(g, n_vertices, d_density, d_normals);
		N2_LAUNCH_CHECK();
	}
	return N2_OK;
}

// ---------------------------------------------------------------------------
// The lattice the mesh is extracted from: Testbed::get_density_on_grid (src/testbed_nerf.cu:4082-4133) with
// generate_grid_samples_nerf_uniform (:586-598) and grid_samples_half_to_float (:682-696): positions
// (x, y, z) / res * (aabb.max - aabb.min) + aabb.min, the field's SDF (row 0 of NerfNetwork::sdf) widened to fp32.
// ---------------------------------------------------------------------------
typedef _Float16 hf;

__global__ void __launch_bounds__(MC_BLOCK) mc_lattice_positions_kernel(McGrid g, uint64_t first, uint32_t count, uint32_t padded,
                                                                        float* __restrict__ positions) {
	const uint32_t i = blockIdx.x * MC_BLOCK + threadIdx.x;
	if (i >= padded) return;
	float* p = positions + (size_t)i * 3;
	if (i >= count) { p[0] = p[1] = p[2] = 0.5f; return; }
	const uint64_t idx = first + i;
	const uint32_t c[3] = {(uint32_t)(idx % g.rx), (uint32_t)((idx / g.rx) % g.ry), (uint32_t)(idx / ((uint64_t)g.rx * g.ry))};
	const uint32_t r[3] = {g.rx, g.ry, g.rz};
#pragma unroll
	for (int d = 0; d < 3; ++d) p[d] = ((float)c[d] * (1.f / (float)r[d])) * g.scale[d] + g.offset[d];
}
// positions and the network's output for the fields whose points are written out; the fused kernels keep 44 bytes per point
// there, and their weight fragments behind it
N2_API uint64_t n2_density_on_grid_scratch_bytes(uint32_t chunk) { return m256(12ull * chunk) + m256(32ull * chunk) + m256(n2_lattice_frag_bytes()); }

N2_API int n2_density_on_grid(n2_field_t* field, n2_stream_t stream, const uint32_t res[3], const float aabb_min[3], const float aabb_max[3],
                              float* d_density, void* d_scratch, uint64_t scratch_bytes, uint32_t chunk) {
	uint64_t n;
	if (int rc = mc_check("n2_density_on_grid", res, n)) return rc;
	N2_REQUIRE(field && d_density && d_scratch && aabb_min && aabb_max, "n2_density_on_grid: null argument");
	N2_REQUIRE(chunk >= 8 && chunk % 8 == 0, "n2_density_on_grid: chunk %u must be a positive multiple of 8", chunk);
	N2_REQUIRE(reinterpret_cast<uintptr_t>(d_scratch) % 256 == 0 && scratch_bytes >= n2_density_on_grid_scratch_bytes(chunk),
	           "n2_density_on_grid: scratch must be 256-byte aligned and hold %llu bytes", (unsigned long long)n2_density_on_grid_scratch_bytes(chunk));
	hipStream_t s = n2_stream(stream);
	float* positions = reinterpret_cast<float*>(d_scratch);
	hf* mlp_out = reinterpret_cast<hf*>(reinterpret_cast<unsigned char*>(d_scratch) + m256(12ull * chunk));
	McGrid g;
	g.rx = res[0]; g.ry = res[1]; g.rz = res[2]; g.thresh = 0.f;
	// here scale is the aabb's extent (the division by the resolution is part of the position formula)
	for (int d = 0; d < 3; ++d) { g.scale[d] = aabb_max[d] - aabb_min[d]; g.offset[d] = aabb_min[d]; }
	int rc = N2_OK;
	N2Lattice lat;
	for (int d = 0; d < 3; ++d) { lat.res[d] = res[d]; lat.inv_res[d] = 1.f / (float)res[d]; lat.extent[d] = g.scale[d]; lat.corner[d] = g.offset[d]; }
	if (n2_field_sdf_row0_lattice(field, stream, lat, chunk, d_scratch, reinterpret_cast<unsigned char*>(d_scratch) + m256(12ull * chunk) + m256(32ull * chunk), d_density, &rc)) return rc;
	// lattice points arrive x fastest: neighbouring lanes in neighbouring cells
	n2_grid_set_point_order(n2_field_encoding(field), 1);
	for (uint64_t first = 0; first < n && rc == N2_OK; first += chunk) {
		const uint32_t m = (uint32_t)((n - first < chunk) ? n - first : chunk), m8 = (m + 7) / 8 * 8;
		mc_lattice_positions_kernel<<<mgrid(m8), dim3(MC_BLOCK), 0, s>>>(g, first, m, m8, positions);
		// the padded tail of the last chunk (m8 - m points at most 7) is evaluated but not kept
		rc = n2_field_sdf_row0(field, stream, positions, 3, 1, m8, m, d_density + first, reinterpret_cast<n2_half*>(mlp_out));
	}
	n2_grid_set_point_order(n2_field_encoding(field), 0);
	if (rc != N2_OK) return rc;
	N2_LAUNCH_CHECK();
	return N2_OK;
}
