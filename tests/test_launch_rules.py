"""The sizes of launches (neus2_amd/csrc/launch_rules.h), compiled with the host compiler: no GPU needed."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WRAPPERS = """
#include "launch_rules.h"
extern "C" void lattice_slab(const uint32_t* res, uint64_t points, uint32_t* out) {
	const N2LatticeSlab s = n2_lattice_slab(res, points);
	out[0] = s.nx; out[1] = s.ny; out[2] = s.nz;
}
extern "C" uint64_t lattice_slab_points(uint64_t rest, uint64_t words, uint32_t n_fine, int large, uint32_t* in_scratch) {
	return n2_lattice_slab_points(rest, words, n_fine, large, *in_scratch);
}
extern "C" int lattice_large_slabs(uint64_t all, uint64_t words, uint32_t n_fine) { return n2_lattice_large_slabs(all, words, n_fine); }
extern "C" uint32_t lattice_fine_walk(uint32_t runs, uint32_t nz) { return n2_lattice_fine_walk(runs, nz); }
extern "C" uint32_t lattice_fine_waves(uint32_t runs, uint32_t nz) { return n2_lattice_fine_waves(runs, nz); }
extern "C" uint32_t lattice_walk(uint32_t runs, uint32_t nz, uint32_t per_simd) { return n2_lattice_walk(runs, nz, per_simd); }
extern "C" int gather_visits(uint32_t by_xcd_max, uint32_t n, uint32_t n_levels, uint32_t points_per_block, uint32_t* visits, uint32_t* grid) {
	const N2GatherGrid g = n2_gather_grid(by_xcd_max, n, n_levels, points_per_block);
	grid[0] = g.x; grid[1] = g.y;
	const uint32_t tiles = n / points_per_block + (n % points_per_block != 0u);
	if (visits == nullptr) return 0;
	for (uint32_t y = 0; y < g.y; ++y)
		for (uint32_t x = 0; x < g.x; ++x) {
			uint32_t level = 0, tile = 0;
			if (!n2_gather_item(x, y, g.y, n_levels, tiles, level, tile)) continue;
			if (level >= n_levels || tile >= tiles) return 1;
			++visits[level * tiles + tile];
		}
	return 0;
}
extern "C" void lattice_chunks(uint32_t first, uint32_t last, uint32_t* out) { n2_lattice_chunks(first, last, out[0], out[1]); }
extern "C" uint32_t walked_levels(const float* scale, float step) { return n2_lattice_walked_levels(scale, step); }
extern "C" uint32_t row_levels(const float* scale, uint32_t nx, float step_x, float reach, float step_z) { return n2_lattice_row_levels(scale, nx, step_x, reach, step_z); }
extern "C" int by_rows(uint32_t rows, uint32_t walked, uint64_t points) { return n2_lattice_by_rows(rows, walked, points); }
extern "C" uint32_t bin_points_per_thread(uint32_t levels, uint32_t n) { return n2_bin_points_per_thread(levels, n, 512); }
extern "C" uint32_t bin_single_points(uint32_t levels) { return n2_bin_single_points(levels, 512); }
extern "C" uint32_t turns(uint32_t first, uint32_t second, uint32_t group, uint32_t* blocks) {
	const N2Turns t = n2_turns(first, second, group);
	*blocks = t.blocks;
	return t.every;
}
extern "C" uint32_t turn(uint32_t block, uint32_t every, uint32_t group, uint32_t* second) {
	bool s;
	const uint32_t at = n2_turn(block, every, group, s);
	*second = s;
	return at;
}
extern "C" void rows_of_blocks(uint32_t blocks, uint32_t threads, uint32_t* out) {
	const N2GatherGrid g = n2_rows_of_blocks(blocks, threads);
	out[0] = g.x; out[1] = g.y;
}
extern "C" uint32_t run_tile(uint32_t group, uint32_t groups, uint32_t run, uint32_t part_shift, uint32_t tiles) { return n2_run_tile(group, groups, run, part_shift, tiles); }
extern "C" uint64_t run_base(uint32_t first_tile, uint32_t tile_records) { return n2_run_base(first_tile, tile_records); }
extern "C" uint32_t run_place(uint32_t first_tile, uint32_t tile, uint32_t tile_records) { return n2_run_place(first_tile, tile, tile_records); }
extern "C" int sdf_one_pass(uint32_t n) { return n2_sdf_one_pass(n); }
extern "C" int adam_lists(uint64_t n_params, uint32_t n_levels, uint64_t batch) { return n2_adam_lists(n_params, n_levels, batch); }
extern "C" int optimiser_streams(uint64_t state_bytes, uint64_t batch, int listed) { return n2_optimiser_streams(state_bytes, batch, listed); }
extern "C" int jacobian_streams(uint32_t n, uint32_t rows) { return n2_jacobian_streams(n, rows); }
extern "C" int whole_lines(uint32_t n, uint32_t bytes) { return n2_rows_of_whole_lines(n, bytes); }
extern "C" int step_stores_stream(uint32_t n, uint32_t rows) { return n2_step_jacobian_stores_stream(n, rows); }
extern "C" int step_loads_stream(uint32_t n, uint32_t rows) { return n2_step_jacobian_loads_stream(n, rows); }
extern "C" int moments_stream(uint64_t state_bytes, uint64_t batch) { return n2_moments_stream(state_bytes, batch); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.cpp", d / "rules.so"
    src.write_text(WRAPPERS)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "neus2_amd", "csrc"),
                    str(src), "-o", str(so)], check=True, timeout=60)
    return C.CDLL(str(so))


# the smallest scratch, rows longer than it (with and without a whole run in it), rows of two points, the largest lattices,
# a row that alone has more runs than a launch takes
@pytest.mark.parametrize("res", [(2, 2, 2), (512, 512, 512), (96, 4, 3), (1000, 7, 2), (2, 1 << 23, 2), (2, 1 << 15, 1 << 15), (1 << 29, 2, 2), (3, 5, 1 << 27)])
@pytest.mark.parametrize("chunk", [8, 64, 1 << 14, 1 << 22, 1 << 31])
@pytest.mark.parametrize("n_fine", [1, 6, 10])
def test_lattice_slabs_fit_the_scratch_and_the_launch(rules, res, chunk, n_fine):
    points = 11 * chunk // n_fine
    out = (C.c_uint32 * 3)()
    rules.lattice_slab((C.c_uint32 * 3)(*res), C.c_uint64(points), out)
    nx, ny, nz = out
    assert 1 <= nx <= res[0] and 1 <= ny <= res[1] and 1 <= nz <= res[2]
    assert nx * ny * nz <= points
    assert (ny == 1 or nx == res[0]) and (nz == 1 or ny == res[1])  # the slab is one piece of the scratch's rows
    # a launch counts its threads in 32 bits: 64 lanes per run of 64 points and level, in workgroups of four
    assert ((nx + 63) // 64 * ny * nz + 3) // 4 * 256 * n_fine < 1 << 32
    # nothing is given away: the slab is the lattice, or another column, row or plane would not fit one of the two
    runs = (nx + 63) // 64
    if nx < res[0]:
        assert nx == points or nx == points // 64 * 64 or runs == 1 << 22
    elif ny < res[1]:
        assert nx * (ny + 1) > points or runs * (ny + 1) > 1 << 22
    elif nz < res[2]:
        assert nx * ny * (nz + 1) > points or runs * ny * (nz + 1) > 1 << 22


# one point, fewer than the scratch has words, about as many as it takes, 512^3, the largest lattice; down to the smallest scratch
@pytest.mark.parametrize("rest", [1, 7, 88, 1 << 16, 1 << 22, 1 << 27, 1 << 31])
@pytest.mark.parametrize("chunk", [8, 1 << 14, 1 << 20, 1 << 22, 1 << 31])
@pytest.mark.parametrize("n_fine", [0, 1, 6, 12])
def test_features_of_a_slab_fit_the_scratch_and_the_output_behind_it(rules, rest, chunk, n_fine):
    rules.lattice_slab_points.restype = C.c_uint64
    words, k = 11 * chunk, C.c_uint32(99)
    alone = words // max(n_fine, 1)
    for large in (0, 1):
        left, slabs = rest, 0
        while left > 0 and slabs < 1000:
            m = rules.lattice_slab_points(C.c_uint64(left), C.c_uint64(words), n_fine, large, C.byref(k))
            assert min(left, alone) <= m <= left  # never fewer than the scratch alone takes
            assert k.value * m <= words and (k.value == max(n_fine, 1) or k.value < n_fine)
            if k.value < n_fine:
                assert large and m > alone and (n_fine - k.value) * m <= left - m
            left -= m
            slabs += 1
    assert rules.lattice_large_slabs(C.c_uint64(rest), C.c_uint64(words), n_fine) == (n_fine > 0 and rest > 8 * alone)


# one run and plane, small lattices, 512^3, the most runs of a launch, lattices that are all planes
@pytest.mark.parametrize("runs,nz", [(1, 1), (1, 3), (64, 64), (192, 96), (4096, 29), (4096, 88), (1 << 22, 1), (1, 1 << 22), (2, 1 << 21)])
@pytest.mark.parametrize("per_simd", [2, 3])
def test_planes_of_a_wave_are_equal_shares_of_the_slab(rules, runs, nz, per_simd):
    for walk, most in ((rules.lattice_fine_walk(runs, nz), 12), (rules.lattice_walk(runs, nz, per_simd), 24)):
        assert 1 <= walk <= min(most, nz)
        parts = -(-nz // walk)
        assert walk == -(-nz // parts)  # no shorter waves for as many of them


# 64^3, both sides of the line along either number, the smallest, more runs than 32 bits count
@pytest.mark.parametrize("runs,nz,waves", [(64, 64, 5), (1, 1, 5), (160, 64, 5), (161, 64, 6), (1, 10240, 5), (1, 10241, 6), (4096, 29, 6), (1 << 22, 1 << 10, 6)])
def test_waves_of_the_fine_levels(rules, runs, nz, waves):
    assert rules.lattice_fine_waves(runs, nz) == waves


# What the two rules below are made of.  Parameters of the field with tables of 2^14 to 2^22 entries a level (18 bytes of optimiser state each), batch, streamed
@pytest.mark.parametrize("n_params,batch,streams", [
    (506884, 1 << 14, 0), (506884, 1 << 16, 0), (506884, 1 << 18, 1), (3507780, 1 << 16, 0), (3507780, 1 << 18, 1), (12612212, 1 << 12, 0),
    (12612212, 20480, 0), (12612212, 28672, 1), (12612212, 1 << 18, 1), (24146548, 1 << 12, 1), (85050820, 1 << 12, 1), (1 << 31, 1 << 31, 1)])
def test_moments_are_streamed_where_state_and_samples_exceed_the_cache(rules, n_params, batch, streams):
    assert rules.moments_stream(C.c_uint64(18 * n_params), C.c_uint64(batch)) == streams


# The optimiser of a training step: the field with tables of 2^14 to 2^22 entries a level, 18 bytes of state per parameter (24 with the average).  Both sides of each line: a sixth of the
# parameters met (8192 | 8320 samples at the default table, fewer levels meet fewer), the smallest table and the largest batch that are listed, and where lists and whole pieces are streamed
@pytest.mark.parametrize("n_params,n_levels,state,batch,listed,streams", [
    (12612212, 16, 18, 128, 1, 0), (12612212, 16, 18, 3072, 1, 0), (12612212, 16, 18, 3328, 1, 1), (12612212, 16, 18, 8192, 1, 1), (12612212, 16, 18, 8320, 0, 1), (12612212, 16, 18, 20480, 0, 1),
    (12612212, 16, 18, 1 << 18, 0, 1), (12612212, 16, 24, 512, 1, 1), (12612212, 8, 18, 16384, 1, 1), (12612212, 8, 18, 16512, 0, 1), (506884, 16, 18, 128, 0, 0), (506884, 16, 18, 48896, 0, 0),
    (506884, 16, 18, 50048, 0, 1), ((1 << 21) - 4, 16, 18, 1024, 0, 0), (1 << 21, 16, 18, 1280, 1, 0), (1 << 21, 16, 18, 1408, 0, 0), (3507780, 16, 18, 2176, 1, 0), (3507780, 16, 18, 2304, 0, 0),
    (24146548, 16, 18, 15616, 1, 1), (24146548, 16, 18, 16384, 0, 1), (85050820, 16, 18, 40960, 1, 1), (85050820, 16, 18, 41088, 0, 1), (1 << 32, 16, 18, 41088, 0, 1), (1 << 32, 16, 18, 128, 1, 1)])
def test_which_optimiser_a_batch_takes(rules, n_params, n_levels, state, batch, listed, streams):
    assert rules.adam_lists(C.c_uint64(n_params), n_levels, C.c_uint64(batch)) == listed
    assert rules.optimiser_streams(C.c_uint64(state * n_params), C.c_uint64(batch), listed) == streams


# 32 rows of 12 bytes a point: 12 MiB, 64 MiB and 160 MiB from both sides, rows that start lines (a multiple of 32 points) and that do not, the most points
@pytest.mark.parametrize("n,stores,loads,alone", [(8, 0, 0, 0), (32736, 0, 0, 0), (32768, 0, 1, 0), (32776, 0, 0, 0), (174752, 0, 1, 0), (174760, 0, 0, 0), (174768, 0, 1, 1),
                                                  (174784, 0, 1, 1), (174792, 0, 1, 1), (436896, 0, 1, 1), (436928, 1, 1, 1), (436936, 1, 1, 1), (0xFFFFFFF8, 1, 1, 1)])
def test_where_the_jacobian_is_streamed(rules, n, stores, loads, alone):
    assert (rules.step_stores_stream(C.c_uint32(n), 32), rules.step_loads_stream(C.c_uint32(n), 32), rules.jacobian_streams(C.c_uint32(n), 32)) == (stores, loads, alone)


@pytest.mark.parametrize("n,bytes,whole", [(0, 2, 1), (64, 2, 1), (63, 2, 0), (32, 2, 0), (32, 4, 1), (31, 4, 0), (32, 12, 1), (8, 12, 0), (1 << 31, 12, 1), ((1 << 32) - 32, 12, 1), ((1 << 32) - 8, 12, 0)])
def test_rows_that_start_lines(rules, n, bytes, whole):
    assert rules.whole_lines(C.c_uint32(n), bytes) == whole


# one level, fewer levels than XCDs, a last round that is not full, the most levels; one tile, tiles that the XCDs cannot share
# evenly; either side of the line
@pytest.mark.parametrize("n_levels", [1, 3, 8, 11, 16, 32])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 1999, 2000, 2001, 5003])
def test_gather_workgroups_meet_every_level_and_tile_once(rules, n_levels, n):
    tiles = -(-n // 128)
    visits, grid = np.zeros(n_levels * tiles, np.uint32), np.zeros(2, np.uint32)
    assert rules.gather_visits(2000, n, n_levels, 128, visits.ctypes.data_as(C.c_void_p), grid.ctypes.data_as(C.c_void_p)) == 0
    assert (visits == 1).all()
    assert (grid[1] > 1) == (n > 2000 and n_levels > 1)


@pytest.mark.parametrize("n", [1 << 18, (1 << 27) - 8, 1 << 27, 1 << 28, 1 << 30])
def test_gather_launch_of_two_lanes_a_point_stays_below_the_thread_limit(rules, n):
    grid = np.zeros(2, np.uint32)
    rules.gather_visits(1 << 19, n, 16, 128, None, grid.ctypes.data_as(C.c_void_p))
    assert int(grid[0]) * 256 < 1 << 32 and int(grid[1]) < 1 << 16


# lattices over the unit cube with 64 to 512 planes (the default table), a box of a tenth of it, a table of eight levels (the rest have scale 1)
@pytest.mark.parametrize("planes,extent,levels,walked", [(64, 1, 16, 6), (128, 1, 16, 6), (208, 1, 16, 6), (224, 1, 16, 8), (256, 1, 16, 8), (272, 1, 16, 10), (384, 1, 16, 10),
                                                         (512, 1, 16, 10), (64, 0.1, 16, 10), (64, 1, 8, 10), (1 << 20, 1, 16, 10), (2, 1, 16, 6)])
def test_levels_the_lattice_walks(rules, planes, extent, levels, walked):
    scale = [16 * 1.447 ** l - 1 if l < levels else 1.0 for l in range(16)]
    assert rules.walked_levels((C.c_float * 16)(*scale), C.c_float(extent / planes)) == walked


# cells of a run's ends: rising, falling, one cell, negative, and the ends of the 32-bit range (boxes far outside the unit cube)
@pytest.mark.parametrize("first,last", [(0, 0), (3, 4), (8, 519), (519, 8), (-1, 2), (-517, -3), (-2 ** 31, 2 ** 31 - 1), (2 ** 31 - 1, -2 ** 31), (-2 ** 31, 5), (0, 2 ** 31 - 1),
                                        (2 ** 31 - 1, 2 ** 31 - 1), (-2 ** 31, -2 ** 31)])
def test_lattice_chunks_hold_every_cell_of_the_run(rules, first, last):
    out = (C.c_uint32 * 2)()
    rules.lattice_chunks(C.c_uint32(first % 2 ** 32), C.c_uint32(last % 2 ** 32), out)
    lo, chunks = C.c_int32(out[0]).value, out[1]
    a, b = min(first, last), max(first, last)
    assert lo % 4 == 0 and lo <= a < lo + 4 and lo + 4 * (chunks - 1) <= b + 1 < lo + 4 * chunks


# the unit cube at several sizes, part of a run, a box upside down along x and along z, one as large as its cells' numbers are exact, no box
@pytest.mark.parametrize("nx,lo,hi,planes,down", [(512, 0, 1, 512, 1), (400, 0, 1, 400, 1), (64, 0, 1, 64, 1), (2, 0, 1, 512, 1), (33, 0, 1, 300, 1), (200, 1, 0, 200, 1), (200, 0, 1, 200, -1),
                                                  (512, -1.5, 2.5, 512, 1), (512, 4e3, 4e3 + 1, 512, 1), (512, 3e5, 3e5 + 1, 512, 1), (512, 0, float("nan"), 512, 1), (512, -2.0 ** 40, 2.0 ** 40, 8, 1)])
def test_runs_of_the_levels_walked_by_rows_fit_a_wave(rules, nx, lo, hi, planes, down):
    """The vertices that any 64 points of such a level meet, cells as the kernels round them, are 64 at most; no plane is left out."""
    f = np.float32
    scale = [float(f(16 * 1.447 ** l - 1)) for l in range(16)]
    inv, ext = f(1) / f(nx), f(hi) - f(lo)
    step_z = f(down) / f(planes)
    reach = max(abs(f(lo)), abs(f(lo) + ext))
    n = rules.row_levels((C.c_float * 16)(*scale), C.c_uint32(nx), C.c_float(abs(float(inv * ext))), C.c_float(float(reach)), C.c_float(float(step_z)))
    assert n <= 10 and (n == 0 or (np.isfinite(hi) and down > 0))
    x = (np.arange(nx).astype(f) * inv * ext + f(lo)).astype(f)
    z = (np.arange(planes).astype(f) * abs(step_z)).astype(f)
    for s in scale[:n]:
        cell, plane = (np.floor((v.astype(np.float64) * f(s) + 0.5).astype(f)) for v in (x, z))  # one fused multiply-add
        for at in range(0, nx, 64):
            run = cell[at:at + 64]
            assert run.max() + 1 - run.min() < 64
        assert np.diff(plane).max(initial=0) <= 1
    if (lo, hi, down) == (0, 1, 1):
        assert n >= {512: 10, 400: 9, 64: 4}.get(nx, 0)


@pytest.mark.parametrize("rows,walked,points,want", [(4, 6, 64 ** 3, 0), (5, 6, 80 ** 3, 1), (4, 6, 512 * 512 * 64, 1), (4, 10, 64 * 512 * 512, 0), (5, 10, 80 * 512 * 400, 0),
                                                     (8, 10, 256 * 256 * 512, 1), (10, 10, 512 ** 3, 1), (0, 6, 1 << 31, 0), (3, 6, 1 << 31, 0)])
def test_which_lattices_are_walked_by_rows(rules, rows, walked, points, want):
    assert rules.by_rows(C.c_uint32(rows), C.c_uint32(walked), C.c_uint64(points)) == want


@pytest.mark.parametrize("levels", [1, 4, 5, 8, 16, 32])
def test_one_point_per_thread_while_all_sorting_workgroups_run_at_once(rules, levels):
    line = rules.bin_single_points(C.c_uint32(levels))
    assert levels * (line // 512) <= 768 < levels * (line // 512 + 1) and line % 512 == 0
    assert [rules.bin_points_per_thread(C.c_uint32(levels), C.c_uint32(n)) for n in (1, line, line + 1, 1 << 31)] == [1, 1, 2, 2]


# one tile, few of them in parts, an ordinary batch, the last one whose level of single records 32 bits count, the first one that they do not, the largest; whole and split buckets
@pytest.mark.parametrize("n,part_shift", [(8, 6), (5000, 2), (1 << 18, 0), (1 << 29, 0), ((1 << 29) + 1024, 0), (1 << 30, 0)])
@pytest.mark.parametrize("tile_records", [8192, 4096])
@pytest.mark.parametrize("group,groups", [(0, 1), (0, 32), (31, 32)])
def test_places_of_a_levels_records_beyond_32_bits(rules, n, part_shift, tile_records, group, groups):
    """What a wave's lanes count from its addresses leads to their tiles' records, of which 64 runs lie within 32 bits."""
    rules.run_base.restype, rules.run_place.restype = C.c_uint64, C.c_uint32
    tiles = -(-n // 1024)
    groups, group = min(groups, tiles), min(group, tiles - 1)
    runs = -(-(tiles - group) // groups) << part_shift
    for stride in (8, 12, 16):
        for first in {w + k * 64 * stride for w in (0, 1, stride - 1) for k in (0, 1, (runs - 1) // (64 * stride))}:
            first_tile = rules.run_tile(group, groups, first, part_shift, tiles)
            base = rules.run_base(first_tile, tile_records)
            for lane in range(64):
                run = first + stride * lane
                tile = rules.run_tile(group, groups, run, part_shift, tiles)
                assert tile == min(group + groups * (run >> part_shift), tiles - 1)
                if run < runs:
                    assert base + rules.run_place(first_tile, tile, tile_records) == tile * tile_records <= (tiles - 1) * tile_records


@pytest.mark.parametrize("n,fits", [(8, 1), (1 << 18, 1), (1 << 26, 1), (71582784, 1), (71582792, 0), (1 << 27, 0), (1 << 28, 0)])
def test_one_pass_of_the_sdf_network_while_its_offsets_fit_32_bits(rules, n, fits):
    """The last lane's place in the Jacobian: row 4 of its scalar base, the last point, three floats each."""
    assert rules.sdf_one_pass(C.c_uint32(n)) == fits == ((4 * n + n - 1) * 12 + 11 < 1 << 32)


# sorting workgroups and those of the input gradient (600 points, 2^14, one level), gathering workgroups and those that sort (groups of the XCDs)
@pytest.mark.parametrize("first,second,group", [(32, 2, 1), (512, 32, 1), (1, 2, 1), (5, 3, 1), (32, 32, 8), (160, 80, 8), (24, 13, 8), (1, 1, 8), (7, 100, 8)])
def test_workgroups_of_two_kinds_are_all_met_once(rules, first, second, group):
    blocks, kind = C.c_uint32(), C.c_uint32()
    every = rules.turns(C.c_uint32(first), C.c_uint32(second), C.c_uint32(group), C.byref(blocks))
    seen = [[], []]
    for b in range(blocks.value):
        at = rules.turn(C.c_uint32(b), C.c_uint32(every), C.c_uint32(group), C.byref(kind))
        assert at % group == b % group  # the XCD is the workgroup's own
        seen[kind.value].append(at)
    for got, n in zip(seen, (first, second)):
        assert [k for k in sorted(got) if k < n] == list(range(n))


# launches that fit one row, by one workgroup less, exactly and by one more; the second order's launch for 2^28 points of sixteen levels; the largest batch of 32 levels
@pytest.mark.parametrize("blocks,threads", [(1, 512), (8388599, 512), (8388600, 512), (8388601, 512), (3 * (1 << 28) // 1024 * 16, 512), (3 * (1 << 30) // 1024 * 32, 512), (1 << 31, 1024)])
def test_rows_of_workgroups_stay_below_the_thread_limit(rules, blocks, threads):
    out = (C.c_uint32 * 2)()
    rules.rows_of_blocks(C.c_uint32(blocks), C.c_uint32(threads), out)
    x, y = out
    assert x * threads < 1 << 32 and y < 1 << 16 and blocks <= x * y < blocks + 16 * y
    assert y == 1 or x % 8 == 0
    assert (y == 1) == (blocks <= 8388600 * 512 // threads // 8 * 8)
