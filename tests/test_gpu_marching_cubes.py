"""Marching cubes and the SDF lattice on the GPU against the oracle, through the C ABI."""
import os

import numpy as np
import pytest
import torch

from gpu_util import RTOL, assert_close, dev, host, q16
from oracle import marching_cubes as omc
from test_oracle_marching_cubes import check_closed_oriented, sphere_lattice

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def test_case_table_equals_the_oracles():
    from neus2_amd.mesh import case_table
    np.testing.assert_array_equal(case_table(), omc.TRIANGLE_TABLE)


@pytest.mark.parametrize("res,kind", [((40, 48, 32), "sphere"), ((17, 9, 33), "noise"), ((2, 2, 2), "noise"), ((64, 64, 64), "two"),
                                      ((100, 24, 10), "noise"), ((130, 9, 7), "noise"), ((96, 80, 72), "sphere")])  # rows that end inside a wave's 64 points
def test_mesh_matches_oracle(res, kind):
    from neus2_amd.mesh import marching_cubes
    rng = np.random.default_rng(res[0])
    if kind == "sphere":
        f, thresh = sphere_lattice(res), 0.0
    elif kind == "two":  # two overlapping balls, threshold off zero
        f = np.maximum(sphere_lattice(res, (0.4, 0.5, 0.5), 0.2), sphere_lattice(res, (0.65, 0.55, 0.45), 0.15))
        thresh = 0.01
    else:  # every case of the table, ambiguous faces included
        f, thresh = rng.standard_normal((res[2], res[1], res[0])).astype(np.float32), 0.1
    lo, hi = (-0.5, 0.0, 0.25), (1.5, 1.0, 0.75)
    want_v, want_t = omc.marching_cubes(f, res, thresh, lo, hi)
    v, t, n = marching_cubes(dev(f), thresh, lo, hi)
    assert v.shape == (len(want_v), 3) and t.shape == (len(want_t), 3)
    np.testing.assert_array_equal(host(v), want_v)                      # bit-exact vertex positions, same numbering
    np.testing.assert_array_equal(host(t).view(np.uint32), want_t)      # same triangles in the same order
    want_n = omc.vertex_normals(want_v, want_t)
    np.testing.assert_allclose(host(n), want_n, rtol=1e-4, atol=1e-6 * max(1.0, float(np.abs(want_n).max())))
    if kind in ("sphere", "two"):
        assert check_closed_oriented(host(v), host(t).astype(np.int64)) == 2


@pytest.mark.parametrize("res", [(63, 6, 5), (64, 6, 5), (65, 6, 5), (128, 30, 12), (129, 40, 11),  # one point short of a word of 64, exact, one over; several blocks of words
                                 # several rows to a word: every pitch, rows that fill it and do not, planes of part of a word, of whole ones, of one row more
                                 (2, 2, 5), (2, 32, 7), (2, 33, 7), (3, 17, 9), (4, 15, 6), (5, 8, 6), (8, 9, 70), (9, 4, 5), (9, 3, 5), (15, 7, 40), (15, 6, 300),
                                 (16, 7, 5), (17, 65, 4)])
def test_rows_of_words(res):
    """Noise: every word of points owns something, so the points of a block fill the emitting kernel's list several times."""
    from neus2_amd.mesh import marching_cubes
    f = np.random.default_rng(res[0] + res[1]).standard_normal((res[2], res[1], res[0])).astype(np.float32)
    want_v, want_t = omc.marching_cubes(f, res, 0.0, (0, 0, 0), (1, 1, 1))
    v, t, n = marching_cubes(dev(f), 0.0)
    np.testing.assert_array_equal(host(v), want_v)
    np.testing.assert_array_equal(host(t).view(np.uint32), want_t)
    want_n = omc.vertex_normals(want_v, want_t)
    np.testing.assert_allclose(host(n), want_n, rtol=1e-4, atol=1e-6 * max(1.0, float(np.abs(want_n).max())))
    assert marching_cubes(dev(f), 0.0, want_normals=False)[2] is None


@pytest.mark.parametrize("res", [(512, 512, 128), (320, 64, 16)])
def test_a_plane_through_every_block_of_words(res):
    """More blocks that own something than workgroups emit at a time, and waves that count whole blocks: one vertex per row, two triangles per square."""
    from neus2_amd.mesh import marching_cubes
    rx, ry, rz = res
    f = (torch.arange(rx, device="cuda") - 200.25).expand(rz, ry, rx).contiguous()
    v, t, n = marching_cubes(f, 0.0, (0, 0, 0), res)  # (one unit per cell)
    assert v.shape == (ry * rz, 3) and t.shape == (2 * (ry - 1) * (rz - 1), 3)
    v, t, n = (a.cpu().view(*s, 3) for a, s in ((v, (rz, ry)), (t, (rz - 1, ry - 1, 2)), (n, (rz, ry))))
    assert bool((v[..., 0] == 200.25).all())
    assert torch.equal(v[..., 1], torch.arange(ry).float().expand(rz, ry)) and torch.equal(v[..., 2], torch.arange(rz).float().view(-1, 1).expand(rz, ry))
    z, y = torch.meshgrid(torch.arange(rz - 1), torch.arange(ry - 1), indexing="ij")
    corner = (z * ry + y).int()
    assert torch.equal(t.reshape(rz - 1, ry - 1, 6).amin(-1), corner) and torch.equal(t.reshape(rz - 1, ry - 1, 6).amax(-1), corner + ry + 1)
    assert bool((n[..., 1:] == 0).all()) and bool((n[1:-1, 1:-1, 0].abs() == 6).all())  # six triangles of twice the area one


@pytest.mark.parametrize("inside_first", [False, True])
@pytest.mark.parametrize("res,axis,at", [((64, 512, 6), 1, 256), ((64, 512, 6), 1, 255), ((128, 64, 10), 2, 4), ((128, 64, 10), 2, 3), ((128, 64, 10), 2, 8), ((256, 128, 5), 0, 64), ((256, 128, 5), 0, 63),
                                         ((130, 100, 9), 2, 8), ((512, 512, 700), 2, 699), ((512, 512, 700), 2, 513), ((512, 512, 1100), 2, 1030)])
def test_a_plane_between_blocks_without_a_surface(res, axis, at, inside_first):
    """A plane across `axis` between the points at - 1 and at, where blocks of 256 words begin and end, all bits of the others the same; with more than 8192 and 16 384 blocks."""
    from neus2_amd.mesh import marching_cubes
    x = torch.arange(res[axis], device="cuda", dtype=torch.float32) - (at - 0.25)
    shape = [1, 1, 1]
    shape[2 - axis] = res[axis]
    f = (-x if inside_first else x).view(shape).expand(res[2], res[1], res[0]).contiguous()
    v, t, n = marching_cubes(f, 0.0, (0, 0, 0), res)
    others = [res[d] for d in range(3) if d != axis]
    assert v.shape == (others[0] * others[1], 3) and t.shape == (2 * (others[0] - 1) * (others[1] - 1), 3)
    want = torch.stack(torch.meshgrid(*[torch.arange(r, device="cuda").float() if d != 2 - axis else torch.tensor([at - 0.25], device="cuda") for d, r in enumerate(reversed(res))], indexing="ij")[::-1], -1)
    assert torch.equal(v, want.reshape(-1, 3))
    assert torch.equal(t.long().reshape(-1).unique(), torch.arange(len(v), device="cuda"))


def test_meshes_counted_by_several_threads_at_once():
    """Each call waits for totals of its own."""
    from concurrent.futures import ThreadPoolExecutor

    from neus2_amd.mesh import marching_cubes
    fields = [dev(np.random.default_rng(k).standard_normal((6 + k % 5, 9 + k % 7, 20 + k)).astype(np.float32)) for k in range(40)]
    want = [tuple(host(a) for a in marching_cubes(f, 0.0)) for f in fields]

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            out = [marching_cubes(fields[(k + q) % 40], 0.0) for q in range(4)]
            torch.cuda.current_stream().synchronize()
            return [tuple(host(a) for a in o) for o in out]
    with ThreadPoolExecutor(40) as pool:
        for k, got in enumerate(pool.map(work, range(40))):
            for q, o in enumerate(got):
                for a, b in zip(o, want[(k + q) % 40]):
                    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("res", [(70, 9, 11), (192, 5, 4), (64, 3, 2), (7, 9, 11), (15, 6, 5)])  # rows that end inside a word and with one, shared words
def test_triangles_are_those_of_the_counted_density(res):
    """The second pass with another density and threshold moves vertices; its triangles stay those that the first pass counted."""
    import ctypes as C

    from neus2_amd import capi
    from neus2_amd.mesh import _f3, _stream, _u3, marching_cubes
    L = capi.lib()
    L.n2_marching_cubes_workspace_bytes.restype = C.c_uint64
    rng = np.random.default_rng(sum(res))
    f, other = (dev(rng.standard_normal(res[::-1]).astype(np.float32)) for _ in range(2))
    v, t, _ = marching_cubes(f, 0.1)
    assert 0 <= int(t.min()) and int(t.max()) < len(v)
    nbytes = int(L.n2_marching_cubes_workspace_bytes(_u3(res)))
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    box = _u3(res), _f3((0, 0, 0)), _f3((1, 1, 1))
    for density, thresh in ((f, 0.1), (f, 0.7), (other, 0.1), (torch.zeros_like(f), 0.0)):
        nv, nt = C.c_uint32(), C.c_uint32()
        capi.check(L.n2_marching_cubes_count(_stream(), *box, C.c_float(0.1), capi.ptr(f), capi.ptr(ws), C.c_uint64(nbytes), C.byref(nv), C.byref(nt)), "count")
        verts, normals = (torch.empty((nv.value, 3), device="cuda") for _ in range(2))
        idx = torch.full((nt.value, 3), -1, dtype=torch.int32, device="cuda")
        capi.check(L.n2_marching_cubes_emit(_stream(), *box, C.c_float(thresh), capi.ptr(density), capi.ptr(ws), capi.ptr(verts), capi.ptr(idx), capi.ptr(normals), nv, nt), "emit")
        assert torch.equal(idx, t)
        assert torch.equal(verts, v) == (density is f and thresh == 0.1)


def test_totals_in_pinned_and_in_other_host_memory():
    """A kernel writes them where both variables are pinned; else they are copied, and nothing beside them is written."""
    import ctypes as C

    from neus2_amd import capi
    from neus2_amd.mesh import _f3, _stream, _u3, marching_cubes
    L = capi.lib()
    L.n2_marching_cubes_workspace_bytes.restype = C.c_uint64
    pinned, pageable = torch.empty(24, dtype=torch.int32, pin_memory=True), torch.empty(24, dtype=torch.int32)
    for k in range(6):
        f = dev(np.random.default_rng(k).standard_normal((9 + k, 8, 21 + k)).astype(np.float32))
        v, t, _ = marching_cubes(f, 0.0)
        res = _u3(f.shape[::-1])
        nbytes = int(L.n2_marching_cubes_workspace_bytes(res))
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        for a, b in ((pinned, pinned), (pageable, pageable), (pinned, pageable), (pageable, pinned)):
            pinned.fill_(-1)
            pageable.fill_(-1)
            at = [C.c_uint32.from_address(a.data_ptr() + 4 * 5), C.c_uint32.from_address(b.data_ptr() + 4 * (11 + k))]
            capi.check(L.n2_marching_cubes_count(_stream(), res, _f3((0, 0, 0)), _f3((1, 1, 1)), C.c_float(0), capi.ptr(f), capi.ptr(ws),
                                                 C.c_uint64(nbytes), C.byref(at[0]), C.byref(at[1])), "n2_marching_cubes_count")
            assert (at[0].value, at[1].value) == (len(v), len(t))
            assert int((pinned == -1).sum() + (pageable == -1).sum()) == 46


@pytest.mark.parametrize("res", [(2, 2, 2), (9, 8, 21), (65, 64, 3), (17, 1500, 1500)])  # one block of words, short rows, several blocks, more than the scan takes in a round
@pytest.mark.parametrize("busy", [False, True])  # nothing in front, or more work than the wait for the totals alone lasts
def test_totals_that_are_waited_for_alone(res, busy):
    import ctypes as C

    from neus2_amd import capi
    from neus2_amd.mesh import _f3, _stream_address, _u3, marching_cubes
    L = capi.lib()
    L.n2_marching_cubes_workspace_bytes.restype = C.c_uint64
    x, y, z = (torch.arange(r, device="cuda") for r in res)
    f = (torch.sin(1.7 * x + 1)[None, None, :] + torch.sin(0.11 * y)[None, :, None] + torch.sin(0.13 * z + 2)[:, None, None]).contiguous()
    v, t, n = marching_cubes(f, 0.0)
    nbytes = int(L.n2_marching_cubes_workspace_bytes(_u3(res)))
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    head = (_stream_address(), _u3(res), _f3((0, 0, 0)), _f3((1, 1, 1)), 0.0, f.data_ptr(), ws.data_ptr())
    load = torch.zeros(1 << 28, device="cuda")
    for totals in (torch.empty(2, dtype=torch.int32, pin_memory=True), torch.empty(2, dtype=torch.int32)):
        totals.fill_(7)
        torch.cuda.synchronize()
        for _ in range(20 if busy else 0):
            load.add_(1.0)
        capi.check(L.n2_marching_cubes_count_totals(*head, nbytes, totals.data_ptr(), totals.data_ptr() + 4), "count_totals")
        assert totals.tolist() == [len(v), len(t)]
        verts, normals, idx = torch.zeros_like(v), torch.zeros_like(n), torch.zeros_like(t)
        capi.check(L.n2_marching_cubes_emit(*head, verts.data_ptr() or None, idx.data_ptr() or None, normals.data_ptr() or None, len(v), len(t)), "emit")
        assert torch.equal(verts, v) and torch.equal(idx, t) and torch.equal(normals, n)


def test_too_many_vertices_leave_nothing_under_way():
    """A caller that is told so goes on with no second pass, and may free the workspace: the call has waited for the stream, not for the totals alone."""
    import ctypes as C

    from neus2_amd import capi
    from neus2_amd.mesh import _f3, _stream_address, _u3
    L = capi.lib()
    L.n2_marching_cubes_workspace_bytes.restype = C.c_uint64
    side = 576  # every edge between neighbours is cut: 3 * 576 * 576 * 575 = 1.07 * 2^29 vertices
    x = torch.arange(side, device="cuda", dtype=torch.int16)
    f = (((x[None, None, :] + x[None, :, None] + x[:, None, None]) & 1).float() - 0.5).contiguous()
    res = _u3((side, side, side))
    nbytes = int(L.n2_marching_cubes_workspace_bytes(res))
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    totals = torch.empty(2, dtype=torch.int32, pin_memory=True)
    stream = torch.cuda.current_stream()
    torch.cuda.synchronize()
    for count in (L.n2_marching_cubes_count_totals, L.n2_marching_cubes_count):
        rc = count(_stream_address(), res, _f3((0, 0, 0)), _f3((1, 1, 1)), 0.0, f.data_ptr(), ws.data_ptr(), nbytes, totals.data_ptr(), totals.data_ptr() + 4)
        assert stream.query()
        assert rc != 0 and b"vertices exceed" in L.n2_last_error()


def test_empty_lattice_and_errors():
    from neus2_amd import capi
    from neus2_amd.mesh import marching_cubes
    v, t, n = marching_cubes(torch.full((8, 8, 8), -1.0, device="cuda"), 0.0)
    assert v.shape == (0, 3) and t.shape == (0, 3)
    with pytest.raises(capi.N2Error):
        marching_cubes(torch.zeros((1, 8, 8), device="cuda"), 0.0)
    with pytest.raises(capi.N2Error):
        marching_cubes(torch.zeros((8, 8, 8), device="cuda", dtype=torch.float16), 0.0)


# rows that end inside a run of 64 points, slabs of part of a plane (and of part of a row), steps
# of many cells of the fine levels (their rows are then gathered, not staged), several slabs of several planes, a box that
# sticks out of the unit cube, a grid of 8 levels with dense ones among those the walk does not keep, eight and ten levels walked
@pytest.mark.parametrize("res,chunk,box,levels", [((70, 9, 5), 1 << 14, (0, 1), 16), ((130, 20, 6), 512, (0.2, 0.9), 16), ((96, 4, 3), 64, (0, 1), 16),
                                                  ((16, 16, 40), 1 << 14, (0, 1), 16), ((320, 12, 33), 1 << 14, (0.4, 0.5), 16), ((40, 33, 21), 4096, (-0.2, 1.1), 16),
                                                  ((64, 30, 20), 1 << 14, (0, 1), 8), ((70, 5, 256), 1 << 14, (0, 1), 16), ((66, 4, 300), 4096, (0, 1), 16)])
def test_lattice_equals_the_same_points_queried(res, chunk, box, levels):
    """density_on_grid (rows of lattice points walked along z) against NerfNetwork::sdf on the same positions."""
    from neus2_amd.mesh import density_on_grid
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork(n_levels=levels)
    gen = torch.Generator(device="cuda").manual_seed(res[0])
    o = net.param_offsets()
    p = torch.randn(o[4], device="cuda", generator=gen) * 0.1
    net.set_params(p.half(), None)
    net.reserve(max(1 << 14, (res[0] * res[1] * res[2] + 7) // 8 * 8))
    lo, hi = (box[0], box[0] + 0.01, box[0]), (box[1], box[1], box[1] - 0.01)
    d = density_on_grid(net._h, res, lo, hi, chunk=chunk)
    z, y, x = np.meshgrid(*(np.arange(r, dtype=np.float32) for r in reversed(res)), indexing="ij")
    ext = np.asarray(hi, np.float32) - np.asarray(lo, np.float32)
    pos = np.stack([(c * np.float32(np.float32(1.0) / np.float32(r))) * e + np.float32(b) for c, r, e, b in zip((x, y, z), res, ext, lo)]).reshape(3, -1)
    n = pos.shape[1]
    padded = np.full((3, (n + 7) // 8 * 8), 0.5, np.float32)
    padded[:, :n] = pos
    want = host(net.sdf(dev(padded)))[0, :n].reshape(res[2], res[1], res[0])
    assert_close(host(d), want, rtol=RTOL, what="SDF lattice", outlier_frac=1e-3)


# Steps of 1 / side and planes of 1 / side: every number of levels that is walked by rows (sides 80 to 512; four only on large lattices), rows that
# end inside a run, several slabs, all three widths of the fine levels' rows; more levels walked along z than along x, boxes upside
# down along z and x, and one far from the unit cube (four vertices gathered per point and plane).  `part` of the box that is evaluated.
@pytest.mark.parametrize("side,res,part,chunk", [(80, (80, 6, 80), 1, 1 << 14), (112, (112, 4, 56), 0.5, 1 << 14), (150, (75, 5, 40), (0.5, 40 / 150), 1 << 11), (210, (70, 9, 66), (70 / 210, 66 / 210), 1 << 14),
                                                 (304, (152, 4, 38), (0.5, 0.125), 1 << 12), (416, (104, 5, 52), (0.25, 0.125), 1 << 14), (512, (130, 6, 64), (130 / 512, 0.125), 1 << 14),
                                                 (64, (512, 512, 64), (1, 1), 1 << 22), (512, (64, 6, 128), (1, 0.25), 1 << 14), (512, (130, 6, 64), (130 / 512, -0.125), 1 << 14),
                                                 (512, (130, 6, 64), (-130 / 512, 0.125), 1 << 14), (512, (66, 4, 64), (66 / 512, 0.125, 3e4), 1 << 14)])
def test_lattices_walked_by_rows_equal_the_same_points_queried(side, res, part, chunk):
    from neus2_amd.mesh import density_on_grid
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork()
    p = torch.randn(net.param_offsets()[4], device="cuda", generator=torch.Generator(device="cuda").manual_seed(side)) * 0.1
    net.set_params(p.half(), None)
    net.reserve(max(1 << 16, chunk))
    part = part if isinstance(part, tuple) else (part, part)
    at = part[2] if len(part) == 3 else 0.0
    f = np.float32
    lo = np.array([at + (0.3 if part[0] < 1 else 0), 0.2, 0.4 if abs(part[1]) < 1 else 0], f)
    hi = lo + np.array([part[0], res[1] / 300, part[1]], f)
    d = density_on_grid(net._h, res, tuple(lo), tuple(hi), chunk=chunk)
    keep = [np.arange(r) if r < 300 else np.unique(np.linspace(0, r - 1, 23).astype(int)) for r in res]  # of a large lattice some rows
    z, y, x = np.meshgrid(*(k.astype(f) for k in reversed(keep)), indexing="ij")
    ext = hi - lo
    pos = np.stack([(c * f(f(1.0) / f(r))) * e + b for c, r, e, b in zip((x, y, z), res, ext, lo)]).reshape(3, -1)
    n = pos.shape[1]
    padded = np.full((3, (n + 7) // 8 * 8), 0.5, f)
    padded[:, :n] = pos
    net.reserve(max(1 << 16, chunk, padded.shape[1]))
    want = host(net.sdf(dev(padded)))[0, :n].reshape(z.shape)
    got = host(d)[np.ix_(*reversed(keep))]
    assert_close(got, want, rtol=RTOL, what="SDF lattice", outlier_frac=1e-3)


# The finest level's row that a run of 64 points meets, in chunks of four entries: each number of words a lane takes, and both sides of where it becomes one
# more, wide loads begin and the points gather for themselves; by waves of three planes, whose loads are wide always, and of five.
@pytest.mark.parametrize("rows", [(6, 9), (160, 130)])
@pytest.mark.parametrize("chunks", [2, 16, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129])
def test_fine_rows_of_every_length(chunks, rows):
    from neus2_amd.mesh import density_on_grid
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork()
    f = np.float32
    scale = net.encoding().level_table()[0][15]
    res = (64, *rows)
    lo = np.array([0.3, 0.2, 0.1], f)

    def met(extent):
        x = (np.arange(64, dtype=f) * f(f(1.0) / f(64))) * f(extent) + lo[0]
        cell = np.floor(x.astype(np.float64) * float(scale) + 0.5).astype(int)
        return (cell[-1] + 1 - (cell[0] & ~3)) // 4 + 1

    extent = next(f(e) for e in np.arange(1, 1500) * 1e-4 if met(e) == chunks)
    hi = lo + np.array([extent, 0.7, 0.8], f)
    p = torch.randn(net.param_offsets()[4], device="cuda", generator=torch.Generator(device="cuda").manual_seed(chunks)) * 0.1
    net.set_params(p.half(), None)
    n = res[0] * res[1] * res[2]
    net.reserve((n + 7) // 8 * 8)
    d = density_on_grid(net._h, res, tuple(lo), tuple(hi), chunk=1 << 22)
    z, y, x = np.meshgrid(*(np.arange(r, dtype=f) for r in reversed(res)), indexing="ij")
    ext = hi - lo
    padded = np.full((3, (n + 7) // 8 * 8), 0.5, f)
    padded[:, :n] = np.stack([(c * f(f(1.0) / f(r))) * e + b for c, r, e, b in zip((x, y, z), res, ext, lo)]).reshape(3, -1)
    want = host(net.sdf(dev(padded)))[0, :n].reshape(z.shape)
    assert_close(host(d), want, rtol=RTOL, what="SDF lattice", outlier_frac=1e-3)


# The features of a slab lie in the scratch and, behind the slab, in the output: slabs that take both, the output alone (a scratch of less than a plane),
# planes in parts at the end, gathered and by rows, an output that starts anywhere; no fine level at all
@pytest.mark.parametrize("res,chunk,levels", [((70, 9, 60), 512, 16), ((70, 9, 60), 64, 16), ((130, 7, 33), 8, 16), ((300, 11, 90), 4096, 16), ((96, 33, 300), 1 << 14, 16),
                                              ((64, 8, 40), 256, 4)])
def test_a_lattice_in_slabs_equals_the_lattice_at_once(res, chunk, levels):
    import ctypes as C
    from neus2_amd import capi
    from neus2_amd.mesh import density_on_grid
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork(n_levels=levels)
    p = torch.randn(net.param_offsets()[4], device="cuda", generator=torch.Generator(device="cuda").manual_seed(res[0])) * 0.1
    net.set_params(p.half(), None)
    n = res[0] * res[1] * res[2]
    net.reserve((n + 7) // 8 * 8)
    whole = density_on_grid(net._h, res, (0, 0, 0), (1, 0.3, 0.4), chunk=(n + 7) // 8 * 8).flatten()
    L = capi.lib()
    L.n2_density_on_grid_scratch_bytes.restype = C.c_uint64
    nbytes = int(L.n2_density_on_grid_scratch_bytes(C.c_uint32(chunk)))
    scratch = torch.full((nbytes + 256,), 0x7B, dtype=torch.uint8, device="cuda")
    out = torch.full((n + 130,), 7.0, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for _ in range(2):  # the second time over the results of the first
        capi.check(L.n2_density_on_grid(net._h, stream, (C.c_uint32 * 3)(*res), (C.c_float * 3)(0, 0, 0), (C.c_float * 3)(1, 0.3, 0.4), C.c_void_p(out.data_ptr() + 4),
                                        C.c_void_p(scratch.data_ptr()), C.c_uint64(nbytes), C.c_uint32(chunk)), "n2_density_on_grid")
        assert torch.equal(out[1:1 + n], whole)
        assert (out[0] == 7) and (out[1 + n:] == 7).all() and (scratch[nbytes:] == 0x7B).all()


# levels switched off, among those that are walked too, whose entries may hold anything; walked by rows, and gathered
@pytest.mark.parametrize("res,active", [((130, 6, 64), 4), ((130, 6, 64), 9), ((130, 6, 64), 12), ((40, 9, 11), 3)])
def test_a_lattice_with_levels_switched_off(res, active):
    from neus2_amd.mesh import density_on_grid
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork()
    o = net.param_offsets()
    p = (torch.randn(o[4], device="cuda", generator=torch.Generator(device="cuda").manual_seed(active)) * 0.1).half()
    net.reserve(1 << 16)
    net.encoding().set_max_level((active - 0.5) / 16)
    active = net.encoding().active_levels()
    assert active < 16
    first = net.encoding().level_table()[3]  # entry that a level starts at
    got = []
    for anything in (0.0, float("nan")):
        p[o[2] + (o[3] - o[2]) // int(first[-1]) * int(first[active]):o[3]] = anything
        net.set_params(p, None)
        got.append(density_on_grid(net._h, res, (0, 0, 0), (130 / 512, 0.02, 0.125)))
    assert torch.isfinite(got[0]).all() and torch.equal(*got)


# rows longer than the chunk, down to the smallest one: slabs of a few runs, and of less than one
@pytest.mark.parametrize("res,chunk", [((513, 3, 5), 64), ((200, 4, 3), 8)])
def test_lattice_of_rows_longer_than_the_chunk(res, chunk):
    """The values do not depend on where the lattice is cut, also where a row does not fit a slab."""
    from neus2_amd.mesh import density_on_grid
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork()
    p = torch.randn(net.param_offsets()[4], device="cuda", generator=torch.Generator(device="cuda").manual_seed(res[0])) * 0.1
    net.set_params(p.half(), None)
    net.reserve(1 << 14)
    whole = density_on_grid(net._h, res, chunk=1 << 14)
    assert torch.equal(whole, density_on_grid(net._h, res, chunk=chunk))


def test_sdf_lattice_and_mesh_of_the_initial_sphere(oracle, tmp_path):
    """get_density_on_grid + marching cubes on the geometric-init network: the zero level set of its SDF is a sphere of
    radius ~0.1 around the cube centre (sdf ~ |x - 0.5| - 0.1)."""
    from neus2_amd.mesh import density_on_grid, marching_cubes, marching_cubes_resolution, save_mesh
    from neus2_amd.training import Trainer, default_config
    from oracle.field import Field
    tr = Trainer(default_config(target_batch_size=4096, max_rays_per_batch=256, max_samples=1 << 16))
    tr.initialize_params(seed=5, sdf_mlp_weights=np.load(os.path.join(GOLD, "sdf_mlp_weights_48.npy")))
    assert marching_cubes_resolution(40) == (48, 48, 48) and marching_cubes_resolution(64, (0, 0, 0), (1, 0.5, 0.25)) == (64, 32, 16)
    res = (48, 32, 48)
    lo, hi = (0.25, 0.3, 0.25), (0.75, 0.7, 0.75)
    d = density_on_grid(tr._field, res, lo, hi, chunk=1 << 14)  # several chunks, the last one partial
    # lattice positions as the reference computes them, SDF from the oracle's field
    z, y, x = np.meshgrid(np.arange(res[2], dtype=np.float32), np.arange(res[1], dtype=np.float32), np.arange(res[0], dtype=np.float32), indexing="ij")
    ext = np.asarray(hi, np.float32) - np.asarray(lo, np.float32)
    pos = np.stack([(x * np.float32(1.0 / res[0])) * ext[0] + np.float32(lo[0]), (y * np.float32(1.0 / res[1])) * ext[1] + np.float32(lo[1]),
                    (z * np.float32(1.0 / res[2])) * ext[2] + np.float32(lo[2])]).reshape(3, -1)
    want = Field(fp16=True).sdf_values(host(tr.params), pos)[0].reshape(res[2], res[1], res[0])
    assert_close(host(d), want, rtol=RTOL, what="SDF lattice", outlier_frac=1e-3)
    v, t, n = marching_cubes(d, 0.0, lo, hi)
    vv, tt = host(v), host(t).astype(np.int64)
    assert len(tt) > 500 and check_closed_oriented(vv, tt) == 2
    r = np.linalg.norm(vv - 0.5, axis=1)
    assert abs(r.mean() - 0.1) < 0.03 and r.std() < 0.04  # 64 random neurons: a lumpy sphere
    # OBJ and PLY as the reference writes them
    for ext_ in ("obj", "ply"):
        p = tmp_path / f"mesh.{ext_}"
        save_mesh(p, vv, host(n), tt)
        text = p.read_text().splitlines()
        if ext_ == "obj":
            assert sum(l.startswith("v ") for l in text) == len(vv) and sum(l.startswith("vn ") for l in text) == len(vv)
            faces = [l for l in text if l.startswith("f ")]
            assert len(faces) == len(tt)
            a, b, c = (int(tok.split("//")[0]) - 1 for tok in faces[0].split()[1:])
            assert (a, b, c) == (tt[0][2], tt[0][1], tt[0][0])  # reversed winding, 1-based
        else:
            assert text[0] == "ply" and f"element vertex {len(vv)}" in text and f"element face {len(tt)}" in text
            assert len(text) == text.index("end_header") + 1 + len(vv) + len(tt)


def test_lattice_larger_than_the_last_level_cache():
    """A lattice whose density is streamed (512 x 512 x 256 points) holds the mesh of the smaller lattice it contains."""
    from neus2_amd.mesh import marching_cubes
    x, y, z = ((torch.arange(r, device="cuda") - c) / 512 for r, c in ((512, 250.3), (512, 260.1), (256, 62.4)))
    d = 0.1 - (x[None, None, :] ** 2 + y[None, :, None] ** 2 + z[:, None, None] ** 2).sqrt()  # all of it below plane 128
    big = marching_cubes(d.contiguous(), 0.0, (0, 0, 0), (1, 1, 0.5))
    small = marching_cubes(d[:128].contiguous(), 0.0, (0, 0, 0), (1, 1, 0.25))
    assert big[0].shape[0] > 10000
    for a, b in zip(big, small):
        assert torch.equal(a, b)
