"""GPU parity of the hash-grid kernels against the CPU oracle, through the C ABI."""
import numpy as np
import pytest
import torch

from gpu_util import RTOL, assert_close, dev, host, q16, rel_l2

pytestmark = pytest.mark.gpu

CFG = dict(n_levels=16, log2_hashmap_size=19, base_resolution=16, per_level_scale=1.447)


@pytest.fixture(scope="module")
def setup(oracle):
    from neus2_amd.tcnn_api import GridEncoding
    og = oracle.Grid(CFG["n_levels"], CFG["log2_hashmap_size"], CFG["base_resolution"], CFG["per_level_scale"])
    gg = GridEncoding(**CFG)
    assert gg.n_params() == og.n_params
    rng = np.random.default_rng(0)
    params = q16(rng.uniform(-1, 1, og.n_params))
    d_params = dev(params, torch.float16)
    d_grads = torch.zeros_like(d_params)
    gg.set_params(d_params, d_grads)
    return og, gg, params, d_params, d_grads


def test_config1_indices_bit_exact(setup):
    """The benchmark's plumbing configuration: 2^14 points U[0,1)^3, seed 0: every corner index of every level identical."""
    og, gg, *_ = setup
    xyz = np.random.default_rng(0).random((3, 1 << 14), dtype=np.float32)
    ref, _ = og.indices(xyz)
    got = host(gg.corner_indices(dev(xyz))).view(np.uint32)
    assert np.array_equal(got, ref)


def test_indices_bit_exact_edge_positions(setup):
    og, gg, *_ = setup
    edge = np.array([0.0, 1.0, np.nextafter(np.float32(1), np.float32(0)), 0.5, 1e-8, 0.25, 0.999999, 1.0 / 3], np.float32)
    xyz = np.stack(np.meshgrid(edge, edge, edge, indexing="ij")).reshape(3, -1).astype(np.float32)
    # plus vertices of several levels, where floor() sits on a knife edge
    extra = [((np.arange(40, dtype=np.float32) - 0.5) / s) for s in og.scale[[0, 3, 9, 15]]]
    e = np.clip(np.concatenate(extra), 0, 1).astype(np.float32)
    xyz = np.concatenate([xyz, np.stack([e, e[::-1], e])], axis=1)
    ref, _ = og.indices(xyz)
    got = host(gg.corner_indices(dev(xyz))).view(np.uint32)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_forward_values_and_ragged_sizes(setup, n):
    og, gg, params, *_ = setup
    xyz = np.random.default_rng(n).random((3, n), dtype=np.float32)
    ref, ref_j = og.forward(params, xyz, want_dy_dx=True)
    out, dy_dx = gg.forward(dev(xyz), prepare_input_gradients=True)
    assert_close(host(out), ref, what="grid forward")
    # dy_dx is fp32 on both sides; differences of fp16 table values times scale
    assert_close(host(dy_dx), ref_j, rtol=1e-4, what="dy_dx")
    out2, none = gg.forward(dev(xyz))
    # the two instantiations may round a tie differently: at most one fp16 ulp apart
    assert none is None
    assert_close(host(out2), host(out), rtol=1e-3, what="forward without dy_dx")


def test_forward_accepts_nerf_coordinate_rows(setup):
    """7 floats per point (xyz, dt, dir), the column-major batch the reference feeds (nerf.h:76-102)."""
    og, gg, params, *_ = setup
    n = 3000
    rng = np.random.default_rng(7)
    coords = rng.random((n, 7), dtype=np.float32)
    out_rows, _ = gg.forward(dev(coords))
    out_soa, _ = gg.forward(dev(np.ascontiguousarray(coords[:, :3].T)))
    assert torch.equal(out_rows, out_soa)


def test_forward_empty_batch(setup):
    _, gg, *_ = setup
    out, _ = gg.forward(torch.zeros((3, 0), dtype=torch.float32, device="cuda"))
    assert out.shape == (32, 0)


def test_forward_small_uniform_params_config1(setup, oracle):
    """Config 1's parameter distribution U(-1e-4, 1e-4), seed 0."""
    og, gg, _, d_params, d_grads = setup
    rng = np.random.default_rng(0)
    p = q16(rng.uniform(-1e-4, 1e-4, og.n_params))
    from neus2_amd.tcnn_api import GridEncoding
    g2 = GridEncoding(**CFG)
    dp = dev(p, torch.float16)
    g2.set_params(dp, None)
    xyz = rng.random((3, 1 << 14), dtype=np.float32)
    out, _ = g2.forward(dev(xyz))
    # fp16 subnormal spacing (6e-8) dominates at this magnitude: absolute floor of one subnormal ulp
    ref = og.forward(p, xyz)
    assert np.abs(host(out) - ref).max() <= 6e-8 + RTOL * np.abs(ref).max()


def test_backward_param_scatter_and_input_grad(setup):
    og, gg, params, d_params, d_grads = setup
    n = 1 << 14
    rng = np.random.default_rng(11)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((32, n)))
    ref_grad, ref_dx = og.backward(params, xyz, dy)
    d_xyz = dev(xyz)
    _, ctx = gg.forward(d_xyz, prepare_input_gradients=True)
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_IGNORE, GRAD_OVERWRITE
    d_grads.fill_(7.0)  # Overwrite must discard this
    dx = gg.backward(ctx, d_xyz, dev(dy, torch.float16), want_input_grad=True, mode=GRAD_OVERWRITE)
    got = host(d_grads)
    assert_close(host(dx), ref_dx, rtol=1e-4, what="dL_dx")
    # fp16 atomics round after every addition: the error of an entry that received
    # k contributions grows like sqrt(k) half-ulps, so coarse levels get a wider band
    for l in range(16):
        a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
        k = 8.0 * n / max(1, int(og.entries[l]))
        tol = RTOL * max(1.0, np.sqrt(k))
        assert rel_l2(got[a:b], ref_grad[a:b]) < tol, (l, rel_l2(got[a:b], ref_grad[a:b]), tol)
    # Accumulate adds a second copy; Ignore leaves the buffer alone
    gg.backward(ctx, d_xyz, dev(dy, torch.float16), mode=GRAD_ACCUMULATE)
    got2 = host(d_grads)
    assert rel_l2(got2, 2 * ref_grad) < 2e-2
    before = d_grads.clone()
    dx2 = gg.backward(ctx, d_xyz, dev(dy, torch.float16), want_input_grad=True, mode=GRAD_IGNORE)
    assert torch.equal(before, d_grads) and torch.equal(dx, dx2)


def test_backward_backward_input(setup):
    og, gg, params, d_params, d_grads = setup
    n = 1 << 13
    rng = np.random.default_rng(13)
    xyz = rng.random((3, n), dtype=np.float32)
    g = q16(rng.standard_normal((32, n)) * 0.1)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    ref_grad, ref_out, ref_din = og.backward_backward_input(params, xyz, v, g)
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_IGNORE, GRAD_OVERWRITE
    d_xyz, d_v, d_g = dev(xyz), dev(v), dev(g, torch.float16)
    out, din = gg.backward_backward_input(d_xyz, d_v, d_g, want_dL_ddLdy=True, want_dL_dx=True, mode=GRAD_OVERWRITE)
    assert_close(host(out), ref_out, what="dL_ddLdy")
    assert_close(host(din), ref_din, rtol=1e-3, what="second-order dL_dx")
    got = host(d_grads)
    for l in range(16):
        a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
        k = 8.0 * n / max(1, int(og.entries[l]))
        tol = RTOL * max(1.0, np.sqrt(k))
        assert rel_l2(got[a:b], ref_grad[a:b]) < tol, (l, rel_l2(got[a:b], ref_grad[a:b]), tol)
    # the reference's call: Accumulate on top of the first-order gradients, outputs optional
    base = q16(rng.standard_normal(og.n_params) * 1e-3)
    d_grads.copy_(dev(base, torch.float16))
    out2, none = gg.backward_backward_input(d_xyz, d_v, d_g, want_dL_ddLdy=True, want_dL_dx=False, mode=GRAD_ACCUMULATE)
    # (a different kernel serves calls that also ask for the second-order dL_dx: same values up to fp16 rounding)
    assert none is None
    assert_close(host(out2), ref_out, what="dL_ddLdy without dL_dx")
    assert rel_l2(host(d_grads), base + ref_grad) < 1e-2
    before = d_grads.clone()
    gg.backward_backward_input(d_xyz, d_v, d_g, mode=GRAD_IGNORE)
    assert torch.equal(before, d_grads)


@pytest.mark.parametrize("cfg", [(6, 12, 4, 1.6), (5, 4, 2, 1.5), (8, 14, 4, 2.0), (14, 19, 16, 1.4472692012786865)])
def test_other_table_shapes(oracle, cfg):
    """Small tables exercise the true-modulo index paths; 14 levels is the reference's shipped config."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    og = oracle.Grid(*cfg)
    gg = GridEncoding(n_levels=cfg[0], log2_hashmap_size=cfg[1], base_resolution=cfg[2], per_level_scale=cfg[3])
    rng = np.random.default_rng(17)
    params = q16(rng.uniform(-1, 1, og.n_params))
    dp = dev(params, torch.float16)
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    n = 2049
    xyz = rng.random((3, n), dtype=np.float32)
    ref_idx, _ = og.indices(xyz)
    assert np.array_equal(host(gg.corner_indices(dev(xyz))).view(np.uint32), ref_idx)
    out, ctx = gg.forward(dev(xyz), prepare_input_gradients=True)
    assert_close(host(out), og.forward(params, xyz), what="forward")
    dy = q16(rng.standard_normal((og.n_out, n)))
    ref_grad, ref_dx = og.backward(params, xyz, dy)
    dx = gg.backward(ctx, dev(xyz), dev(dy, torch.float16), want_input_grad=True, mode=GRAD_OVERWRITE)
    assert_close(host(dx), ref_dx, rtol=1e-4, what="dL_dx")
    assert rel_l2(host(dg), ref_grad) < 2e-2


@pytest.mark.parametrize("cfg", [(6, 12, 4, 1.6), (5, 4, 2, 1.5), (8, 14, 4, 2.0), (14, 19, 16, 1.4472692012786865),
                                 (16, 19, 32, 1.4472692012786865), (4, 21, 512, 1.9)])
def test_sorted_scatter_other_table_shapes(oracle, cfg):
    """The bucketed scatter on other tables: one bucket per level (2^12 entries), four buckets (2^14: no multiple of the
    8 XCDs), tiny tables with a true modulo, the 14-level config, hashed levels whose resolution exceeds the 12 index bits
    a pair record relies on (base 32: 5646 and 8170 cells, one record per corner there), and a table too large for the
    bucket plan (2^21 entries: falls back to the atomic scatter)."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    og = oracle.Grid(*cfg)
    gg = GridEncoding(n_levels=cfg[0], log2_hashmap_size=cfg[1], base_resolution=cfg[2], per_level_scale=cfg[3])
    rng = np.random.default_rng(23)
    params = q16(rng.uniform(-1, 1, og.n_params))
    dp = dev(params, torch.float16)
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    n = 3 * 4096 + 13 * 8
    assert gg.reserve_scatter_workspace(1 << 14) == (cfg[1] <= 19)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((og.n_out, n)))
    g2 = q16(rng.standard_normal((og.n_out, n)) * 0.1)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    ref1, _ = og.backward(params, xyz, dy, want_dx=False)
    ref, _, _ = og.backward_backward_input(params, xyz, v, g2, grad=ref1.copy(), want_dinput=False)
    dg.fill_(7.0)
    gg.backward_fused(dev(xyz), dev(dy, torch.float16), dev(v), dev(g2, torch.float16), want_dL_ddLdy=False, mode=GRAD_OVERWRITE)
    got = host(dg)
    for l in range(cfg[0]):
        a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
        k = 8.0 * n / max(1, int(og.entries[l]))
        tol = RTOL * (1.0 if cfg[1] <= 19 else max(1.0, np.sqrt(k)))  # the atomic fallback adds in fp16
        assert rel_l2(got[a:b], ref[a:b]) < tol, (l, rel_l2(got[a:b], ref[a:b]), tol)


def test_sorted_scatter_split_buckets(oracle):
    """A small table under a large batch: every level has fewer buckets than the batch needs workgroups, so buckets are
    split over several workgroups whose fp32 images a combine launch adds in a fixed order (both record kinds: the dense
    levels' single records and the hashed levels' pair records).  Against the oracle, accumulate mode included, and two
    runs give the same bits."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    cfg = (6, 12, 4, 1.6)
    og = oracle.Grid(*cfg)
    gg = GridEncoding(n_levels=cfg[0], log2_hashmap_size=cfg[1], base_resolution=cfg[2], per_level_scale=cfg[3])
    rng = np.random.default_rng(29)
    params = q16(rng.uniform(-1, 1, og.n_params))
    dp = dev(params, torch.float16)
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    n = 40 * 1024 + 77  # 8 n / 65536 = 5 workgroups per bucket
    assert gg.reserve_scatter_workspace(n)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((og.n_out, n)) * 0.05)
    g2 = q16(rng.standard_normal((og.n_out, n)) * 0.01)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    ref1, _ = og.backward(params, xyz, dy, want_dx=False)
    ref, _, _ = og.backward_backward_input(params, xyz, v, g2, grad=ref1.copy(), want_dinput=False)
    d_xyz, d_dy, d_v, d_g2 = dev(xyz), dev(dy, torch.float16), dev(v), dev(g2, torch.float16)

    def check(got, want, what):
        for l in range(cfg[0]):
            a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
            assert rel_l2(got[a:b], want[a:b]) < RTOL, (what, l, rel_l2(got[a:b], want[a:b]))

    dg.fill_(7.0)
    gg.backward_fused(d_xyz, d_dy, d_v, d_g2, want_dL_ddLdy=False, mode=GRAD_OVERWRITE)
    first = dg.clone()
    check(host(dg), ref, "overwrite")
    gg.backward_fused(d_xyz, d_dy, d_v, d_g2, want_dL_ddLdy=False, mode=GRAD_ACCUMULATE)
    check(host(dg), 2 * ref, "accumulate")
    dg.fill_(-3.0)
    gg.backward_fused(d_xyz, d_dy, d_v, d_g2, want_dL_ddLdy=False, mode=GRAD_OVERWRITE)
    assert torch.equal(dg, first)


def test_errors_are_reported_not_launched():
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding, N2Error
    gg = GridEncoding(**CFG)
    x = torch.rand((3, 16), device="cuda")
    with pytest.raises(N2Error, match="set_params"):
        gg.forward(x)
    p = torch.zeros(gg.n_params(), dtype=torch.float16, device="cuda")
    gg.set_params(p, None)
    out, ctx = gg.forward(x, prepare_input_gradients=True)
    with pytest.raises(N2Error, match="gradient buffer"):
        gg.backward(ctx, x, torch.zeros((32, 16), dtype=torch.float16, device="cuda"), mode=GRAD_OVERWRITE)
    with pytest.raises(N2Error):
        gg.forward(x.double())


@pytest.mark.parametrize("n", [1 << 13, 1001])
def test_backward_fused_equals_first_plus_second_order(setup, n):
    """One scatter pass == backward(Overwrite) followed by backward_backward_input(Accumulate)."""
    og, gg, params, d_params, d_grads = setup
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE
    rng = np.random.default_rng(21)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((32, n)))
    g2 = q16(rng.standard_normal((32, n)) * 0.1)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    ref1, _ = og.backward(params, xyz, dy, want_dx=False)
    ref, ref_out, _ = og.backward_backward_input(params, xyz, v, g2, grad=ref1.copy(), want_dinput=False)
    d_grads.fill_(3.0)
    out = gg.backward_fused(dev(xyz), dev(dy, torch.float16), dev(v), dev(g2, torch.float16), mode=GRAD_OVERWRITE)
    assert_close(host(out), ref_out, what="fused dL_ddLdy")
    got = host(d_grads)
    for l in range(16):
        a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
        k = 8.0 * n / max(1, int(og.entries[l]))
        tol = RTOL * max(1.0, np.sqrt(k))
        assert rel_l2(got[a:b], ref[a:b]) < tol, (l, rel_l2(got[a:b], ref[a:b]), tol)
    none = gg.backward_fused(dev(xyz), dev(dy, torch.float16), dev(v), dev(g2, torch.float16), want_dL_ddLdy=False,
                             mode=GRAD_ACCUMULATE)
    assert none is None and rel_l2(host(d_grads), 2 * ref) < 2e-2


@pytest.mark.parametrize("n", [1, 1025, (1 << 15) + 1, 70001])  # one record, a second tile, one tile past the few-tiles kernel, tiles taken in several turns
def test_sorted_scatter_batch_sizes(oracle, n):
    """The reduce kernel's two forms and its walk over tiles, overwriting and accumulating."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    og = oracle.Grid(CFG["n_levels"], CFG["log2_hashmap_size"], CFG["base_resolution"], CFG["per_level_scale"])
    gg = GridEncoding(**CFG)
    rng = np.random.default_rng(n)
    dp = dev(q16(rng.uniform(-1, 1, og.n_params)), torch.float16)
    dg = torch.full_like(dp, 9.0)
    gg.set_params(dp, dg)
    assert gg.reserve_scatter_workspace(n)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((32, n)))
    ref, _ = og.backward(host(dp), xyz, dy, want_dx=False)
    for mode, times in ((GRAD_OVERWRITE, 1), (GRAD_ACCUMULATE, 2)):
        gg.backward(None, dev(xyz), dev(dy, torch.float16), mode=mode)
        got = host(dg)
        for l in range(16):
            a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
            assert rel_l2(got[a:b], times * ref[a:b]) < RTOL, (mode, l)


@pytest.mark.parametrize("n", [3, 200, 40000])  # the kernel for few records and the other one
@pytest.mark.parametrize("levels,log2_size,base", [(1, 19, 16), (1, 16, 64), (1, 16, 37), (2, 19, 16)])  # dense, hashed, a number of buckets that is no multiple of eight
def test_sorted_scatter_is_exact_for_values_of_all_sizes(n, levels, log2_size, base):
    """Points in the middle of their cells: every record is dL_dy / 8, exactly, and the sums are exact until they are rounded, from the smallest fp16
    values to those above 128 that do not fit the short form; infinite values stay infinite, values that are no number count as zero."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(n_levels=levels, log2_hashmap_size=log2_size, base_resolution=base, per_level_scale=1.0)
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = torch.zeros(gg.n_params(), device="cuda").half()
    dg = torch.full_like(dp, 5.0)
    gg.set_params(dp, dg)
    assert gg.reserve_scatter_workspace(n)
    x = torch.randint(0, base - 1, (3, n), device="cuda", generator=gen).float() / (base - 1)
    size = torch.randint(-18, 9, (2 * levels, n), device="cuda", generator=gen)
    size = torch.where(torch.rand(size.shape, device="cuda", generator=gen) < 0.02, size + 5, size)
    dy = torch.ldexp(torch.randint(-7, 8, size.shape, device="cuda", generator=gen).float(), size)  # (multiples of 2^-18, up to 7 * 2^13)
    dy[0, 0] = float("inf")
    dy[1, n // 2] = float("nan")
    dy = dy.half()
    at = gg.corner_indices(x).long()
    offsets = gg.level_table()[3]
    want = torch.zeros((dg.numel() // 2, 2), device="cuda", dtype=torch.float64)
    special = torch.zeros_like(want)
    for l in range(levels):
        for f in range(2):
            rec = (dy[2 * l + f].double() / 8)
            special[:, f].index_add_(0, at[l].reshape(-1) + int(offsets[l]), rec.isinf().double().repeat(8))
            rec = torch.where(rec.isfinite(), rec, 0.0)
            want[:, f].index_add_(0, at[l].reshape(-1) + int(offsets[l]), rec.repeat(8))
    for mode, times in ((GRAD_OVERWRITE, 1), (GRAD_ACCUMULATE, 2)):
        gg.backward(None, x, dy, mode=mode)
        got = dg.reshape(-1, 2)
        once = want.float().half()
        ref = once if times == 1 else (want.float() + once.float()).half()
        ref = torch.where(special > 0, float("inf"), ref.float()).half()
        skip = torch.isinf(once) & (special == 0) if times == 2 else torch.zeros_like(special, dtype=torch.bool)
        bad = (got != ref) & ~skip
        assert not bad.any(), (mode, int(bad.sum()), got[bad][:4], ref[bad][:4], want[bad][:4])


# the kernel for few records, the same with more records in a bucket than claims (an image by ranges), the other one
@pytest.mark.parametrize("n,within", [(200, None), (3000, 6), (40000, None)])
@pytest.mark.parametrize("levels,log2_size,base", [(1, 19, 16), (1, 16, 64), (1, 16, 37), (2, 6, 16)])  # dense, hashed, levels that keep an image, buckets split over several workgroups
def test_infinite_records_are_neither_cancelled_nor_wrapped(n, within, levels, log2_size, base):
    """An entry with infinite records of one sign has an infinite gradient, however many there are (two, every 64th point) and however large finite ones of the
    other sign (up to 65504 / 8, over a thousand of them); one with both signs has no number, as the sum has none.  No two points of a run of equal cells that would be merged."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(n_levels=levels, log2_hashmap_size=log2_size, base_resolution=base, per_level_scale=1.0)
    gen = torch.Generator(device="cuda").manual_seed(n + base)
    dp = torch.zeros(gg.n_params(), device="cuda").half()
    dg = torch.full_like(dp, 5.0)
    gg.set_params(dp, dg)
    assert gg.reserve_scatter_workspace(n)
    cells = torch.randint(0, within or base - 1, (3, n), device="cuda", generator=gen)
    i = torch.arange(n, device="cuda")
    dy = torch.randn((2 * levels, n), device="cuda", generator=gen)
    for k, cell, values in ((3, 2, (65504.0, -65504.0)), (5, 6, (-65504.0, 65504.0)), (7, 10, (65504.0, 1.0))):  # every eighth point: three cells with large values
        cells[:, i % 8 == k] = cell
        dy[:, i % 8 == k] = torch.tensor(values * levels, device="cuda").view(-1, 1)
    inf = float("inf")
    for start, pair in ((3, (-inf, inf)), (5, (inf, -inf)), (7, (-inf, -inf))):  # of those points every 64th, and so more than one of 200
        dy[:, start::64] = torch.tensor(pair * levels, device="cuda").view(-1, 1)
    dy[0, 15] = inf  # both signs at the third one
    dy = dy.half()
    x = (cells.float() / (base - 1)).contiguous()
    at = gg.corner_indices(x).long()
    offsets = gg.level_table()[3]
    ref = torch.zeros((dg.numel() // 2, 2), device="cuda", dtype=torch.float64)
    marks = torch.zeros((2,) + ref.shape, device="cuda", dtype=torch.float64)
    for l in range(levels):
        to = at[l].reshape(-1) + int(offsets[l])
        for f in range(2):
            rec = dy[2 * l + f].double() / 8
            ref[:, f].index_add_(0, to, torch.where(rec.isfinite(), rec, 0.0).repeat(8))
            for sign in range(2):
                marks[sign, :, f].index_add_(0, to, (rec == (-inf if sign else inf)).double().repeat(8))
    assert (marks.amax((1, 2)) >= 2).all() and bool(((marks[0] > 0) & (marks[1] > 0)).any())
    want = torch.where(marks[0] > 0, inf, torch.where(marks[1] > 0, -inf, ref))
    want = torch.where((marks[0] > 0) & (marks[1] > 0), float("nan"), want).half()
    for mode in (GRAD_OVERWRITE, GRAD_ACCUMULATE, GRAD_OVERWRITE):  # (the second order of calls: nothing stays marked)
        gg.backward(None, x, dy, mode=mode)
        got = dg.reshape(-1, 2)
        special = ~want.isfinite()
        same = (got == want) | (got.isnan() & want.isnan())
        assert bool(same[special].all()), (mode, got[special & ~same][:4], want[special & ~same][:4])
        if mode == GRAD_OVERWRITE:
            assert bool(got[~special].isfinite().all())
            assert rel_l2(host(got[~special]), host(want[~special])) < RTOL
    dy = torch.where(dy.isfinite(), dy, torch.zeros_like(dy))
    gg.backward(None, x, dy, mode=GRAD_OVERWRITE)
    fits = ref.half().isfinite()
    assert rel_l2(host(dg.reshape(-1, 2)[fits]), host(ref[fits])) < RTOL


@pytest.mark.parametrize("n", [200, 40000])  # the kernel for few records and the other one
@pytest.mark.parametrize("levels,log2_size,base", [(1, 19, 16), (1, 16, 64), (1, 16, 37)])  # dense, hashed, buckets of several sizes
def test_an_accumulating_scatter_rounds_to_fp32_and_then_to_fp16(n, levels, log2_size, base):
    """1024 + (0.5 + 2^-24) is 1024.5 in fp32 and, of two neighbours at the same distance, the even 1024 in fp16; in one rounding it would be 1025."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GridEncoding
    gg = GridEncoding(n_levels=levels, log2_hashmap_size=log2_size, base_resolution=base, per_level_scale=1.0)
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = torch.zeros(gg.n_params(), device="cuda").half()
    dg = torch.full_like(dp, 1024.0)
    gg.set_params(dp, dg)
    assert gg.reserve_scatter_workspace(n)
    cells = torch.randint(0, base - 1, (3, n), device="cuda", generator=gen)
    cells[:, n // 3::n // 3] = 2
    i = torch.arange(n, device="cuda")
    dy = torch.where(i == n // 3, 4.0, torch.where(i == n // 3 * 2, 2.0 ** -21, 0.0)).expand(2 * levels, n).half().contiguous()  # (a record is an eighth of it)
    x = (cells.float() / (base - 1)).contiguous()
    at = gg.corner_indices(x)[0].long()
    ref = torch.zeros(dg.numel() // 2, device="cuda", dtype=torch.float64).index_add_(0, at.reshape(-1), dy[0].double().repeat(8) / 8)
    assert int((ref == 0.5 + 2.0 ** -24).sum()) == 8
    gg.backward(None, x, dy, mode=GRAD_ACCUMULATE)
    want = (ref.float() + 1024.0).half()
    assert bool((want == 1024.0).all()) and torch.equal(dg.reshape(-1, 2), want[:, None].expand(-1, 2))


# full buckets of pair records in front of the others: split, whole, in accumulating launches of more items than run at one time; behind them; single records alone;
# the last batch whose few records' items are taken in turn, and the first one with a workgroup for each
@pytest.mark.parametrize("levels,log2_size,n", [(4, 14, 40000), (5, 16, 70000), (16, 16, 140000), (5, 19, 70000), (2, 19, 40000), (16, 19, 16896), (16, 19, 16897)])
def test_sorted_scatter_with_either_kind_of_records_first(oracle, levels, log2_size, n):
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    cfg = {**CFG, "n_levels": levels, "log2_hashmap_size": log2_size}
    og = oracle.Grid(cfg["n_levels"], cfg["log2_hashmap_size"], cfg["base_resolution"], cfg["per_level_scale"])
    gg = GridEncoding(**cfg)
    rng = np.random.default_rng(n)
    dp = dev(q16(rng.uniform(-1, 1, og.n_params)), torch.float16)
    dg = torch.full_like(dp, 9.0)
    gg.set_params(dp, dg)
    assert gg.reserve_scatter_workspace(n)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((2 * levels, n)))
    ref, _ = og.backward(host(dp), xyz, dy, want_dx=False)
    for mode, times in ((GRAD_OVERWRITE, 1), (GRAD_ACCUMULATE, 2)):
        gg.backward(None, dev(xyz), dev(dy, torch.float16), mode=mode)
        got = host(dg)
        for l in range(levels):
            a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
            assert rel_l2(got[a:b], times * ref[a:b]) < RTOL, (mode, l)


@pytest.mark.parametrize("n,room", [(512, 512), (513, 513), (513, 70000), (16384, 16384), (16384, 16385)])
def test_sorted_scatter_tiles_of_one_and_two_points_per_thread(oracle, n, room):
    """The sums are exact, so the size of a tile leaves no trace: a batch equals the one that has points without a gradient behind it, up to where
    tiles are larger; in a workspace that is just large enough and in a larger one."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(**CFG)
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = (torch.rand(gg.n_params(), device="cuda", generator=gen) * 2 - 1).half()
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    large = 24576 + 1024  # (two points per thread, the batches one)
    x = torch.rand((3, large), device="cuda", generator=gen)
    dy, g2, v = (torch.randn((w, large), device="cuda", generator=gen) for w in (32, 32, 3))
    dy[:, n:] = 0
    g2[:, n:] = 0
    got = []
    for points, space in ((n, room), (large, large)):
        gg.set_params(dp, dg)
        assert gg.reserve_scatter_workspace(space)
        dg.fill_(9.0)
        out = gg.backward_fused(x[:, :points].contiguous(), dy[:, :points].half().contiguous(), v[:, :points].contiguous(), g2[:, :points].half().contiguous(), mode=GRAD_OVERWRITE)
        got.append((dg.clone(), out[:, :n].clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and bool((got[0][0] != 0).any())


# edges of the workgroups that take the input gradient along, tiles of one and of two points per thread, streamed Jacobians, tables of other widths, and
# a scatter that has no workspace and so takes nothing along
@pytest.mark.parametrize("n,levels,room", [(1, 16, True), (511, 16, True), (513, 16, True), (24576, 16, True), (24577, 16, True), (180001, 16, True), (5003, 1, True), (5003, 3, True), (5003, 16, False)])
def test_input_gradient_beside_the_scatter(n, levels, room):
    """Both gradients from one call are those of two."""
    from neus2_amd.tcnn_api import GRAD_IGNORE, GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(**{**CFG, "n_levels": levels})
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = (torch.rand(gg.n_params(), device="cuda", generator=gen) * 2 - 1).half()
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    if room:
        assert gg.reserve_scatter_workspace(n)
    x = torch.rand((3, n), device="cuda", generator=gen)
    dy = torch.randn((2 * levels, n), device="cuda", generator=gen).half()
    _, ctx = gg.forward(x, prepare_input_gradients=True)
    dx = gg.backward(ctx, x, dy, want_input_grad=True, mode=GRAD_OVERWRITE)
    both = dg.clone()
    assert torch.equal(dx, gg.backward(ctx, x, dy, want_input_grad=True, mode=GRAD_IGNORE)) and bool((dx != 0).any())
    dg.fill_(9.0)
    gg.backward(None, x, dy, mode=GRAD_OVERWRITE)
    if room:
        assert torch.equal(both, dg)
    else:  # atomics add in the order of their arrival, a rounding to fp16 each
        assert rel_l2(host(both), host(dg)) < RTOL


# one point, the edges of a wave, of a workgroup and of the tiles (claims up to 24 576 points), batches above the size whose gathers are dealt by XCD; levels dealt in short turns;
# both orders in the launch and the second alone
@pytest.mark.parametrize("n,levels", [(1, 16), (63, 16), (65, 16), (511, 16), (513, 16), (5003, 16), (24576, 16), (24577, 16), (140001, 16), (600001, 16), (5003, 1), (5003, 3), (513, 7)])
@pytest.mark.parametrize("first", [False, True])
def test_second_order_output_beside_the_scatter(n, levels, first):
    """dL_ddLdy is the same with and without scratch space for the sorted scatter, whose launch gathers it, up to the rounding of its fp32 sums; the parameters' gradients
    are those of a call without it."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    sorting, adding = (GridEncoding(**{**CFG, "n_levels": levels}) for _ in range(2))
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = (torch.rand(sorting.n_params(), device="cuda", generator=gen) * 2 - 1).half()
    dg = torch.zeros_like(dp)
    assert sorting.reserve_scatter_workspace(n)
    x, v = torch.rand((3, n), device="cuda", generator=gen), torch.randn((3, n), device="cuda", generator=gen) * 1e-3
    dy, g2 = (torch.randn((2 * levels, n), device="cuda", generator=gen).half() for _ in range(2))
    for off in ("none", "level", "per point"):
        per_point = torch.randint(0, 2, (n,), device="cuda", generator=gen).float() if off == "per point" else None

        def call(grid, want):
            grid.set_params(dp, dg)
            grid.set_max_level(0.5 if off == "level" else 1000.0)
            grid.set_max_level_gpu(per_point)
            dg.fill_(9.0)
            if first:
                out = grid.backward_fused(x, dy, v, g2, want_dL_ddLdy=want, mode=GRAD_OVERWRITE)
            else:
                out, _ = grid.backward_backward_input(x, v, g2, want_dL_ddLdy=want, mode=GRAD_OVERWRITE)
            return out, dg.clone()

        got, grads = call(sorting, True)
        # eight products and their sum in fp32 on both sides (2^-24 each of values up to 4096 * 5e-3 * 2), one rounding to fp16 each
        torch.testing.assert_close(got.float(), call(adding, True)[0].float(), rtol=2.0 ** -10, atol=2e-5)
        assert (off != "none" or bool((got != 0).any())) and torch.equal(grads, call(sorting, False)[1])


# batches whose buckets hold few records, up to the last one and the next; points that all fall into a few cells, in turn (no runs to merge), so that
# single buckets hold more records than sums can be claimed for; tables of few and of small buckets
@pytest.mark.parametrize("n,where,table", [(1, "anywhere", (16, 19)), (511, "anywhere", (16, 19)), (5003, "anywhere", (16, 19)), (16384, "anywhere", (16, 19)), (24576, "anywhere", (16, 19)), (24577, "anywhere", (16, 19)),
                                           (512, "two cells", (16, 19)), (2048, "two cells", (16, 19)), (2050, "two cells", (16, 19)), (24576, "two cells", (16, 19)),
                                           (9001, "outside", (16, 19)), (100, "anywhere", (6, 12)), (128, "two cells", (6, 12)), (7000, "anywhere", (1, 19)), (300, "anywhere", (3, 6))])
def test_sorted_scatter_of_few_records(n, where, table):
    """The sums are exact, so how a bucket is summed leaves no trace: a batch equals the one that has points without a gradient behind it, which is
    large enough for the other kernel.  Overwriting, accumulating, with levels switched off, and for both layouts of the positions."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(**{**CFG, "n_levels": table[0], "log2_hashmap_size": table[1]})
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = (torch.rand(gg.n_params(), device="cuda", generator=gen) * 2 - 1).half()
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    large = 70000
    x = torch.rand((3, large), device="cuda", generator=gen)
    if where == "two cells":
        x = 0.3 + 0.4 * (torch.arange(large, device="cuda") % 2) + 1e-5 * x
    elif where == "outside":
        x = x * 1.5 - 0.25
    dy, g2, v = (torch.randn((w, large), device="cuda", generator=gen) for w in (2 * table[0], 2 * table[0], 3))
    dy[:, n:] = 0
    g2[:, n:] = 0
    for mode, level, rows in ((GRAD_OVERWRITE, 1000.0, True), (GRAD_ACCUMULATE, 1000.0, True), (GRAD_OVERWRITE, 0.4, True), (GRAD_OVERWRITE, 1000.0, False)):
        gg.set_max_level(level)
        got = []
        for points in (n, large):
            gg.set_params(dp, dg)
            assert gg.reserve_scatter_workspace(points)
            dg.fill_(3.0)
            at = x[:, :points].contiguous() if rows else x[:, :points].t().contiguous()
            a, b, c = dy[:, :points].half().contiguous(), v[:, :points].contiguous(), g2[:, :points].half().contiguous()
            if rows:
                gg.backward_fused(at, a, b, c, want_dL_ddLdy=False, mode=mode)
            else:
                gg.backward(None, at, a, mode=mode)
            got.append(dg.clone())
        assert torch.equal(got[0], got[1]) and bool((got[0] != (3.0 if mode == GRAD_ACCUMULATE else 0.0)).any()), (mode, level, rows)


# one point, a wave and a few, the kernel for few records and the other one
@pytest.mark.parametrize("n", [1, 70, 5003, 40001])
@pytest.mark.parametrize("second", [False, True])
def test_points_that_a_mask_leaves_out_of_the_scatter_may_hold_anything(n, second):
    """Points along lines, whose runs of equal cells are summed across lanes, every third one switched off: what those hold reaches no other point's gradient."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(**CFG)
    gen = torch.Generator(device="cuda").manual_seed(n)
    dp = (torch.rand(gg.n_params(), device="cuda", generator=gen) * 2 - 1).half()
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    assert gg.reserve_scatter_workspace(n)
    off = torch.arange(n, device="cuda") % 3 == 2
    x = (0.2 + 0.6 * torch.arange(n, device="cuda") / n).repeat(3, 1) + torch.tensor([[0.0], [0.01], [0.02]], device="cuda")
    dy, g2, v = (torch.randn((w, n), device="cuda", generator=gen) for w in (32, 32, 3))
    gg.set_max_level_gpu(torch.where(off, -1.0, 1.0))
    got = []
    for bad in (False, True):
        fill = lambda t, value: torch.where(off, torch.full_like(t, value), t).contiguous()
        a = (fill(x, float("nan") if bad else 0.5), fill(dy, float("inf") if bad else 0.0).half(), fill(v, float("nan") if bad else 0.0), fill(g2, float("-inf") if bad else 0.0).half())
        dg.fill_(9.0)
        if second:
            gg.backward_fused(a[0], a[1], a[2], a[3], want_dL_ddLdy=False, mode=GRAD_OVERWRITE)
        else:
            gg.backward(None, a[0], a[1], mode=GRAD_OVERWRITE)
        got.append(dg.clone())
    assert torch.equal(got[0], got[1]) and bool(torch.isfinite(got[0].float()).all()) and bool((got[0] != 0).any())


# the last batch of one point per thread and the next one, workspaces that are just large enough and larger; buckets of up to 65536 records are whole
@pytest.mark.parametrize("levels,log2_size,line,whole", [(16, 19, 24576, True), (7, 16, 55808, True), (7, 14, 55808, False), (2, 6, 196608, False)])
def test_sorted_scatter_at_the_line_between_the_tiles(levels, log2_size, line, whole):
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    gg = GridEncoding(**{**CFG, "n_levels": levels, "log2_hashmap_size": log2_size})
    gen = torch.Generator(device="cuda").manual_seed(levels)
    dp = (torch.rand(gg.n_params(), device="cuda", generator=gen) * 2 - 1).half()
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    x = torch.rand((3, line + 1), device="cuda", generator=gen)
    dy, g2, v = (torch.randn((w, line + 1), device="cuda", generator=gen) for w in (2 * levels, 2 * levels, 3))
    dy[:, line:] = 0
    g2[:, line:] = 0
    got = []
    for points, space in ((line, line), (line, line + 1), (line + 1, line + 1)):
        assert gg.reserve_scatter_workspace(space)
        dg.fill_(9.0)
        gg.backward_fused(x[:, :points].contiguous(), dy[:, :points].half().contiguous(), v[:, :points].contiguous(), g2[:, :points].half().contiguous(), want_dL_ddLdy=False, mode=GRAD_OVERWRITE)
        got.append(dg.clone())
    assert torch.equal(got[0], got[1]) and bool((got[0] != 0).any()) and bool(torch.isfinite(got[0].float()).all())
    if whole:
        assert torch.equal(got[0], got[2])
    else:  # fp32 images of a bucket's parts, and other tiles make other parts: some entries round to the next fp16 number, 2^-10 of the entry away
        assert float((got[0].float() - got[2].float()).norm() / got[2].float().norm()) < 2 ** -10


@pytest.mark.parametrize("kind", ["uniform", "clustered", "rays"])
def test_sorted_scatter_path(oracle, kind):
    """With a scatter workspace, batches go through the run-length kernel (coarsest levels) and the
    LDS counting sort (the others): fp32 / exact accumulation, tighter agreement with the fp32 oracle than the
    atomic path, on uniform points, on points packed into a few cells (the contention case) and on points in ray
    order (consecutive samples share cells on the coarse levels, so runs are merged before they are written)."""
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding
    og = oracle.Grid(CFG["n_levels"], CFG["log2_hashmap_size"], CFG["base_resolution"], CFG["per_level_scale"])
    gg = GridEncoding(**CFG)
    rng = np.random.default_rng(31)
    params = q16(rng.uniform(-1, 1, og.n_params))
    dp = dev(params, torch.float16)
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    n = 3 * 4096 + 520  # not a multiple of the 1024-point tile
    assert gg.reserve_scatter_workspace(1 << 15)
    if kind == "uniform":
        xyz = rng.random((3, n), dtype=np.float32)
    elif kind == "clustered":
        xyz = (0.4 + 0.02 * rng.random((3, n))).astype(np.float32)
    else:
        per_ray = 97  # not a divisor of the 32-sample runs a lane walks
        n_rays = (n + per_ray - 1) // per_ray
        o = 0.3 + 0.4 * rng.random((n_rays, 1, 3))
        d = rng.standard_normal((n_rays, 1, 3))
        d /= np.linalg.norm(d, axis=-1, keepdims=True)
        k = np.arange(per_ray).reshape(1, per_ray, 1) - per_ray // 2
        xyz = np.clip(o + d * k * (np.sqrt(3.0) / 1024), 0, 1).reshape(-1, 3)[:n].T.astype(np.float32).copy()
    dy = q16(rng.standard_normal((32, n)))
    g2 = q16(rng.standard_normal((32, n)) * 0.1)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    ref1, _ = og.backward(params, xyz, dy, want_dx=False)
    ref, ref_out, _ = og.backward_backward_input(params, xyz, v, g2, grad=ref1.copy(), want_dinput=False)
    d_xyz, d_dy, d_v, d_g2 = dev(xyz), dev(dy, torch.float16), dev(v), dev(g2, torch.float16)

    def check(got, want, what):
        for l in range(16):
            a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
            # every contribution is rounded to fp16 once, sums are fp32, one final rounding
            assert rel_l2(got[a:b], want[a:b]) < RTOL, (what, l, rel_l2(got[a:b], want[a:b]))

    dg.fill_(9.0)
    gg.backward(None, d_xyz, d_dy, mode=GRAD_OVERWRITE)
    check(host(dg), ref1, "first order")
    dg.fill_(9.0)
    out = gg.backward_fused(d_xyz, d_dy, d_v, d_g2, mode=GRAD_OVERWRITE)
    assert_close(host(out), ref_out, what="fused dL_ddLdy")
    check(host(dg), ref, "fused")
    gg.backward_fused(d_xyz, d_dy, d_v, d_g2, want_dL_ddLdy=False, mode=GRAD_ACCUMULATE)
    check(host(dg), 2 * ref, "fused accumulate")
    # second-order only, accumulated on top
    _, ref2, _ = None, None, None
    base = host(dg).copy()
    ref_bbi, _, _ = og.backward_backward_input(params, xyz, v, g2, want_dinput=False)
    gg.backward_backward_input(d_xyz, d_v, d_g2, mode=GRAD_ACCUMULATE)
    check(host(dg), base + ref_bbi, "second order accumulate")
    # untouched entries stay exactly zero after Overwrite
    gg.backward(None, d_xyz, d_dy, mode=GRAD_OVERWRITE)
    got = host(dg)
    assert (got[ref1 == 0] == 0).all()


@pytest.mark.parametrize("run", [1, 2, 3, 5, 8, 9, 16, 40])  # around the steps of the sum over a run, and longer than a row of 16 lanes
def test_sorted_scatter_merges_runs_of_one_length(oracle, run):
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    og = oracle.Grid(CFG["n_levels"], CFG["log2_hashmap_size"], CFG["base_resolution"], CFG["per_level_scale"])
    gg = GridEncoding(**CFG)
    rng = np.random.default_rng(run)
    params = q16(rng.uniform(-1, 1, og.n_params))
    dp = dev(params, torch.float16)
    dg = torch.full_like(dp, 9.0)
    gg.set_params(dp, dg)
    n = 1500  # a second tile, and in it a second point of some threads
    assert gg.reserve_scatter_workspace(n)
    xyz = np.repeat(rng.random((3, (n + 4) // run + 1), dtype=np.float32), run, axis=1)[:, :n + 4][:, 4:].copy()  # (runs start off the rows)
    dy, g2 = q16(rng.standard_normal((32, n))), q16(rng.standard_normal((32, n)) * 0.1)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    ref1, _ = og.backward(params, xyz, dy, want_dx=False)
    ref, _, _ = og.backward_backward_input(params, xyz, v, g2, grad=ref1.copy(), want_dinput=False)
    gg.backward(None, dev(xyz), dev(dy, torch.float16), mode=GRAD_OVERWRITE)
    first = host(dg).copy()
    gg.backward_fused(dev(xyz), dev(dy, torch.float16), dev(v), dev(g2, torch.float16), want_dL_ddLdy=False, mode=GRAD_OVERWRITE)
    for l in range(16):
        a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
        assert rel_l2(first[a:b], ref1[a:b]) < RTOL and rel_l2(host(dg)[a:b], ref[a:b]) < RTOL, l


def test_sorted_scatter_pair_records_edge_cells(oracle):
    """Hashed levels sort one record per pair of x-neighbour corners; the second corner's place in the bucket is the
    first one's xor 2^(t+1) - 1, t = trailing one bits of the cell's x.  Cells whose x ends in 0 .. 11 one bits (the
    longest carries a 12-bit index can take), the first and the last cell of every level, against the oracle; and points
    outside the unit cube that carry a zero gradient change nothing."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, GridEncoding
    og = oracle.Grid(CFG["n_levels"], CFG["log2_hashmap_size"], CFG["base_resolution"], CFG["per_level_scale"])
    gg = GridEncoding(**CFG)
    rng = np.random.default_rng(41)
    params = q16(rng.uniform(-1, 1, og.n_params))
    dp = dev(params, torch.float16)
    dg = torch.zeros_like(dp)
    gg.set_params(dp, dg)
    n = 2 * 4096 + 264
    assert gg.reserve_scatter_workspace(1 << 14)
    xyz = rng.random((3, n), dtype=np.float32)
    # x coordinates in the middle of cells 2^k - 1 (k = 0 .. 11), 0 and res - 2 of the finest levels
    j = 0
    for level in (15, 14, 11, 8, 5):
        scale = float(og.scale[level])
        res = int(og.resolution[level])
        for cell in [0, res - 2] + [(1 << k) - 1 for k in range(13) if (1 << k) - 1 <= res - 2]:
            for rep in range(4):
                xyz[0, j] = np.float32((cell + 0.1 + 0.2 * rep) / scale)
                j += 1
    assert j < 4096
    dy = q16(rng.standard_normal((32, n)))
    stray = slice(n - 200, n)
    xyz[:, stray] = rng.uniform(-3, 4, (3, 200)).astype(np.float32)
    xyz[0, n - 200:n - 100] = rng.uniform(1.001, 40, 100).astype(np.float32)  # cells beyond the 12 index bits
    dy[:, stray] = 0
    inside = slice(0, n - 200)
    ref, _ = og.backward(params, np.ascontiguousarray(xyz[:, inside]), np.ascontiguousarray(dy[:, inside]), want_dx=False)
    dg.fill_(9.0)
    gg.backward(None, dev(xyz), dev(dy, torch.float16), mode=GRAD_OVERWRITE)
    got = host(dg)
    for l in range(16):
        a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
        assert rel_l2(got[a:b], ref[a:b]) < RTOL, (l, rel_l2(got[a:b], ref[a:b]))
    assert (got[ref == 0] == 0).all()


def _level_tols(og, n):
    return [RTOL * max(1.0, np.sqrt(8.0 * n / max(1, int(og.entries[l])))) for l in range(og.n_levels)]


@pytest.mark.parametrize("kind", ["global", "per_point", "progressive"])
@pytest.mark.parametrize("bucketed", [False, True])
def test_level_mask(setup, oracle, kind, bucketed):
    """Switched-off levels: zero features and dy_dx, no gradient, zero dL_ddLdy rows; everything else as unmasked.
    Expected values = the oracle on inputs whose switched-off (level, point) rows are zeroed."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE
    og, gg, params, d_params, d_grads = setup
    n = 3 * 4096 + 40 if bucketed else 3000
    rng = np.random.default_rng(77)
    xyz = rng.random((3, n), dtype=np.float32)
    dy = q16(rng.standard_normal((32, n)))
    g2 = q16(rng.standard_normal((32, n)) * 0.1)
    v = (rng.standard_normal((3, n)) * 1e-3).astype(np.float32)
    keep = None
    try:
        if bucketed:
            assert gg.reserve_scatter_workspace(1 << 14)
        if kind == "global":
            gg.set_max_level(0.5)
            assert gg.active_levels() == 9
            off = oracle.level_mask(16, n, 0.5)
        elif kind == "per_point":
            frac = (rng.random(n) * 2).astype(np.float32)  # the reference draws random_val * 2 per ray
            keep = dev(frac)
            gg.set_max_level_gpu(keep)
            off = oracle.level_mask(16, n, frac)
            assert 0.2 < off.mean() < 0.4
        else:
            gg.set_progressive(0.2, 0.02, 100)
            gg.set_training_step(1234)
            want = oracle.progressive_levels(16, 0.2, 0.02, 100, 1234)
            assert gg.active_levels() == want == 7
            off = oracle.level_mask(16, n, 1.0, valid_levels=want)
        off_rows = np.repeat(off, 2, axis=0)
        ref_y, ref_j = og.forward(params, xyz, want_dy_dx=True)
        ref_y[off_rows] = 0
        ref_j[off_rows] = 0
        d_xyz = dev(xyz)
        y, ctx = gg.forward(d_xyz, prepare_input_gradients=True)
        assert_close(host(y), ref_y, what="masked grid output")
        assert_close(host(ctx), ref_j, rtol=1e-4, what="masked dy_dx")
        assert (host(y)[off_rows] == 0).all() and (host(ctx)[off_rows] == 0).all()
        dy_m, g2_m = dy.copy(), g2.copy()
        dy_m[off_rows] = 0
        g2_m[off_rows] = 0
        ref1, ref_dx = og.backward(params, xyz, dy_m)
        ref, ref_out, _ = og.backward_backward_input(params, xyz, v, g2_m, grad=ref1.copy(), want_dinput=False)
        ref_out[off_rows] = 0
        d_grads.fill_(5.0)
        dx = gg.backward(ctx, d_xyz, dev(dy, torch.float16), want_input_grad=True, mode=GRAD_OVERWRITE)
        assert_close(host(dx), ref_dx, rtol=1e-4, what="masked dL_dx")
        got1 = host(d_grads)
        d_grads.fill_(5.0)
        out = gg.backward_fused(d_xyz, dev(dy, torch.float16), dev(v), dev(g2, torch.float16), mode=GRAD_OVERWRITE)
        got = host(d_grads)
        assert_close(host(out), ref_out, what="masked dL_ddLdy")
        assert (host(out)[off_rows] == 0).all()
        for l, tol in enumerate(_level_tols(og, n)):
            a, b = int(og.offset[l]) * 2, int(og.offset[l + 1]) * 2
            for g, r, what in ((got1, ref1, "first order"), (got, ref, "fused")):
                if np.abs(r[a:b]).max() == 0:
                    assert (g[a:b] == 0).all(), (what, l)  # a level nobody uses: Overwrite leaves zeros
                else:
                    assert rel_l2(g[a:b], r[a:b]) < tol, (what, l, rel_l2(g[a:b], r[a:b]), tol)
        # the second-order kernel that also returns dL_dx
        out2, din = gg.backward_backward_input(d_xyz, dev(v), dev(g2, torch.float16), want_dL_ddLdy=True, want_dL_dx=True,
                                               mode=GRAD_OVERWRITE)
        _, _, ref_din = og.backward_backward_input(params, xyz, v, g2_m)
        assert_close(host(out2), ref_out, what="masked dL_ddLdy (dL_dx variant)")
        assert_close(host(din), ref_din, rtol=1e-3, what="masked second-order dL_dx")
    finally:
        gg.set_max_level(1.0)
        gg.set_max_level_gpu(None)
        gg.set_progressive(1.0, 0.0, 0)
        if bucketed:
            from neus2_amd import capi
            import ctypes as C
            capi.lib().n2_grid_set_workspace(gg._h, None, C.c_uint64(0), C.c_uint32(0))
    assert gg.active_levels() == 16


def test_lattice_order_forward(setup):
    """The one-lane-per-point forward that n2_grid_set_point_order selects for lattice-ordered inference: same values as
    the oracle (and as the default kernel up to fp32 summation order), also with a level mask and ragged sizes."""
    og, gg, params, d_params, d_grads = setup
    r = 40
    z, y, x = np.meshgrid(np.arange(r), np.arange(r), np.arange(r), indexing="ij")
    xyz = (np.stack([x, y, z]).reshape(3, -1)[:, :r ** 3 - 13] / np.float32(r)).astype(np.float32)
    ref = og.forward(params, xyz)
    try:
        gg.set_point_order(True)
        y1, _ = gg.forward(dev(xyz))
        assert_close(host(y1), ref, what="lattice-order forward")
        gg.set_max_level(0.25)
        y2, _ = gg.forward(dev(xyz))
        ref2 = ref.copy()
        ref2[10:] = 0  # limit 4: levels 0..4 stay
        assert_close(host(y2), ref2, what="lattice-order forward, masked")
        assert (host(y2)[10:] == 0).all()
    finally:
        gg.set_point_order(False)
        gg.set_max_level(1.0)
    y0, _ = gg.forward(dev(xyz))
    assert rel_l2(host(y1), host(y0)) < 1e-3


@pytest.mark.parametrize("levels", [16, 14, 5])  # whole rounds of eight levels over the XCDs, a cut last round, nothing but that
@pytest.mark.parametrize("n", [1, 129, 3000])
def test_forward_by_level_costs_equals_the_default_deal(levels, n):
    """How the levels are dealt to the XCDs never shows in the results."""
    import ctypes as C

    from neus2_amd import capi
    from neus2_amd.tcnn_api import GridEncoding
    g = GridEncoding(levels, 2, 14, 8, 1.5)
    gen = torch.Generator(device="cuda").manual_seed(levels)
    p = torch.rand(g.n_params(), device="cuda", generator=gen).half()
    g.set_params(p, None)
    x = torch.rand((3, n), device="cuda", generator=gen)
    a, ja = g.forward(x, prepare_input_gradients=True)
    capi.check(capi.lib().n2_grid_set_level_costs(g._h, (C.c_float * levels)(*[1.0 + 3 * (l % 3) for l in range(levels)])))
    b, jb = g.forward(x, prepare_input_gradients=True)
    assert torch.equal(a, b) and torch.equal(ja, jb) and bool(a.abs().sum() > 0)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257])
@pytest.mark.parametrize("masked", [False, True])
def test_a_point_is_encoded_the_same_beside_any_neighbour(setup, n, masked):
    """Two adjacent lanes share the gathers of their points: bit for bit the same with another partner, one that is not a
    number or whose levels are switched off among them, and with none."""
    og, gg, params, *_ = setup
    rng = np.random.default_rng(n)
    xyz = (rng.random((3, n + 1)) * 1.1 - 0.05).astype(np.float32)
    xyz[:, 0] = np.nan
    frac = (rng.random(n + 1) * 2).astype(np.float32)
    keep = [dev(frac), dev(np.ascontiguousarray(frac[1:]))]
    try:
        outs = []
        for x, f in ((xyz, keep[0]), (np.ascontiguousarray(xyz[:, 1:]), keep[1])):
            if masked:
                gg.set_max_level_gpu(f)
            outs.append(gg.forward(dev(x), prepare_input_gradients=True))
    finally:
        gg.set_max_level_gpu(None)
    (a, ja), (b, jb) = outs
    assert torch.equal(a[:, 1:], b) and torch.equal(ja[:, 1:], jb) and bool(b.abs().sum() > 0)
