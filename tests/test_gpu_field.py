"""GPU parity of the NeuS field (NerfNetwork forward / backward / sdf / density) against the oracle."""
import os

import numpy as np
import pytest
import torch

from gpu_util import RTOL, assert_close, assert_grad_close, dev, host, q16, rel_l2

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
FLIP = 2e-4


def make(oracle, seed=0, geometric_init=False, **cfg):
    from neus2_amd.tcnn_api import NerfNetwork
    from oracle.field import Field
    of = Field(fp16=True, **cfg)
    gf = NerfNetwork(**cfg)
    assert gf.n_params() == of.n_params
    assert gf.param_offsets() == [of.off_sdf, of.off_rgb, of.off_grid, of.off_var, of.n_params]
    rng = np.random.default_rng(seed)
    p = np.zeros(of.n_params, np.float32)
    if geometric_init and of.sdf_in_w == 48:
        p[:of.off_rgb] = np.load(os.path.join(GOLD, "sdf_mlp_weights_48.npy"))
        p[of.off_grid:of.off_var] = rng.uniform(-1e-4, 1e-4, of.grid.n_params)
    else:
        p[:of.off_rgb] = rng.standard_normal(of.off_rgb) * 0.2
        p[of.off_grid:of.off_var] = rng.uniform(-0.5, 0.5, of.grid.n_params)
    p[of.off_rgb:of.off_grid] = rng.standard_normal(of.off_grid - of.off_rgb) * 0.2
    p[of.off_var] = 0.3
    p = q16(p)
    dp = dev(p, torch.float16)
    dg = torch.zeros_like(dp)
    gf.set_params(dp, dg)
    return of, gf, p, dp, dg, rng


def rand_coords(rng, n):
    c = rng.random((n, 7)).astype(np.float32)
    d = rng.standard_normal((n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    c[:, 4:7] = (d + 1) / 2
    c[:, 3] = 0
    return c


@pytest.mark.parametrize("geo", [False, True])
def test_forward_full_config(oracle, geo):
    of, gf, p, *_, rng = make(oracle, seed=1, geometric_init=geo)
    n = 4096
    coords = rand_coords(rng, n)
    ref, _ = of.forward(p, coords)
    out = host(gf.forward(dev(coords))).T
    # rows 11..15 are unused colour-net outputs but still defined: compare everything
    for name, rows in (("rgb", slice(0, 3)), ("sdf", slice(3, 4)), ("normal", slice(4, 7)), ("variance", slice(7, 8)),
                       ("dir", slice(8, 11)), ("tail", slice(11, 16))):
        assert_close(out[rows], ref[rows], what=f"field output {name}", outlier_frac=FLIP)
    if geo:
        r = np.linalg.norm(coords[:, :3] - 0.5, axis=1)
        assert np.corrcoef(out[3], r)[0, 1] > 0.75  # the sphere of the geometric init


def test_backward_full_config(oracle):
    of, gf, p, dp, dg, rng = make(oracle, seed=2)
    n = 8192
    coords = rand_coords(rng, n)
    # magnitudes chosen so that batch-summed gradients stay inside the fp16 range of the gradient buffer
    dL = q16(rng.standard_normal((16, n)) * np.array([.1, .1, .1, .1, 3, 3, 3, .1, .003, .003, .003, 0, 0, 0, 0, 0])[:, None])
    ref_out, ctx = of.forward(p, coords)
    ref = of.backward(p, ctx, dL, ek_batch_size=n)
    from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE
    d_coords = dev(coords)
    gf.forward(d_coords)
    dg.fill_(5.0)
    d_dL = dev(np.ascontiguousarray(dL.T), torch.float16)
    gf.backward(d_coords, d_dL, ek_batch_size=n, mode=GRAD_OVERWRITE)
    got = host(dg)
    assert_grad_close(got[of.off_sdf:of.off_rgb], ref[of.off_sdf:of.off_rgb], what="SDF MLP gradients (1st + 2nd order)",
                      rtol=2 * RTOL)
    assert_grad_close(got[of.off_rgb:of.off_grid], ref[of.off_rgb:of.off_grid], what="colour MLP gradients", rtol=2 * RTOL)
    # one fp16 rounding of a sum accumulated in fp32
    var_floor = 1e-5 * float(np.abs(dL[7]).sum()) + 1e-6
    assert abs(got[of.off_var] - ref[of.off_var]) <= RTOL * abs(ref[of.off_var]) + var_floor, (got[of.off_var], ref[of.off_var])
    for l in range(16):
        a = of.off_grid + 2 * int(of.grid.offset[l])
        b = of.off_grid + 2 * int(of.grid.offset[l + 1])
        k = 8.0 * n / max(1, int(of.grid.entries[l]))
        tol = 2 * RTOL * max(1.0, np.sqrt(k))
        assert rel_l2(got[a:b], ref[a:b]) < tol, (l, rel_l2(got[a:b], ref[a:b]), tol)
    # Accumulate doubles everything
    gf.backward(d_coords, d_dL, ek_batch_size=n, mode=GRAD_ACCUMULATE)
    got2 = host(dg)
    assert rel_l2(got2[:of.off_grid], 2 * ref[:of.off_grid]) < 3 * RTOL
    assert rel_l2(got2[of.off_grid:of.off_var], 2 * ref[of.off_grid:of.off_var]) < 2e-2
    # ... the variance gradient too (every backward sums its own batch, nothing is left over from the first call)
    assert abs(got2[of.off_var] - 2 * ref[of.off_var]) <= 3 * RTOL * abs(ref[of.off_var]) + 2 * var_floor, (got2[of.off_var], ref[of.off_var])


def test_backward_reference_14_level_config(oracle):
    """configs/nerf/base.json ships 14 levels -> SDF net input width 32 (the second weight fixture)."""
    cfg = dict(n_levels=14, log2_hashmap_size=19, base_resolution=16, per_level_scale=1.4472692012786865)
    of, gf, p, dp, dg, rng = make(oracle, seed=3, **cfg)
    assert of.sdf_in_w == 32
    n = 2048
    coords = rand_coords(rng, n)
    dL = q16(rng.standard_normal((16, n)))
    ref_out, ctx = of.forward(p, coords)
    out = host(gf.forward(dev(coords))).T
    assert_close(out[:11], ref_out[:11], what="14-level output", outlier_frac=FLIP)
    ref = of.backward(p, ctx, dL, ek_batch_size=1 << 18)
    gf.backward(dev(coords), dev(np.ascontiguousarray(dL.T), torch.float16), ek_batch_size=1 << 18)
    got = host(dg)
    assert_grad_close(got[:of.off_grid], ref[:of.off_grid], what="MLP gradients", rtol=2 * RTOL)
    assert rel_l2(got[of.off_grid:of.off_var], ref[of.off_grid:of.off_var]) < 1e-2


def test_sdf_and_density(oracle):
    of, gf, p, *_, rng = make(oracle, seed=4)
    n = 4096
    xyz = rng.random((3, n), dtype=np.float32)
    ref = of.sdf_values(p, xyz)
    got = host(gf.sdf(dev(xyz)))
    assert_close(got, ref, what="NerfNetwork::sdf", outlier_frac=FLIP)
    refd = of.density(p, xyz)
    gotd = host(gf.density(dev(xyz)))
    assert_close(gotd[0], refd[0], rtol=5e-3, what="NerfNetwork::density")
    # the row-per-point layout gives the same answer
    rows = np.zeros((n, 7), np.float32)
    rows[:, :3] = xyz.T
    assert torch.equal(gf.sdf(dev(rows)), gf.sdf(dev(xyz)))


@pytest.mark.parametrize("n", [8, 32, 40, 1000, 6144, 6152, 8192, 8200])
@pytest.mark.parametrize("levels,active", [(16, 1.0), (14, 1.0), (16, 0.5), (9, 1.0)])
def test_small_queries_equal_the_same_points_in_a_large_one(n, levels, active):
    """Queries of up to 8192 points are one launch: bit for bit what the gather and network launches give."""
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork(n_levels=levels)
    gen = torch.Generator(device="cuda").manual_seed(n + levels)
    net.set_params((torch.randn(net.param_offsets()[4], device="cuda", generator=gen) * 0.1).half(), None)
    if active < 1.0:
        net.encoding().set_max_level(active)
    many = torch.rand((16384, 3), device="cuda", generator=gen) * 1.2 - 0.1
    few = many[:n].contiguous()
    for query in (net.sdf, net.density):
        want = query(many)[:, :n]
        assert torch.equal(query(few).view(torch.int16), want.contiguous().view(torch.int16))
        assert torch.equal(query(few.T.contiguous()).view(torch.int16), want.contiguous().view(torch.int16))


@pytest.mark.parametrize("levels", [1, 6])  # input rows of 16 columns: four elements a load reach into the next row, and of the last one into W_out
def test_small_queries_of_narrow_networks_equal_the_same_points_in_a_large_one(levels):
    test_small_queries_equal_the_same_points_in_a_large_one(72, levels, 1.0)


@pytest.mark.parametrize("n", [8, 32, 40, 64, 72, 264])  # pairs across a wave's halves: no second half, a part of it, all, a wave more, a workgroup more
@pytest.mark.parametrize("active", [1.0, 0.5])
def test_small_batches_equal_the_same_samples_in_a_large_one(n, active):
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork()
    gen = torch.Generator(device="cuda").manual_seed(n)
    p = ((torch.rand(net.n_params(), device="cuda", generator=gen) - 0.5) * 0.4).half()
    net.set_params(p, torch.zeros_like(p))
    net.encoding().set_max_level(active)
    coords = torch.rand((512, 7), device="cuda", generator=gen)
    large = net.forward(coords)
    assert torch.equal(net.forward(coords[:n].contiguous()), large[:n]) and bool(torch.isfinite(large.float()).all())


# the last batch whose levels are all gathered and the first whose two coarsest are the network kernel's, the last and first with three more from blocks; tiles of 32 samples that are
# not whole; as few levels as that takes, and fewer; levels switched off, of these as well; tables that fill an LDS with the fragments and such that do not (base resolutions 24 and 32);
# a fifth level that is hashed, all of them but one
@pytest.mark.parametrize("n,cfg,active", [((3 << 15) - 8, {}, 1.0), (3 << 15, {}, 1.0), ((3 << 15) + 8, {}, 1.0), ((1 << 18) - 8, {}, 1.0), (1 << 18, {}, 1.0), ((1 << 18) + 8, {}, 1.0), (700008, {}, 1.0),
                                          ((1 << 17) + 24, dict(n_levels=3), 1.0), ((1 << 17) + 24, dict(n_levels=2), 1.0), ((1 << 18) + 24, dict(n_levels=6), 1.0), ((1 << 18) + 24, dict(n_levels=5), 1.0),
                                          ((1 << 18) + 24, {}, 0.25), ((1 << 18) + 24, {}, 0.1875), ((1 << 18) + 24, {}, 0.125), ((1 << 18) + 24, {}, 0.0625), ((1 << 17) + 24, {}, 0.0625), ((1 << 18) + 24, {}, 0.0),
                                          ((1 << 18) + 24, dict(base_resolution=24, per_level_scale=1.1), 1.0), ((1 << 18) + 24, dict(base_resolution=32), 1.0),
                                          ((1 << 18) + 24, dict(log2_hashmap_size=17), 1.0), ((1 << 18) + 24, dict(log2_hashmap_size=13), 1.0)])
def test_large_queries_equal_their_parts(n, cfg, active):
    """Bit for bit what smaller queries give, whose levels are all gathered."""
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork(**cfg)
    gen = torch.Generator(device="cuda").manual_seed(n)
    params = ((torch.rand(net.n_params(), device="cuda", generator=gen) - 0.5) * 0.3).half()
    net.set_params(params)
    net.encoding().set_max_level(active)
    x = torch.rand((3, n), device="cuda", generator=gen) * 1.2 - 0.1
    part = 1 << 15
    for query, points in ((net.sdf, x), (net.density, x.t().contiguous())):
        got = query(points)
        for a in range(0, n, part):
            want = query(x[:, a:a + part].contiguous())
            assert torch.equal(got[:, a:a + part].view(torch.int16), want.view(torch.int16)), a


# both sides of where rows and outputs pass by the caches, and a size beyond whose rows do not start lines
@pytest.mark.parametrize("n", [(3 << 18) - 32, 3 << 18, (3 << 18) + 8, (3 << 18) + 32])
def test_streamed_queries_equal_their_parts(n):
    test_large_queries_equal_their_parts(n, {}, 1.0)


# one tile past the line at which a query's and a forward's levels are no longer dealt to the XCDs
@pytest.mark.parametrize("levels", [16, 14, 1])
def test_batches_past_the_deal_by_xcd_equal_their_parts(levels):
    from neus2_amd.tcnn_api import NerfNetwork
    net = NerfNetwork(n_levels=levels)
    gen = torch.Generator(device="cuda").manual_seed(levels)
    net.set_params((torch.randn(net.param_offsets()[4], device="cuda", generator=gen) * 0.1).half(), None)
    n, part = (1 << 19) + 8, 1 << 17
    net.reserve(n)
    x = torch.rand((3, n), device="cuda", generator=gen)
    whole = net.sdf(x[:, :(5 << 16) + 8].contiguous()).clone()
    pieces = [net.sdf(x[:, a:a + part].contiguous()).clone() for a in range(0, (5 << 16) + 8, part)]
    assert torch.equal(whole, torch.cat(pieces, 1)[:, :whole.shape[1]])
    coords = torch.rand((n, 7), device="cuda", generator=gen)
    out = net.forward(coords).clone()
    assert torch.equal(out, torch.cat([net.forward(coords[a:a + part].contiguous()).clone() for a in range(0, n, part)]))
    enc = net.encoding()
    y, _ = enc.forward(x)
    assert torch.equal(y, torch.cat([enc.forward(x[:, a:a + part].contiguous())[0] for a in range(0, n, part)], 1))


def test_stream_lookup_follows_the_current_stream():
    from neus2_amd.tcnn_api import _stream
    side = torch.cuda.Stream()
    for s in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(s):
            assert (_stream().value or 0) == s.cuda_stream == torch.cuda.current_stream().cuda_stream


def test_field_errors(oracle):
    from neus2_amd.tcnn_api import N2Error, NerfNetwork
    gf = NerfNetwork()
    c = torch.rand((64, 7), device="cuda")
    with pytest.raises(N2Error, match="set_params"):
        gf.forward(c)
    gf.set_params(torch.zeros(gf.n_params(), dtype=torch.float16, device="cuda"), None)
    gf.forward(c)
    with pytest.raises(N2Error, match="gradient buffer"):
        gf.backward(c, torch.zeros((64, 16), dtype=torch.float16, device="cuda"))
    with pytest.raises(N2Error, match="multiple of 8"):
        gf.forward(torch.rand((12, 7), device="cuda"))
    assert gf.forward(torch.rand((0, 7), device="cuda")).shape == (0, 16)


def test_select_equals_forward_on_the_selected_samples(oracle):
    """n2_field_select: backward over samples picked from the last forward (with repeats and gaps, odd and even counts)
    gives exactly the gradients of a forward over those samples' coordinates followed by the same backward."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE, N2Error
    of, gf, p, dp, dg, rng = make(oracle, seed=6)
    n_src = 6000
    coords = rand_coords(rng, n_src)
    d_coords = dev(coords)
    for n in (4096, 5000):  # (smaller batches scatter with fp16 atomics, whose order of arrival is not reproducible)
        idx = np.sort(rng.integers(0, n_src, n)).astype(np.int32)
        idx[-40:] = idx[:40]  # roll-over style repeats, out of order
        dL = q16(rng.standard_normal((n, 16)) * np.array([.1, .1, .1, .1, 3, 3, 3, .1, .003, .003, .003, 0, 0, 0, 0, 0]))
        d_dL = dev(dL, torch.float16)
        sub = dev(coords[idx])
        gf.forward(sub)
        dg.fill_(3.0)
        gf.backward(sub, d_dL, ek_batch_size=n, mode=GRAD_OVERWRITE)
        want = dg.clone()
        gf.forward(d_coords)
        gf.select(dev(idx, torch.int32), n_src)
        dg.fill_(3.0)  # (the three spare variance slots are never written)
        gf.backward(sub, d_dL, ek_batch_size=n, mode=GRAD_OVERWRITE)
        assert torch.equal(dg, want), n
    # the batch of a backward must be the selection (or the forward) that precedes it
    with pytest.raises(N2Error):
        gf.backward(d_coords, dev(q16(rng.standard_normal((n_src, 16))), torch.float16), ek_batch_size=n_src)
    with pytest.raises(N2Error):
        gf.select(dev(idx, torch.int32), n_src + 8)


def test_padding_rows_follow_the_batch_size(oracle):
    """The inputs of the two networks are padded to 48 rows; the padding rows are cleared once per batch size and never
    written again.  Starting from a workspace full of NaNs, batches of changing sizes (the rows move with the row pitch),
    the SDF-only path and a backward through a selection all agree with the oracle."""
    from neus2_amd.tcnn_api import GRAD_OVERWRITE
    of, gf, p, dp, dg, rng = make(oracle, seed=11)
    gf.reserve(8192)
    gf._ws.fill_(0xFF)  # every fp16 of the workspace is a NaN
    for n in (4096, 2048, 8192, 4096):
        coords = rand_coords(rng, n)
        ref, ctx = of.forward(p, coords)
        out = host(gf.forward(dev(coords))).T
        assert np.isfinite(out[:11]).all(), n
        assert_close(out[:11], ref[:11], what=f"field output at n={n}", outlier_frac=FLIP)
        xyz = np.ascontiguousarray(coords[: n // 2, :3])
        sdf = host(gf.sdf(dev(xyz)))
        assert np.isfinite(sdf[0]).all()
        assert_close(sdf[0], of.sdf_values(p, xyz.T.copy())[0], what=f"sdf at n={n // 2}", outlier_frac=FLIP)
    # a backward through a selection of half the last batch
    n = 4096
    coords = rand_coords(rng, n)
    gf.forward(dev(coords))
    pick = np.sort(rng.choice(n, n // 2, replace=False)).astype(np.int32)
    gf.select(torch.from_numpy(pick).cuda(), n)
    dL = q16(rng.standard_normal((16, n // 2)) * np.array([.1, .1, .1, .1, 3, 3, 3, .1, .003, .003, .003, 0, 0, 0, 0, 0])[:, None])
    sub = np.ascontiguousarray(coords[pick])
    _, ctx = of.forward(p, sub)
    ref = of.backward(p, ctx, dL, ek_batch_size=n // 2)
    gf.backward(dev(sub), dev(np.ascontiguousarray(dL.T), torch.float16), ek_batch_size=n // 2, mode=GRAD_OVERWRITE)
    got = host(dg)
    assert np.isfinite(got).all()
    assert_grad_close(got[of.off_sdf:of.off_rgb], ref[of.off_sdf:of.off_rgb], what="SDF MLP gradients", rtol=2 * RTOL)
    assert_grad_close(got[of.off_rgb:of.off_grid], ref[of.off_rgb:of.off_grid], what="colour MLP gradients", rtol=2 * RTOL)


def test_direction_encoding_rows(oracle):
    """The degree-4 spherical-harmonics rows of the colour net's input on their own: with every other input column of
    the colour net's first layer zeroed, the output depends on the direction only through the 16 SH rows, and a net whose
    hidden layers pass values through unchanged hands them to the output."""
    from neus2_amd.tcnn_api import NerfNetwork
    from oracle.field import Field
    of, gf = Field(fp16=True), NerfNetwork()
    rng = np.random.default_rng(4)
    p = np.zeros(of.n_params, np.float32)
    # colour net: W0 [64][48] picks SH row k (input column 16 + k) into neurons 2k (+) and 2k + 1 (-), the second layer is
    # the identity, the output layer recombines relu(x) - relu(-x) = x for the first 16 SH values
    W0 = np.zeros((64, 48), np.float32)
    W1 = np.eye(64, dtype=np.float32)
    Wo = np.zeros((16, 64), np.float32)
    for k in range(16):
        W0[2 * k, 16 + k], W0[2 * k + 1, 16 + k] = 1.0, -1.0
        Wo[k, 2 * k], Wo[k, 2 * k + 1] = 1.0, -1.0
    p[of.off_rgb:of.off_grid] = np.concatenate([W0.ravel(), W1.ravel(), Wo.ravel()])
    p[of.off_sdf:of.off_rgb] = rng.standard_normal(of.off_rgb) * 0.1
    p[of.off_grid:of.off_var] = rng.uniform(-0.1, 0.1, of.grid.n_params)
    p = q16(p)
    dp = dev(p, torch.float16)
    gf.set_params(dp, torch.zeros_like(dp))
    n = 4096
    coords = rand_coords(rng, n)
    out = host(gf.forward(dev(coords))).T
    sh = oracle.sh4(np.ascontiguousarray(coords[:, 4:7].T))           # pinned by scipy.special.sph_harm_y
    # rows 0..2 and 11..15 of the output are the colour net's own rows (3..10 are overwritten by sdf, normal, ...)
    for r in (0, 1, 2, 11, 12, 13, 14, 15):
        assert_close(out[r], q16(sh[r]), rtol=RTOL, what=f"SH row {r}", scale=1.0)


@pytest.mark.parametrize("n_levels", [15, 17, 20, 22])  # networks of 48 inputs, whose encodings have 30 to 44 rows
def test_backward_of_more_levels_than_the_fused_kernels_take(oracle, n_levels):
    of, gf, p, dp, dg, rng = make(oracle, seed=13, n_levels=n_levels, log2_hashmap_size=14, per_level_scale=1.2)
    assert of.sdf_in_w == 48
    n = 2048
    coords = rand_coords(rng, n)
    dL = q16(rng.standard_normal((16, n)) * np.array([.1, .1, .1, .1, 3, 3, 3, .1, .003, .003, .003, 0, 0, 0, 0, 0])[:, None])
    _, ctx = of.forward(p, coords)
    ref = of.backward(p, ctx, dL, ek_batch_size=n)
    gf.reserve(n)
    gf._ws.fill_(0x3C)  # (nothing may be left from another call: halves of 1.06)
    d_coords = dev(coords)
    gf.forward(d_coords)
    gf.backward(d_coords, dev(np.ascontiguousarray(dL.T), torch.float16), ek_batch_size=n)
    got = host(dg)
    assert_grad_close(got[:of.off_rgb], ref[:of.off_rgb], what="SDF MLP gradients", rtol=2 * RTOL)
    for l in range(n_levels):
        a, b = (of.off_grid + 2 * int(of.grid.offset[l + k]) for k in range(2))
        k = 8.0 * n / max(1, int(of.grid.entries[l]))
        tol = 2 * RTOL * max(1.0, np.sqrt(k))
        assert rel_l2(got[a:b], ref[a:b]) < tol, (l, rel_l2(got[a:b], ref[a:b]), tol)


@pytest.mark.parametrize("infinite", ["all", "even_x"])
def test_slopes_that_are_no_numbers_count_as_zero(oracle, infinite):
    """Infinite entries of one level and feature: differences of two of them are no numbers and add nothing to the normal; a difference to a finite
    entry is the largest slope a block holds, (2^19 - 1) 2^-19 of the level's scale where it is the block's own exponent."""
    of, gf, p, dp, dg, rng = make(oracle, seed=12, log2_hashmap_size=14)
    n, w = 512, of.sdf_in_w
    coords = rand_coords(rng, n)
    coords[:, :3] = 0.1 + 0.8 * coords[:, :3]
    W0, Wo = p[:64 * w].reshape(64, w), p[64 * w:of.off_rgb].reshape(16, 64)
    W0[:, 3] = q16(np.where(rng.random(64) < 0.5, -1, 1) * (0.1 + rng.random(64)))  # the sign alone decides about a neuron
    res, off = int(of.grid.resolution[0]), of.off_grid + 2 * int(of.grid.offset[0])
    level = p[off:off + 2 * int(of.grid.entries[0])].reshape(-1, 2)
    level[:, 0] = 0
    J = of.grid.forward(p[of.off_grid:of.off_var], np.ascontiguousarray(coords[:, :3].T), want_dy_dx=True)[1].astype(np.float64)
    assert not J[0].any()
    level[:, 0] = np.where((np.arange(len(level)) % res % 2 == 0) | (infinite == "all"), np.inf, 0.25)
    if infinite == "even_x":
        cell = np.floor(coords[:, 0] * of.grid.scale[0] + np.float32(0.5)).astype(int)
        J[0, :, 0] = np.where(cell % 2 == 0, -1, 1) * (2 ** 19 - 1) / 2 ** 19 * float(of.grid.scale[0])
    g = q16(W0.T.astype(np.float64) @ (Wo[0].astype(np.float64) * (W0[:, 3] > 0)))
    want = np.einsum("k,knd->dn", g[3:3 + of.enc_w].astype(np.float64), J) + g[:3, None]
    dp.copy_(dev(p, torch.float16))
    got = host(gf.forward(dev(coords))).T[4:7]
    assert_close(got, want.astype(np.float32), what="normal")


@pytest.mark.parametrize("n_levels", [16, 12, 20])  # the fused kernels, others of them, and the separate ones
def test_captured_steps_and_the_padding_rows(n_levels):
    """A batch size that is first met under capture: a step outside the graph comes before the first replay.  Queries between replays, which use the padding's place."""
    from neus2_amd.tcnn_api import NerfNetwork
    n = 1000
    gen = torch.Generator(device="cuda").manual_seed(n_levels)
    net = NerfNetwork(n_levels, 14)
    P = (torch.randn(net.n_params(), device="cuda", generator=gen) * 0.2).half()
    G = torch.zeros_like(P)
    net.set_params(P, G)
    coords = torch.rand((n, 7), device="cuda", generator=gen)
    dL = (torch.randn((n, 16), device="cuda", generator=gen) * 0.01).half()
    x = torch.rand((3, 16384), device="cuda", generator=gen)
    def step():
        y = net.forward(coords)
        net.backward(coords, dL)
        return y
    net.reserve(16384)
    want = [step().clone(), G.clone()]
    assert all(bool(torch.isfinite(t).all()) for t in want)
    net.sdf(x)  # (another batch size: nothing counts as cleared any more)
    net.reserve(16392)  # a workspace of its own for this batch size ...
    net._ws.fill_(255)  # ... and what memory that nothing has written may hold: no numbers
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        y = step()
    torch.cuda.synchronize()
    got = [step(), G]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    for k in range(3):
        net.sdf(x)
        y.zero_()
        G.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[0]) and torch.equal(G, want[1]), k
