"""SDF network with the eikonal second-order path (grid + 48-64-16 MLP, loss = mean|sdf| + 0.1 mean(|grad sdf| - 1)^2):
forward, normals and every parameter gradient against the same composition of the oracle's pieces."""
import os

import numpy as np
import pytest
import torch

from gpu_util import RTOL, assert_close, assert_grad_close, dev, host, q16, rel_l2

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


@pytest.mark.parametrize("kind", ["uniform", "rays"])
def test_sdf_eikonal_step_matches_oracle(oracle, kind):
    from neus2_amd.sdf_net import SdfNet
    rng = np.random.default_rng(7)
    n = 8192
    net = SdfNet(max_batch=n)
    P = q16(rng.uniform(-0.01, 0.01, net.grid.n_params()))  # gradient norms around 1 +- a few tenths; larger tables overflow fp16 gradients
    W = q16(np.load(os.path.join(GOLD, "sdf_mlp_weights_48.npy")) + rng.normal(0, 0.05, 4096))
    if kind == "uniform":
        x = rng.random((3, n), dtype=np.float32)
    else:
        o = 0.3 + 0.4 * rng.random((n // 64, 1, 3))
        d = rng.standard_normal((n // 64, 1, 3))
        d /= np.linalg.norm(d, axis=-1, keepdims=True)
        x = np.clip(o + d * (np.arange(64).reshape(1, 64, 1) - 32) * (np.sqrt(3.0) / 1024), 0, 1).reshape(-1, 3).T.astype(np.float32).copy()
    dP, dW = dev(P, torch.float16), dev(W, torch.float16)
    gP, gW = torch.zeros_like(dP), torch.zeros_like(dW)
    net.set_params(dP, gP, dW, gW)
    ctx = net.forward(dev(x))
    loss = float(net.loss_backward(ctx, ek_weight=0.1, loss_scale=128.0).item())
    from oracle.sdf_step import sdf_eikonal_step
    ref = sdf_eikonal_step(P, W, x, 0.1, 128.0)
    assert_close(host(ctx["sdf"]), ref["sdf"], what="sdf", outlier_frac=1e-3)
    assert_close(host(ctx["normal"]), ref["normal"], what="normal", outlier_frac=2e-3)
    assert abs(loss - ref["loss"]) <= 2e-3 * abs(ref["loss"])
    assert_grad_close(host(gW), ref["mlp_grad"], what="MLP gradient", rtol=5e-3)
    got = host(gP)
    for l in range(16):
        a, b = int(ref["offset"][l]) * 2, int(ref["offset"][l + 1]) * 2
        assert rel_l2(got[a:b], ref["grid_grad"][a:b]) < 5e-3, (l, rel_l2(got[a:b], ref["grid_grad"][a:b]))


@pytest.mark.parametrize("n_levels,n", [(16, 1), (16, 255), (16, 5003), (3, 257), (13, 1000), (20, 777), (16, 180000)])
def test_normals_and_loss_in_one_pass_equal_the_two_calls(n_levels, n):
    """n2_sdf_normals_and_eikonal_loss against n2_grid_backward and n2_sdf_eikonal_loss, bit for bit: fewer rows than a lane
    holds at once, more (20 levels), and a Jacobian that is streamed (180000 points)."""
    import ctypes as C
    from neus2_amd import capi
    from neus2_amd.capi import check, ptr
    from neus2_amd.tcnn_api import GRAD_IGNORE, GridEncoding, _stream
    L = capi.lib()
    gen = torch.Generator(device="cuda").manual_seed(n)
    enc = GridEncoding(n_levels, 2, 14, 16, 1.3)
    P = (torch.randn(enc.n_params(), device="cuda", generator=gen) * 0.01).half()
    enc.set_params(P, None)
    x = torch.rand((3, n), device="cuda", generator=gen)
    rows, in_w = 2 * n_levels, (3 + 2 * n_levels + 15) // 16 * 16
    _, dy_dx = enc.forward(x, prepare_input_gradients=True)
    g = torch.randn((in_w, n), device="cuda", generator=gen).half()
    y = torch.randn((16, n), device="cuda", generator=gen).half()
    ws = torch.empty(int(L.n2_sdf_eikonal_workspace_bytes(C.c_uint32(n))), dtype=torch.uint8, device="cuda")
    outs = []
    for one in (False, True):
        normal, v = (torch.full((3, n), 7.0, device="cuda") for _ in range(2))
        dL_dy, v_in = torch.full((16, n), 7.0, device="cuda").half(), torch.full((in_w, n), 7.0, device="cuda").half()
        loss = torch.zeros(1, device="cuda")
        head = (_stream(), C.c_uint32(n), C.c_uint32(rows), C.c_uint32(in_w), ptr(y), ptr(g))
        tail = (ptr(normal), C.c_float(0.1), C.c_float(128.0), ptr(dL_dy), ptr(v), ptr(v_in), ptr(loss), ptr(ws), C.c_uint64(ws.numel()))
        if one:
            check(L.n2_sdf_normals_and_eikonal_loss(*head, ptr(dy_dx), *tail), "n2_sdf_normals_and_eikonal_loss")
        else:
            normal_enc = enc.backward(dy_dx, x, g[3:3 + rows].contiguous(), want_input_grad=True, mode=GRAD_IGNORE)
            # (in 64 bits first: the input gradient is a sum of 32-bit products of `rows` terms)
            ref = (g[3:3 + rows].double()[:, :, None] * dy_dx.double()).sum(0).t()
            assert float((normal_enc.double() - ref).norm() / ref.norm()) < 1e-6
            check(L.n2_sdf_eikonal_loss(*head, ptr(normal_enc), *tail, ptr(dy_dx)), "n2_sdf_eikonal_loss")
        outs.append((normal, v, dL_dy, v_in, loss))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
