"""What a user of this framework has it do, at the sizes and options it is used with: training steps, the operators a program
composes itself, queries, occupancy-grid updates and mesh extraction, all through the Python entry points.

listed() and draw() give the cases, prepare() what a program holds before the call, run() one call, work() the bytes and
operations the call cannot do without, tolerance() what another correct implementation at the same precision may differ by."""
import functools
import math

import torch

from neus2_amd import scene
from neus2_amd.mesh import density_on_grid, marching_cubes
from neus2_amd.sdf_net import SdfNet
from neus2_amd.tcnn_api import GRAD_ACCUMULATE, GRAD_OVERWRITE, GridEncoding, NerfNetwork, generate_training_samples, pack_cameras
from neus2_amd.training import GRID_CELLS, OccupancyGrid, Trainer, default_config, next_multiple

MARCH_STEP = math.sqrt(3.0) / 1024.0  # the sample generator's fixed step: consecutive samples of a ray are this far apart


def listed():
    return [
        # the training step the benchmark quotes: early in training every marched sample is kept, the batch is 2^18
        dict(name="train 2^18", kind="train", target=1 << 18, trained=False),
        # late in training: the occupancy grid has closed in on the surface, a step marches three samples for each it keeps
        dict(name="train 2^18 trained", kind="train", target=1 << 18, trained=True),
        # a small batch, as for previews and tests: launches and the optimiser's pass over the table count
        dict(name="train 2^14", kind="train", target=1 << 14, trained=False),
        # the encoding alone, forward with the Jacobian and backward to parameters and positions, uniform points
        dict(name="grid 2^18", kind="grid", n=1 << 18, order="uniform", second=False),
        # the same on few points along rays, an odd number of them, with the second-order pass
        dict(name="grid 5003 second order", kind="grid", n=5003, order="rays", second=True),
        # the SDF network with the eikonal term: forward, normals, first- and second-order backward
        dict(name="sdf net 2^18", kind="sdf_net", n=1 << 18, order="uniform"),
        # the whole field as an operator inside a caller's own loop, a ragged batch
        dict(name="field 52344", kind="field", n=52344),
        # a handful of distance queries (collision tests, probes): latency
        dict(name="query 1000", kind="query", n=1000, what="sdf"),
        # many density queries in no order
        dict(name="query 2^20", kind="query", n=1 << 20, what="density"),
        # one full sweep of the occupancy grid, as before each of the first training steps
        dict(name="occupancy 128^3", kind="occupancy", n_uniform=GRID_CELLS, n_nonuniform=0),
        # mesh extraction, first half: the SDF on the lattice
        dict(name="lattice 512^3", kind="lattice", rx=512, ry=512, rz=512),
        # mesh extraction, second half: marching cubes over the lattice, with normals
        dict(name="mesh 512^3", kind="mesh", rx=512, ry=512, rz=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "grid", "grid", "sdf_net", "field", "query", "occupancy", "lattice", "mesh"])
    if kind == "train":
        return dict(kind=kind, target=_log(rng, 1 << 12, 1 << 18) // 128 * 128, trained=rng.random() < 0.5)
    if kind == "grid":
        return dict(kind=kind, n=_log(rng, 200, 1 << 18), order=rng.choice(["uniform", "rays"]), second=rng.random() < 0.5)
    if kind == "sdf_net":
        return dict(kind=kind, n=_log(rng, 1 << 10, 1 << 18) // 8 * 8, order=rng.choice(["uniform", "rays"]))
    if kind == "field":
        return dict(kind=kind, n=_log(rng, 1 << 10, 1 << 18) // 8 * 8)
    if kind == "query":
        return dict(kind=kind, n=_log(rng, 64, 1 << 21) // 8 * 8, what=rng.choice(["sdf", "density"]))
    if kind == "occupancy":
        n = _log(rng, 1 << 17, GRID_CELLS)
        return dict(kind=kind, n_uniform=n, n_nonuniform=0) if rng.random() < 0.5 else dict(kind=kind, n_uniform=n // 2, n_nonuniform=n // 2)
    sides = [16 * rng.randint(4, 32) for _ in range(3)]  # mesh extraction rounds each side up to a multiple of 16
    return dict(kind=kind, rx=sides[0], ry=sides[1], rz=sides[2])


# ---------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(gen, shape, lo, hi):
    return torch.rand(shape, device="cuda", generator=gen) * (hi - lo) + lo


def _normal(gen, shape):
    return torch.randn(shape, device="cuda", generator=gen)


def _grid_parameters(gen, encoding):
    """Table entries as training leaves them: the finer the level, the smaller, so that every level adds about as much to the
    distance's gradient."""
    scale, _, entries, _ = encoding.level_table()
    return torch.cat([_normal(gen, 2 * int(e)) * (0.3 / float(s)) for s, e in zip(scale, entries)])


def _sdf_weights(gen, in_width):
    """An SDF network whose row 0 is close to |x - 0.5|: first-layer directions spread over the sphere, equal weights behind
    the ReLUs, and small encoding columns."""
    k = torch.arange(64, device="cuda", dtype=torch.float64)
    z = 1 - 2 * (k + 0.5) / 64
    phi = k * math.pi * (3 - math.sqrt(5)) + float(torch.rand(1, device="cuda", generator=gen)) * 2 * math.pi
    r = torch.sqrt(1 - z * z)
    w0 = _normal(gen, (64, in_width)) * 0.05
    w0[:, :3] = torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], 1).float()
    w1 = _normal(gen, (16, 64)) * 0.15
    w1[0] = 4.0 / 64
    return torch.cat([w0.reshape(-1), w1.reshape(-1)])


def _field_parameters(gen, encoding, offsets, variance):
    """The field's parameter vector: geometric SDF network, Xavier colour network, table, variance."""
    in_width = (offsets[1] - offsets[0]) // 64 - 16
    xavier = [_uniform(gen, (o, i), -1, 1).reshape(-1) * math.sqrt(6.0 / (o + i)) for o, i in ((64, 48), (64, 64), (16, 64))]
    p = torch.cat([_sdf_weights(gen, in_width), *xavier, _grid_parameters(gen, encoding)])
    return torch.cat([p, torch.full((offsets[4] - offsets[3],), variance, device="cuda")])


def _positions(gen, n, order):
    """[3, n] positions in the unit cube: anywhere, or in runs of 40 along rays through it."""
    if order == "uniform":
        return _uniform(gen, (3, n), 0, 1)
    rays = (n + 39) // 40
    d = _normal(gen, (3, rays, 1))
    d = d / d.norm(dim=0, keepdim=True)
    start = _uniform(gen, (3, rays, 1), 0.1, 0.9)
    x = start + d * (torch.arange(40, device="cuda") * MARCH_STEP)
    return x.reshape(3, -1)[:, :n].clamp(0, 1).contiguous()


@functools.lru_cache(maxsize=None)
def _cameras():
    return scene.cameras_on_sphere(64, 512)


@functools.lru_cache(maxsize=None)
def _shell(band):
    return scene.sphere_bitfield(radius=0.3, band=band)


def _images(gen):
    """The training images: a lit, textured sphere of radius 0.3 in front of nothing, RGBA with premultiplied alpha."""
    phase = _uniform(gen, (3,), 0, 6)
    light = _normal(gen, (3,))
    light = light / light.norm()
    out = []
    for cam in _cameras():
        w, h = cam["res"]
        m = torch.from_numpy(cam["xform"].reshape(3, 4)).cuda()
        px = ((torch.arange(w, device="cuda") + 0.5) / w - 0.5) * w / float(cam["focal"][0])
        py = ((torch.arange(h, device="cuda") + 0.5) / h - 0.5) * h / float(cam["focal"][1])
        d = px[None, :, None] * m[:, 0] + py[:, None, None] * m[:, 1] + m[:, 2]
        d = d / d.norm(dim=-1, keepdim=True)
        oc = m[:, 3] - 0.5
        b = (d * oc).sum(-1)
        disc = b * b - ((oc * oc).sum() - 0.09)
        hit = (disc > 0).float()[..., None]
        nrm = (oc + (-b - disc.clamp(min=0).sqrt())[..., None] * d) / 0.3
        albedo = 0.5 + 0.5 * torch.sin(nrm * torch.tensor([9.0, 7.0, 5.0], device="cuda") + phase)
        rgb = albedo * (0.25 + 0.75 * (nrm * light).sum(-1, keepdim=True).clamp(0, 1)) * hit
        out.append(torch.cat([rgb, hit], -1).reshape(-1, 4))
    return torch.cat(out)


def _rays(case):
    # what the ray budget's feedback settles at: 52 samples a ray in a wide shell, 7 kept of 20 on a trained field
    return next_multiple(case["target"] * (0.1375 if case["trained"] else 1 / 52.5), 128)


def _prepare_train(case, gen, seed):
    """A training run that goes on: parameters and optimiser state as a snapshot restores them."""
    trained, target, n_rays = case["trained"], case["target"], _rays(case)
    cfg = default_config(target_batch_size=target, learning_rate=1e-4 if trained else 1e-3)
    cfg.field.sdf_bias = -0.3 if trained else -0.1
    tr = Trainer(cfg)
    cams, images = pack_cameras(_cameras()), _images(gen)
    bits = torch.from_numpy(_shell(0.0115 if trained else 0.03)).cuda()
    tr.set_scene(cams, 64, images, bits)
    p = _field_parameters(gen, tr.encoding(), tr.offsets, 0.85 if trained else 0.3)
    tr.set_parameters(p.cpu().numpy())
    marched = generate_training_samples(n_rays, 0, 0, cams, 64, images, (1.0, 1.0, 1.0), bits, cfg.max_samples)["sample_counter"]
    n_inference = next_multiple(min(int(marched), cfg.max_samples), 128)
    for _ in range(2):  # the feedback also switches the depth rounds on when a step marches far more than it keeps
        tr.step(n_rays=n_rays, n_inference=n_inference)
        tr.update_budget()
    s = tr.optimizer_state()
    m1, m2 = (tr._view(a, tr.n_params, torch.float32) for a in (s.first_moments, s.second_moments))
    steps = tr._view(s.param_steps, tr.n_params, torch.int16 if s.param_steps_bits == 16 else torch.int32)
    # gradients of the sizes these batches give, hundreds of steps old
    m1.copy_(_normal(gen, tr.n_params) * 2e-7)
    m2.copy_(_uniform(gen, tr.n_params, 0.5e-12, 2e-12))
    steps.fill_(500)
    tr.set_parameters(p.cpu().numpy())
    return dict(case=case, trainer=tr, n_rays=n_rays, n_inference=n_inference, m1=m1, m2=m2)


def _prepare_grid(case, gen, seed):
    n = case["n"]
    enc = GridEncoding()
    params = _grid_parameters(gen, enc).half()
    grads = torch.zeros_like(params)
    enc.set_params(params, grads)
    enc.reserve_scatter_workspace(n)
    return dict(case=case, enc=enc, grads=grads, x=_positions(gen, n, case["order"]), dy=_normal(gen, (32, n)).half(), v=_normal(gen, (3, n)))


def _prepare_sdf_net(case, gen, seed):
    n = case["n"]
    net = SdfNet(max_batch=n)
    params, weights = _grid_parameters(gen, net.grid).half(), _sdf_weights(gen, net.in_w).half()
    grid_grads, mlp_grads = torch.zeros_like(params), torch.zeros_like(weights)
    net.set_params(params, grid_grads, weights, mlp_grads)
    return dict(case=case, net=net, grid_grads=grid_grads, mlp_grads=mlp_grads, x=_positions(gen, n, case["order"]))


def _field(gen, n, gradients):
    net = NerfNetwork()
    params = _field_parameters(gen, net.encoding(), net.param_offsets(), 0.3).half()
    grads = torch.zeros_like(params) if gradients else None
    net.set_params(params, grads)
    net.reserve(n)
    return net, grads


def _prepare_field(case, gen, seed):
    n = case["n"]
    net, grads = _field(gen, n, True)
    x = _positions(gen, n, "rays")
    d = _normal(gen, (3, n))
    d = d / d.norm(dim=0, keepdim=True) * 0.5 + 0.5
    coords = torch.cat([x, torch.full((1, n), MARCH_STEP, device="cuda"), d]).t().contiguous()
    dl = _normal(gen, (n, 16)) * 0.05
    dl[:, 11:] = 0
    return dict(case=case, net=net, grads=grads, coords=coords, dl=dl.half())


def _prepare_query(case, gen, seed):
    net, _ = _field(gen, case["n"], False)
    return dict(case=case, net=net, x=_positions(gen, case["n"], "uniform"))


def _prepare_occupancy(case, gen, seed):
    cfg = default_config(target_batch_size=1 << 12, max_rays_per_batch=1 << 8, max_samples=1 << 21)
    cfg.field.sdf_bias = -0.3
    tr = Trainer(cfg)
    tr.set_parameters(_field_parameters(gen, tr.encoding(), tr.offsets, 0.5).cpu().numpy())
    occ = OccupancyGrid(1, seed=seed)
    occ.update(tr._field, GRID_CELLS, 0)  # the grid as the updates before this one have left it
    return dict(case=case, trainer=tr, occ=occ)


def _prepare_lattice(case, gen, seed):
    cfg = default_config(target_batch_size=1 << 12, max_rays_per_batch=1 << 8, max_samples=1 << 22)
    tr = Trainer(cfg)
    tr.set_parameters(_field_parameters(gen, tr.encoding(), tr.offsets, 0.3).cpu().numpy())
    return dict(case=case, trainer=tr)


def _prepare_mesh(case, gen, seed):
    """A distance lattice of a bumpy sphere, somewhere near the middle and in some unit of length."""
    x, y, z = ((torch.arange(r, device="cuda") / r - 0.5) for r in (case["rx"], case["ry"], case["rz"]))
    d = (x[None, None, :] ** 2 + y[None, :, None] ** 2 + z[:, None, None] ** 2).sqrt_().sub_(0.3)
    d += 0.02 * torch.sin(17 * x + 1)[None, None, :] * torch.sin(13 * y + 2)[None, :, None] * torch.sin(11 * z + 3)[:, None, None]
    shift = [int(s * r) for s, r in zip(_uniform(gen, (3,), -0.12, 0.12).tolist(), d.shape)]
    return dict(case=case, density=torch.roll(d, shift, (0, 1, 2)) * float(_uniform(gen, (1,), 0.5, 2)))


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _generator(seed), seed)


# ---------------------------------------------------------------------------------------------------------------------
# one call
# ---------------------------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        tr = state["trainer"]
        tr.step(n_rays=state["n_rays"], n_inference=state["n_inference"])
        return dict(master=tr.master, params=tr.params, grads=tr.grads, m1=state["m1"], m2=state["m2"])
    if kind == "grid":
        enc, x, dy = state["enc"], state["x"], state["dy"]
        out, ctx = enc.forward(x, prepare_input_gradients=True)
        dx = enc.backward(ctx, x, dy, want_input_grad=True, mode=GRAD_OVERWRITE)
        if not case["second"]:
            return dict(out=out, dy_dx=ctx, dx=dx, grads=state["grads"])
        second, _ = enc.backward_backward_input(x, state["v"], dy, want_dL_ddLdy=True, mode=GRAD_ACCUMULATE)
        return dict(out=out, dy_dx=ctx, dx=dx, second=second, grads=state["grads"])
    if kind == "sdf_net":
        net = state["net"]
        ctx = net.forward(state["x"])
        loss = net.loss_backward(ctx)
        return dict(loss=loss, sdf=ctx["sdf"], normal=ctx["normal"], grid_grads=state["grid_grads"], mlp_grads=state["mlp_grads"])
    if kind == "field":
        net = state["net"]
        out = net.forward(state["coords"])
        net.backward(state["coords"], state["dl"])
        return dict(out=out, grads=state["grads"])
    if kind == "query":
        return getattr(state["net"], case["what"])(state["x"])
    if kind == "occupancy":
        occ = state["occ"]
        occ.update(state["trainer"]._field, case["n_uniform"], case["n_nonuniform"])
        return dict(density=occ.density_grid, bits=occ.bitfield, mean=occ.mean)
    if kind == "lattice":
        return density_on_grid(state["trainer"]._field, (case["rx"], case["ry"], case["rz"]), chunk=1 << 22)
    vertices, triangles, normals = marching_cubes(state["density"], 0.0)
    return dict(vertices=vertices, triangles=triangles, normals=normals)


# ---------------------------------------------------------------------------------------------------------------------
# what a call cannot do without
# ---------------------------------------------------------------------------------------------------------------------
# entries per level of the default encoding: 16 levels growing by 1.447 from 16, dense while they fit, at most 2^19
_ENTRIES = [min(-(-int(math.ceil(16 * 1.447 ** l - 1) + 1) ** 3 // 8) * 8, 1 << 19) for l in range(16)]
_SDF_FORWARD, _SDF_GRADIENT, _RGB_FORWARD = 8192, 8192, 16384                # flop a sample
_RGB_BACKWARD, _SDF_BACKWARD, _SDF_SECOND = 2 * 16384, 2 * 8192, 14336


def _touched(n):
    """Table entries that n points (about four new ones a point and level) meet: bytes of them are moved, not of the others."""
    return sum(e * (1 - math.exp(-4.0 * n / e)) for e in _ENTRIES)


def work(case):
    kind = case["kind"]
    table = 4 * sum(_ENTRIES)  # bytes of the fp16 table, and of its gradient
    if kind == "train":
        n = case["target"]
        marched = _rays(case) * (20 if case["trained"] else 52)
        # parameters, both moments and counters of what the batch met, read and written; the gradient written and read whole
        return dict(bytes=2 * _touched(n) * 32 + 2 * table,
                    flops=marched * (_SDF_FORWARD + _SDF_GRADIENT + _RGB_FORWARD) + n * (_RGB_BACKWARD + _SDF_BACKWARD + _SDF_SECOND))
    if kind in ("lattice", "mesh"):
        points = case["rx"] * case["ry"] * case["rz"]
        if kind == "lattice":
            return dict(bytes=4 * points + table, flops=_SDF_FORWARD * points)
        surface = 4 * math.pi * 0.09 * (case["rx"] * case["ry"] + case["ry"] * case["rz"] + case["rx"] * case["rz"]) / 2
        return dict(bytes=4 * points + surface * (24 + 24), flops=0)
    if kind == "occupancy":
        n = case["n_uniform"] + case["n_nonuniform"]
        return dict(bytes=min(table, 4 * _touched(n)) + 8 * GRID_CELLS + GRID_CELLS / 7, flops=_SDF_FORWARD * n)
    n = case["n"]
    if kind == "query":
        return dict(bytes=4 * _touched(n) + n * (12 + 32), flops=_SDF_FORWARD * n)
    rows = 12 + 64 + 384 + 64 + 12 if kind == "grid" else 0  # positions, features, Jacobian, their gradient, positions' gradient
    if kind == "grid":
        return dict(bytes=4 * _touched(n) + table + n * (rows + ((12 + 64) if case["second"] else 0)), flops=n * 16 * 8 * (30 if case["second"] else 20))
    if kind == "sdf_net":
        return dict(bytes=4 * _touched(n) + table + n * (12 + 2 + 12), flops=n * (_SDF_FORWARD + _SDF_GRADIENT + _SDF_BACKWARD + _SDF_SECOND))
    return dict(bytes=4 * _touched(n) + table + n * (28 + 32 + 32),
                flops=n * (_SDF_FORWARD + _SDF_GRADIENT + _RGB_FORWARD + _RGB_BACKWARD + _SDF_BACKWARD + _SDF_SECOND))


def tolerance(case):
    """fp16 activations and gradients through two or three layers; integers and the mesh's fp32 positions have no such excuse."""
    kind = case["kind"]
    if kind == "mesh":
        return dict(rel=1e-6, max=1e-3)
    if kind == "grid":
        return dict(rel=1e-3, max=0.05)  # fp32 interpolation, one rounding to fp16; table gradients are sums of such roundings
    if kind == "occupancy":
        return dict(rel=2e-3, max=0.2, differ=1e-3)  # a cell's bit is a comparison with the mean density
    if kind in ("query", "lattice"):
        return dict(rel=2e-3, max=0.05)
    # a ReLU at zero may fall to either side: few single values of the gradients move by much
    return dict(rel=5e-3, max=0.9)
