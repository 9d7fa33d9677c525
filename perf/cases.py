"""The work a user of this framework has it do, as cases that can be timed and compared.

Every case goes through the package's public entry points with what the path meets
in earnest: rays of look-at cameras at radius 3 around a unit-sphere scene, points
that are samples along those rays (neighbouring points share grid cells), and
networks that are past their geometric initialisation (every hash level and every
encoder column of the first layer takes part).  Ranges: 512 to 8192 rays a step, 96
samples a ray, hash grids of 2^14 to 2^22 entries with 2 to 8 features, every stage
of the coarse-to-fine schedule, float32 and bfloat16 compute.

    listed()            the cases that stand for each path
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the caller's program holds before the call
    run(state)          one pass
    work(case)          bytes and operations one pass cannot do without
    exact(case, seed)   the outputs in 64 bits, from plain torch
"""
import copy
import functools
import math
import random

import torch

from neuralangelo_amd import mesh, misc, nerf_util
from neuralangelo_amd.encoding import Encoding, growth_rate
from neuralangelo_amd.mcubes import lattice_marching_cubes
from neuralangelo_amd.model import Model, default_config

SAMPLES = 96      # samples per ray of the default configuration: 64 + 2 x 16
BACKGROUND = 32   # background samples per ray
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a viewer's or a debugging probe's query of the encoder alone: latency
        dict(name="encode_small_f32", op="encode", points=4096, log2_T=19, F=4, active=16,
             dtype="f32", backward=False),
        # the encoder as a drop-in for tcnn.Encoding in a float32 trainer
        dict(name="encode_grad_f32", op="encode", points=262147, log2_T=19, F=4, active=16,
             dtype="f32", backward=True),
        # the same at the full table and the full step's point count, bf16
        dict(name="encode_grad_bf16", op="encode", points=786432, log2_T=22, F=8, active=16,
             dtype="bf16", backward=True),
        # mesh extraction: the float32 field on one 128^3 block (+1 shared point per axis)
        dict(name="lattice_f32", op="lattice", nx=129, ny=129, nz=129, log2_T=22, F=8, active=16,
             dtype="f32"),
        # one 512-ray step of a float32 trainer (the reference's default batch): the SDF
        # field with its 4-tap gradients, forward and backward
        dict(name="field_f32", op="field", rays=512, log2_T=19, F=4, active=16, dtype="f32"),
        # the same in the middle of the coarse-to-fine schedule, bf16, with the Hessian
        dict(name="field_bf16", op="field", rays=2048, log2_T=21, F=8, active=9, dtype="bf16"),
        # the colour network of a full step, forward and backward
        dict(name="colour_bf16", op="colour", rays=8192, dtype="bf16"),
        # the background network of a 1024-ray step, forward and backward
        dict(name="background_bf16", op="background", rays=1024, dtype="bf16"),
        # the hierarchical sampling of a full step (coarse distances, two SDF passes)
        dict(name="sample_bf16", op="sample", rays=8192, log2_T=22, F=8, active=16, dtype="bf16"),
        # a preview image of 32 x 32 pixels, float32: one whole call with many small launches
        dict(name="render_f32", op="render", size=32, log2_T=19, F=4, dtype="f32"),
        # a whole training step (render, losses, gradients) over packed rays of uneven
        # sample counts at the full table, about as many samples as 8192 dense rays
        dict(name="train_bf16", op="train", rays=8192, log2_T=22, F=8, dtype="bf16"),
        # marching cubes over a whole extraction lattice in 128^3 blocks
        dict(name="mc_1024", op="mc", nx=1024, ny=1024, nz=1024, block=128, shapes=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["encode", "encode", "lattice", "field", "field", "colour", "background",
                     "sample", "render", "train", "mc"])
    dtype = rng.choice(["f32", "bf16"])
    log2_T = rng.choice([14, 17, 18, 19, 20, 21, 22])
    F = rng.choice([2, 4, 8])
    active = rng.randint(4, 16)
    if op == "encode":
        return dict(op=op, points=_log_int(rng, 512, 786432), log2_T=log2_T, F=F, active=active,
                    dtype=dtype, backward=rng.random() < 0.6)
    F = rng.choice([4, 8])
    if op == "lattice":
        n = [_log_int(rng, 24, 129) for _ in range(3)]
        return dict(op=op, nx=n[0], ny=n[1], nz=n[2], log2_T=log2_T, F=F, active=active,
                    dtype=dtype)
    if op == "field":
        return dict(op=op, rays=_log_int(rng, 64, 4096 if dtype == "bf16" else 2048),
                    log2_T=log2_T, F=F, active=active, dtype=dtype)
    if op == "colour":
        return dict(op=op, rays=_log_int(rng, 64, 8192 if dtype == "bf16" else 2048), dtype=dtype)
    if op == "background":
        return dict(op=op, rays=_log_int(rng, 64, 8192 if dtype == "bf16" else 2048), dtype=dtype)
    if op == "sample":
        return dict(op=op, rays=_log_int(rng, 64, 8192), log2_T=log2_T, F=F, active=active,
                    dtype=dtype)
    if op == "render":
        return dict(op=op, size=rng.randint(12, 96), log2_T=log2_T, F=F, dtype=dtype)
    if op == "train":
        return dict(op=op, rays=_log_int(rng, 256, 8192), log2_T=log2_T, F=F, dtype="bf16")
    n = [_log_int(rng, 64, 768) for _ in range(3)]
    return dict(op=op, nx=n[0], ny=n[1], nz=n[2], block=rng.choice([64, 128, 0]),
                shapes=rng.randint(3, 32))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed, salt=0):
    return torch.Generator(device=_device()).manual_seed(int(seed) * 1000003 + salt)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=_device())


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=_device())


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


@functools.lru_cache(maxsize=2)
def _base_encoding(log2_T, F, dtype):
    cfg = dict(otype="HashGrid", n_levels=16, n_features_per_level=F, log2_hashmap_size=log2_T,
               base_resolution=32, per_level_scale=growth_rate(5, 11, 16))
    return Encoding(3, cfg, dtype=DTYPES[dtype]).to(_device())


@functools.lru_cache(maxsize=2)
def _base_model(log2_T, F, dtype, background, size):
    cfg_data = dict(train=dict(image_size=[size, size]), val=dict(image_size=[size, size]))
    m = Model(default_config(log2_T=log2_T, F=F, background=background), cfg_data=cfg_data,
              compute_dtype=DTYPES[dtype])
    m.cfg_render["rand_rays"] = 1024
    return m.to(_device())


def _fill_table(params, enc, g):
    """Table values of a network in training: a level's features shrink with its cells,
    so every level adds about the same slope to the field."""
    F = enc.n_features_per_level
    for lv in range(enc.n_levels):
        a, b = enc.offsets[lv] * F, enc.offsets[lv + 1] * F
        amp = 0.5 / enc.resolutions[lv]
        params[a:b].uniform_(-amp, amp, generator=g)


def _gates(g, n):
    """Biases of trained ReLU layers: a unit is on or off for most inputs of a scene."""
    b = _randn(g, n)
    return b.sign() * (0.25 + 0.25 * b.abs())


def _model(case, g, background=False, active=16, size=32):
    """A copy of the configured model with weights of a network in training."""
    m = copy.deepcopy(_base_model(case.get("log2_T", 14), case.get("F", 8), case["dtype"],
                                  background, size))
    with torch.no_grad():
        _fill_table(m.neural_sdf.tcnn_encoding.params, m.neural_sdf.tcnn_encoding, g)
        hid = 256
        l0, l1 = m.neural_sdf.mlp.linears
        for lin in (l0, l1):
            lin.weight_v.copy_(_randn(g, *lin.weight_v.shape) * math.sqrt(2 / hid))
            lin.weight_g.copy_(lin.weight_v.norm(dim=1, keepdim=True)
                               * (0.9 + 0.2 * _rand(g, hid, 1)))
            lin.bias.copy_(0.02 * _randn(g, hid))
        head = m.neural_sdf.mlp.linear_sdf
        head.weight.copy_(math.sqrt(math.pi / hid) * (1 + 0.05 * _randn(g, 1, hid)))
        head.bias.fill_(-0.5)
        for lin in m.neural_rgb.mlp.linears:
            k = lin.in_features
            lin.weight_v.copy_((2 * _rand(g, *lin.weight_v.shape) - 1) * math.sqrt(3 / k))
            lin.weight_g.copy_(lin.weight_v.norm(dim=1, keepdim=True))
            lin.bias.copy_(_gates(g, lin.bias.shape[0]))
        m.s_var.fill_(4.0)
        if background:
            for stack in (m.background_nerf.mlp_feat, m.background_nerf.mlp_rgb):
                for lin in stack.linears:
                    k = lin.in_features
                    lin.weight.copy_((2 * _rand(g, *lin.weight.shape) - 1) * math.sqrt(3 / k))
                    lin.bias.copy_(_gates(g, lin.bias.shape[0]))
    sdf = m.neural_sdf
    sdf.active_levels = sdf.anneal_levels = active
    sdf.set_normal_epsilon()
    m.progress = 1.0
    return m.train()


def _rays(n, g, aim=0.9):
    """Rays of cameras at radius 3 towards points within `aim` of the scene's middle."""
    cams = _unit(_randn(g, max(1, n // 512), 3)) * 3.0
    pick = torch.arange(n, device=_device()) % cams.shape[0]
    center = cams[pick].contiguous()
    at = _unit(_randn(g, n, 3)) * (aim * _rand(g, n, 1) ** (1 / 3))
    return center, _unit(at - center)


def _sorted_dists(n_rays, n, g):
    """Sorted distances across the unit sphere, denser near the surface half way."""
    u = torch.sort(_rand(g, n_rays, n), dim=1).values
    u = 0.5 + 0.5 * (2 * u - 1).sign() * (2 * u - 1).abs() ** 1.5
    return 2.1 + 1.8 * u


def _ray_points(rays, g, n=SAMPLES):
    center, unit = _rays(rays, g)
    d = _sorted_dists(rays, n, g)
    return center, unit, d, (center[:, None] + unit[:, None] * d[..., None])


def _upstream(g, *shape):
    """Upstream gradients as rendering gives them: a few samples of a ray carry most, and
    neighbours pull the same way."""
    return (1 + _randn(g, *shape)) * _rand(g, *shape[:-1], 1) ** 4 * 1e-3


def _camera(g):
    """World-to-camera pose [1,3,4] of a camera at radius 3 looking at the origin."""
    c = _unit(_randn(g, 3)) * 3.0
    fwd = -_unit(c)
    right = _unit(torch.linalg.cross(fwd, torch.tensor([0.0, 0.0, 1.0], device=c.device)))
    rot = torch.stack([right, torch.linalg.cross(fwd, right), fwd], dim=0)
    return torch.cat([rot, -(rot * c).sum(-1, keepdim=True)], dim=1)[None].contiguous()


def _intrinsics(size):
    f = 0.5 * size / math.tan(math.radians(50.0) / 2)
    return torch.tensor([[[f, 0.0, size / 2], [0.0, f, size / 2], [0.0, 0.0, 1.0]]],
                        device=_device())


def _lattice_axes(n):
    intv = 2.0 / 1024
    return [-1.0 + 0.37 + intv * torch.arange(k, dtype=torch.float32, device=_device()) for k in n]


def _packed(rays, g):
    """Rays with 0 to 192 samples each, about 96 on average; one in eight is empty."""
    center, unit = _rays(rays, g)
    at = torch.arange(rays, device=_device())
    counts = torch.where(at % 8 == 0, 0, (at * 220 // rays).clamp(max=192))
    counts = counts[torch.randperm(rays, generator=g, device=_device())]
    offsets = torch.zeros(rays + 1, dtype=torch.int32, device=_device())
    offsets[1:] = counts.cumsum(0).to(torch.int32)
    ray = torch.repeat_interleave(torch.arange(rays, device=_device()), counts)
    near, far = nerf_util.intersect_with_sphere(center, unit)
    lo = near.nan_to_num(2.0)[ray, 0]
    hi = far.nan_to_num(4.0)[ray, 0]
    u = _rand(g, ray.numel())
    order = torch.argsort(ray.double() + 0.999 * u.double())
    return center, unit, offsets, (lo + u[order] * (hi - lo)).contiguous()


def _mc_volume(case, g):
    """A signed distance volume, a union of spheres with fine surface detail.  The shapes
    belong to the case (so its mesh has as many vertices for every seed); the seed scales
    every lattice value, as another network of the same object would."""
    dev, n = _device(), (case["nx"], case["ny"], case["nz"])
    top = max(n)
    ax = [(2.0 / top) * torch.arange(k, dtype=torch.float32, device=dev) - k / top for k in n]
    vol = torch.full(n, 4.0, device=dev)
    x, y, z = ax[0][:, None, None], ax[1][None, :, None], ax[2][None, None, :]
    shape = random.Random("%d %d %d %d" % (*n, case["shapes"]))
    for k in range(case["shapes"]):
        c = [shape.uniform(-0.8, 0.8) * m / top for m in n]
        d2 = (x - c[0]) ** 2 + (y - c[1]) ** 2
        vol = torch.minimum(vol, (d2 + (z - c[2]) ** 2).sqrt_().sub_(shape.uniform(0.06, 0.3)))
    w = shape.uniform(40.0, 80.0)
    vol += 0.004 * (torch.sin(w * x) * torch.sin(w * y)) * torch.sin(w * z)
    return vol.mul_(torch.rand(n, generator=g, device=dev).add_(0.5)), ax


def prepare(case, seed):
    g = _generator(seed)
    op = case["op"]
    s = dict(op=op, case=case)
    if op == "encode":
        enc = copy.deepcopy(_base_encoding(case["log2_T"], case["F"], case["dtype"]))
        with torch.no_grad():
            _fill_table(enc.params, enc, g)
        enc.active_levels = case["active"]
        rays = -(-case["points"] // SAMPLES)
        pts = _ray_points(rays, g)[3].reshape(-1, 3)[:case["points"]]
        s.update(enc=enc, x=((pts + 2.0) / 4.0).contiguous())
        if case["backward"]:
            s["dy"] = _upstream(g, case["points"], enc.n_output_dims).to(enc.dtype)
    elif op == "lattice":
        m = _model(case, g, active=case["active"])
        s.update(sdf=m.neural_sdf, axes=_lattice_axes((case["nx"], case["ny"], case["nz"])))
    elif op == "field":
        m = _model(case, g, active=case["active"])
        pts = _ray_points(case["rays"], g)[3].reshape(-1, 3)
        P = pts.shape[0]
        s.update(sdf=m.neural_sdf, pts=pts, hess=case["dtype"] == "bf16",
                 dsdf=_upstream(g, P, 1), dgrad=0.1 * _upstream(g, P, 3),
                 dhess=1e-4 * _upstream(g, P, 3),
                 dfeat=_upstream(g, P, 280).to(DTYPES[case["dtype"]])[:, :256])
    elif op == "colour":
        m = _model(case, g)
        R = case["rays"]
        _, unit, _, pts = _ray_points(R, g)
        # the features as the SDF network hands them over: columns of the colour rows
        rows = (0.3 * _randn(g, R * SAMPLES, 280).abs()).to(DTYPES[case["dtype"]])
        s.update(rgb=m.neural_rgb, pts=pts, unit=unit,
                 feats=rows[:, :256].unflatten(0, (R, SAMPLES)).requires_grad_(True),
                 normals=_randn(g, R, SAMPLES, 3).requires_grad_(True),
                 dout=_upstream(g, R, SAMPLES, 3))
    elif op == "background":
        m = _model(case, g, background=True)
        R = case["rays"]
        center, unit = _rays(R, g)
        inv = 1.0 - (torch.arange(BACKGROUND, device=_device()) + _rand(g, R, BACKGROUND)) / BACKGROUND
        pts = center[:, None] + unit[:, None] * (3.9 / (inv + 1e-5))[..., None]
        s.update(bg=m.background_nerf, pts=pts, unit=unit[:, None],
                 drgb=_upstream(g, R, BACKGROUND, 3), ddensity=_upstream(g, R, BACKGROUND, 1)[..., 0])
    elif op == "sample":
        m = _model(case, g, active=case["active"])
        # rays that meet the surface, as under a foreground mask
        center, unit = _rays(case["rays"], g, aim=0.4)
        near, far, _ = m.get_dist_bounds(center, unit)
        s.update(model=m, center=center, unit=unit, near=near, far=far,
                 rands=_rand(g, case["rays"], 64))
    elif op == "render":
        m = _model(case, g, size=case["size"])
        s.update(model=m, data=dict(pose=_camera(g), intr=_intrinsics(case["size"]),
                                    idx=torch.zeros(1, dtype=torch.long, device=_device())))
    elif op == "train":
        m = _model(case, g)
        center, unit, offsets, dists = _packed(case["rays"], g)
        s.update(model=m, center=center, unit=unit, offsets=offsets, dists=dists,
                 target=_rand(g, case["rays"], 3))
    elif op == "mc":
        vol, ax = _mc_volume(case, g)
        s.update(vol=vol, axes=ax, intv=2.0 / max(vol.shape))
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _clear(module):
    for p in module.parameters():
        p.grad = None


def _grads(module):
    return {k: p.grad for k, p in module.named_parameters() if p.grad is not None}


def _run_encode(s):
    enc = s["enc"]
    if not s["case"]["backward"]:
        with torch.no_grad():
            return enc(s["x"])
    enc.params.grad = None
    out = enc(s["x"])
    out.backward(s["dy"])
    return dict(out=out, grad=enc.params.grad)


def _run_lattice(s):
    return mesh.lattice_sdf(s["sdf"].sdf_nograd, s["axes"], s["axes"][0].device)


def _run_field(s):
    net = s["sdf"]
    _clear(net)
    sdf, feat, taps, delta = net.forward_with_taps(s["pts"])
    grad, hess = net.gradients_from_taps(taps, sdf, sdf, s["hess"], delta)
    outs, ups = [sdf, feat, grad], [s["dsdf"], s["dfeat"], s["dgrad"]]
    if s["hess"]:
        outs, ups = outs + [hess], ups + [s["dhess"]]
    torch.autograd.backward(outs, ups)
    return dict(sdf=sdf, feat=feat, gradient=grad, hessian=hess, grads=_grads(net))


def _run_colour(s):
    net = s["rgb"]
    _clear(net)
    s["feats"].grad = s["normals"].grad = None
    rgb = net(s["pts"], s["normals"], s["unit"], s["feats"], None, normals_are_gradients=True)
    rgb.backward(s["dout"])
    return dict(rgb=rgb, dfeats=s["feats"].grad, dnormals=s["normals"].grad, grads=_grads(net))


def _run_background(s):
    net = s["bg"]
    _clear(net)
    rgb, density = net(s["pts"], s["unit"], None)
    torch.autograd.backward([rgb, density], [s["drgb"], s["ddensity"]])
    return dict(rgb=rgb, density=density, grads=_grads(net))


def _run_sample(s):
    return s["model"].sample_dists_all(s["center"], s["unit"], s["near"], s["far"],
                                       stratified=True, rands=s["rands"])


def _run_render(s):
    out = s["model"].inference(s["data"])
    return {k: out[k] for k in ("rgb_map", "opacity_map", "depth_map", "normal_map")}


def _run_train(s):
    m = s["model"]
    _clear(m)
    out = m.render_rays_packed(s["center"], s["unit"], s["dists"], s["offsets"])
    eik, curv = misc.sdf_losses(out["gradients"], out["hessians"], out["outside"])
    loss = 3 * torch.nn.functional.l1_loss(out["rgb"], s["target"]) + 0.1 * eik + 5e-4 * curv
    loss.backward()
    return dict(loss=loss, rgb=out["rgb"], weights=out["weights"], grads=_grads(m))


def _run_mc(s):
    return lattice_marching_cubes(s["vol"], s["case"]["block"], 0.0, axes=s["axes"],
                                  intv=s["intv"])


def run(state):
    return globals()["_run_" + state["op"]](state)


# ---------------------------------------------------------------------------
# bytes and operations
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _levels(log2_T):
    """Per level: float32 scale, resolution, first entry, entries, whether it is hashed
    (Instant-NGP's level table, 16 levels from 2^5 to 2^11)."""
    import numpy as np
    log2s = np.float32(np.log2(np.float64(np.float32(growth_rate(5, 11, 16)))))
    out, first = [], 0
    for lv in range(16):
        e = np.float32(np.exp2(np.float64(np.float32(np.float32(lv) * log2s))))
        scale = np.float32(np.float32(e * np.float32(32)) - np.float32(1))
        res = int(np.ceil(scale)) + 1
        size = min((res ** 3 + 7) // 8 * 8, 1 << log2_T)
        out.append((float(scale), res, first, size, res ** 3 > size))
        first += size
    return out, first


def _entries(points, log2_T, active):
    """Table entries that `points` samples along rays touch, each counted once (neighbours
    share corners: about two entries a point and level)."""
    return sum(min(2 * points, size) for _, _, _, size, _ in _levels(log2_T)[0][:active])


def _lattice_entries(n, log2_T, active):
    """Table entries that a block of lattice points 1/2048 of the volume apart touches."""
    total = 0
    for _, res, _, size, _ in _levels(log2_T)[0][:active]:
        total += min(size, math.prod(k * res // 2048 + 2 for k in n))
    return total


def _packed_samples(rays):
    return sum(min(i * 220 // rays, 192) for i in range(rays) if i % 8)


def work(case):
    op, b = case["op"], 2 if case.get("dtype") == "bf16" else 4
    if op == "mc":
        n = case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=4.0 * n, flops=0.0)
    if op == "colour":
        P = case["rays"] * SAMPLES
        per = 278 * 256 + 3 * 256 * 256 + 256 * 3
        return dict(bytes=P * (12.0 + 2 * 256 * b + 24 + 24), flops=6.0 * P * per)
    if op == "background":
        P = case["rays"] * BACKGROUND
        per = 84 * 256 + 5 * 256 * 256 + 340 * 256 + 256 * 257 + 272 * 128 + 128 * 3
        return dict(bytes=P * (12.0 + 2 * 16), flops=6.0 * P * per)
    L, F, T = 16, case["F"], case["log2_T"]
    act = case.get("active", 16)
    width = L * F
    params = _levels(T)[1] * F
    if op == "encode":
        P = case["points"]
        e = _entries(P, T, act) * F
        n = P * (12.0 + width * b) + e * b
        if case["backward"]:
            n += P * (width * b) + 4.0 * params
        return dict(bytes=n, flops=2.0 * 8 * P * act * F * (2 if case["backward"] else 1))
    layer0 = (width + 3) * 256
    if op == "lattice":
        P = case["nx"] * case["ny"] * case["nz"]
        e = _lattice_entries((case["nx"], case["ny"], case["nz"]), T, act)
        return dict(bytes=4.0 * P + e * F * b, flops=2.0 * P * (layer0 + 256))
    if op == "sample":
        P = case["rays"] * 80
        return dict(bytes=case["rays"] * (24.0 + 8 + 256 + 4 * SAMPLES)
                    + _entries(P, T, act) * F * b, flops=2.0 * P * (layer0 + 256))
    field = 5 * layer0 + 256 * 256 + 5 * 256
    if op == "field":
        P = case["rays"] * SAMPLES
        e = _entries(P, T, act) * F
        n = P * (12.0 + 2 * (4 + 256 * b + 12)) + e * b + 4.0 * params
        return dict(bytes=n + (24.0 * P if case["dtype"] == "bf16" else 0), flops=6.0 * P * field)
    colour = 278 * 256 + 3 * 256 * 256 + 256 * 3
    if op == "render":
        R = case["size"] ** 2
        P = R * SAMPLES
        return dict(bytes=R * 32.0 + _entries(5 * P, T, 16) * F * b,
                    flops=2.0 * (R * 80 * (layer0 + 256) + P * (field + colour)))
    P = _packed_samples(case["rays"])
    e = _entries(P, T, 16) * F
    return dict(bytes=P * 8.0 + case["rays"] * 48.0 + e * b + 4.0 * params,
                flops=6.0 * P * (field + colour))


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
_TAPS = ((1, -1, -1), (-1, -1, 1), (-1, 1, -1), (1, 1, 1))


class _Lookup64(torch.autograd.Function):
    """table[i], adding the rows' gradients to table.grad in place (plain indexing would
    make a gradient of the whole table for every corner); `tag` only ties it to the graph."""

    @staticmethod
    def forward(ctx, tag, table, i):
        ctx.table, ctx.i = table, i
        return table[i]

    @staticmethod
    def backward(ctx, dy):
        if ctx.table.grad is None:
            ctx.table.grad = torch.zeros_like(ctx.table)
        ctx.table.grad.index_add_(0, ctx.i, dy)
        return torch.zeros((), dtype=dy.dtype, device=dy.device), None, None


def _encode64(u, table, log2_T, active):
    """Hash encoding [P, 16 F] of unit-cube points u (float64) from the table [entries, F]."""
    F = table.shape[1]
    tag = torch.zeros((), dtype=u.dtype, device=u.device, requires_grad=True)
    out = []
    for lv, (scale, res, first, size, hashed) in enumerate(_levels(log2_T)[0]):
        if lv >= active:
            out.append(torch.zeros(u.shape[0], F, dtype=u.dtype, device=u.device))
            continue
        pos = u * scale + 0.5
        cell = pos.floor()
        t = pos - cell
        cell = cell.long() & 0xffffffff
        acc = 0
        for c in range(8):
            x, y, z = [(cell[:, d] + ((c >> d) & 1)) & 0xffffffff for d in range(3)]
            if hashed:
                i = (x ^ ((y * 2654435761) & 0xffffffff) ^ ((z * 805459861) & 0xffffffff)) % size
            else:
                i = ((x + y * res + z * (res * res)) & 0xffffffff) % size
            w = 1
            for d in range(3):
                w = w * (t[:, d] if (c >> d) & 1 else 1 - t[:, d])
            acc = acc + w[:, None] * _Lookup64.apply(tag, table, first + i)
        out.append(acc)
    return torch.cat(out, dim=1)


def _softplus64(x):
    return torch.nn.functional.softplus(x, beta=100, threshold=1e9)


class _Net64:
    """The networks of a model in float64, by plain torch, on its own parameter copies."""

    def __init__(self, model, active=16):
        self.p = {k: v.detach().double().requires_grad_(True) for k, v in model.named_parameters()}
        enc = model.neural_sdf.tcnn_encoding
        self.table = enc.params.detach().double().view(-1, enc.n_features_per_level)
        self.T, self.active = enc.log2_hashmap_size, active
        self.eps = float(model.neural_sdf.normal_eps) / math.sqrt(3)

    def weight(self, name):
        v = self.p[name + ".weight_v"]
        return v * (self.p[name + ".weight_g"] / v.norm(dim=1, keepdim=True))

    def enc(self, x):
        return _encode64((x + 2.0) / 4.0, self.table, self.T, self.active)

    def sdf(self, x, feat=False):
        m = "neural_sdf.mlp."
        h = torch.cat([x, self.enc(x)], dim=1) @ self.weight(m + "linears.0").t()
        h = _softplus64(h + self.p[m + "linears.0.bias"])
        sdf = h @ self.p[m + "linear_sdf.weight"].t() + self.p[m + "linear_sdf.bias"]
        if not feat:
            return sdf
        f = _softplus64(h @ self.weight(m + "linears.1").t() + self.p[m + "linears.1.bias"])
        return sdf, f

    def gradients(self, x, sdf):
        k = torch.tensor(_TAPS, dtype=torch.float64, device=x.device)
        s = [self.sdf(x + k[i] * self.eps) for i in range(4)]
        grad = sum(k[i] * s[i] for i in range(4)) / (4 * self.eps)
        trace = ((s[0] + s[1] + s[2] + s[3]) / 2 - 2 * sdf) / self.eps ** 2
        return grad, trace.expand(-1, 3) / 3

    def colour(self, x, view, normal, feat):
        h = torch.cat([x, _sh64(view), normal, feat], dim=1)
        for i in range(5):
            n = "neural_rgb.mlp.linears.%d" % i
            h = h @ self.weight(n).t() + self.p[n + ".bias"]
            h = h.relu() if i < 4 else h.sigmoid()
        return h

    def grads(self, prefix=""):
        if self.table.grad is not None:
            self.p["neural_sdf.tcnn_encoding.params"].grad = self.table.grad.view(-1)
        return {k[len(prefix):]: v.grad for k, v in self.p.items()
                if k.startswith(prefix) and v.grad is not None}


def _sh64(d):
    """Real spherical harmonics to degree 3."""
    x, y, z = d.unbind(-1)
    pi = math.pi
    a, b = math.sqrt(3 / (4 * pi)), math.sqrt(15 / (4 * pi))
    c, e = math.sqrt(35 / (32 * pi)), math.sqrt(21 / (32 * pi))
    f, q = math.sqrt(105 / (4 * pi)), math.sqrt(7 / (16 * pi))
    xx, yy, zz = x * x, y * y, z * z
    return torch.stack([
        torch.full_like(x, 0.5 / math.sqrt(pi)), -a * y, a * z, -a * x, b * x * y, -b * y * z,
        math.sqrt(5 / (16 * pi)) * (2 * zz - xx - yy), -b * x * z, b / 2 * (xx - yy),
        -c * y * (3 * xx - yy), f * x * y * z, -e * y * (4 * zz - xx - yy),
        q * z * (2 * zz - 3 * xx - 3 * yy), -e * x * (4 * zz - xx - yy), f / 2 * z * (xx - yy),
        -c * x * (xx - 3 * yy)], dim=-1)


def _pieces(n, step):
    return [slice(i, min(i + step, n)) for i in range(0, n, step)]


def _exact_encode(s, case):
    enc, x = s["enc"], s["x"].double()
    table = enc.params.detach().double().view(-1, case["F"])
    out = []
    for k in _pieces(x.shape[0], 1 << 16):
        o = _encode64(x[k], table, case["log2_T"], case["active"])
        if case["backward"]:
            o.backward(s["dy"][k].double())
        out.append(o.detach())
    out = torch.cat(out)
    return dict(out=out, grad=table.grad.view(-1)) if case["backward"] else out


@torch.no_grad()
def _exact_lattice(s, case):
    net = _Net64(s["model64"], case["active"])
    x = torch.stack(torch.meshgrid(*s["axes"], indexing="ij"), dim=-1).double()
    f = x.view(-1, 3)
    return torch.cat([net.sdf(f[k]) for k in _pieces(f.shape[0], 1 << 16)]).view(x.shape[:-1])


def _exact_field(s, case):
    net, pts = _Net64(s["model64"], case["active"]), s["pts"].double()
    got = []
    for k in _pieces(pts.shape[0], 1 << 14):
        sdf, feat = net.sdf(pts[k], feat=True)
        grad, hess = net.gradients(pts[k], sdf)
        loss = (sdf * s["dsdf"][k].double()).sum() + (feat * s["dfeat"][k].double()).sum() \
            + (grad * s["dgrad"][k].double()).sum()
        if s["hess"]:
            loss = loss + (hess * s["dhess"][k].double()).sum()
        loss.backward()
        got.append([t.detach() for t in (sdf, feat, grad, hess)])
    sdf, feat, grad, hess = [torch.cat(t) for t in zip(*got)]
    return dict(sdf=sdf, feat=feat, gradient=grad, hessian=hess if s["hess"] else None,
                grads=net.grads("neural_sdf."))


def _exact_colour(s, case):
    net = _Net64(s["model64"])
    P = case["rays"] * SAMPLES
    pts, unit = s["pts"].double().view(P, 3), s["unit"].double().repeat_interleave(SAMPLES, 0)
    got = []
    for k in _pieces(P, 1 << 16):
        feats = s["feats"].detach().reshape(P, 256)[k].double().requires_grad_(True)
        raw = s["normals"].detach().view(P, 3)[k].double().requires_grad_(True)
        rgb = net.colour(pts[k], unit[k], torch.nn.functional.normalize(raw, dim=-1), feats)
        rgb.backward(s["dout"].view(P, 3)[k].double())
        got.append((rgb.detach(), feats.grad, raw.grad))
    rgb, df, dn = [torch.cat(t).view(case["rays"], SAMPLES, -1) for t in zip(*got)]
    return dict(rgb=rgb, dfeats=df, dnormals=dn, grads=net.grads("neural_rgb."))


def _exact_background(s, case):
    net = _Net64(s["model64"])
    P = case["rays"] * BACKGROUND
    pts, unit = s["pts"].double().view(P, 3), s["unit"].double().expand_as(s["pts"]).reshape(P, 3)
    freq = math.pi * 2.0 ** torch.arange(10, dtype=torch.float64, device=pts.device)
    got = []
    for k in _pieces(P, 1 << 16):
        r = pts[k].norm(dim=-1, keepdim=True)
        q = torch.cat([pts[k] / r, 1 / r], dim=-1)
        a = q[..., None] * freq
        x = torch.cat([q, torch.stack([a.sin(), a.cos()], dim=-2).reshape(q.shape[0], -1)], dim=-1)
        h = x
        for i in range(8):
            n = "background_nerf.mlp_feat.linears.%d" % i
            h = (torch.cat([h, x], dim=-1) if i == 4 else h) @ net.p[n + ".weight"].t() \
                + net.p[n + ".bias"]
            h = h.relu() if i < 7 else h
        density = torch.nn.functional.softplus(h[:, 0], threshold=1e9)
        c = torch.cat([h[:, 1:].relu(), _sh64(unit[k])], dim=-1)
        for i in range(2):
            n = "background_nerf.mlp_rgb.linears.%d" % i
            c = c @ net.p[n + ".weight"].t() + net.p[n + ".bias"]
            c = c.sigmoid() if i else c.relu()
        loss = (c * s["drgb"].view(P, 3)[k].double()).sum() \
            + (density * s["ddensity"].view(P)[k].double()).sum()
        loss.backward()
        got.append((c.detach(), density.detach()))
    rgb, density = [torch.cat(t) for t in zip(*got)]
    return dict(rgb=rgb.view(case["rays"], BACKGROUND, 3),
                density=density.view(case["rays"], BACKGROUND),
                grads=net.grads("background_nerf."))


def _front64(alphas):
    """alpha_i times the product of (1 - alpha_j) over the samples before it."""
    t = torch.cumprod(1 - alphas, dim=-1)
    return alphas * torch.cat([torch.ones_like(t[..., :1]), t[..., :-1]], dim=-1)


def _resample64(d, s, inv_s, n):
    """One hierarchical round: n distances drawn from the weights of the SDF values s."""
    step = d[:, 1:] - d[:, :-1]
    cos = (s[:, 1:] - s[:, :-1]) / (step + 1e-5)
    cos = torch.minimum(torch.cat([torch.zeros_like(cos[:, :1]), cos[:, :-1]], dim=1), cos)
    mid = 0.5 * (s[:, 1:] + s[:, :-1])
    a = torch.sigmoid((mid - 0.5 * cos * step) * inv_s)
    b = torch.sigmoid((mid + 0.5 * cos * step) * inv_s)
    w = _front64(((a - b) / (a + 1e-5)).clamp(0, 1))
    cdf = torch.cumsum(w / w.sum(1, keepdim=True).clamp_min(1e-12), dim=1)
    cdf = torch.cat([torch.zeros_like(cdf[:, :1]), cdf], dim=1)
    u = ((torch.arange(n, dtype=d.dtype, device=d.device) + 0.5) / n).expand(d.shape[0], n)
    i = torch.searchsorted(cdf, u.contiguous(), right=True)
    lo, hi = (i - 1).clamp(min=0), i.clamp(max=cdf.shape[1] - 1)
    t = (u - cdf.gather(1, lo)) / (cdf.gather(1, hi) - cdf.gather(1, lo) + 1e-8)
    return d.gather(1, lo) + t * (d.gather(1, hi) - d.gather(1, lo))


def _sample64(net, center, unit, near, far, u):
    """64 stratified distances and two rounds of 16 more, sorted [R, 96]."""
    d = (torch.arange(64, dtype=center.dtype, device=center.device) + u) / 64 * (far - near) + near
    at = lambda t: net.sdf((center[:, None] + unit[:, None] * t[..., None]).view(-1, 3)).view(t.shape)  # noqa: E731
    s = at(d)
    for k in range(2):
        fine = _resample64(d, s, 64 * 2 ** k, 16)
        both, order = torch.cat([d, fine], dim=1).sort(dim=1, stable=True)
        if k == 0:
            s = torch.cat([s, at(fine)], dim=1).gather(1, order)
        d = both
    return d


@torch.no_grad()
def _exact_sample(s, case):
    net = _Net64(s["model64"], case["active"])
    c, v, near, far, u = [s[k].double() for k in ("center", "unit", "near", "far", "rands")]
    return torch.cat([_sample64(net, c[k], v[k], near[k], far[k], u[k])
                      for k in _pieces(c.shape[0], 1024)])[..., None]


def _alphas64(inv_s, view, sdf, grad, step):
    """NeuS alphas past the end of the cosine annealing."""
    cos = -(-(view * grad).sum(-1)).relu()
    a = torch.sigmoid((sdf - 0.5 * cos * step) * inv_s)
    b = torch.sigmoid((sdf + 0.5 * cos * step) * inv_s)
    return ((a - b) / (a + 1e-5)).clamp(0, 1)


def _bounds64(c, v):
    cv = (c * v).sum(-1, keepdim=True)
    root = (cv ** 2 - ((c * c).sum(-1, keepdim=True) - 1)).sqrt()
    outside = root.isnan()
    near = torch.where(outside, torch.ones_like(cv), (-cv - root).relu())
    return near, torch.where(outside, torch.full_like(cv, 1.2), -cv + root), outside


@torch.no_grad()
def _exact_render(s, case):
    net, n = _Net64(s["model64"]), case["size"]
    pose, intr = s["data"]["pose"][0].double(), s["data"]["intr"][0].double()
    at = torch.arange(n, dtype=torch.float64, device=pose.device) + 0.5
    y, x = torch.meshgrid(at, at, indexing="ij")
    cam = torch.stack([x, y, torch.ones_like(x)], dim=-1).view(-1, 3) @ intr.inverse().t()
    rot, t = pose[:, :3], pose[:, 3]
    ray = cam @ rot
    centers = (-t @ rot).expand_as(ray)
    maps = []
    for k in _pieces(n * n, 256):
        c, v = centers[k], _unit(ray[k])
        near, far, outside = _bounds64(c, v)
        d = _sample64(net, c, v, near, far, 0.5)
        R, N = d.shape
        pts = (c[:, None] + v[:, None] * d[..., None]).view(-1, 3)
        view = v[:, None].expand(R, N, 3)
        sdf, feat = net.sdf(pts, feat=True)
        grad, _ = net.gradients(pts, sdf)
        rgb = net.colour(pts, view.reshape(-1, 3), torch.nn.functional.normalize(grad, dim=-1),
                         feat).view(R, N, 3)
        sdf = torch.where(outside, torch.full_like(d, 1000.0), sdf.view(R, N))
        step = torch.cat([d, far], dim=1)[:, 1:] - d
        w = _front64(_alphas64(net.p["s_var"].exp(), view, sdf, grad.view(R, N, 3), step))
        total = lambda q: (q * w[..., None]).sum(1)  # noqa: E731
        maps.append((total(rgb), w.sum(1, keepdim=True),
                     total(d[..., None]) / ray[k].norm(dim=-1, keepdim=True),
                     -total(grad.view(R, N, 3)) @ rot.t()))
    rgb, opacity, depth, normal = [torch.cat(t).view(1, n, n, -1).movedim(-1, 1)
                                   for t in zip(*maps)]
    return dict(rgb_map=rgb, opacity_map=opacity, depth_map=depth, normal_map=normal)


def _exact_train(s, case):
    net = _Net64(s["model64"])
    off = s["offsets"].long()
    counts, R, S = off[1:] - off[:-1], off.numel() - 1, int(off[-1])
    c_all, v_all, d_all = s["center"].double(), s["unit"].double(), s["dists"].double()
    rgbs, weights, total = [], [], 0
    for k in _pieces(R, 128):
        n, a = counts[k], int(off[k.start])
        r = torch.repeat_interleave(torch.arange(n.numel(), device=n.device), n)
        c, v, d = c_all[k], v_all[k], d_all[a:a + r.numel()]
        _, far, outside = _bounds64(c, v)
        pts, out = c[r] + v[r] * d[:, None], outside[r]
        sdf, feat = net.sdf(pts, feat=True)
        sdf = torch.where(out, torch.full_like(sdf, 1000.0), sdf)
        grad, hess = net.gradients(pts, sdf)
        rgb = net.colour(pts, v[r], torch.nn.functional.normalize(grad, dim=-1), feat)
        last = torch.ones_like(r, dtype=torch.bool)
        last[:-1] = r[1:] != r[:-1]
        step = torch.where(last, far[r, 0], torch.cat([d[1:], d[:1]])) - d
        alpha = _alphas64(net.p["s_var"].exp(), v[r], sdf[:, 0], grad, step)
        pad = torch.zeros(n.numel(), max(1, int(n.max())), dtype=alpha.dtype, device=alpha.device)
        at = torch.arange(r.numel(), device=r.device) - (off[k] - a)[r]
        w = _front64(pad.index_put((r, at), alpha))[r, at]
        ray = torch.zeros(n.numel(), 3, dtype=w.dtype, device=w.device).index_add(
            0, r, rgb * w[:, None])
        inside = (~out[:, 0]).double()
        eik = ((grad.norm(dim=-1) - 1) ** 2 * inside).sum() / S
        curv = (hess.sum(-1).abs() * inside).sum() / S
        loss = 3 * (ray - s["target"][k].double()).abs().sum() / (3 * R) + 0.1 * eik + 5e-4 * curv
        loss.backward()
        total = total + loss.detach()
        rgbs.append(ray.detach())
        weights.append(w.detach())
    return dict(loss=total, rgb=torch.cat(rgbs), weights=torch.cat(weights), grads=net.grads())


def exact(case, seed):
    if case["op"] == "mc":
        return None  # whole numbers, and vertices that the 64-bit bound holds
    s = prepare(case, seed)
    if case["op"] == "encode":
        return _exact_encode(s, case)
    s["model64"] = s.get("model") or _whole(s, case, seed)
    return globals()["_exact_" + case["op"]](s, case)


def _whole(s, case, seed):
    """The model that prepare() took the case's network from."""
    return _model(case, _generator(seed), background=case["op"] == "background",
                  active=case.get("active", 16))
