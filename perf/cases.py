"""What a user of this framework has it do, as measurable cases.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)`
one more of the same ranges, `prepare(case, seed)` what a program holds before
the call, `run(state)` one pass through the public entry points, `work(case)`
the bytes and operations the pass cannot do without, `exact(case, seed)` the
same outputs from plain torch in 64 bits (positions in the grid, the march and
the sample points follow the fp32 definition of the method, everything after
them is computed in fp64).

Fields are spheres with a rough hash-grid part (geometric initialisation plus
seeded noise on the weights and the table), seen by a ring of cameras: the
state training converges to, without training it.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from supernormal_amd import nerfacc
from supernormal_amd.fields import SDFNetwork, SingleVarianceNetwork
from supernormal_amd.fused import FlatParams
from supernormal_amd.scene import Dataset
from supernormal_amd.step import SyncFreeStep
from supernormal_amd.tcnn import Encoding

DEV = "cuda"

# the grids and networks of the repository's three workloads
WORKLOADS = {
    "sphere128": dict(levels=8, features=2, log2_t=15, base=16, scale=1.5, hidden=32, layers=1),
    "tbs612": dict(levels=16, features=2, log2_t=19, base=16, scale=1.38, hidden=64, layers=2),
    "prims1024": dict(levels=16, features=2, log2_t=21, base=16, scale=1.38, hidden=64, layers=2),
}


# --------------------------------------------------------------------------- #
# the cases
# --------------------------------------------------------------------------- #
def _step(net, batch, res, cap, step_size, active, precision, method, size, views):
    return dict(kind="step", **WORKLOADS[net], batch=batch, res=res, cap=cap, step_size=step_size,
                active=active, precision=precision, method=method, width=size[0], height=size[1],
                views=views)


def _sdf(kind, net, n, precision, active=None):
    w = WORKLOADS[net]
    return dict(kind=kind, **w, n=n, precision=precision,
                active=w["levels"] if active is None else active)


def listed():
    return [
        # the smallest training run (256 patches, 8 levels, one hidden layer,
        # fp32, <= 32 samples per ray): what launches and latency cost
        dict(_step("sphere128", 256, 64, 32, 1e-2, 8, "fp32", "dfd", (128, 128), 4),
             name="step_small"),
        # the headline iteration: 18 432 rays, the end of the schedule
        dict(_step("tbs612", 2048, 128, 1024, 1e-3, 16, "fp16", "dfd", (612, 512), 2),
             name="step_late"),
        # the analytic-gradient iteration in the middle of the schedule (10 of
        # 16 levels active, a larger step)
        dict(_step("tbs612", 2048, 128, 1024, 2.5e-3, 10, "fp16", "ad", (612, 512), 2),
             name="step_ad_mid"),
        # the large single-object run: 73 728 rays, T = 2^21, 256^3 cells
        dict(_step("prims1024", 8192, 256, 1024, 1e-3, 16, "fp16", "dfd", (1024, 1024), 1),
             name="step_large"),
        # the field trained through autograd (the host-synchronised iteration
        # and a caller's own losses): matrix-core MLP, a late iteration's points
        dict(_sdf("sdf_train", "tbs612", 1204317, "fp16"), name="sdf_train_fp16"),
        # the same in fp32 (the default precision), an early iteration's points
        dict(_sdf("sdf_train", "tbs612", 299593, "fp32"), name="sdf_train_fp32"),
        # the analytic x-gradient and its double backward through autograd, fp32
        dict(_sdf("sdf_grad", "tbs612", 160003, "fp32"), name="sdf_grad_fp32"),
        # field queries without gradient over a 128^3 grid's cells: occupancy
        # updates and mesh extraction
        dict(_sdf("sdf_eval", "tbs612", 1 << 21, "fp16"), name="sdf_eval_grid"),
        # the tinycudann drop-in on its own, gradients to table and positions
        dict(kind="encode", **{k: v for k, v in WORKLOADS["tbs612"].items()
                               if k not in ("hidden", "layers")}, n=262147, name="encode_train"),
        # the NerfAcc drop-ins on their own: marching a batch of rays ...
        dict(kind="march", rays=2048, res=128, step_size=1e-3, cap=0, name="march"),
        # ... patch weights, accumulation and their backward ...
        dict(kind="weights", patches=2048, patch=9, mean=64, name="patch_weights"),
        # ... and the occupancy grid's update after the warm-up
        dict(kind="occ", res=128, name="occ_update"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "sdf_train", "sdf_train", "sdf_grad", "sdf_eval", "encode",
                       "march", "weights", "occ"])
    if kind == "step":
        net = rng.choice(["sphere128", "tbs612", "tbs612"])
        w = WORKLOADS[net]
        small = net == "sphere128"
        return _step(net, _log(rng, 100, 600) if small else _log(rng, 256, 2500),
                     rng.choice([32, 64]) if small else rng.choice([64, 128]),
                     rng.choice([24, 32, 48]) if small else 1024,
                     1e-2 if small else 10 ** rng.uniform(-3.0, -2.0),
                     rng.randint(2, w["levels"]), rng.choice(["fp16", "fp32"]),
                     rng.choice(["dfd", "dfd", "ad"]), (128, 128) if small else (306, 256), 2)
    if kind in ("sdf_train", "sdf_grad", "sdf_eval"):
        net = rng.choice(["sphere128", "tbs612"])
        hi = {"sdf_train": 1200000, "sdf_grad": 300000, "sdf_eval": 4000000}[kind]
        return _sdf(kind, net, _log(rng, 1000, hi),
                    "fp32" if kind == "sdf_grad" else rng.choice(["fp16", "fp32"]),
                    rng.randint(1, WORKLOADS[net]["levels"]))
    if kind == "encode":
        return dict(kind="encode", levels=rng.choice([8, 14, 16]), features=rng.choice([1, 2, 2, 4]),
                    log2_t=rng.randint(15, 20), base=rng.choice([16, 32]),
                    scale=rng.choice([1.3195079107728942, 1.38, 1.5]), n=_log(rng, 1000, 400000))
    if kind == "march":
        return dict(kind="march", rays=_log(rng, 100, 9000), res=rng.choice([64, 100, 128]),
                    step_size=10 ** rng.uniform(-3.0, -2.0), cap=rng.choice([0, 0, 96, 1024]))
    if kind == "weights":
        return dict(kind="weights", patches=_log(rng, 100, 9000), patch=rng.choice([1, 4, 9, 25]),
                    mean=_log(rng, 4, 100))
    return dict(kind="occ", res=rng.randint(24, 127))


# --------------------------------------------------------------------------- #
# inputs (plain torch, from the seed alone)
# --------------------------------------------------------------------------- #
RADIUS = 0.36  # covers about a fifth of a view


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _grid(case):
    """Per level: (scale, resolution, table entries, first entry, dense)."""
    out, off = [], 0
    l2 = math.log2(float(np.float32(case["scale"])))
    for lv in range(case["levels"]):
        sc = float(np.float32(2.0 ** (lv * l2) * case["base"] - 1.0))
        res = math.ceil(sc) + 1
        size = min((min(res ** 3, 0xffffffff // 2) + 7) // 8 * 8, 1 << case["log2_t"])
        out.append((sc, res, size, off, res ** 3 <= size))
        off += size
    return out, off


def _table(case, g):
    """Table values whose contribution to the gradient is alike on every level."""
    grid, n = _grid(case)
    t = torch.rand(n, case["features"], generator=g, device=DEV) * 2 - 1
    for sc, _, size, off, _ in grid:
        t[off:off + size] *= 0.02 * grid[0][0] / sc
    return t.reshape(-1)


def _parameters(case, seed):
    """A field's parameters by state-dict name: a sphere's geometric
    initialisation, encoding columns and table as training leaves them."""
    g = _gen(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    H, n_hidden, E = case["hidden"], case["layers"], case["levels"] * case["features"]
    p = {"encoding.params": _table(case, g)}
    dims = [3 + E] + [H] * n_hidden + [1]
    for lv in range(len(dims) - 1):
        if lv == len(dims) - 2:
            W, b = math.sqrt(math.pi) / math.sqrt(H) + 1e-3 * rn(1, H), torch.full((1,), -RADIUS, device=DEV)
        else:
            W, b = rn(H, dims[lv]) * math.sqrt(2.0 / H), 1e-3 * rn(H)
            if lv == 0:
                W[:, 3:] = 0.05 * rn(H, E)
        p[f"lin{lv}.bias"] = b
        p[f"lin{lv}.weight_g"] = W.norm(dim=1, keepdim=True) * (1 + 0.01 * rn(W.shape[0], 1))
        p[f"lin{lv}.weight_v"] = W
    # slope 1 and the zero set at RADIUS, on the average over directions
    u = F.normalize(torch.randn(4096, 3, generator=g, device=DEV), dim=1)
    lo, hi = (_smooth(p, u * (RADIUS + h)).mean() for h in (-0.1, 0.1))
    p[f"lin{lv}.weight_g"] *= 0.2 / (hi - lo)
    p[f"lin{lv}.bias"] *= 0.2 / (hi - lo)
    p[f"lin{lv}.bias"] -= _smooth(p, u * RADIUS).mean()
    return p


def _smooth(p, x):
    """The field at x without its encoding columns, in fp32."""
    n = sum(k.endswith("bias") for k in p)
    for lv in range(n):
        v = p[f"lin{lv}.weight_v"]
        W = p[f"lin{lv}.weight_g"] * v / v.norm(dim=1, keepdim=True)
        x = F.linear(x, W[:, :x.shape[1]], p[f"lin{lv}.bias"])
        if lv < n - 1:
            x = F.softplus(x, beta=100)
    return x[:, 0]


def _points(n, seed, step=1e-3):
    """Sample points of 3x3 patches as the march gives them: runs of samples
    through the surface, the patch's 9 rays beside each other."""
    g = _gen(seed + 7)
    s = -(-n // 9)
    cnt = (16 + 110 * torch.rand(s // 16 + 1, generator=g, device=DEV)).long()
    ray = torch.repeat_interleave(torch.arange(len(cnt), device=DEV), cnt)[:s]
    j = torch.arange(s, device=DEV) - (torch.cumsum(cnt, 0) - cnt)[ray]
    u = F.normalize(torch.randn(len(cnt), 3, generator=g, device=DEV), dim=1)
    d = F.normalize(-u + 0.6 * (torch.rand(len(cnt), 3, generator=g, device=DEV) - 0.5), dim=1)
    e1 = F.normalize(torch.linalg.cross(d, u.roll(1, 1)), dim=1)
    e2 = torch.linalg.cross(d, e1)
    k = torch.arange(9, device=DEV)
    off = (e1[:, None] * (k % 3 - 1)[None, :, None] + e2[:, None] * (k // 3 - 1)[None, :, None]) * 1.6e-3
    c = RADIUS * u[ray] + d[ray] * (j * step - 0.03)[:, None]
    return (c[:, None] + off[ray]).reshape(-1, 3)[:n].contiguous()


def _cells(n, seed):
    """Jittered cells of a grid over [-1, 1]^3 in order (the first n)."""
    g = _gen(seed + 7)
    r = math.ceil(n ** (1 / 3))
    i = torch.arange(n, device=DEV)
    c = torch.stack([i // (r * r), i // r % r, i % r], 1).float()
    return (c + torch.rand(n, 3, generator=g, device=DEV)) / r * 2 - 1


def _views(case, seed):
    """Normal maps [n,H,W,3], masks, intrinsics and poses (numpy, fp32 maps on
    the GPU) of the sphere seen by cameras on a ring."""
    n, W, H = case["views"], case["width"], case["height"]
    f = 0.5 * W / math.tan(math.radians(35.0) / 2)
    K = np.eye(4)
    K[0, 0], K[1, 1], K[0, 2], K[1, 2] = f, f, (W - 1) / 2.0, (H - 1) / 2.0
    rot = np.random.RandomState(seed % (1 << 31)).uniform(0, 2 * math.pi)
    poses, normals, masks = [], [], []
    ys, xs = torch.meshgrid(torch.arange(H, device=DEV, dtype=torch.float64),
                            torch.arange(W, device=DEV, dtype=torch.float64), indexing="ij")
    pix = torch.stack([(xs - K[0, 2]) / f, (ys - K[1, 2]) / f, torch.ones_like(xs)], -1)
    pix = pix / pix.norm(dim=-1, keepdim=True)
    g = _gen(seed + 3)
    for i in range(n):
        el, az = math.radians((0.0, 25.0, -25.0, 45.0)[i % 4]), rot + 2 * math.pi * i / n
        eye = 2.5 * np.array([math.cos(el) * math.sin(az), -math.sin(el), -math.cos(el) * math.cos(az)])
        fwd = -eye / np.linalg.norm(eye)
        right = np.cross(fwd, [0.0, 1.0, 0.0])
        right /= np.linalg.norm(right)
        P = np.eye(4)
        P[:3, 0], P[:3, 1], P[:3, 2], P[:3, 3] = right, np.cross(fwd, right), fwd, eye
        o = torch.as_tensor(eye, device=DEV)
        d = pix @ torch.as_tensor(P[:3, :3], device=DEV).T
        b = (d * o).sum(-1)
        disc = b * b - (o @ o - RADIUS ** 2)
        m = disc > 0
        nrm = (o + d * (-b - disc.clamp_min(0).sqrt())[..., None]) / RADIUS
        nrm = nrm + 0.02 * torch.randn(nrm.shape, generator=g, device=DEV)
        normals.append(torch.where(m[..., None], F.normalize(nrm, dim=-1), 0.0).float())
        masks.append(m.float())
        poses.append(P)
    return torch.stack(normals), torch.stack(masks), np.stack([K] * n), np.stack(poses)


def _occupied(p, res):
    """Occupied cells of the field's smooth part (bool [res]^3)."""
    a = (torch.arange(res, device=DEV) + 0.5) / res * 2 - 1
    x = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    return (torch.sigmoid(-80 * _smooth(p, x)) > 0.1).reshape(res, res, res)


def _rays(case, seed):
    """Centre rays of random pixels towards the sphere's neighbourhood, with
    the unit sphere's entry and exit, and its occupied cells.  A case has one
    scene; the seed turns it (a permutation of the axes) and orders the rays,
    so that the number of samples is the case's."""
    n, res = case["rays"], case["res"]
    g = _gen(n * 1000 + res)
    o = 2.5 * F.normalize(torch.randn(n, 3, generator=g, device=DEV), dim=1)
    d = F.normalize(1.2 * (torch.rand(n, 3, generator=g, device=DEV) - 0.5) - o, dim=1)
    b, c = (o * d).sum(1), (o * o).sum(1) - 1
    q = (b * b - c).clamp_min(0).sqrt()
    a = (torch.arange(res, device=DEV) + 0.5) / res * 2 - 1
    r = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).norm(dim=-1)
    bump = 0.05 * torch.randn(res, res, res, generator=g, device=DEV)
    near = -b - q + torch.rand(n, generator=g, device=DEV) * case["step_size"]
    occ = r + 0.1 * bump < RADIUS + 0.03
    turn = [(0, 1, 2), (1, 2, 0), (2, 0, 1), (0, 2, 1), (2, 1, 0), (1, 0, 2)][seed % 6]
    order = torch.randperm(n, generator=_gen(seed), device=DEV)
    pick = lambda t: t[order][:, turn].contiguous() if t.dim() == 2 else t[order]
    return pick(o), pick(d), pick(near), pick(q - b), occ.permute(turn).contiguous()


def _alphas(case, seed):
    """Opacities of patches' samples, ray indices, normals and the cotangents.
    A case has one distribution of samples per patch; the seed orders it."""
    n, P = case["patches"], case["patch"]
    g = _gen(n)
    r = lambda *s: torch.rand(*s, generator=g, device=DEV)
    cnt = torch.where(r(n) < 0.35, torch.zeros(n, device=DEV), -2 * case["mean"] * torch.log(1 - 0.999 * r(n))).long()
    g = _gen(seed)
    cnt = cnt[torch.randperm(n, generator=g, device=DEV)]
    ri = torch.repeat_interleave(torch.arange(n, device=DEV), cnt)
    s = len(ri)
    j = torch.arange(s, device=DEV) - (torch.cumsum(cnt, 0) - cnt)[ri]
    t = (j.float() / cnt[ri].float() - 0.25)[:, None] * 12 + r(s, P)
    a = 0.14 * torch.sigmoid(t)
    nrm = F.normalize(torch.randn(s, P, 3, generator=g, device=DEV), dim=-1)
    g_w = torch.randn(n, P, 1, generator=g, device=DEV) / (n * P)
    return a[..., None].contiguous(), ri, nrm, g_w, torch.randn(n, P, 3, generator=g, device=DEV) / (n * P)


def _occ(case, seed):
    """An occupancy grid's values and the cells of an update after the warm-up:
    a quarter of all drawn uniformly, and as many occupied ones."""
    g = _gen(seed)
    n = case["res"] ** 3
    occs = torch.rand(n, generator=g, device=DEV) ** 6
    occupied = torch.nonzero(occs > 0.1)[:, 0]
    cells = torch.cat([torch.randint(n, (n // 4,), generator=g, device=DEV),
                       occupied[torch.randint(len(occupied), (n // 4,), generator=g, device=DEV)]])
    return occs, cells, torch.rand(len(cells), 3, generator=g, device=DEV)


def _density(x):
    """The update's evaluation function: a sphere's occupancy."""
    return torch.sigmoid(-80 * (x.norm(dim=-1, keepdim=True) - RADIUS))


def _cotangents(n, seed):
    g = _gen(seed + 5)
    a = torch.randn(n, generator=g, device=DEV) * 1e-6
    return a, torch.randn(n, 3, generator=g, device=DEV) * 1e-6


# --------------------------------------------------------------------------- #
# prepare, run
# --------------------------------------------------------------------------- #
def _encoding_config(case):
    return dict(otype="HashGrid", n_levels=case["levels"], n_features_per_level=case["features"],
                log2_hashmap_size=case["log2_t"], base_resolution=case["base"],
                per_level_scale=case["scale"])


def _network(case, params):
    net = SDFNetwork(d_in=3, d_out=1, d_hidden=case["hidden"], n_layers=case["layers"],
                     skip_in=[-1], bias=RADIUS, weight_norm=True, input_concat=True,
                     encoding_config=_encoding_config(case)).to(DEV)
    net.load_state_dict(params)
    net.mlp_precision = case["precision"]
    for _ in range(case["active"]):
        net.increase_bandwidth()
    return net


VARIANCE = 0.5  # inv_s = exp(10 v) = 148


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind)
    if kind == "step":
        params = _parameters(case, seed)
        net = _network(case, params)
        var = SingleVarianceNetwork(VARIANCE).to(DEV)
        grid = nerfacc.OccupancyGrid([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0], case["res"]).to(DEV)
        grid.binary.copy_(_occupied(params, case["res"]))
        flat = FlatParams(list(net.parameters()) + list(var.parameters()), DEV)
        normals, masks, K, poses = _views(case, seed)
        ds = Dataset.from_arrays(normals, masks, K, poses, DEV)
        st.update(net=net, var=var, flat=flat, step_size=case["step_size"], step=SyncFreeStep(
            net, var, grid, flat, ds, case["batch"], 3, case["cap"], precision=case["precision"],
            seed=seed, method=case["method"], device=DEV))
    elif kind in ("sdf_train", "sdf_grad", "sdf_eval"):
        st["net"] = _network(case, _parameters(case, seed))
        st["x"] = (_cells if kind == "sdf_eval" else _points)(case["n"], seed)
        st["a"], st["v"] = _cotangents(case["n"], seed)
    elif kind == "encode":
        st["enc"] = Encoding(3, _encoding_config(case)).to(DEV)
        with torch.no_grad():
            st["enc"].params.copy_(_table(case, _gen(seed)))
        st["x"] = _points(case["n"], seed).requires_grad_(True)
        st["g"] = torch.randn(case["n"], case["levels"] * case["features"], generator=_gen(seed + 5),
                              device=DEV) * 1e-6
    elif kind == "march":
        o, d, near, far, occ = _rays(case, seed)
        st["grid"] = nerfacc.OccupancyGrid([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0], case["res"]).to(DEV)
        st["grid"].binary.copy_(occ)
        st.update(o=o, d=d, near=near, far=far, step_size=case["step_size"], cap=case["cap"])
    elif kind == "weights":
        a, st["ri"], st["nrm"], st["g_w"], st["g_n"] = _alphas(case, seed)
        st["alpha"], st["n"] = a.requires_grad_(True), case["patches"]
    else:
        occs, st["cells"], st["jitter"] = _occ(case, seed)
        st["grid"] = nerfacc.OccupancyGrid([-1.0, -1.0, -1.0, 1.0, 1.0, 1.0], case["res"]).to(DEV)
        st["grid"].occs.copy_(occs)
    return st


def run(st):
    kind = st["kind"]
    if kind == "step":
        # one iteration in graph mode; the next one's march runs ahead, as in training
        losses = st["step"].step(LR, st["step_size"], next_step_size=st["step_size"])
        return dict(losses=losses, grad={k: p.grad for k, p in st["net"].named_parameters()},
                    grad_variance=st["var"].variance.grad,
                    weights={k: p.data for k, p in st["net"].named_parameters()},
                    variance=st["var"].variance.data)
    if kind in ("sdf_train", "sdf_grad"):
        net = st["net"]
        named = list(net.named_parameters())
        if kind == "sdf_train":
            f, g = net.fused_sdf(st["x"]), None
            grads = torch.autograd.grad([f], [p for _, p in named], [st["a"]])
        else:
            f, g = net.fused_sdf_and_gradient(st["x"])
            grads = torch.autograd.grad([f, g], [p for _, p in named], [st["a"], st["v"]])
        return dict(sdf=f, gradient=g, grad={k: t for (k, _), t in zip(named, grads)})
    if kind == "sdf_eval":
        with torch.no_grad():
            return st["net"].fused_sdf(st["x"])
    if kind == "encode":
        out = st["enc"](st["x"])
        gx, gp = torch.autograd.grad([out], [st["x"], st["enc"].params], [st["g"]])
        return dict(out=out, gx=gx, gp=gp)
    if kind == "march":
        ri, t0, t1 = nerfacc.ray_marching(st["o"], st["d"], t_min=st["near"], t_max=st["far"],
                                          grid=st["grid"], render_step_size=st["step_size"],
                                          max_samples_per_ray=st["cap"])
        return dict(ri=ri, t0=t0, t1=t1)
    if kind == "weights":
        w = nerfacc.render_weight_from_alpha_patch_based(st["alpha"], st["ri"], n_rays=st["n"])
        ws = nerfacc.accumulate_along_rays_patch_based(w, st["ri"], n_patches=st["n"])
        cn = nerfacc.accumulate_along_rays_patch_based(w, st["ri"], values=st["nrm"],
                                                       n_patches=st["n"])
        ga, = torch.autograd.grad([ws, cn], [st["alpha"]], [st["g_w"], st["g_n"]])
        return dict(w=w, ws=ws, cn=cn, ga=ga)
    st["grid"].update_cells(st["cells"], st["jitter"], _density)
    return dict(occs=st["grid"].occs, binary=st["grid"].binary)


# a learning rate of the warm-up's first steps: a pass leaves the field's
# surface where it is, so that repeated passes are the same work
LR = 1e-7


# --------------------------------------------------------------------------- #
# what a pass cannot do without
# --------------------------------------------------------------------------- #
def _visible(case):
    """Visible centre samples of a step, about: a fifth of the rays meet the
    sphere, from the shell in front of it to where the transmittance ends
    (or the sample capacity)."""
    depth = 0.03 + 18.4 / math.exp(10 * VARIANCE)
    return 0.22 * case["batch"] * min(1.3 * depth / case["step_size"], case["cap"])


def work(case):
    kind = case["kind"]
    if kind == "march":
        m = 0.5 * case["rays"] * min(0.7 / case["step_size"], case["cap"] or 1e9)
        return dict(bytes=case["rays"] * 32 + m * 16 + case["res"] ** 3, flops=m * 20)
    if kind == "weights":
        s = 1.3 * case["patches"] * case["mean"]
        return dict(bytes=s * (case["patch"] * 24 + 8) + case["patches"] * case["patch"] * 32,
                    flops=s * case["patch"] * 24)
    if kind == "occ":
        n = case["res"] ** 3
        return dict(bytes=n * 9 + n // 2 * 20, flops=n * 20)
    E, f = case["levels"] * case["features"], case["features"]
    table = 4 * f * _grid(case)[1]
    if kind == "encode":
        n = case["n"]
        return dict(bytes=2 * table + n * (24 + 8 * E), flops=n * case["levels"] * 8 * (10 + 6 * f))
    H, A = case["hidden"], case["active"]
    mlp = 2 * ((3 + E) * H + (case["layers"] - 1) * H * H + H)
    enc = A * 8 * (8 + 2 * f)
    if kind == "sdf_eval":
        return dict(bytes=table + case["n"] * 16, flops=case["n"] * (mlp + enc))
    if kind == "sdf_train":
        return dict(bytes=2 * table + case["n"] * 20, flops=case["n"] * (3 * mlp + 2 * enc))
    if kind == "sdf_grad":
        return dict(bytes=2 * table + case["n"] * 44, flops=case["n"] * (8 * mlp + 5 * enc))
    n = 9 * _visible(case) * 1.02
    per = (8 * mlp + 5 * enc) if case["method"] == "ad" else (3 * mlp + 2 * enc)
    # parameters, gradients and moments of the optimiser, the patches' pixels
    return dict(bytes=8 * table + case["batch"] * 9 * 120, flops=n * per)


# --------------------------------------------------------------------------- #
# 64-bit results
# --------------------------------------------------------------------------- #
def _encode64(case, x, table, active):
    """The encoding of x [N,3] (fp64 holding fp32 values); the position in the
    grid is the method's fp32 one, its derivative the level's scale."""
    grid, _ = _grid(case)
    f, M = case["features"], 0xffffffff
    t = table.reshape(-1, f)
    out = []
    for lv, (sc, res, size, off, dense) in enumerate(grid):
        if lv >= active:
            out.append(torch.zeros(x.shape[0], f, dtype=torch.float64, device=x.device))
            continue
        p = (x.detach() * sc + 0.5).float()
        cell = torch.floor(p)
        fr = (p - cell).double()
        if x.requires_grad:
            fr = fr + sc * (x - x.detach())
        gi = cell.long() & M
        acc = 0.0
        for c in range(8):
            b = (c & 1, c >> 1 & 1, c >> 2 & 1)
            q = [gi[:, k] + b[k] & M for k in range(3)]
            if dense:
                i = (q[0] + (q[1] * res & M) + (q[2] * (res * res & M) & M) & M) % size
            else:
                i = (q[0] ^ (q[1] * 2654435761 & M) ^ (q[2] * 805459861 & M)) & (size - 1)
            w = 1.0
            for k in range(3):
                w = w * (fr[:, k] if b[k] else 1 - fr[:, k])
            acc = acc + w[:, None] * t.index_select(0, i + off)
        out.append(acc)
    return torch.cat(out, 1)


def _field64(case, p, x, active):
    h = torch.cat([x, _encode64(case, x, p["encoding.params"], active)], 1)
    n = case["layers"] + 1
    for lv in range(n):
        v = p[f"lin{lv}.weight_v"]
        h = F.linear(h, p[f"lin{lv}.weight_g"] * v / v.norm(dim=1, keepdim=True), p[f"lin{lv}.bias"])
        if lv < n - 1:
            h = F.softplus(h, beta=100)
    return h[:, 0]


def _leaves(params):
    return {k: v.double().requires_grad_(True) for k, v in params.items()}


CHUNK = 1 << 18


def _sdf64(case, p, x, want_gradient):
    """(sdf, gradient or None) of x, chunk by chunk, without a graph."""
    fs, gs = [], []
    for s in range(0, x.shape[0], CHUNK):
        xc = x[s:s + CHUNK].double()
        if want_gradient:
            xc.requires_grad_(True)
            f = _field64(case, p, xc, case["active"])
            gs.append(torch.autograd.grad(f.sum(), xc)[0])
        else:
            with torch.no_grad():
                f = _field64(case, p, xc, case["active"])
        fs.append(f.detach())
    return torch.cat(fs), torch.cat(gs) if want_gradient else None


def _backward64(case, p, x, a, v):
    """Gradients of sum a sdf (+ v . gradient) to the parameters, chunk by chunk."""
    for s in range(0, x.shape[0], CHUNK):
        xc = x[s:s + CHUNK].double()
        if v is not None:
            xc.requires_grad_(True)
        f = _field64(case, p, xc, case["active"])
        J = (a[s:s + CHUNK] * f).sum()
        if v is not None:
            J = J + (v[s:s + CHUNK] * torch.autograd.grad(f.sum(), xc, create_graph=True)[0]).sum()
        # (the last bias does not enter the gradient)
        for q, g in zip(p.values(), torch.autograd.grad(J, list(p.values()), allow_unused=True)):
            if g is not None:
                q.grad = g if q.grad is None else q.grad + g


def _march32(o, d, near, far, occ, step, cap):
    """The march of rays over [-1, 1]^3 (fp32, the method's operations): dense
    starts and ends [R, J] and counts."""
    R, res, f32 = o.shape[0], occ.shape[0], torch.float32
    st = torch.tensor(step, dtype=f32, device=DEV)
    inv = 1.0 / d
    t0 = near.clone()
    t1 = t0 + st
    tm = (t0 + t1) * 0.5
    j = torch.zeros(R, dtype=torch.int64, device=DEV)
    a0, a1 = [torch.zeros(R, cap, dtype=f32, device=DEV) for _ in range(2)]
    rows, sgn = torch.arange(R, device=DEV), torch.copysign(torch.ones_like(d), d)
    while True:
        act = (tm < far) & (j < cap)
        if not bool(act.any()):
            return a0, a1, j
        x = o + tm[:, None] * d
        u = (x + 1.0) * 0.5
        inside = ((x >= -1) & (x <= 1)).all(1)
        c = (torch.nan_to_num(u) * float(res)).int().clamp(0, res - 1).long()
        hit = act & inside & occ[c[:, 0], c[:, 1], c[:, 2]]
        k = j.clamp(max=cap - 1)
        a0[rows, k] = torch.where(hit, t0, a0[rows, k])
        a1[rows, k] = torch.where(hit, t1, a1[rows, k])
        j = j + hit.long()
        un = u * float(res)
        nb = torch.floor((un + 0.5) + 0.5 * sgn)
        dist = ((((nb - un) * inv) * (1.0 / res)) * 2.0).amin(1).clamp_min(0.0)
        target = torch.minimum(tm + dist, far)
        skip = act & ~hit
        tt, more = tm, skip
        while bool(more.any()):
            tt = torch.where(more, tt + st, tt)
            more = more & (tt < target)
        n0 = torch.where(skip, tt - st * 0.5, torch.where(hit, t1, t0))
        n1 = torch.where(skip, tt + st * 0.5, torch.where(hit, t1 + st, t1))
        tm = torch.where(skip, tt, torch.where(hit, (n0 + n1) * 0.5, tm))
        t0, t1 = n0, n1


def _sample32(case, seed):
    """The patches an iteration draws: fp32 rays, their marching planes, V^-1,
    normals, masks, and the centre rays' jittered entry and exit."""
    normals, masks, K, poses = _views(case, seed)
    g, B, W, H = _gen(seed), case["batch"], case["width"], case["height"]
    draw_ = lambda lo, hi: torch.randint(lo, hi, (B,), device=DEV, generator=g)
    cx, cy, sel = draw_(1, W - 2), draw_(1, H - 2), draw_(0, case["views"])
    u = torch.rand((B,), generator=g, device=DEV, dtype=torch.float32)
    k = torch.arange(9, device=DEV)
    xs, ys = cx[:, None] + k % 3 - 1, cy[:, None] + k // 3 - 1
    Ki = torch.inverse(torch.as_tensor(K, dtype=torch.float32, device=DEV))[sel][:, None]
    R = torch.as_tensor(poses, dtype=torch.float32, device=DEV)[sel][:, None]
    fx, fy = xs.float(), ys.float()
    p = torch.stack([(Ki[..., r, 0] * fx + Ki[..., r, 1] * fy) + Ki[..., r, 2] for r in range(3)], -1)
    p = p / torch.sqrt((p[..., 0] ** 2 + p[..., 1] ** 2) + p[..., 2] ** 2)[..., None]
    d = torch.stack([(R[..., r, 0] * p[..., 0] + R[..., r, 1] * p[..., 1]) + R[..., r, 2] * p[..., 2]
                     for r in range(3)], -1)
    o = R[..., :3, 3].expand(d.shape).contiguous()
    dot = lambda a, b: (a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1]) + a[..., 2] * b[..., 2]
    oc, dc = o[:, 4].contiguous(), d[:, 4].contiguous()
    aa, bb, cc = dot(dc, dc), 2.0 * dot(oc, dc), dot(oc, oc) - 1.0
    mid, q = 0.5 * (-bb) / aa, torch.sqrt(bb * bb - 4.0 * aa * cc) / (2.0 * aa)
    step = torch.tensor(case["step_size"], dtype=torch.float32, device=DEV)
    Rd, dd = R.double(), d.double()
    V = torch.stack([dd, Rd[..., :3, 0].expand(dd.shape), Rd[..., :3, 1].expand(dd.shape)], -2)
    return dict(o=o, d=d, oc=oc, dc=dc, near=(mid - q) + u * step, far=mid + q,
                plane=R[:, 0, :3, 2], vinv=torch.inverse(V), normal=normals[sel[:, None], ys, xs],
                mask=(masks[sel[:, None], ys, xs] > 0.5).double(), dot=dot)


def _alpha64(fs, fe, inv_s):
    c, e = torch.sigmoid(fs * inv_s), torch.sigmoid(fe * inv_s)
    return ((c - e + 1e-5) / (c + 1e-5)).clip(0.0, 1.0)


def _exclusive(a, dim):
    """Products of 1 - a before each sample along dim."""
    T = torch.cumprod(1 - a, dim)
    return torch.cat([torch.ones_like(T.narrow(dim, 0, 1)), T.narrow(dim, 0, T.shape[dim] - 1)], dim)


def _dense(flat, where):
    """Rows of a dense [B, J, ...] array from its valid entries' values."""
    out = torch.zeros(where.shape + flat.shape[1:], dtype=flat.dtype, device=flat.device)
    out[where] = flat
    return out


def _step64(case, seed):
    params = _parameters(case, seed)
    p = _leaves(params)
    q = _sample32(case, seed)
    B, J = case["batch"], case["cap"]
    t0, t1, cnt = _march32(q["oc"], q["dc"], q["near"], q["far"], _occupied(params, case["res"]),
                           case["step_size"], J)
    valid = torch.arange(J, device=DEV)[None] < cnt[:, None]

    def ends(t0, t1, valid):
        """Samples whose end is not the next sample's start."""
        nxt = torch.zeros_like(valid)
        nxt[:, :-1] = valid[:, 1:] & (t1[:, :-1] == t0[:, 1:])
        return valid & ~nxt

    def end_values(fs, flat_e, own):
        """A sample's end: its own value where `own`, else the next start's."""
        nxt = torch.cat([fs[:, 1:], fs[:, -1:]], 1)
        own_e = _dense(flat_e, own)
        return torch.where(own.reshape(own.shape + (1,) * (fs.dim() - 2)), own_e, nxt)

    var = torch.tensor(VARIANCE, dtype=torch.float32).double().to(DEV).requires_grad_(True)
    inv_s = torch.exp(10 * var).clip(1e-6, 1e6).detach().requires_grad_(True)
    # the visible samples of the centre rays
    own = ends(t0, t1, valid)
    at = lambda t, m: (q["oc"][:, None] + q["dc"][:, None] * t[..., None])[m]
    f, _ = _sdf64(case, p, torch.cat([at(t0, valid), at(t1, own)]), False)
    n = int(valid.sum())
    fs = _dense(f[:n], valid)
    a = torch.where(valid, _alpha64(fs, end_values(fs, f[n:], own), inv_s.detach()), 0.0)
    keep = valid & (_exclusive(a, 1) >= 1e-8)
    cnt = keep.sum(1)
    J = max(1, int(cnt.max()))
    order = torch.argsort((~keep).to(torch.int8), dim=1, stable=True)[:, :J]
    t0, t1 = t0.gather(1, order), t1.gather(1, order)
    valid = torch.arange(J, device=DEV)[None] < cnt[:, None]
    # the patches' samples: fp32 points on the marching planes
    own = ends(t0, t1, valid)
    dcn = q["dot"](q["dc"], q["plane"])[:, None, None]
    dkn = q["dot"](q["d"], q["plane"][:, None])[:, None]
    ts, te = (t0[..., None] * dcn) / dkn, (t1[..., None] * dcn) / dkn
    xs, xe = (q["o"][:, None] + q["d"][:, None] * t[..., None] for t in (ts, te))
    pts = torch.cat([xs[valid].reshape(-1, 3), xe[own].reshape(-1, 3)])
    S = int(valid.sum())
    ad = case["method"] == "ad"
    f, gp = _sdf64(case, p, pts, ad)
    f.requires_grad_(True)
    fs = _dense(f[:S * 9].reshape(-1, 9), valid)
    fe = end_values(fs, f[S * 9:].reshape(-1, 9), own)
    if ad:
        gp.requires_grad_(True)
        G = _dense(gp[:S * 9].reshape(-1, 9, 3), valid)
    else:
        shape = fs.shape[:2] + (3, 3)
        o, d = q["o"].double()[:, None], q["d"].double()[:, None]
        x = (o + d * ts.double()[..., None]).reshape(shape + (3,))
        h, w = (x[:, :, 1:] - x[:, :, :-1]).norm(dim=-1), (x[:, :, :, 1:] - x[:, :, :, :-1]).norm(dim=-1)
        g = fs.reshape(shape)
        dx = torch.stack([(g[..., 1] - g[..., 0]) / w[..., 0],
                          (g[..., 2] - g[..., 0]) / (w[..., 0] + w[..., 1]),
                          (g[..., 2] - g[..., 1]) / w[..., 1]], -1)
        dy = torch.stack([(g[:, :, 1] - g[:, :, 0]) / h[:, :, 0],
                          (g[:, :, 2] - g[:, :, 0]) / (h[:, :, 0] + h[:, :, 1]),
                          (g[:, :, 2] - g[:, :, 1]) / h[:, :, 1]], 2)
        dt = torch.where(valid[..., None], te.double() - ts.double(), 1.0)
        proj = torch.stack([(fe - fs) / dt, dx.reshape(fs.shape), dy.reshape(fs.shape)], -1)
        G = (q["vinv"][:, None] * proj[..., None, :]).sum(-1)
    v3 = valid[..., None]
    a = torch.where(v3, _alpha64(fs, fe, inv_s), 0.0)
    wt = a * _exclusive(a, 1)
    G = torch.where(v3[..., None], G, 0.0)
    ws, cn = wt.sum(1), (wt[..., None] * G).sum(1)
    m = q["mask"]
    l_n = (((cn - q["normal"].double()) * m[..., None]) ** 2).sum() / (m.sum() + 1e-5)
    l_m = F.binary_cross_entropy(ws.clip(1e-5, 1 - 1e-5), m)
    # (a sample's gradient is never exactly zero; the padding's is)
    nrm = torch.where(v3, (G ** 2).sum(-1), 1.0).sqrt()
    l_e = ((nrm - 1) ** 2).sum() / (S * 9)
    back = torch.autograd.grad(l_n + l_m + l_e, [f, inv_s] + ([gp] if ad else []))
    _backward64(case, p, pts, back[0], back[2] if ad else None)
    g_var = back[1] * 10 * inv_s.detach()
    adam = lambda w, g: w - LR * g / (g.abs() + 1e-8)  # the first step: m / sqrt(v) = g / |g|
    losses = torch.stack([l_n, l_m, l_e, back[1]]).detach()
    return dict(losses=losses, grad={k: w.grad for k, w in p.items()}, grad_variance=g_var,
                weights={k: adam(w.detach(), w.grad) for k, w in p.items()},
                variance=adam(var.detach(), g_var))


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _step64(case, seed)
    if kind in ("sdf_train", "sdf_grad", "sdf_eval"):
        p = _leaves(_parameters(case, seed))
        x = (_cells if kind == "sdf_eval" else _points)(case["n"], seed)
        f, g = _sdf64(case, p, x, kind == "sdf_grad")
        if kind == "sdf_eval":
            return f
        a, v = (t.double() for t in _cotangents(case["n"], seed))
        _backward64(case, p, x, a, v if kind == "sdf_grad" else None)
        return dict(sdf=f, gradient=g, grad={k: w.grad for k, w in p.items()})
    if kind == "encode":
        st = dict(x=_points(case["n"], seed).double().requires_grad_(True),
                  t=_table(case, _gen(seed)).double().requires_grad_(True))
        g = torch.randn(case["n"], case["levels"] * case["features"], generator=_gen(seed + 5),
                        device=DEV) * 1e-6
        out = _encode64(case, st["x"], st["t"], case["levels"])
        gx, gp = torch.autograd.grad([out], [st["x"], st["t"]], [g.double()])
        return dict(out=out.detach(), gx=gx, gp=gp)
    if kind == "weights":
        a, ri, nrm, g_w, g_n = (t.double() if t.is_floating_point() else t for t in _alphas(case, seed))
        a.requires_grad_(True)
        cnt = torch.bincount(ri, minlength=case["patches"])
        where = torch.arange(max(1, int(cnt.max())), device=DEV)[None] < cnt[:, None]
        A = _dense(a[..., 0], where)
        w = (A * _exclusive(A, 1))[where][..., None]
        acc = lambda s: torch.zeros((case["patches"],) + s.shape[1:], dtype=s.dtype,
                                    device=DEV).index_add(0, ri, s)
        ws, cn = acc(w), acc(w * nrm)
        ga, = torch.autograd.grad([ws, cn], [a], [g_w, g_n])
        return dict(w=w.detach(), ws=ws.detach(), cn=cn.detach(), ga=ga)
    if kind == "occ":
        occs, cells, jitter = _occ(case, seed)
        r = case["res"]
        c = torch.stack([cells // (r * r), cells // r % r, cells % r], 1).double()
        occ = _density((c + jitter.double()) / r * 2 - 1)[:, 0]
        new = torch.full((r ** 3,), -1.0, dtype=torch.float64, device=DEV).scatter_reduce(
            0, cells, occ, "amax")
        return dict(occs=torch.where(new >= 0, torch.maximum(occs.double() * 0.95, new), occs.double()),
                    binary=None)
    return None  # the march's samples are fp32 and compared as they are
