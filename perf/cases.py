"""The work a user of this package has it do, as cases that can be prepared, run and checked.

A case is a dict of plain values; ``kind`` names the path and the other entries its
sizes, types and options.  Every path goes through the package's public Python entry
points: the drop-in modules and functions a training or rendering program calls
(HashGridEncoder, nerf_mlp, NeRF, march_rays, integrate_rays, render_rays_inference)
and the Trainer's step.

Inputs follow what the paths meet in use: encoder and field points are consecutive
samples of rays at the marcher's step (2 sqrt 3 / 1024), occupancy grids are a few
balls of 128^3 cells, camera rays come from a sphere of radius 4 with the 800x800 /
1111 px camera's field of view, and the trainer steps on views of the 8-blob scene.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from jaxngp_amd import volrend
from jaxngp_amd.encoders import HashGridEncoder
from jaxngp_amd.nerfs import MLP_LAYERS, N_PARAMS, NeRF, nerf_mlp
from jaxngp_amd.renderer import make_near_far_from_bound, make_rays_worldspace, render_rays_inference
from jaxngp_amd.scene import BlobScene, Camera, look_at_poses, make_views
from jaxngp_amd.train import TrainConfig, Trainer

G = 128  # occupancy grid cells per axis
DIAG = 1024  # marching steps per diagonal
STEP = 2 * math.sqrt(3.0) / DIAG  # the marcher's step at bound 1
MLP_FLOPS = 2 * sum(a * b for _, _, a, b in MLP_LAYERS)  # per sample, forward


def listed():
    return [
        # The training batch's table lookup and its gradient through the drop-in encoder:
        # 2^18 ray samples, the field's grid (L 16, F 2, T 2^19), f32.
        {"name": "encoder_train_f32", "kind": "encoder", "points": 1 << 18, "log2_T": 19, "dtype": "f32"},
        # The same on the half-precision path, with a batch that is no multiple of anything.
        {"name": "encoder_ragged_f16", "kind": "encoder", "points": 77_777, "log2_T": 19, "dtype": "f16"},
        # The smallest encoder calls: a few rays' samples (debugging, fine-tuning on few rays).
        {"name": "encoder_small_f32", "kind": "encoder", "points": 1_023, "log2_T": 19, "dtype": "f32"},
        # The field's MLPs, forward and backward, on the training batch.
        {"name": "mlp_train", "kind": "mlp", "samples": 1 << 18},
        # ... and on a handful of ragged samples, where launches count.
        {"name": "mlp_small", "kind": "mlp", "samples": 1_237},
        # Density/colour queries of a trained field without autograd (mesh extraction,
        # baking, evaluation): a large f32 block, and a small ragged half-precision one.
        {"name": "field_query_f32", "kind": "field", "points": (1 << 20) + 13, "dtype": "f32"},
        {"name": "field_query_f16_small", "kind": "field", "points": 9_001, "dtype": "f16"},
        # The training marcher at the reference's batch shape (n_rays = total_samples = 2^18).
        {"name": "march_train", "kind": "march", "rays": 1 << 18, "samples": 1 << 18},
        # Compositing and its gradient: 4,096 ragged rays of up to 128 samples, about 2^18 slots.
        {"name": "integrate_train", "kind": "integrate", "rays": 1 << 12, "max_samples": 128},
        # The whole training step (rays, march, field, compositing, loss, backward, Adam,
        # grid cadence) at the benchmark's batch, f32.
        {"name": "train_step_f32", "kind": "train", "samples": 1 << 18, "precision": "fp32", "guided": False},
        # The same on the half-precision path with proposal-placed samples.
        {"name": "train_step_guided_f16", "kind": "train", "samples": 1 << 18, "precision": "fp16", "guided": True},
        # One 800x800 frame of the ray-pool renderer, f32 field.
        {"name": "render_800_f32", "kind": "render", "size": 800, "dtype": "f32"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["encoder", "mlp", "field", "march", "integrate", "train", "render"])
    if kind == "encoder":
        return {"kind": kind, "points": _log_uniform(rng, 500, 1 << 18), "log2_T": rng.choice([17, 19, 19, 20]),
                "dtype": rng.choice(["f32", "f32", "f16"])}
    if kind == "mlp":
        return {"kind": kind, "samples": _log_uniform(rng, 500, 1 << 18)}
    if kind == "field":
        return {"kind": kind, "points": _log_uniform(rng, 2_000, 1 << 20), "dtype": rng.choice(["f32", "f16"])}
    if kind == "march":
        s = _log_uniform(rng, 1 << 13, 1 << 18)
        return {"kind": kind, "rays": _log_uniform(rng, 500, s), "samples": s}
    if kind == "integrate":
        return {"kind": kind, "rays": _log_uniform(rng, 200, 1 << 12), "max_samples": rng.randint(16, 512)}
    if kind == "train":
        return {"kind": kind, "samples": _log_uniform(rng, 1 << 14, 1 << 18), "precision": rng.choice(["fp32", "fp16"]),
                "guided": rng.random() < 0.4}
    return {"kind": "render", "size": _log_uniform(rng, 64, 640), "dtype": rng.choice(["f32", "f32", "f16"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _ray_samples(n, gen):
    """n points in [-1, 1]^3 that are runs of 192 consecutive marching samples, and the
    rays' unit directions per point."""
    dev = _dev()
    per = 192
    rays = -(-n // per)
    centre = (torch.rand(rays, 3, generator=gen, device=dev) - 0.5) * 1.1
    d = torch.randn(rays, 3, generator=gen, device=dev)
    d = d / torch.linalg.norm(d, dim=-1, keepdim=True)
    t = (torch.arange(per, device=dev) - per / 2) * STEP
    xyz = centre[:, None, :] + t[None, :, None] * d[:, None, :]
    dirs = d[:, None, :].expand(rays, per, 3)
    return xyz.reshape(-1, 3)[:n].contiguous(), dirs.reshape(-1, 3)[:n].contiguous()


def _table_(table, gen, scale):
    with torch.no_grad():
        table.copy_((torch.rand(table.shape, generator=gen, device=table.device) - 0.5) * (2 * scale))


def _field(dtype, seed, gen):
    """A field with a trained one's spread: features of order 0.1, densities around 20."""
    half = dtype == "f16"
    m = NeRF(bound=1.0, device=_dev(), seed=int(seed) % 2 ** 31, table_dtype=torch.float16 if half else torch.float32)
    _table_(m.position_encoder.table, gen, 0.5)
    with torch.no_grad():
        density_head = m.mlp_params[2048:3072].view(64, 16)  # density_mlp/Dense_1
        density_head[:, 0] = density_head[:, 0] * 6 + 0.8
    if half:
        m.mlp_half = m.mlp_params.detach().half()
    return m


def _grid_coords():
    """Cell centres of the 128^3 grid in Morton order, [G^3, 3] in [-1, 1]."""
    idx = torch.arange(G ** 3, dtype=torch.int32, device=_dev()).view(torch.uint32)
    v = volrend.morton3d_invert(idx).view(torch.int32).float()
    return (v + 0.5) / G * 2 - 1


def _ball_bits(gen):
    """Bitfield of six balls (radius 0.1 to 0.35) inside [-1, 1]^3."""
    p = _grid_coords()
    density = torch.zeros(G ** 3, device=_dev())
    c = (torch.rand(6, 3, generator=gen, device=_dev()) - 0.5) * 1.2
    r = 0.1 + 0.25 * torch.rand(6, generator=gen, device=_dev())
    for k in range(6):
        density = torch.maximum(density, (((p - c[k]) ** 2).sum(-1) < r[k] ** 2).float())
    return volrend.packbits(0.5, density)[1]


def _camera_rays(n, gen):
    """Rays from a sphere of radius 4 towards the scene, with their AABB entry and exit."""
    dev = _dev()
    v = torch.randn(n, 3, generator=gen, device=dev)
    o = 4 * v / torch.linalg.norm(v, dim=-1, keepdim=True)
    d = (torch.rand(n, 3, generator=gen, device=dev) - 0.5) * 2 - o
    d = d / torch.linalg.norm(d, dim=-1, keepdim=True)
    t0, t1 = make_near_far_from_bound(1.0, o, d)
    return o.contiguous(), d.contiguous(), t0, t1


def _blob_density(scene, p):
    x = p.double()
    out = torch.zeros(x.shape[0], dtype=torch.float64, device=x.device)
    for c, r, s in zip(scene.centers, scene.radii, scene.peaks):
        d2 = ((x - torch.as_tensor(c, device=x.device)) ** 2).sum(-1)
        out += float(s) * torch.exp(-d2 / (2 * float(r) ** 2))
    return out.float()


def _encoder(case, gen):
    half = case["dtype"] == "f16"
    enc = HashGridEncoder(L=16, T=1 << case["log2_T"], F=2, N_min=16, N_max=2048,
                          param_dtype=torch.float16 if half else torch.float32, device=_dev(), generator=gen)
    _table_(enc.table, gen, 0.5)
    return enc


def prepare(case, seed):
    kind, gen, dev = case["kind"], _gen(seed), _dev()
    if kind == "encoder":
        enc = _encoder(case, gen)
        pos, _ = _ray_samples(case["points"], gen)
        g = torch.randn(case["points"], 32, generator=gen, device=dev)
        return {"kind": kind, "encoder": enc, "pos": pos, "g": g}
    if kind == "mlp":
        n = case["samples"]
        field = _field("f32", seed, gen)
        enc = torch.randn(n, 32, generator=gen, device=dev) * 0.2
        _, dirs = _ray_samples(n, gen)
        g = torch.randn(n, 4, generator=gen, device=dev) * torch.tensor([1e-4, 1e-2, 1e-2, 1e-2], device=dev)
        return {"kind": kind, "enc": enc.requires_grad_(), "dirs": dirs, "g": g,
                "params": field.mlp_params.detach().clone().requires_grad_()}
    if kind == "field":
        xyz, dirs = _ray_samples(case["points"], gen)
        return {"kind": kind, "model": _field(case["dtype"], seed, gen), "xyz": xyz, "dirs": dirs}
    if kind == "march":
        o, d, t0, t1 = _camera_rays(case["rays"], gen)
        noise = torch.rand(case["rays"], generator=gen, device=dev)
        return {"kind": kind, "args": (case["samples"], DIAG, 1, G, 1.0, 0.0, o, d, t0, t1, noise, _ball_bits(gen))}
    if kind == "integrate":
        n, most = case["rays"], case["max_samples"]
        total = n * most // 2 + 7
        ns = torch.randint(0, most + 1, (n,), generator=gen, device=dev)
        start = torch.cumsum(ns, 0) - ns
        ns = torch.minimum(ns, torch.clamp(total - 7 - start, min=0))  # rays past the last slot are empty
        start = torch.cumsum(ns, 0) - ns
        used = int(ns.sum())  # the slots after them belong to no ray, as the marcher leaves them
        ray = torch.zeros(total, dtype=torch.int64, device=dev)
        ray[:used] = torch.repeat_interleave(torch.arange(n, device=dev), ns)
        k = torch.arange(total, device=dev) - start[ray]
        z = 2.5 + torch.rand(n, generator=gen, device=dev)[ray] + k * STEP
        # densities of a trained field: near empty in front, opaque within the ray
        sigma = torch.exp(torch.randn(total, generator=gen, device=dev) * 1.5 + 1.0 + 3.0 * k / most)
        rgb = torch.rand(total, 3, generator=gen, device=dev)
        drgbs = torch.cat([sigma[:, None], rgb], 1).contiguous()
        u32 = lambda t: t.to(torch.int32).contiguous().view(torch.uint32)
        return {"kind": kind, "start": u32(start), "ns": u32(ns), "dss": torch.full((total,), STEP, device=dev),
                "z": z.float().contiguous().requires_grad_(), "drgbs": drgbs.requires_grad_(),
                "bgs": torch.rand(n, 3, generator=gen, device=dev).requires_grad_(),
                "g": torch.randn(n, 4, generator=gen, device=dev) * 1e-3}
    if kind == "train":
        scene = BlobScene.random(seed=int(seed) % 1000, n_blobs=8)
        cam = Camera(width=200, height=200, fx=277.75, fy=277.75, cx=100.0, cy=100.0)
        data = make_views(scene, cam, look_at_poses(8, seed=int(seed) % 1000), dev, n_steps=64)
        cfg = TrainConfig(total_samples=case["samples"], precision=case["precision"], proposal=case["guided"],
                          proposal_guided=case["guided"], seed=1_000_000_007 + int(seed))
        tr = Trainer(data, cfg, device=dev)
        # a run past the all-cells phase of the grid cadence, its grid on the scene
        tr.step_count = 1_000
        g = tr.grid
        g.density = torch.where(g.density < 0, g.density, _blob_density(scene, _grid_coords()))
        tr.threshold_ogrid()
        return {"kind": kind, "trainer": tr}
    if kind == "render":
        s = case["size"]
        f = 1111.0 * s / 800
        cam = Camera(width=s, height=s, fx=f, fy=f, cx=s / 2, cy=s / 2)
        pose = torch.as_tensor(look_at_poses(1, seed=int(seed) % 2 ** 31, golden=False)[0], dtype=torch.float32,
                               device=dev)
        return {"kind": kind, "model": _field(case["dtype"], seed, gen), "camera": cam, "pose": pose,
                "bits": _ball_bits(gen)}
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "encoder":
        enc = state["encoder"]
        out, _ = enc(state["pos"], 1.0)
        (dtable,) = torch.autograd.grad(out, (enc.table,), state["g"])
        return {"encodings": out, "dtable": dtable}
    if kind == "mlp":
        out = nerf_mlp(state["enc"], state["dirs"], state["params"])
        denc, dparams = torch.autograd.grad(out, (state["enc"], state["params"]), state["g"])
        return {"drgbs": out, "denc": denc, "dparams": dparams}
    if kind == "field":
        with torch.no_grad():
            return {"drgbs": state["model"](state["xyz"], state["dirs"], None)[0]}
    if kind == "march":
        out = volrend.march_rays(*state["args"])
        return dict(zip(("measured", "valid", "n_samples", "start", "indices", "xyzs", "dirs", "dss", "z_vals"), out))
    if kind == "integrate":
        measured, rgbds, opac = volrend.integrate_rays(0.3, state["start"], state["ns"], state["bgs"], state["dss"],
                                                       state["z"], state["drgbs"])
        dbgs, dz, ddrgbs = torch.autograd.grad(rgbds, (state["bgs"], state["z"], state["drgbs"]), state["g"])
        return {"measured": measured, "rgbds": rgbds, "opacities": opac, "dbgs": dbgs, "dz": dz, "ddrgbs": ddrgbs}
    if kind == "train":
        tr = state["trainer"]
        tr.step()
        m = tr.model
        return {"loss": tr.b["loss"], "dtable": tr.b["dtable"], "dparams": tr.b["dparams"],
                "table": m.position_encoder.table, "params": m.mlp_params}
    o, d = make_rays_worldspace(state["camera"], state["pose"])
    rgbd, bg = render_rays_inference(state["model"], o, d, state["bits"])
    return {"rgbd": rgbd, "bg": bg}


# ---------------------------------------------------------------------------
# the work of one pass: each input read once, each output written once
# ---------------------------------------------------------------------------

def _table_rows(log2_T):
    rows = 0
    for i in range(16):
        r = math.ceil(16 * 128 ** (i / 15) - 1) + 1
        rows += min(-(-r ** 3 // 8) * 8, 1 << log2_T)
    return rows


def work(case):
    kind = case["kind"]
    if kind == "encoder":
        n, rows, e = case["points"], _table_rows(case["log2_T"]), 2 if case["dtype"] == "f16" else 4
        touched = min(rows, n * 16 * 8)  # rows read (the forward) at most; the whole gradient is written
        return {"bytes": n * (12 + 2 * 128) + 2 * e * (touched + rows), "flops": n * 16 * 8 * 2 * 4}
    if kind == "mlp":
        return {"bytes": case["samples"] * (2 * 128 + 12 + 2 * 16) + 2 * 4 * N_PARAMS,
                "flops": case["samples"] * 3 * MLP_FLOPS}
    if kind == "field":
        n, e = case["points"], 2 if case["dtype"] == "f16" else 4
        return {"bytes": n * 40 + 2 * e * min(_table_rows(19), n * 128), "flops": n * (MLP_FLOPS + 512)}
    if kind == "march":
        return {"bytes": case["samples"] * 36 + case["rays"] * 45 + G ** 3 // 8, "flops": case["samples"] * 30}
    if kind == "integrate":
        s = case["rays"] * case["max_samples"] // 2
        return {"bytes": s * (24 + 44) + case["rays"] * (40 + 68), "flops": s * 60}
    if kind == "train":
        s, e = case["samples"], 2 if case["precision"] == "fp16" else 4
        # the table read and its gradient written, Adam's moments and weights read and written
        return {"bytes": _table_rows(19) * 2 * (2 * e + 4 + 6 * 4) + s * 300, "flops": s * 4 * MLP_FLOPS}
    n = case["size"] ** 2
    e = 2 if case["dtype"] == "f16" else 4
    samples = n * 20  # composited samples a pixel on these scenes, background pixels among them
    return {"bytes": n * (24 + 16 + 12) + _table_rows(19) * 2 * e, "flops": samples * MLP_FLOPS}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _levels(log2_T):
    """(scale, resolution, row offset, dense) of the sixteen levels and the row count."""
    b = math.exp((math.log(2048) - math.log(16)) / 15)
    out, off = [], 0
    for i in range(16):
        scale = 16 * b ** i - 1
        res = math.ceil(scale) + 1
        rows = -(-res ** 3 // 8) * 8
        dense = rows <= 1 << log2_T
        rows = rows if dense else 1 << log2_T
        out.append((float(np.float32(scale)), res, off, dense))
        off += rows
    return out, off


def _corners(pos, level, T, n_rows):
    """Row indices and weights [8][N] of every point at one level."""
    scale, res, off, dense = level
    s = (pos.double() + 1) / 2 * scale + 0.5
    f = torch.floor(s)
    r = s - f
    v = f.long()
    for c in range(8):
        o = ((c >> 2) & 1, (c >> 1) & 1, c & 1)
        x, y, z = (v[:, a] + o[a] for a in range(3))
        if dense:
            h = x + y * res + z * res * res
        else:
            h = (x ^ ((y * 2654435761) & 0xFFFFFFFF) ^ ((z * 805459861) & 0xFFFFFFFF))
        w = torch.ones(pos.shape[0], dtype=torch.float64, device=pos.device)
        for a in range(3):
            w = w * (r[:, a] if o[a] else 1 - r[:, a])
        yield torch.clamp(h % T + off, max=n_rows - 1), w


def _encode64(pos, table, log2_T):
    levels, rows = _levels(log2_T)
    out = torch.zeros(pos.shape[0], 32, dtype=torch.float64, device=pos.device)
    for l, level in enumerate(levels):
        for idx, w in _corners(pos, level, 1 << log2_T, rows):
            out[:, 2 * l:2 * l + 2] += table[idx].double() * w[:, None]
    return out


def _encode64_grad(pos, g, log2_T):
    levels, rows = _levels(log2_T)
    out = torch.zeros(rows, 2, dtype=torch.float64, device=pos.device)
    for l, level in enumerate(levels):
        gl = g[:, 2 * l:2 * l + 2].double()
        for idx, w in _corners(pos, level, 1 << log2_T, rows):
            out.index_add_(0, idx, gl * w[:, None])
    return out


def _sh4(d):
    x, y, z = d.unbind(-1)
    xy, xz, yz, x2, y2, z2 = x * y, x * z, y * z, x * x, y * y, z * z
    return torch.stack([
        0.28209479177387814 * torch.ones_like(x), -0.48860251190291987 * y, 0.48860251190291987 * z,
        -0.48860251190291987 * x, 1.0925484305920792 * xy, -1.0925484305920792 * yz,
        0.94617469575755997 * z2 - 0.31539156525251999, -1.0925484305920792 * xz,
        0.54627421529603959 * (x2 - y2), 0.59004358992664352 * y * (-3 * x2 + y2), 2.8906114426405538 * xy * z,
        0.45704579946446572 * y * (1 - 5 * z2), 0.3731763325901154 * z * (5 * z2 - 3),
        0.45704579946446572 * x * (1 - 5 * z2), 1.4453057213202769 * z * (x2 - y2),
        0.59004358992664352 * x * (-x2 + 3 * y2)], -1)


class _TruncExp(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return torch.exp(x)

    @staticmethod
    def backward(ctx, g):
        (x,) = ctx.saved_tensors
        return g * torch.exp(torch.clamp(x, -15, 15))


def _mlp64(enc, dirs, params):
    w, at = [], 0
    for _, _, fi, fo in MLP_LAYERS:
        w.append(params[at:at + fi * fo].view(fi, fo))
        at += fi * fo
    o = torch.relu(enc @ w[0]) @ w[1]
    h = torch.relu(torch.relu(torch.cat([o, _sh4(dirs)], -1) @ w[2]) @ w[3])
    return torch.cat([_TruncExp.apply(o[:, :1]), torch.sigmoid(h @ w[4])], -1)


def _integrate64(s):
    """Compositing with the stop at T <= 1e-4 and the reference's gradient, on rays
    padded to the longest."""
    start, ns = (s[k].view(torch.int32).long() for k in ("start", "ns"))
    n, total = start.shape[0], s["dss"].shape[0]
    most = max(1, int(ns.max()))
    k = torch.arange(most, device=start.device)[None]
    own = k < ns[:, None]
    at = torch.where(own, start[:, None] + k, 0)
    sig, rgb = s["drgbs"].detach().double()[at][..., 0], s["drgbs"].detach().double()[at][..., 1:]
    z, ds = s["z"].detach().double()[at], s["dss"].double()[at]
    bg, g = s["bgs"].detach().double(), s["g"].double()
    om = torch.where(own, torch.exp(-sig * ds), 1.0)
    after = torch.cumprod(om, 1)
    T = torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], 1)  # before each sample
    live = own & (T > 1e-4)
    w = torch.where(live, T * (1 - om), 0.0)
    T_end = torch.where(live, after, 1.0).amin(1)
    c = torch.cat([rgb, z[..., None]], -1)
    parts = torch.cumsum(w[..., None] * c, 1)
    acc = parts[:, -1]
    stop = T_end <= 1e-4
    bg4 = torch.cat([bg, torch.zeros_like(bg[:, :1])], -1)
    rgbd = torch.where(stop[:, None], acc / (1 - T_end)[:, None], acc + T_end[:, None] * bg4)
    rest = torch.where(1 - T_end >= 1 - 1e-4, 0.0, T_end)
    inner = (torch.where(live, after, 0.0)[..., None] * c - (rgbd[:, None] - parts)
             - bg4[:, None] * rest[:, None, None]) * g[:, None]
    dsig = ds * inner.sum(-1)
    dsig = torch.clamp(z * z, max=1.0) * dsig + torch.where((sig > 4e-5) & (z < 0.3), 1e-4, 0.0)
    dz = torch.zeros(total, dtype=torch.float64, device=z.device)
    dd = torch.zeros(total, 4, dtype=torch.float64, device=z.device)
    dz[at[live]] = (w * g[:, None, 3])[live]
    dd[at[live]] = torch.cat([dsig[..., None], w[..., None] * g[:, None, :3]], -1)[live]
    return {"measured": None, "rgbds": rgbd, "opacities": 1 - T_end,
            "dbgs": torch.where(stop, 0.0, T_end)[:, None] * g[:, :3], "dz": dz, "ddrgbs": dd}


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("encoder", "mlp", "field", "integrate"):
        return None  # the marcher's outputs follow its f32 steps; whole steps and frames compose the others
    s = prepare(case, seed)
    if kind == "encoder":
        table = s["encoder"].table.detach()
        return {"encodings": _encode64(s["pos"], table, case["log2_T"]),
                "dtable": _encode64_grad(s["pos"], s["g"], case["log2_T"])}
    if kind == "mlp":
        e, p = s["enc"].detach().double().requires_grad_(), s["params"].detach().double().requires_grad_()
        out = _mlp64(e, s["dirs"].double(), p)
        denc, dparams = torch.autograd.grad(out, (e, p), s["g"].double())
        return {"drgbs": out.detach(), "denc": denc, "dparams": dparams}
    if kind == "field":
        m = s["model"]
        params = (m.mlp_half if m.mlp_half is not None else m.mlp_params.detach()).double()
        with torch.no_grad():
            enc = _encode64(s["xyz"], m.position_encoder.table.detach(), 19)
            return {"drgbs": _mlp64(enc, s["dirs"].double(), params)}
    return _integrate64(s)
