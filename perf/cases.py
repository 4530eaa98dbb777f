"""The workloads this library's speed is measured on.

Each case is one pass through the public entry points as a program calls
them: whole frames (FramePipeline, GuiFrame), training steps (RadianceField),
and the single stages of both (fused render, volume building, ray traversal
and sampling, the training-only tree kernels, compositing, the FastNerf
inference surface).  Sizes come from the frame configurations of
sailor_amd.pipeline and sailor_amd.gui and from the tests, with odd ones
between.  Scenes are seeded capsule performers like those of
sailor_amd.scenes, ray-cast on the GPU so that many can be made quickly.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from sailor_amd import InferNerf, scenes
from sailor_amd import VoxelEncoding as VE
from sailor_amd import voxel_encoding_helper as VH
from sailor_amd.gui import GuiFrame
from sailor_amd.model import CONFIG_MODELS, NerfWeights, fastnerf_params
from sailor_amd.pipeline import FrameConfig, FramePipeline
from sailor_amd.render import PackedModel, render_rays
from sailor_amd.train import RadianceField

DEV = "cuda"
HALF = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ---------------------------------------------------------------------------
# cases
def listed():
    return [
        # the real-time frame of the benchmark: 512^2 from 4 RGBD views of
        # 1024^2, replayed from a graph as a viewer does
        dict(name="frame_bf16_512", kind="frame", prec="bf16", views=4, img=1024, dim=256, rate=8,
             target=512, S=48, model="c2", graph=True),
        # the small plain-precision frame, launched call by call
        dict(name="frame_fp32_256", kind="frame", prec="fp32", views=4, img=512, dim=128, rate=8,
             target=256, S=64, model="c1", graph=False),
        # the GUI's frame loop at its own settings (FastNerf + upsampling)
        dict(name="gui_fp16_512", kind="gui", views=4, img=512, dim=128, rate=4, target=512, S=32),
        # a full training batch: 8 target views of 256^2 rays
        dict(name="train_bf16_8x256", kind="train", prec="bf16", R=524288, S=48, views=4, img=1024,
             hit=0.28),
        # a small training step of random rays, plain precision
        dict(name="train_fp32_2000", kind="train", prec="fp32", R=2000, S=48, views=3, img=512,
             hit=0.6),
        # one fused render of a tile with more than 4 source views
        dict(name="render_fp16_6views", kind="render", prec="fp16", R=40001, S=48, views=6,
             img=1024, model="c2", hit=0.5, early_exit=False),
        # a handful of rays (a picked region, a progressive tile): latency
        dict(name="render_bf16_500", kind="render", prec="bf16", R=500, S=24, views=2, img=512,
             model="c1", hit=0.7, early_exit=True),
        # a new frame fused into the volume and its tree rebuilt, drop-in calls
        dict(name="build_256", kind="build", views=4, img=1024, dim=256, rate=8),
        # target rays through the tree, sampled and sorted, drop-in calls
        dict(name="rays_320", kind="rays", views=4, img=512, dim=128, rate=4, target=320, S=48),
        # the training-only tree path on random rays
        dict(name="octree_train_20000", kind="octree", views=4, img=512, dim=128, rate=8, R=20000,
             S=48, C=8),
        # the compositing the training differentiates, forward and backward
        dict(name="composite_occ_65536", kind="composite", op="tensor_occ", R=65536, S=48, F=16),
        # FastNerf's inference surface, the size of a large call
        dict(name="infer_fp16_65536", kind="infer", R=65536, S=48, views=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "gui", "train", "render", "build", "rays", "octree", "composite",
                       "infer"])
    if kind == "frame":
        prec = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        return dict(kind=kind, prec=prec, views=rng.randint(2, 4), img=rng.randint(400, 1024),
                    dim=8 * rng.randint(16, 32), rate=8,
                    target=rng.randint(100, 256 if prec == "fp32" else 512),
                    S=8 * rng.randint(3, 8), model="c1" if prec == "fp32" else
                    rng.choice(["c1", "c2"]), graph=rng.random() < 0.5)
    if kind == "gui":
        return dict(kind=kind, views=rng.randint(2, 4), img=rng.randint(256, 512),
                    dim=4 * rng.randint(20, 32), rate=4, target=rng.randint(200, 512),
                    S=rng.randint(16, 40))
    if kind == "train":
        prec = rng.choice(["bf16", "bf16", "fp32"])
        return dict(kind=kind, prec=prec, R=_log(rng, 500, 30000 if prec == "fp32" else 300000),
                    S=16 * rng.randint(1, 4), views=rng.randint(2, 4), img=rng.randint(400, 1024),
                    hit=round(rng.uniform(0.2, 0.9), 2))
    if kind == "render":
        prec = rng.choice(["bf16", "fp16", "fp32"])
        return dict(kind=kind, prec=prec, R=_log(rng, 300, 8000 if prec == "fp32" else 60000),
                    S=8 * rng.randint(2, 8), views=rng.randint(2, 7), img=rng.randint(400, 1024),
                    model=rng.choice(["c1", "c2"]), hit=round(rng.uniform(0.3, 1.0), 2),
                    early_exit=rng.random() < 0.3)
    if kind == "build":
        rate = rng.choice([4, 8])
        return dict(kind=kind, views=rng.randint(2, 6), img=rng.randint(400, 1024),
                    dim=rate * rng.randint(96 // rate, 256 // rate), rate=rate)
    if kind == "rays":
        rate = rng.choice([4, 8])
        return dict(kind=kind, views=4, img=512, dim=rate * rng.randint(96 // rate, 160 // rate),
                    rate=rate, target=rng.randint(64, 320), S=rng.randint(16, 64))
    if kind == "octree":
        return dict(kind=kind, views=4, img=512, dim=8 * rng.randint(12, 20), rate=8,
                    R=_log(rng, 1000, 20000), S=rng.randint(16, 64), C=rng.randint(1, 12))
    if kind == "composite":
        return dict(kind=kind, op=rng.choice(["tensor_occ", "tensor_density", "infer"]),
                    R=_log(rng, 500, 65536), S=rng.randint(16, 64), F=rng.randint(1, 32))
    return dict(kind="infer", R=_log(rng, 700, 65536), S=rng.randint(16, 48),
                views=rng.randint(2, 4))


# ---------------------------------------------------------------------------
# inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 40) + 17)


def _f32(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV)


def _ray_capsule(o, d, a, b, r):
    """Nearest hit distance of unit rays d [N,3] from o [3] with the capsule
    (segment a-b, radius r); inf where missed."""
    ba, oa = b - a, o - a
    baba, bard, baoa = ba @ ba, d @ ba, oa @ ba
    rdoa, oaoa = d @ oa, oa @ oa
    A = baba - bard * bard
    Bq = baba * rdoa - baoa * bard
    C = baba * oaoa - baoa * baoa - r * r * baba
    h = Bq * Bq - A * C
    inf = torch.full_like(rdoa, math.inf)
    t = (-Bq - h.clamp_min(0).sqrt()) / A
    y = baoa + t * bard
    best = torch.where((h >= 0) & (y > 0) & (y < baba) & (t > 0), t, inf)
    for cap in (a, b):
        oc = o - cap
        bb = d @ oc
        hh = bb * bb - (oc @ oc - r * r)
        ts = -bb - hh.clamp_min(0).sqrt()
        best = torch.where((hh > 0) & (ts > 0) & (ts < best), ts, best)
    return best


def _scene(seed, views, img):
    """A capsule performer seen by a ring of `views` RGBD cameras: depth with
    2 mm noise, quantised to 0.1 mm, 1 % of the pixels missing."""
    rng = np.random.default_rng(int(seed) % (1 << 40) + 1000)
    r = rng.uniform(0.05, 0.15, 10)
    a = rng.uniform(scenes.BOX_MIN + r[:, None], scenes.BOX_MAX - r[:, None])
    b = rng.uniform(scenes.BOX_MIN + r[:, None], scenes.BOX_MAX - r[:, None])
    col = rng.uniform(0.0, 1.0, (10, 3))
    cams = scenes.ring_cameras(views, img * 1.172, img, img)
    g = _gen(seed)
    d64 = lambda x: torch.as_tensor(np.asarray(x, np.float64), device=DEV)
    depth, rgb, mask = [], [], []
    for cam in cams:
        K, R, T = d64(cam.K), d64(cam.R), d64(cam.T)
        px = torch.arange(img, device=DEV, dtype=torch.float64)
        x = ((px - K[0, 2]) / K[0, 0])[None, :].expand(img, img)
        y = ((px - K[1, 2]) / K[1, 1])[:, None].expand(img, img)
        dc = torch.stack([x, y, torch.ones_like(x)], -1).reshape(-1, 3)
        nrm = dc.norm(dim=1)
        d = (dc / nrm[:, None]) @ R
        o = -(R.T @ T)
        best = torch.full((img * img,), math.inf, dtype=torch.float64, device=DEV)
        c = torch.zeros((img * img, 3), dtype=torch.float64, device=DEV)
        for i in range(10):
            t = _ray_capsule(o, d, d64(a[i]), d64(b[i]), float(r[i]))
            near = t < best
            best = torch.where(near, t, best)
            c = torch.where(near[:, None], d64(col[i]), c)
        hit = torch.isfinite(best)
        z = torch.where(hit, best / nrm, torch.zeros_like(best))
        z = z + 0.002 * torch.randn(z.shape, generator=g, device=DEV, dtype=torch.float64)
        z = (z * 10000.0).round().clamp(0, 65535) / 10000.0
        z[~hit | (torch.rand(z.shape, generator=g, device=DEV) < 0.01)] = 0.0
        depth.append(z.reshape(img, img).float())
        rgb.append(c.T.reshape(3, img, img).float())
        mask.append(hit.reshape(img, img).float())
    depth, rgb, mask = torch.stack(depth), torch.stack(rgb), torch.stack(mask)
    sc = scenes.Scene(int(seed), a, b, r, col, cams, None, depth.cpu().numpy(), rgb.cpu().numpy(),
                      mask.cpu().numpy())
    return sc, depth, rgb, mask


def _frame_config(c, model):
    return FrameConfig("case", c["views"], c["img"], c["img"] * 1.172, c["dim"], c["rate"],
                       c["target"], c["target"] * 1.172, c["S"], model)


def _target(seed, size):
    """A novel view on the ring, between two source cameras."""
    phase = np.random.default_rng(int(seed) % (1 << 40) + 5).uniform(0.3, 1.2)
    return scenes.target_camera(size, size, size * 1.172, phase)


def _prepare_frame(c, seed):
    cfg = _frame_config(c, c["model"])
    mc = CONFIG_MODELS[c["model"]]
    p = FramePipeline(cfg, prec=c["prec"], device=DEV)
    sc = _scene(seed, c["views"], c["img"])[0]
    fm = torch.randn((c["views"], mc.F, mc.Hf, mc.Wf), generator=_gen(seed + 3), device=DEV)
    p.load_scene(sc, fm.cpu().numpy(), _target(seed, c["target"]))
    if c["graph"]:
        p.capture()
    return p


def _prepare_gui(c, seed):
    frame = GuiFrame(_frame_config(c, "c1"), frame_id=int(seed) % (1 << 20), device=DEV)
    return frame


def _ellipsoid_rays(seed, R, S, hit, random_pixels):
    """R target rays [1,R,6] of a ring camera with S sorted sample distances
    each around the surface of an ellipsoid performer, -1 where the ray has
    none (about 1 - hit of them): raster order of a square image, or random
    pixels as a training batch picks them."""
    g = _gen(seed + 11)
    side = int(math.ceil(math.sqrt(R)))
    cam = _target(seed, side)
    K, RT = (torch.as_tensor(np.asarray(m, np.float64), device=DEV) for m in (cam.K, cam.RT))
    o = -(RT[:, :3].T @ RT[:, 3])
    # pixels spread over the box whose share `hit` the ellipsoid covers
    half = side * 1.172 / 2.5 * math.sqrt(0.4 * 1.0 * math.pi / hit) / 2.0
    n = torch.arange(R, device=DEV, dtype=torch.float64)
    if random_pixels:
        uv = torch.rand((R, 2), generator=g, device=DEV, dtype=torch.float64)
    else:
        uv = torch.stack([(n % side + 0.5) / side, ((n / side).floor() + 0.5) / side], -1)
    px = K[0, 2] + (uv - 0.5) * 2.0 * half
    d = torch.stack([(px[:, 0] - K[0, 2]) / K[0, 0], (px[:, 1] - K[1, 2]) / K[1, 1],
                     torch.ones_like(n)], -1)
    d = (d / d.norm(dim=1, keepdim=True)) @ RT[:, :3]
    axes = torch.tensor([0.4, 1.0, 0.4], dtype=torch.float64, device=DEV)
    oo = (o - torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64, device=DEV)) / axes
    dd = d / axes
    qa, qb, qc = (dd * dd).sum(1), dd @ oo, oo @ oo - 1.0
    disc = qb * qb - qa * qc
    t0 = (-qb - disc.clamp_min(0).sqrt()) / qa
    band = torch.rand((R, S), generator=g, device=DEV, dtype=torch.float64).sort(-1)[0]
    t = t0[:, None] + 0.16 * band - 0.06
    t = torch.where(disc[:, None] > 0, t, torch.full_like(t, -1.0)).float()
    rays = torch.cat([o.expand(R, 3), d], -1).float()
    zdir = RT[2:3, :3].float()
    return t[None].contiguous(), rays[None].contiguous(), zdir.contiguous()


def _render_inputs(c, seed, model, random_pixels):
    mc = CONFIG_MODELS[model]
    t, rays, zdir = _ellipsoid_rays(seed, c["R"], c["S"], c["hit"], random_pixels)
    cams = scenes.ring_cameras(c["views"], c["img"] * 1.172, c["img"], c["img"])
    K, RT = _f32([[x.K for x in cams]]), _f32([[x.RT for x in cams]])
    fm = torch.randn((1, c["views"], mc.Hf, mc.Wf, mc.F), generator=_gen(seed + 3), device=DEV)
    bbox = _f32(scenes.fixed_cube(2.2)[None])
    return t, rays, K, RT, (c["img"], c["img"]), fm, bbox, zdir


def _weights(model, seed):
    """Xavier weights with small biases, as a trained model has some."""
    mc = CONFIG_MODELS[model]
    w = NerfWeights.init(mc.F, mc.H, seed=int(seed) % 100000)
    rng = np.random.default_rng(int(seed) % (1 << 40) + 77)
    w.dense_b = [rng.normal(0, 0.05, b.shape).astype(np.float32) for b in w.dense_b]
    w.sigma_b = float(np.float32(rng.normal(-1.0, 0.2)))
    return w


def _prepare_train(c, seed):
    w = _weights("c1", seed)
    field = RadianceField(w, c["prec"], DEV)
    args = _render_inputs(c, seed, "c1", c["R"] < 100000)
    target = torch.rand((1, c["R"], 3), generator=_gen(seed + 7), device=DEV)
    valid = (args[0][..., :1] >= 0).float()
    return dict(field=field, args=args, target=target * valid, n=3.0 * float(valid.sum()),
                opt=torch.optim.SGD(field.parameters(), lr=1e-3), w=w)


def _prepare_render(c, seed):
    args = list(_render_inputs(c, seed, c["model"], False))
    w = _weights(c["model"], seed)
    if c["prec"] != "fp32":
        args[5] = args[5].to(HALF[c["prec"]])
    return dict(args=args, w=w, model=PackedModel(w, c["prec"], DEV),
                early_exit=c["early_exit"])


def _volume_inputs(c, seed):
    sc, depth, rgb, mask = _scene(seed, c["views"], c["img"])
    K, RT = _f32(sc.K()), _f32(sc.RT())
    d, dc = c["dim"], c["dim"] // c["rate"]
    i32 = dict(dtype=torch.int32, device=DEV)
    vols = ([torch.empty((1, n, n, n), **i32) for n in (d, dc)],
            [torch.zeros((1,), **i32) for _ in range(2)])
    return dict(data=(rgb, depth[:, None], mask[:, None], K, RT), vols=vols, rate=c["rate"],
                tree=VH.OcTreeOptions(levels=2, batch_size=1, rate=c["rate"], vol_dim=d,
                                      device=DEV + ":0"))


def _build(s):
    occ, num, tsdf, color, origin, bbox, size = VH.integrate_depths(
        s["data"], s["vols"], 1, _tsdf_th_low=13.5, _tsdf_th_high=13.5, _level_volumes=2,
        _volume_res_rate=s["rate"])
    s["tree"].init_octree(occ, num, size, bbox)
    return occ, num, tsdf, color, origin, bbox, size


def _prepare_build(c, seed):
    s = _volume_inputs(c, seed)
    s["nodes"] = torch.zeros((c["dim"] ** 3 // 8, 6), device=DEV)
    return s


def _prepare_rays(c, seed):
    s = _volume_inputs(c, seed)
    _build(s)
    cam = _target(seed, c["target"])
    s.update(K=_f32(cam.K[None, None]), R=_f32(cam.R[None, None]), T=_f32(cam.T[None, None]),
             size=c["target"], S=c["S"],
             noise=torch.rand((1, c["target"] ** 2, c["S"]), generator=_gen(seed + 9), device=DEV))
    return s


def _prepare_octree(c, seed):
    s = _volume_inputs(c, seed)
    _build(s)
    g = _gen(seed + 9)
    img = c["img"]
    cam = _target(seed, img)
    R, S, C = c["R"], c["S"], c["C"]
    xy = torch.randint(img // 4, 3 * img // 4, (1, 1, R, 2), generator=g, device=DEV)
    s.update(K=_f32(cam.K[None, None]), R=_f32(cam.R[None, None]), T=_f32(cam.T[None, None]),
             size=img, xy=xy.to(torch.int32), S=S, img=img, views=c["views"],
             noise=torch.rand((1, R, S), generator=g, device=DEV),
             feats=torch.randn((1, C, R, S, 8), generator=g, device=DEV).requires_grad_(),
             grad=torch.randn((1, C, R, S), generator=g, device=DEV))
    return s


def _prepare_composite(c, seed):
    g = _gen(seed)
    R, S, F = c["R"], c["S"], c["F"]
    t = (2.0 + 0.5 * torch.rand((1, R, S), generator=g, device=DEV)).sort(-1)[0]
    # occupancies of a trained model: mostly small, a few surfaces
    occ = torch.sigmoid(3.0 * torch.randn((1, R, S, 1), generator=g, device=DEV) - 3.0)
    if c["op"] == "tensor_density":
        occ = 40.0 * occ
    feats = torch.randn((1, R, S, F), generator=g, device=DEV)
    valid = torch.rand((1, R), generator=g, device=DEV) < 0.8
    grads = [torch.randn((1, R, n), generator=g, device=DEV) for n in (F, 1, 1, 1)]
    grads[2], grads[3] = 0.1 * grads[2], 0.1 * grads[3]
    return dict(op=c["op"], t=t, sigma=occ.requires_grad_(), feats=feats.requires_grad_(),
                valid=valid, grads=grads)


def _prepare_infer(c, seed):
    g = _gen(seed)
    R, S, V = c["R"], c["S"], c["views"]
    n = V * R * S
    rand = lambda *s: torch.rand(*s, generator=g, device=DEV)
    randn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    pd, pc, _ = fastnerf_params(int(seed) % 100000)
    return dict(t=(1.0 + 2.0 * rand((1, R, S))).sort(-1)[0], z=2.0 * rand((n, 1)) - 1.0,
                ps=(2.0 * randn((n, 1))).clamp(-1, 1), geo=randn((n, 16)), rgb=rand((n, 3)),
                frgb=randn((n, 16)),
                dirs=torch.nn.functional.normalize(randn((n, 3)), dim=-1),
                pd=torch.from_numpy(pd).to(DEV), pc=torch.from_numpy(pc).to(DEV), R=R, S=S, V=V)


PREPARE = dict(frame=_prepare_frame, gui=_prepare_gui, train=_prepare_train,
               render=_prepare_render, build=_prepare_build, rays=_prepare_rays,
               octree=_prepare_octree, composite=_prepare_composite, infer=_prepare_infer)


def prepare(case, seed):
    return dict(kind=case["kind"], s=PREPARE[case["kind"]](case, int(seed)))


# ---------------------------------------------------------------------------
# one pass
def _run_frame(p):
    p.replay()
    return dict(rgb=p.rgb, depth=p.depth, aux=p.aux, samples=p.sorted, tsdf=p.tsdf, occ=p.occ0)


def _run_gui(g):
    rgb, depth, detail = g.render()
    return dict(rgb=rgb, depth=depth, detail=detail)


def _run_train(s):
    field = s["field"]
    s["opt"].zero_grad()
    rgb, depth, aux = field(*s["args"])
    loss = ((rgb - s["target"]) ** 2).sum() / s["n"]
    loss.backward()
    grads = [p.grad for p in field.flat_params()]
    s["opt"].step()
    return dict(rgb=rgb.detach(), depth=depth, aux=aux, grads=grads)


def _run_render(s):
    out = render_rays(*s["args"], s["model"], early_exit=s["early_exit"])
    return dict(rgb=out["rgb"], depth=out["depth"], aux=out["aux"])


def _run_build(s):
    occ, num, tsdf, color, origin, bbox, size = _build(s)
    # the program keeps the nodes in a table of its own, sized for any scene
    nodes = s["tree"].get_all_nodes()
    s["nodes"][:nodes.shape[0]].copy_(nodes)
    return dict(occ=occ, num=num, tsdf=tsdf, color=color, bbox=bbox, size=size,
                nodes=s["nodes"])


def _run_rays(s):
    rays = VE.rays_calculating(s["K"], s["R"], s["T"], s["size"], 0).view(1, -1, 6)
    tree = s["tree"]
    idx, t0, t1, length = tree.ray_intersection(rays[..., :3], rays[..., 3:],
                                                instersect_start_level=0)
    sidx, st = tree.ray_voxels_points_sampling_coarse(idx, t0, t1, s["noise"], length,
                                                      instersect_start_level=0,
                                                      n_sampled_points=s["S"])
    depths, order = tree.sort_sampling(st)
    return dict(rays=rays, idx=idx, t0=t0, t1=t1, length=length, sidx=sidx, samples=st,
                sorted=depths, order=order)


def _run_octree(s):
    rays = VE.rays_calculating(s["K"], s["R"], s["T"], s["size"], 0)
    rays = VE.rays_selecting(rays, s["xy"], 0)[:, 0]
    ori, dirs = rays[..., :3].contiguous(), rays[..., 3:].contiguous()
    tree = s["tree"]
    hits = tree.ray_intersection(ori, dirs, instersect_start_level=0, only_voxel_traversal=False)
    idx, t0, t1, length = hits[:4]
    sidx, st = tree._ray_voxels_sampling_points(idx, t0, t1, length, s["noise"], 0, s["S"])
    out = VH.voxel_trilinear_interpolation(tree.get_octree(), ori, dirs, st, sidx, s["feats"])
    grad, = torch.autograd.grad(out, s["feats"], s["grad"])
    xy, z = tree._project_sampled_xyz(ori, dirs, st, sidx, s["data"][3], s["data"][4], s["img"],
                                      s["img"], s["views"])
    return dict(hits=list(hits), sidx=sidx, samples=st, out=out.detach(), grad=grad, xy=xy, z=z)


def _run_composite(s):
    if s["op"] == "infer":
        with torch.no_grad():
            return list(VH.volume_render_infer(s["t"], s["sigma"], s["feats"], 1e-4))
    fn = VH.volume_render_torch.forward_occ if s["op"] == "tensor_occ" \
        else VH.volume_render_torch.forward
    out = fn(s["t"], s["sigma"], s["feats"], 4.0, s["valid"])
    grads = torch.autograd.grad(out, (s["sigma"], s["feats"]), s["grads"])
    return dict(out=[o.detach() for o in out], grads=list(grads))


def _run_infer(s):
    return list(InferNerf.infer_nerf(s["t"], s["z"], s["ps"], s["geo"], s["rgb"], s["frgb"],
                                     s["dirs"], s["pd"], s["pc"], 1, s["R"], s["S"], s["V"],
                                     s["V"], 0))


RUN = dict(frame=_run_frame, gui=_run_gui, train=_run_train, render=_run_render,
           build=_run_build, rays=_run_rays, octree=_run_octree, composite=_run_composite,
           infer=_run_infer)


def run(state):
    return RUN[state["kind"]](state["s"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
def _mlp_flops(model):
    mc = CONFIG_MODELS[model]
    return 2 * ((63 + mc.F) * mc.H + 3 * mc.H * mc.H)


def _hydra_flops(F, V):
    return 2 * 2 * V * 6 * F * 32 + 2 * (F * 64 + 64 * 32 + 32 * 3)


def work(case):
    c, kind = case, case["kind"]
    V, S = c.get("views", 0), c.get("S", 0)
    if kind in ("frame", "gui", "build"):
        # depth and colour maps read, 16 B per voxel written, read again by
        # the tree; per target ray its samples
        vox = c["dim"] ** 3
        nbytes = V * c["img"] ** 2 * 8 + vox * 20
        if kind == "build":
            return dict(bytes=nbytes, flops=vox * V * 40)
        R = c["target"] ** 2
        nbytes += R * (24 + 4 + 16 * S + 24)
        if kind == "frame":
            mc = CONFIG_MODELS[c["model"]]
            nbytes += V * mc.Hf * mc.Wf * mc.F * 4
            return dict(bytes=nbytes, flops=0.3 * R * (S * V * _mlp_flops(c["model"])
                                                       + _hydra_flops(mc.F, V)))
        nbytes += V * (128 * 128 * 32 + 1024 * 1024 * 19) * 4 + R * 48
        return dict(bytes=nbytes, flops=0.3 * R * (S * V * 27000 + S * 16500 + 4 * 29632))
    if kind in ("train", "render"):
        model = c.get("model", "c1")
        mc = CONFIG_MODELS[model]
        item = 4 if c["prec"] == "fp32" or kind == "train" else 2
        nbytes = c["R"] * (S * 4 + 24 + 24) + V * mc.Hf * mc.Wf * mc.F * item
        flops = c["hit"] * c["R"] * (S * V * _mlp_flops(model) + _hydra_flops(mc.F, V))
        return dict(bytes=nbytes, flops=flops * (3 if kind == "train" else 1))
    if kind == "rays":
        R = c["target"] ** 2
        return dict(bytes=R * (24 + 4 + 1024 * 12 + S * 20), flops=R * 2000)
    if kind == "octree":
        R, n = c["R"], c["R"] * S
        return dict(bytes=R * (24 + 12 * (512 + 3 * c["dim"] // c["rate"]))
                    + n * (12 + c["C"] * 72 + V * 12), flops=n * (c["C"] * 36 + V * 40))
    if kind == "composite":
        n = c["R"] * S
        train = c["op"] != "infer"
        return dict(bytes=n * (8 + 4 * c["F"]) * (2 if train else 1) + c["R"] * (c["F"] + 3) * 8,
                    flops=n * (6 + 2 * c["F"]) * (3 if train else 1))
    n = V * c["R"] * S
    return dict(bytes=n * 160 + c["R"] * (4 * S + 136),
                flops=n * 2 * (18 * 64 + 3 * 64 * 64 + 18 * 16 + 16 * 8)
                + c["R"] * S * 2 * (2 * 64 * 64 + 64) + c["R"] * V * 23040)


def tolerance(case):
    kind = case["kind"]
    if kind in ("build", "rays", "octree"):
        # voxel lists, nodes, hits and samples are one-rounding-per-operation
        # float32 arithmetic and reproduce bit for bit
        return "exact"
    # the others: about four times what the library's outputs are off their
    # 64-bit values
    if kind == "composite":
        return dict(rel=2e-6, max=1e-4)      # 32-bit sums over a ray: 2e-7
    if kind == "infer":
        return dict(rel=1e-3, max=0.1)       # half-rounded layer inputs: 2.6e-4
    if kind == "gui":
        return dict(rel=2e-3, max=0.5)       # the same, then colours picked by depth: 5e-4
    if kind == "train":
        # gradients also move where a rounding crosses a ReLU's kink
        return dict(rel=2e-3, max=0.1) if case["prec"] == "fp32" else dict(rel=1e-2, max=0.4)
    # colours: 2.6e-6, 1.1e-3 and 1.5e-4 off
    return dict(fp32=dict(rel=1e-5, max=1e-3), bf16=dict(rel=5e-3, max=0.2),
                fp16=dict(rel=1e-3, max=0.1))[case["prec"]]


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
def _d(a):
    return torch.as_tensor(a).detach().to(device=DEV, dtype=torch.float64)


def _params64(w, grad=False):
    leaf = lambda a: _d(np.asarray(a)).clone().requires_grad_(grad)
    flat = [*map(leaf, w.dense_w), *map(leaf, w.dense_b), leaf(w.sigma_w),
            leaf(np.array([np.float32(w.sigma_b)]))]
    flat += [leaf(st[k]) for st in w.hydra for k in ("q", "k", "v", "fc", "w1", "b1", "w2", "b2")]
    flat += [leaf(x) for wb in w.rgb for x in wb]
    return flat


def _sample64(fmap, K, RT, x, img_hw):
    """Bilinear features of one view's map [Hf,Wf,F] at world points x [N,3]."""
    p = x @ RT[:, :3].T + RT[:, 3]
    behind = p[:, 2:] < 0.01
    scr = (p / torch.where(behind, torch.ones_like(p[:, 2:]), p[:, 2:])) @ K.T
    half = torch.tensor([img_hw[1] // 2, img_hw[0] // 2], dtype=x.dtype, device=x.device)
    grid = torch.where(behind, torch.full_like(scr[:, :2], -2.0), (scr[:, :2] - half) / half)
    return torch.nn.functional.grid_sample(
        fmap.permute(2, 0, 1)[None], grid[None, None], mode="bilinear", padding_mode="zeros",
        align_corners=True)[0, :, 0].T


def _render64(P, t, rays, K, RT, img_hw, fmap, bbox, zdir):
    """Valid rays t [N,S], rays [N,6] -> rgb, depth, (weight, alpha) sums."""
    N, S = t.shape
    V = K.shape[0]
    x = (rays[:, None, :3] + t[..., None] * rays[:, None, 3:]).reshape(-1, 3)
    q = (x - 0.5 * (bbox[:, 0] + bbox[:, 1])) * (2.0 / (bbox[:, 1] - bbox[:, 0]))
    pe = [q]
    for f in range(10):
        pe += [torch.sin(q * 2.0 ** f), torch.cos(q * 2.0 ** f)]
    pe = torch.cat(pe, -1)
    feats = [_sample64(fmap[v], K[v], RT[v], x, img_hw) for v in range(V)]
    mean = 0
    for f in feats:
        h = torch.cat([pe, f], -1)
        for layer in range(4):
            h = torch.relu(h @ P[layer].T + P[4 + layer])
        mean = mean + h / V
    alpha = torch.sigmoid(mean @ P[8] + P[9]).reshape(N, S)
    T = torch.cumprod(torch.cat([torch.ones_like(alpha[:, :1]), 1.0 - alpha], 1), 1)
    # a ray ends with the sample that takes its transmittance below 1e-4
    w = torch.where(T[:, :-1].detach() < 1e-4, torch.zeros_like(alpha), alpha * T[:, :-1])
    tok = torch.stack([(w[..., None] * f.reshape(N, S, -1)).sum(1) for f in feats], 1)
    for st in range(2):
        q_, k_, v_, fc, w1, b1, w2, b2 = P[10 + 8 * st:18 + 8 * st]
        norm = lambda z: z / z.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        kv = (norm(tok @ k_.T) * (tok @ v_.T)).sum(1, keepdim=True)
        out = (norm(tok @ q_.T) * kv) @ fc.T + tok
        tok = torch.relu(out @ w1.T + b1) @ w2.T + b2 + out
    r = P[26:]
    h = torch.relu(tok[:, 0] @ r[0].T + r[1])
    h = torch.relu(h @ r[2].T + r[3])
    rgb = torch.sigmoid(h @ r[4].T + r[5])
    depth = (w * t).sum(1) * (rays[:, 3:] @ zdir)
    return rgb, depth, torch.stack([w.sum(1), (w * alpha).sum(1)], -1)


def _exact_render(c, s, train):
    t, rays, K, RT, img_hw, fmap, bbox, zdir = s["args"]
    P = _params64(s["w"], train)
    idx = torch.nonzero(t[0, :, 0] >= 0).flatten()
    R = t.shape[1]
    rgb, depth, aux = (torch.zeros((1, R, n), dtype=torch.float64, device=DEV) for n in (3, 1, 2))
    K, RT, fmap, bbox, zdir = _d(K[0]), _d(RT[0]), _d(fmap[0]), _d(bbox[0]), _d(zdir[0])
    step = max(1, (100000 if train else 300000) // (c["S"] * c["views"]))
    for part in idx.split(step):
        with torch.set_grad_enabled(train):
            o = _render64(P, _d(t[0, part]), _d(rays[0, part]), K, RT, img_hw, fmap, bbox, zdir)
            if train:
                (((o[0] - _d(s["target"][0, part])) ** 2).sum() / s["n"]).backward()
        rgb[0, part], depth[0, part], aux[0, part] = o[0].detach(), o[1].detach()[:, None], \
            o[2].detach()
    out = dict(rgb=rgb, depth=depth[..., 0], aux=aux)
    if train:
        out["grads"] = [p.grad for p in P]
    return out


def _exact_composite(s):
    t, sigma, feats = _d(s["t"]), _d(s["sigma"])[..., 0], _d(s["feats"])
    train = s["op"] != "infer"
    sigma.requires_grad_(train)
    feats.requires_grad_(train)
    one = torch.ones_like(t[..., :1])
    if s["op"] == "tensor_density":
        e = torch.cat([t[..., 1:] - t[..., :-1], 0 * one], -1) * sigma
        alpha, T = 1.0 - torch.exp(-e), torch.exp(e - torch.cumsum(e, -1))
    else:
        alpha = sigma
        T = torch.cumprod(torch.cat([one, 1.0 - alpha + (1e-6 if train else 0.0)], -1), -1)
        T = T[..., :-1]
    w = alpha * T
    if not train:
        w = torch.where(T < 1e-4, torch.zeros_like(w), w)
    out = [(w[..., None] * feats).sum(2), (w * t).sum(-1, keepdim=True),
           w.sum(-1, keepdim=True), (w * alpha).sum(-1, keepdim=True)]
    if not train:
        return out
    out = [o * s["valid"][..., None] for o in out]
    gs, gf = torch.autograd.grad(out, (sigma, feats), [_d(g) for g in s["grads"]])
    return dict(out=[o.detach() for o in out], grads=[gs[..., None], gf])


def _exact_infer(s):
    pd, pc = _d(s["pd"]), _d(s["pc"])

    def reader(p):
        at = [0]

        def take(*shape):
            n = int(np.prod(shape))
            at[0] += n
            return p[at[0] - n:at[0]].reshape(shape)
        return take
    R, S, V = s["R"], s["S"], s["V"]
    view = lambda x, part: _d(x.reshape(V, R, S, -1)[:, part])
    take = reader(pd)
    dense = [(take(o, i), take(o)) for i, o in
             ((18, 64), (64, 64), (64, 64), (64, 64), (64, 64), (64, 64), (64, 1), (18, 16),
              (16, 8))]
    run_layers = lambda h, layers: [h := torch.relu(h @ w.T + b) for w, b in layers][-1]
    out = []
    for part in torch.arange(R, device=DEV).split(max(1, 1000000 // (S * V))):
        x = torch.cat([view(s["z"], part), view(s["ps"], part), view(s["geo"], part)], -1)
        h = run_layers(run_layers(x, dense[:4]).mean(0), dense[4:6])
        alpha = torch.sigmoid(h @ dense[6][0].T + dense[6][1])[..., 0]
        f = torch.cat([view(s["frgb"], part), view(s["rgb"], part), run_layers(x, dense[7:]),
                       view(s["dirs"], part)], -1)
        T = torch.cumprod(torch.cat([torch.ones_like(alpha[:, :1]), 1.0 - alpha], 1), 1)[:, :-1]
        w = torch.where(T < 1e-4, torch.zeros_like(alpha), alpha * T)
        tok = (w[None, ..., None] * f).sum(2).permute(1, 0, 2)
        take = reader(pc)
        for _ in range(2):
            q, k, v = (tok @ take(32, 30).T for _ in range(3))
            kv = (k / k.norm(dim=-1, keepdim=True) * v).sum(1, keepdim=True)
            res = tok + (q / q.norm(dim=-1, keepdim=True) * kv) @ take(30, 32).T
            h = torch.relu(res @ take(32, 30).T + take(32))
            tok = h @ take(30, 32).T + take(30) + res
        h = run_layers(tok[:, 0], [(take(64, 30), take(64)), (take(32, 64), take(32))])
        out.append(((w * _d(s["t"][0, part])).sum(1, keepdim=True),
                    torch.sigmoid(h @ take(3, 32).T + take(3)), tok[:, 0]))
    return [torch.cat(o)[None] for o in zip(*out)]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "render", "composite", "infer"):
        s = prepare(case, seed)["s"]
        if kind == "composite":
            return _exact_composite(s)
        with torch.no_grad():
            if kind == "infer":
                return _exact_infer(s)
            return _exact_render(case, s, kind == "train")
    # frames, trees and samples hang on float32 roundings (which pixel, which
    # cell): they have no 64-bit counterpart
    return None
