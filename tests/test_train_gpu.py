"""GPU checks of the differentiation form against torch autograd of the
float64 restatement (oracle/nerf_ref.py):
  * Hydra + RGB head backward: dL/d token and the small-weight gradient.
"""
import numpy as np
import pytest
import torch

from oracle import nerf_ref

pytestmark = pytest.mark.gpu

_pipes = {}


def pipe(prec="fp32", model="c1"):
    from sailor_amd.pipeline import FrameConfig, FramePipeline
    cfg = FrameConfig(f"{model}_small", 4, 512, 600.0, 128, 8, 48, 56.25, 64, model)
    if (prec, model) not in _pipes:
        p = FramePipeline.synthetic(cfg, prec=prec)
        p.run()
        torch.cuda.synchronize()
        _pipes[(prec, model)] = p
    return _pipes[(prec, model)]


def _small_layout(w, tensors):
    """Flatten tensors named like NerfWeights.small_buffer's parts."""
    parts = [tensors["sigma_w"], torch.cat([tensors["sigma_b"].reshape(1),
                                            torch.zeros(3, dtype=torch.float64)])]
    for st in tensors["hydra"]:
        parts += [st["q"], st["k"], st["v"], st["fc"], st["w1"], st["b1"], st["w2"], st["b2"]]
    (w1, b1), (w2, b2), (w3, b3) = tensors["rgb"]
    parts += [w1, b1, w2, b2, w3, torch.cat([b3, torch.zeros(1, dtype=torch.float64)])]
    return torch.cat([p.reshape(-1) for p in parts])


@pytest.mark.parametrize("model", ["c1", "c2"])
def test_hydra_backward_matches_autograd(model):
    """F = 32 (c1): the fp32 MFMA backward kernels; F = 64 (c2): the vector
    ALU kernel."""
    from sailor_amd.train import BackwardScratch, hydra_backward, workspace_views
    p = pipe(model=model)
    cfg, w = p.cfg, p.weights
    n_rays = cfg.target * cfg.target
    p.shade()
    torch.cuda.synchronize()
    n_valid, lst, tok = workspace_views(p.render_ws, n_rays, p.mc.F)
    assert n_valid > 50
    g = torch.Generator(device="cpu").manual_seed(5)
    grad_rgb = torch.randn((n_rays, 3), generator=g).cuda()
    scr = BackwardScratch(1, n_rays, p.mc.F, p.mc.H, "cuda")
    dtok, gsmall = hydra_backward(grad_rgb, 1, n_rays, cfg.n_views, p.model, p.render_ws, scr)
    torch.cuda.synchronize()

    D = lambda a: torch.tensor(np.asarray(a), dtype=torch.float64, requires_grad=True)
    hyd = [{k: D(v) for k, v in st.items()} for st in w.hydra]
    rgbw = [(D(a), D(b)) for a, b in w.rgb]
    t64 = tok.double().cpu().requires_grad_()
    rgb = nerf_ref.hydra_rgb(hyd, rgbw, t64)
    # the forward's colour of the listed rays is this function of the tokens
    np.testing.assert_allclose(rgb.detach().numpy(),
                               p.rgb[0][lst.long()].double().cpu().numpy(), atol=2e-5)
    loss = (rgb * grad_rgb[lst.long()].double().cpu()).sum()
    loss.backward()
    np.testing.assert_allclose(dtok[:n_valid].double().cpu().numpy(), t64.grad.numpy(),
                               rtol=1e-4, atol=1e-6)
    zero = lambda n: torch.zeros(n, dtype=torch.float64)
    ref = _small_layout(w, {
        "sigma_w": zero(p.mc.H), "sigma_b": zero(1),
        "hydra": [{k: v.grad for k, v in st.items()} for st in hyd],
        "rgb": [(a.grad, b.grad) for a, b in rgbw]}).numpy()
    got = gsmall.double().cpu().numpy()
    scale = np.max(np.abs(ref))
    assert np.max(np.abs(got - ref)) <= 1e-4 * scale, (np.max(np.abs(got - ref)), scale)


def _grad_errors(got, ref):
    """(max |got - ref| / max |ref|, ||got - ref|| / ||ref||) of one tensor."""
    got = np.asarray(got, np.float64).reshape(-1)
    ref = np.asarray(ref, np.float64).reshape(-1)
    scale = max(np.max(np.abs(ref)), 1e-30)
    return (np.max(np.abs(got - ref)) / scale,
            np.linalg.norm(got - ref) / max(np.linalg.norm(ref), 1e-30))


def _flat_grads(gr):
    """Named flat list of a gradient dict (RenderTrainer.backward layout)."""
    out = [(f"dense_w{l}", gr["dense_w"][l]) for l in range(4)]
    out += [(f"dense_b{l}", gr["dense_b"][l]) for l in range(4)]
    out += [("sigma_w", gr["sigma_w"]), ("sigma_b", gr["sigma_b"])]
    for s, st in enumerate(gr["hydra"]):
        out += [(f"hydra{s}.{k}", v) for k, v in st.items()]
    for i, (a, b) in enumerate(gr["rgb"]):
        out += [(f"rgb{i}.w", a), (f"rgb{i}.b", b)]
    return out


def _oracle_grads(w, p, sub, g, img_hw, dtype, trace=None, mm_dtype=None):
    """Gradients of L = sum(g . rgb) over rays `sub` by torch autograd through
    nerf_ref.render_rays in `dtype` (float64: the target; float32: what fp32
    autograd of the same model reaches)."""
    P = nerf_ref.params_of(w, dtype=dtype, requires_grad=True)
    rgb = nerf_ref.render_rays(
        w, p.sorted[:, sub].cpu().numpy(), p.rays[:, sub].cpu().numpy(), p.K.cpu().numpy(),
        p.RT.cpu().numpy(), p.fmaps_np[None], p.bbox.cpu().numpy(), p.zdir.cpu().numpy(),
        img_hw, dtype=dtype, params=P, trace=trace, mm_dtype=mm_dtype)[0]
    (rgb * torch.from_numpy(g[:, sub]).to(dtype)).sum().backward()
    grads = dict(dense_w=[x.grad for x in P["dense_w"]], dense_b=[x.grad for x in P["dense_b"]],
                 sigma_w=P["sigma_w"].grad, sigma_b=P["sigma_b"].grad,
                 hydra=[{k: v.grad for k, v in st.items()} for st in P["hydra"]],
                 rgb=[(a.grad, b.grad) for a, b in P["rgb"]])
    return rgb.detach(), grads


def _trainer_case(prec, batch_items):
    from sailor_amd.model import NerfWeights
    from sailor_amd.train import RenderTrainer
    p = pipe()
    w = NerfWeights.init(p.mc.F, p.mc.H, perturb_std=0.01)
    w.dense_b = [np.random.default_rng(40 + l).normal(0, 0.01, p.mc.H).astype(np.float32)
                 for l in range(4)]
    tr = RenderTrainer(w, prec, "cuda", batch_items=batch_items)
    img_hw = (p.cfg.img, p.cfg.img)
    out = tr.forward(p.sorted, p.rays, p.K, p.RT, img_hw, p.fmap, p.bbox, p.zdir)
    torch.cuda.synchronize()
    valid = torch.nonzero(p.sorted[0, :, 0] >= 0).flatten().cpu().numpy()
    assert valid.size > 100
    rng = np.random.default_rng(9)
    sub = np.sort(rng.choice(valid, size=min(160, valid.size), replace=False))
    g = np.zeros((1, p.cfg.target ** 2, 3), np.float32)
    g[0, sub] = rng.normal(size=(sub.size, 3)).astype(np.float32)
    return p, w, tr, out, sub, g, img_hw


def _compare(grads, ref, tols):
    rows, bad = [], []
    for i, ((name, got), (_, want)) in enumerate(zip(_flat_grads(grads), _flat_grads(ref))):
        got = got.detach().double().cpu().numpy() if torch.is_tensor(got) else got
        mx, l2 = _grad_errors(got, want.numpy())
        rows.append(f"{name}: l2 {l2:.2e} max {mx:.2e} tol {tols[i]:.2e}")
        if l2 > tols[i]:
            bad.append(name)
    return rows, bad


def test_render_backward_fp32_columns_and_gradients():
    """fp32 differentiation form vs torch autograd of the float64 restatement,
    L = sum(g . rgb) with g non-zero on a random subset of the listed rays.

    1. Per column (ray, sample, view): the layer inputs A_l and deltas D_l the
       kernel hands to the weight-gradient GEMMs equal the restatement's
       layer inputs and dL/d pre-activation.  A delta may differ only where
       a ReLU mask flips: every column whose delta differs by more than 1e-4
       of the largest must hold a pre-activation within 5e-4 of zero at that
       layer or a later one (the float32 encoding alone moves the first
       layer's input by up to ~1e-4), and such columns must be rare (< 1%).
    2. Over the rays free of such flips, every parameter gradient (dense
       layers, occupancy head, Hydra, RGB head) is within relative L2 error
       max(1e-4, 3 x that of float32 autograd of the same restatement): the
       gradient sums cancel heavily, so float32 autograd itself sits up to
       ~1e-3 off the float64 value on some tensors."""
    p, w, tr, out, sub, g, img_hw = _trainer_case("fp32", 100000)
    F, H, S = p.mc.F, p.mc.H, p.cfg.S
    tr.backward(torch.from_numpy(g).cuda(), keep_columns=True)
    torch.cuda.synchronize()
    A, D = [[x.double().cpu().numpy() for x in part] for part in tr.columns]
    from sailor_amd.train import workspace_views
    n_valid, lst, _ = workspace_views(out["workspace"], p.cfg.target ** 2, F)
    pos = {int(r): i for i, r in enumerate(lst.cpu().numpy())}
    idx = np.array([pos[int(r)] for r in sub])
    trace = {}
    rgb64, _ = _oracle_grads(w, p, sub, g, img_hw, torch.float64, trace)
    np.testing.assert_allclose(out["rgb"][0, sub].double().cpu().numpy(), rgb64[0].numpy(),
                               atol=2e-5)
    cols = lambda M, K: M.reshape(n_valid, S, 4, -1)[idx, :, :, :K]      # [N, S, 4, K]
    x0 = torch.stack(trace["x0"], 2).detach().numpy()                     # [N, S, 4, 63+F]
    pre = [torch.stack([trace["pre"][v][l] for v in range(4)], 2).detach().numpy()
           for l in range(4)]
    dpre = [torch.stack([trace["pre"][v][l].grad for v in range(4)], 2).numpy()
            for l in range(4)]
    a0 = cols(A[0], F + 64)
    np.testing.assert_allclose(np.concatenate([a0[..., F:F + 63], a0[..., :F]], -1), x0,
                               atol=2e-4)
    for l in range(1, 4):
        ref = np.maximum(pre[l - 1], 0.0)
        np.testing.assert_allclose(cols(A[l], H), ref, atol=2e-4 * np.abs(ref).max())
    near0 = [np.abs(x).min(-1) < 5e-4 for x in pre]                     # [N, S, 4]
    flip_rays = np.zeros(sub.size, bool)
    n_cols = sub.size * S * 4
    for l in range(4):
        ref = dpre[l]
        err = np.abs(cols(D[l], H) - ref).max(-1)
        off = err > 1e-4 * np.abs(ref).max()
        explained = np.logical_or.reduce(near0[l:])
        assert not (off & ~explained).any(), (l, np.argwhere(off & ~explained)[:5])
        assert off.sum() < 0.01 * n_cols, (l, off.sum())
        flip_rays |= off.any((1, 2))
    clean = sub[~flip_rays]
    assert clean.size >= 0.8 * sub.size, (clean.size, sub.size)
    g2 = np.zeros_like(g)
    g2[0, clean] = g[0, clean]
    tr.batch_items = 128       # several item batches
    grads = tr.backward(torch.from_numpy(g2).cuda())
    torch.cuda.synchronize()
    _, ref = _oracle_grads(w, p, clean, g2, img_hw, torch.float64)
    _, ref32 = _oracle_grads(w, p, clean, g2, img_hw, torch.float32)
    base = [_grad_errors(b.double().numpy(), r.numpy())[1]
            for (_, b), (_, r) in zip(_flat_grads(ref32), _flat_grads(ref))]
    rows, bad = _compare(grads, ref, [max(1e-4, 3 * b) for b in base])
    print(f"flip rays {flip_rays.sum()} of {sub.size}")
    print("\n".join(rows))
    assert not bad, "\n".join(rows)


def test_render_backward_bf16_matches_autograd():
    """bf16 form (bf16 MFMA, fp32 accumulation) vs torch autograd of the
    float64 restatement: every parameter gradient within relative L2 error
    max(1e-2, 3 x that of mixed-precision autograd of the same restatement
    with bf16-rounded layer inputs and weights).  The sums of this loss
    cancel heavily (random-sign dL/d rgb), which makes bf16 rounding of the
    forward alone move some gradients by several percent.  Several item
    batches (256 rays each) exercise the batching."""
    p, w, tr, out, sub, g, img_hw = _trainer_case("bf16", 256)
    grads = tr.backward(torch.from_numpy(g).cuda())
    torch.cuda.synchronize()
    _, ref = _oracle_grads(w, p, sub, g, img_hw, torch.float64)
    _, emu = _oracle_grads(w, p, sub, g, img_hw, torch.float64, mm_dtype=torch.bfloat16)
    base = [_grad_errors(b.numpy(), r.numpy())[1]
            for (_, b), (_, r) in zip(_flat_grads(emu), _flat_grads(ref))]
    rows, bad = _compare(grads, ref, [max(1e-2, 3 * b) for b in base])
    rows = [f"{r} (bf16-input autograd l2 {b:.2e})" for r, b in zip(rows, base)]
    print("\n".join(rows))
    assert not bad, "\n".join(rows)


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_fused_weight_gradients_match_column_form(prec):
    """In-kernel weight-gradient accumulation vs the column form (inputs and
    deltas written per column, then D^T A GEMMs) on the same forward: both
    sum the same LDS values, so they agree to float32 summation order
    (relative L2 <= 1e-5 per tensor), on all listed rays."""
    p, w, tr, out, sub, g, img_hw = _trainer_case(prec, 512)
    gall = np.zeros_like(g)
    valid = torch.nonzero(p.sorted[0, :, 0] >= 0).flatten().cpu().numpy()
    gall[0, valid] = np.random.default_rng(3).normal(size=(valid.size, 3)).astype(np.float32)
    gt = torch.from_numpy(gall).cuda()
    tr.fused = True
    fused = tr.backward(gt)
    fused = {k: ([x.clone() for x in v] if k in ("dense_w", "dense_b") else v)
             for k, v in fused.items()}
    torch.cuda.synchronize()
    tr.fused = False
    cols = tr.backward(gt)
    torch.cuda.synchronize()
    bad = []
    for l in range(4):
        for key in ("dense_w", "dense_b"):
            a = fused[key][l].double().cpu().numpy()
            b = cols[key][l].double().cpu().numpy()
            e = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
            if e > 1e-5:
                bad.append((key, l, e))
    assert not bad, bad


@pytest.mark.parametrize("prec", ["bf16", "fp16"])
@pytest.mark.parametrize("S,V,n", [(16, 4, 1), (32, 1, 37), (48, 3, 300), (64, 2, 515)])
def test_fused_16bit_gradients_over_samples_views_and_rays(prec, S, V, n):
    """The fused form's weight gradients vs float64 products D^T A of the
    column form's matrices at the ends of the 16-bit range: one to four
    16-sample chunks, masked view slots, fewer and more rays than workgroups.
    bf16: both hold the same 16-bit values, so only the float32 summation
    differs (the bound of the comparison above).  fp16: one of the two rounds
    dL/dz w straight to 16 bits (a mixed-precision product), the other by way of
    float32, which differs by an ulp (2^-10) in one element of 2^13: 1e-5 of a
    delta's norm.  That turns the rounding (2^-11) of 1e-5 / 2^-11 = 2 % of the
    next deltas, 7e-5 of their norm at most: bound 1e-4."""
    from sailor_amd.model import NerfWeights
    from sailor_amd.train import RenderTrainer
    p = pipe()
    w = NerfWeights.init(p.mc.F, p.mc.H, perturb_std=0.01)
    w.dense_b = [np.random.default_rng(40 + l).normal(0, 0.01, p.mc.H).astype(np.float32)
                 for l in range(4)]
    tr = RenderTrainer(w, prec, "cuda", batch_items=4096)
    sel = torch.nonzero(p.sorted[0, :, 0] >= 0).flatten()[:n]
    near = p.sorted[:, sel, :1]
    far = p.sorted[:, sel].max(dim=2, keepdim=True).values
    t = (near + (far - near) * torch.linspace(0, 1, S, device="cuda")).contiguous()
    t[:, 1::5] = -1.0   # rays without samples between the others
    tr.forward(t, p.rays[:, sel].contiguous(), p.K[:, :V].contiguous(),
               p.RT[:, :V].contiguous(), (p.cfg.img, p.cfg.img), p.fmap[:, :V].contiguous(),
               p.bbox, p.zdir)
    g = torch.from_numpy(np.random.default_rng(3).normal(size=(1, sel.numel(), 3))
                         .astype(np.float32)).cuda()
    gr = tr.backward(g)
    fused = [x.double().cpu().numpy() for k in ("dense_w", "dense_b") for x in gr[k]]
    tr.backward(g, keep_columns=True)
    A, D = ([m.double().cpu().numpy() for m in ms] for ms in tr.columns)
    from sailor_amd.train import natural_first_layer_grad
    want = [d.T @ x for d, x in zip(D, A)]
    want[0] = natural_first_layer_grad(torch.from_numpy(want[0]), p.mc.F).numpy()
    want += [d.sum(0) for d in D]
    for i, (a, b) in enumerate(zip(fused, want)):
        assert np.isfinite(a).all() and np.abs(b).max() > 0
        assert np.linalg.norm(a - b) <= (1e-5 if prec == "bf16" else 1e-4) * np.linalg.norm(b), i


def test_fused_gradients_match_central_differences():
    """Fused fp32 gradients of L = sum(g . rgb) vs central finite differences
    of the float64 restatement on 12 random parameters: dense weights and
    biases of every layer, occupancy head, Hydra and RGB head.  h = 1e-5
    rather than 1e-3: a bias step moves that unit's pre-activation in every
    column, and with h = 1e-3 the ReLU kinks crossed inside +-h bias the
    difference by several percent; in float64 the smaller step costs no
    accuracy.  Bar: |fd - grad| <= 2e-3 * max|grad| of the tensor + 1e-7 (a
    column whose float32 pre-activation has the other sign than the float64
    one contributes a different ReLU derivative; the per-column test above
    bounds those columns)."""
    from sailor_amd.model import NerfWeights
    p, w, tr, out, sub, g, img_hw = _trainer_case("fp32", 100000)
    sub = sub[:48]
    g2 = np.zeros_like(g)
    g2[0, sub] = g[0, sub]
    grads = tr.backward(torch.from_numpy(g2).cuda())
    torch.cuda.synchronize()
    args = (p.sorted[:, sub].cpu().numpy(), p.rays[:, sub].cpu().numpy(), p.K.cpu().numpy(),
            p.RT.cpu().numpy(), p.fmaps_np[None], p.bbox.cpu().numpy(), p.zdir.cpu().numpy(),
            img_hw)
    gt = torch.from_numpy(g2[:, sub]).double()

    def loss(P):
        with torch.no_grad():
            return float((nerf_ref.render_rays(w, *args, params=P)[0] * gt).sum())
    rng = np.random.default_rng(17)
    picks = [("dense_w", 0), ("dense_w", 1), ("dense_w", 2), ("dense_w", 3), ("dense_b", 1),
             ("dense_b", 3), ("sigma_w", None), ("hydra0", "q"), ("hydra1", "w2"),
             ("hydra1", "b1"), ("rgb", 0), ("rgb", 2)]
    bad = []
    for name, sel in picks:
        P = nerf_ref.params_of(w)
        if name in ("dense_w", "dense_b"):
            ref_t, got_t = P[name][sel], grads[name][sel]
        elif name == "sigma_w":
            ref_t, got_t = P["sigma_w"], grads["sigma_w"]
        elif name.startswith("hydra"):
            s = int(name[-1])
            ref_t, got_t = P["hydra"][s][sel], grads["hydra"][s][sel]
        else:
            ref_t, got_t = P["rgb"][sel][0], grads["rgb"][sel][0]
        got_t = got_t.detach().double().cpu().numpy()
        idx = tuple(int(rng.integers(0, n)) for n in ref_t.shape)
        h = 1e-5
        orig = float(ref_t[idx])
        ref_t[idx] = orig + h
        lp = loss(P)
        ref_t[idx] = orig - h
        lm = loss(P)
        ref_t[idx] = orig
        fd = (lp - lm) / (2 * h)
        tol = 2e-3 * np.abs(got_t).max() + 1e-7
        if abs(fd - got_t[idx]) > tol:
            bad.append((name, sel, idx, fd, float(got_t[idx]), tol))
    assert not bad, bad
