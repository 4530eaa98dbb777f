"""GPU parity of the FastNerf inference surface (sailor_amd.InferNerf, the
drop-in for the reference's InferNerf module) against the float64
restatement oracle/fastnerf_ref.py on seeded inputs with the reference's
packed half parameters.

precision="fp32" (vector ALUs): fp32 arithmetic vs float64 on the same half
parameters, |d| <= 1e-4 + 1e-4 |ref| (NaN colour features where the
reference's epsilon-free normalisation gives 0/0: rays without samples).

precision="fp16" (default; density MLPs on fp16 MFMA): against the
restatement with the density layers' inputs rounded to half
(act_dtype=float16), |d| <= 1e-3 + 1e-3 |ref|: the fp32 and float64 sums
can round an activation to neighbouring halves (2^-11 relative), which moves
the occupancies by ~1e-4.  Against the unrounded float64 values the colour error is
that of half inputs (checked <= 2e-2), and the colour features are nearer
the rounded restatement than the float64 one (it is the one matched).  The
colour path of this form (Hydra stacks and RGB head on fp16 MFMA) rounds
the inputs of those products to half as well."""
import numpy as np
import pytest
import torch

from oracle import fastnerf_ref as fr
from tests import fastnerf_cases as fc
from tests.helpers import graph_us

pytestmark = pytest.mark.gpu


def _cu(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


@pytest.mark.parametrize("B,R,S,Vg,Vt", [(2, 64, 16, 4, 4), (1, 45, 24, 6, 3), (1, 8, 8, 1, 1)])
def test_infer_nerf_matches_float64(B, R, S, Vg, Vt):
    from sailor_amd import InferNerf
    pd, pc, _ = fc.params()
    t, z, ps, geo, rgb, frgb, dirs = fc.nerf_inputs(B, R, S, Vg, Vt)
    d, c, f = InferNerf.infer_nerf(_cu(t), _cu(z).view(-1, 1), _cu(ps).view(-1, 1), _cu(geo),
                                   _cu(rgb), _cu(frgb), _cu(dirs), _cu(pd, torch.float16),
                                   _cu(pc, torch.float16), B, R, S, Vg, Vt, 0,
                                   precision="fp32")
    torch.cuda.synchronize()
    rd, rc, rf = fr.infer_nerf(t, z, ps, geo, rgb, frgb, dirs, pd, pc, B, R, S, Vg, Vt)
    for got, ref in ((d, rd), (c, rc), (f, rf)):
        np.testing.assert_allclose(got.double().cpu().numpy(), ref.numpy(), rtol=1e-4,
                                   atol=1e-4, equal_nan=True)
    # rays without samples: 0/0 in the normalisation gives NaN features; the
    # colour head's max(x, 0) turns them into a finite colour, as in the
    # reference
    dropped = t[..., -1] < 0
    assert np.isnan(f.cpu().numpy()[dropped]).all()
    assert not np.isnan(f.cpu().numpy()[~dropped]).any() and np.isfinite(c.cpu().numpy()).all()


def test_infer_density_matches_float64():
    from sailor_amd import InferNerf
    pd, _, _ = fc.params()
    B, N, V = 2, 777, 4
    _, z, ps, geo, _, _, _ = fc.nerf_inputs(B, N, 1, V, 1, seed=9)
    out = InferNerf.infer_density(_cu(z).view(-1, 1), _cu(ps).view(-1, 1), _cu(geo),
                                  _cu(pd, torch.float16), B, N, V, 0, precision="fp32")
    torch.cuda.synchronize()
    ref = fr.infer_density(z, ps, geo, pd, B, N, V)
    assert out.shape == (B, 1, N)
    np.testing.assert_allclose(out.double().cpu().numpy(), ref.numpy(), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("B,R,S,Vg,Vt", [(2, 64, 16, 4, 4), (1, 45, 24, 6, 3), (1, 8, 8, 1, 1),
                                         (1, 30, 8, 2, 2), (1, 12, 8, 9, 2)])
def test_infer_nerf_fp16_mfma(B, R, S, Vg, Vt):
    """Default precision: 1, 2, 4 and 8 view slots on MFMA, 9 views on the
    fp32 fallback."""
    from sailor_amd import InferNerf
    pd, pc, _ = fc.params()
    t, z, ps, geo, rgb, frgb, dirs = fc.nerf_inputs(B, R, S, Vg, Vt)
    d, c, f = InferNerf.infer_nerf(_cu(t), _cu(z).view(-1, 1), _cu(ps).view(-1, 1), _cu(geo),
                                   _cu(rgb), _cu(frgb), _cu(dirs), _cu(pd, torch.float16),
                                   _cu(pc, torch.float16), B, R, S, Vg, Vt, 0)
    torch.cuda.synchronize()
    act = torch.float16 if Vg <= 8 else None
    rd, rc, rf = fr.infer_nerf(t, z, ps, geo, rgb, frgb, dirs, pd, pc, B, R, S, Vg, Vt,
                               act_dtype=act)
    tol = 1e-3 if act is not None else 1e-4
    for got, ref in ((d, rd), (c, rc), (f, rf)):
        np.testing.assert_allclose(got.double().cpu().numpy(), ref.numpy(), rtol=tol, atol=tol,
                                   equal_nan=True)
    if act is not None:
        _, rc64, rf64 = fr.infer_nerf(t, z, ps, geo, rgb, frgb, dirs, pd, pc, B, R, S, Vg, Vt)
        e64 = np.nanmax(np.abs(c.double().cpu().numpy() - rc64.numpy()))
        f64 = np.nanmax(np.abs(f.double().cpu().numpy() - rf64.numpy()))
        f16 = np.nanmax(np.abs(f.double().cpu().numpy() - rf.numpy()))
        print(f"colour vs float64 {e64:.2e}; features vs float64 {f64:.2e}, vs the rounded "
              f"restatement {f16:.2e}")
        assert e64 <= 2e-2 and f16 <= f64


def test_infer_density_fp16_mfma():
    from sailor_amd import InferNerf
    pd, _, _ = fc.params()
    for B, N, V in ((2, 777, 4), (1, 301, 3), (1, 64, 8)):
        _, z, ps, geo, _, _, _ = fc.nerf_inputs(B, N, 1, V, 1, seed=9)
        out = InferNerf.infer_density(_cu(z).view(-1, 1), _cu(ps).view(-1, 1), _cu(geo),
                                      _cu(pd, torch.float16), B, N, V, 0)
        torch.cuda.synchronize()
        ref = fr.infer_density(z, ps, geo, pd, B, N, V, act_dtype=torch.float16)
        np.testing.assert_allclose(out.double().cpu().numpy(), ref.numpy(), rtol=1e-3,
                                   atol=1e-4)


def test_infer_blending_matches_float64():
    from sailor_amd import InferNerf
    _, _, pb = fc.params()
    rng = np.random.default_rng(4)
    nf = rng.normal(0, 1, (1000, 40)).astype(np.float32)
    rf = rng.normal(0, 1, (1000, 30)).astype(np.float32)
    out = InferNerf.infer_blending(_cu(nf), _cu(rf), _cu(pb, torch.float16), 0)
    torch.cuda.synchronize()
    ref = fr.infer_blending(nf, rf, pb)
    np.testing.assert_allclose(out.double().cpu().numpy(), ref.numpy(), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("V", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("B,N", [(2, 1), (5, 7), (3, 31), (2, 33), (40, 9), (2, 4000)])
def test_batches_share_tiles_of_points(B, N, V):
    """Batches of fewer points than a tile of 32, of more, and more points than
    there are waves: each point's occupancy is the one its batch alone gives, bit
    for bit (a column of an MFMA does not see the others)."""
    from sailor_amd import InferNerf
    pd = _cu(fc.params()[0], torch.float16)
    _, z, ps, geo, _, _, _ = fc.nerf_inputs(B, N, 1, V, 1, seed=N + V)
    z, ps, geo = _cu(z), _cu(ps), _cu(geo)
    got = InferNerf.infer_density(z, ps, geo, pd, B, N, V, 0)
    for b in range(B):
        part = slice(b * V * N, (b + 1) * V * N)
        alone = InferNerf.infer_density(z[part], ps[part], geo[part].contiguous(), pd, 1, N, V, 0)
        assert torch.equal(got[b], alone[0]), b


def test_batches_of_few_points_infer_nerf():
    """The geometry features of the texture views (fewer than the geometry
    views) come out per batch too: depth, colour and features of 5 batches of
    3 rays x 5 samples equal each batch's alone."""
    from sailor_amd import InferNerf
    pd, pc, _ = fc.params()
    B, R, S, Vg, Vt = 5, 3, 5, 4, 2
    t, z, ps, geo, rgb, frgb, dirs = fc.nerf_inputs(B, R, S, Vg, Vt, seed=3)
    g = dict(t=t.reshape(B, -1), z=z.reshape(B, -1), ps=ps.reshape(B, -1), geo=geo.reshape(B, -1),
             rgb=rgb.reshape(B, -1), frgb=frgb.reshape(B, -1), dirs=dirs.reshape(B, -1))
    run = lambda n, s: InferNerf.infer_nerf(
        _cu(g["t"][s]).view(n, R, S), *[_cu(g[k][s]).view(-1, c) for k, c in
                                        (("z", 1), ("ps", 1), ("geo", 16), ("rgb", 3),
                                         ("frgb", 16), ("dirs", 3))],
        _cu(pd, torch.float16), _cu(pc, torch.float16), n, R, S, Vg, Vt, 0)
    whole = run(B, slice(0, B))
    for b in range(B):
        for w, a in zip(whole, run(1, slice(b, b + 1))):
            assert torch.equal(w[b].nan_to_num(7.0), a[0].nan_to_num(7.0)), b


def test_many_short_batches_take_the_time_of_their_points():
    """4096 batches of 33 points take at most 1.6 times what the same points do
    in one batch (measured 1.1; 5 with a workgroup per batch)."""
    from sailor_amd import InferNerf
    pd = _cu(fc.params()[0], torch.float16)
    B, N, V = 4096, 33, 4
    g = torch.Generator(device="cuda").manual_seed(0)
    z = torch.rand(B * V * N, generator=g, device="cuda")
    geo = torch.randn((B * V * N, 16), generator=g, device="cuda")
    many = graph_us(lambda: InferNerf.infer_density(z, z, geo, pd, B, N, V, 0))
    one = graph_us(lambda: InferNerf.infer_density(z, z, geo, pd, 1, B * N, V, 0))
    print(f"{B} batches {many:.1f} us, one {one:.1f} us")
    assert many <= 1.6 * one


@pytest.mark.parametrize("V", [1, 3, 8])
def test_density_features_may_start_on_any_float(V):
    """Geometry features that are a view at an odd float of a larger tensor."""
    from sailor_amd import InferNerf
    pd = _cu(fc.params()[0], torch.float16)
    N = 77
    _, z, ps, geo, _, _, _ = fc.nerf_inputs(1, N, 1, V, 1, seed=V)
    z, ps, geo = _cu(z), _cu(ps), _cu(geo)
    want = InferNerf.infer_density(z, ps, geo, pd, 1, N, V, 0)
    for shift in (1, 2, 3):
        held = torch.empty(geo.numel() + shift, device="cuda")
        odd = held[shift:].view(geo.shape)
        odd.copy_(geo)
        assert odd.data_ptr() % 16 == 4 * shift and odd.is_contiguous()
        assert torch.equal(InferNerf.infer_density(z, ps, odd, pd, 1, N, V, 0), want)
