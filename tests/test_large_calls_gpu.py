"""Calls of more rays than one launch holds lanes for (2^32): every ray is
processed.  Inputs are as small as the entry points allow per ray; the outputs
of the first and last rays are compared with a small call's."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.helpers import scene_inputs, target_rays_np

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.fixture(autouse=True)
def _free():
    yield
    torch.cuda.empty_cache()


def test_compositing_of_more_than_2_26_rows_of_33_samples():
    import sailor_amd.VoxelEncoding as VE
    R, S, n = (1 << 26) + 5, 33, 777
    g = torch.Generator(device="cuda").manual_seed(0)
    t = torch.rand((1, n, S), generator=g, device="cuda").sort(-1)[0]
    s = torch.rand((1, n, S), generator=g, device="cuda") * 0.3
    f = torch.randn((1, n, S, 1), generator=g, device="cuda")
    grads = [torch.randn((1, n, 1), generator=g, device="cuda") for _ in range(4)]

    def big(x):   # n distinct rows at both ends, zeros between
        b = torch.zeros((1, R) + x.shape[2:], device="cuda")
        b[:, :n], b[:, -n:] = x, x
        return b
    small = VE.volume_render_torch_forward(t, s, f, None, True)
    bt, bs, bf = big(t), big(s), big(f)
    for o, r in zip(VE.volume_render_torch_forward(bt, bs, bf, None, True), small):
        assert torch.equal(o[:, :n], r) and torch.equal(o[:, -n:], r)
        assert not o[:, n:-n].any()
    small = VE.volume_render_torch_backward(*grads, t, s, f, None, True)
    for o, r in zip(VE.volume_render_torch_backward(*[big(x) for x in grads], bt, bs, bf, None,
                                                    True), small):
        assert torch.equal(o[:, :n], r) and torch.equal(o[:, -n:], r)


def _tree(rate=4, dim=32):
    from sailor_amd import VoxelEncoding as VE
    inp = scene_inputs(0, 4, 128, 128, 150.0)
    o = orc.integrate(inp["K"], inp["RT"], inp["R"], inp["T"], inp["colors"], inp["depths"],
                      (dim, dim, dim), fixed_bbox=None)
    oc, ocnt = orc.merge(o["occ"], rate)
    n0, n1 = int(o["num_occ"].sum()), int(ocnt.sum())
    tree = VE.MultiLayerOctree(2, 1, rate, 0)
    tree.init_octree([_t(o["occ"]), _t(oc)], [n0, n1],
                     [_t(o["num_occ"].astype(np.int32).reshape(1, 1)),
                      _t(ocnt.astype(np.int32).reshape(1, 1))], [0, n0],
                     _t(o["voxel_size"].reshape(1, 1)), _t(o["vol_bbox"]))
    tree.build_octree()
    return tree


def test_walks_of_more_than_2_29_rays():
    """Rays that miss the volume, 64 rays of a camera at both ends: traversal
    that stops at the first node, sampling of its hits, the recursive traversal
    with its 2 entries a row kept (more overflow, which the status reports)."""
    from sailor_amd._lib import call, ptr, stream_of
    tree = _tree()
    r6 = orc.rays(*target_rays_np(64, 64, 75.0), 64, 64)[0, 0].reshape(-1, 6)[2000:2064]
    n, R = 64, (1 << 29) + 67
    dev, st = torch.device("cuda"), stream_of("cuda")
    f32 = lambda *s: torch.full(s, 7.0, device=dev)
    i32 = lambda *s: torch.full(s, 7, dtype=torch.int32, device=dev)

    def run(R):
        ori, dirs = f32(R, 3), f32(R, 3)   # from (7, 7, 7) away
        for k, x in ((0, ori), (3, dirs)):
            x[:n] = _t(r6[:, k:k + 3])
            x[-n:] = x[:n].clone()
        idx, t0, t1, vl, status = i32(R), f32(R), f32(R), f32(R), torch.zeros_like(i32(4))
        head = [ptr(tree._vols[1]), ptr(tree.node_pos), ptr(tree.node_info),
                tree.node_pos.shape[0], ptr(tree.volume_bbox), ptr(tree.voxel_size), 1, 32, 8, 4]
        call("sailor_octree_voxel_traversal", *head, ptr(ori), ptr(dirs), R, 1, -1, 1, 1,
             ptr(idx), ptr(t0), ptr(t1), ptr(vl), ptr(status), st)
        out = [(idx, -1), (vl, 0.0)]
        noise, si, sz = f32(R), i32(R), f32(R)
        call("sailor_octree_sampling_coarse", ptr(idx), ptr(t0), ptr(t1), ptr(noise), ptr(vl),
             ptr(tree.node_pos), ptr(tree.voxel_size), 1, R, 1, 1, 4, ptr(si), ptr(sz), st)
        ai, az = i32(R), f32(R)
        call("sailor_octree_sampling", ptr(idx), ptr(t0), ptr(t1), ptr(noise), ptr(vl),
             ptr(tree.node_pos), tree.node_pos.shape[0], ptr(tree.voxel_size), 1, R, 1, 1, 1, 2,
             ptr(ai), ptr(az), st)
        out += [(si, -1), (sz, -1.0), (ai, -1), (az, -1.0)]
        ci, c0, c1, fi, f0, f1 = i32(R), f32(R), f32(R), i32(R, 2), f32(R, 2), f32(R, 2)
        length = f32(R)
        call("sailor_octree_traversal", *head, ptr(ori), ptr(dirs), R, 1, 2, -1, 1, ptr(ci),
             ptr(c0), ptr(c1), ptr(fi), ptr(f0), ptr(f1), ptr(length), ptr(status), st)
        return out + [(ci, -1), (fi, -1), (f0, -1.0), (length, 0.0)]
    small = run(2 * n)
    assert (small[0][0] >= 0).any() and (small[2][0] >= 0).any()
    for (o, miss), (r, _) in zip(run(R), small):
        assert torch.equal(o[:n], r[:n]) and torch.equal(o[-n:], r[n:])
        assert bool((o[n:-n] == miss).all())


def test_trace_of_a_target_of_more_than_2_29_pixels():
    """The first and last rows of a 32768 x 16400 target, one sample a ray,
    against the same pixels of a target that has only those rows."""
    from sailor_amd.render import trace_sample
    tree = _tree()
    H, W, S = 16400, 32768, 1
    K, R, T = target_rays_np(H, W, 20000.0)
    K, R, T = (_t(x[0]).float() for x in (K, R, T))
    box, vs = tree.volume_bbox.reshape(1, 3, 2), tree.voxel_size
    noise = torch.full((1, H * W, S), 0.5, device="cuda")
    _, sidx, st, vl = trace_sample(K, R, T.reshape(1, 3), (H, W), tree._vols[1], tree.node_pos,
                                   tree.node_info, box, vs, 32, 4, noise, want_rays=False)
    mid = H // 2 * W
    assert (sidx[0, mid:mid + W] >= 0).any()
    for row in (0, H // 2, H - 1):
        K2 = K.clone()
        K2[0, 1, 2] -= row   # the target whose row 0 is this row
        _, s2, t2, v2 = trace_sample(K2, R, T.reshape(1, 3), (1, W), tree._vols[1], tree.node_pos,
                                     tree.node_info, box, vs, 32, 4, noise[:, :W], want_rays=False)
        part = slice(row * W, (row + 1) * W)
        # a row offset taken off the principal point moves a ray by a rounding
        same = (s2 == sidx[:, part]).float().mean()
        assert same > 0.999, (row, float(same))
        assert ((v2 - vl[:, part]).abs() < 1e-4).float().mean() > 0.999
    del noise
    assert bool(((sidx >= 0) == (st >= 0)).all())
