"""Renders of both forms against the oracle's march, heads and inference compositing of the same rays.  Front to back in
rounds: rays with one to hundreds of samples, thin and opaque fields, chunks of rays larger than a hit batch holds, one
and odd ray counts, boxes that are no cube.  Whole rays: several ray chunks, several hit batches per chunk, several
samples per voxel.  A ray's colour has the same bits in both."""
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import pyoracle as orc  # noqa: E402

import importlib  # noqa: E402

from helpers import assert_close, pkg  # noqa: E402

scenes = importlib.import_module("3dmaker_amd.scenes")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,batch,cascades,bias,hidden,layers", [
    (1, 1 << 14, 1, 0.0, 64, 3),        # whole rays: a hit batch below 2^18.  One ray
    (819, 1 << 14, 1, 0.0, 64, 3),
    (820, 1 << 14, 1, 0.0, 64, 3),
    (2047, 1 << 14, 1, 4.0, 32, 3),     # thin field: no ray saturates
    (5000, 1 << 14, 1, -6.0, 64, 2),    # opaque field
    (777, 1 << 12, 3, 1.0, 64, 4),      # cascades; a colour head outside the MFMA kernels' shapes
    (13107, 1 << 18, 1, 0.0, 64, 3),    # the most rays that go whole at this hit batch, and one more, in rounds
    (13108, 1 << 18, 1, 0.0, 64, 3),
    (13107, (1 << 18) - 16, 1, 0.0, 32, 2),  # a hit batch below the rounds'
    (14001, 1 << 18, 1, 4.0, 32, 3),    # rounds.  Thin field: no ray saturates, many rounds
    (40001, 1 << 18, 1, -6.0, 64, 2),   # opaque field: most rays end in the first round; two chunks of rays
    (15001, 1 << 18, 3, 1.0, 64, 4),    # cascades; a colour head outside the MFMA kernels' shapes
])
def test_render_matches_whole_rays(R, batch, cascades, bias, hidden, layers):
    check(R, batch, cascades, bias, hidden, layers)


@pytest.mark.parametrize("R,K", [(900, 1), (3000, 2), (700, 3)])
def test_whole_rays_in_chunks_and_hit_batches(R, K):
    """One and several samples per voxel: whole rays, here of several chunks of 256 rays."""
    batch = 20 * R if K == 1 else 1 << 12
    N = check(R, batch + 16, 1, 0.0, 64, 2, K=K, chunk=256)
    assert K == 1 or N > 3 * batch        # several hit batches


@pytest.mark.parametrize("mn,mx,cascades", [((-1.3, -1.5, -1.4), (1.4, 1.5, 1.2), 1), ((-1.5,) * 3, (1.5, 1.5, 1.75), 3)])
def test_rounds_in_a_box_that_is_no_cube(mn, mx, cascades):
    check(14003, 1 << 18, cascades, 1.0, 64, 3, mn=mn, mx=mx)


def check(R, batch, cascades, bias, hidden, layers, K=1, chunk=1024, mn=(-1.5,) * 3, mx=(1.5,) * 3):
    print(f"[render rounds] R={R} batch={batch} C={cascades} bias={bias} colour {hidden} x {layers} "
          f"K={K} chunk={chunk} box {mn} {mx}", flush=True)
    P = pkg()
    res, mips, T_ = 64, 4, 1 << 14
    o = P.Nerf.default_options()
    o.gridResolution[:] = [res] * 3
    o.aabbMin[:], o.aabbMax[:] = mn, mx
    o.levelsMipmap, o.numCascades, o.samplesPerVoxel = mips, cascades, K
    o.hashTableSize, o.growthFactor = T_, 1.447
    o.colorHiddenDim, o.colorNumLayers = hidden, layers
    o.batchSize, o.rayChunkSize, o.renderBatchSize = batch, chunk, batch
    o.densityBias = bias
    o.bgColor[:] = [0.25, 0.5, 1.0]
    nerf = P.Nerf(o)
    rng = np.random.default_rng(3)
    table = rng.normal(0, 0.5, 16 * T_ * 2).astype(np.float32)
    nerf.density.load_hashgrid(table)
    l0 = [rng.random((res, res, res)) < (0.5 if c == 0 else 0.02) for c in range(cascades)]
    bits = scenes.pack_grid(l0, mips)
    nerf.set_occupancy(bits)
    nerf.set_memory_mode(True)
    ro, rd = scenes.rays_c4(R, n_cams=8, seed=6)
    d_o, d_d = torch.from_numpy(ro).cuda(), torch.from_numpy(rd).cuda()
    rgb = torch.full((R, 3), -1.0, device="cuda")
    nerf.render(d_o, d_d, R, rgb)
    rgb2 = torch.full((R, 3), -1.0, device="cuda")
    nerf.render(d_o, d_d, R, rgb2)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(rgb.cpu().numpy(), rgb2.cpu().numpy())

    mn, mx = np.float32(mn), np.float32(mx)
    di, near, far = orc.ray_aabb_inv(ro, rd, mn, mx, cascades)
    m = orc.march_hits(ro, rd, di, near, far, bits, [res] * 3, mn, mx, cascades, mips, K, 1 << 24)
    N = int(m["total"])
    cnt, off, t, ridx = m["counts"][:R], m["offsets"][:R], m["t"][:N], m["ray_idx"][:N]
    assert N > 0 or R == 1
    def weights(net, i, h, out, n):
        W = np.zeros(sum((out if l == n - 1 else h) * (i if l == 0 else h) for l in range(n)), np.float32)
        B = np.zeros(sum(out if l == n - 1 else h for l in range(n)), np.float32)
        net.save_weights(W, B)
        return W.astype(np.float16), B

    dW, dB = weights(nerf.density, 32, 64, 16, 2)
    cW, cB = weights(nerf.color, 32, hidden, 8, layers)
    enc = orc.hash_encode(np.ascontiguousarray(m["pos"][:N]), table.astype(np.float16), T_, 16, 16, 1.447)
    y, _ = orc.mlp_forward(enc, dW, dB, 32, 64, 16, 2, save_acts=False)
    cin, sig = orc.sh_gather(rd, ridx, y, bias)
    c, _ = orc.mlp_forward(cin, cW, cB, 32, hidden, 8, layers, out_act=1, save_acts=False)
    want = orc.composite_infer(off, cnt, t, sig, np.ascontiguousarray(c[:, :3]), np.float32([0.25, 0.5, 1.0]))
    want = want["rgb"] if isinstance(want, dict) else want[0]
    assert_close(rgb.cpu().numpy(), want, what="rgb")
    if cascades == 1 and R > 1:
        assert cnt.max() > 17  # more than one round
    nerf.close()
    return N


@pytest.mark.parametrize("hidden,layers", [(32, 3), (64, 2), (64, 4)])   # the last one outside the MFMA heads
def test_a_ray_has_one_colour_however_rays_are_grouped(hidden, layers):
    """The same rays in one call (rounds), in calls small enough to go whole, alone, and with another hit batch: the
    same bits."""
    P = pkg()
    res, mips, T_, R, batch = 64, 4, 1 << 14, 16000, 1 << 18
    small = batch // 20                  # the most rays that go whole
    o = P.Nerf.default_options()
    o.gridResolution[:] = [res] * 3
    o.aabbMin[:], o.aabbMax[:] = [-1.5] * 3, [1.5] * 3
    o.levelsMipmap, o.numCascades, o.samplesPerVoxel = mips, 1, 1
    o.hashTableSize, o.growthFactor = T_, 1.447
    o.colorHiddenDim, o.colorNumLayers = hidden, layers
    o.batchSize, o.rayChunkSize, o.renderBatchSize = batch, 512, 1 << 19
    nerf = P.Nerf(o)
    rng = np.random.default_rng(3)
    nerf.density.load_hashgrid(rng.normal(0, 0.5, 16 * T_ * 2).astype(np.float32))
    nerf.set_occupancy(scenes.pack_grid([rng.random((res, res, res)) < 0.3], mips))
    ro, rd = scenes.rays_c4(R, n_cams=8, seed=6)
    d_o, d_d = torch.from_numpy(ro).cuda(), torch.from_numpy(rd).cuda()

    def render(cuts):
        rgb = torch.full((R, 3), -1.0, device="cuda")
        for a, b in zip(cuts[:-1], cuts[1:]):
            nerf.render(d_o[a:b], d_d[a:b], b - a, rgb[a:b])
        torch.cuda.synchronize()
        return rgb.cpu().numpy()

    whole = render([0, R])
    assert len(np.unique(whole[:, 0])) > R // 2   # colours, not the background
    np.testing.assert_array_equal(render(list(range(0, R, small)) + [R]), whole)
    np.testing.assert_array_equal(render([0, 1, 2, 17, 3000, R]), whole)
    nerf.set_memory_mode(True)                    # a hit batch of 2^19: R <= 2^19 / 20 goes whole
    np.testing.assert_array_equal(render([0, R]), whole)
    nerf.close()
