"""The fused MLP's 16x16x32 kernels at the edges of what they take: input widths that are not a multiple of 32,
padded and full-width inputs and outputs, one to many layers, ragged and tiny batches, both tile counts per wave;
and unaligned rows through the launchers.  Tolerances are those of fp16 operands with fp32 sums (2e-3 abs,
1e-2 rel), scaled to the largest gradient for gradients."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import pyoracle as orc  # noqa: E402

from helpers import assert_close, pkg  # noqa: E402

pytestmark = pytest.mark.gpu


def layer_sizes(i, h, o, n):
    return [((o if l == n - 1 else h), (i if l == 0 else h)) for l in range(n)]


def make(i, h, o, n, seed):
    rng = np.random.default_rng(seed)
    W = [(rng.uniform(-1, 1, s) / np.sqrt(s[1])).astype(np.float32) for s in layer_sizes(i, h, o, n)]
    B = [rng.uniform(-0.1, 0.1, s[0]).astype(np.float32) for s in layer_sizes(i, h, o, n)]
    return W, B


def flat(xs):
    return np.concatenate([x.reshape(-1) for x in xs])


def pointers(ts):
    return torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device="cuda")


@pytest.mark.parametrize("i,h,o,n,act,N,shift", [
    (24, 32, 4, 2, 0, 1, 0), (8, 32, 8, 3, 1, 17, 0), (40, 64, 24, 2, 0, 33, 1), (64, 64, 64, 4, 0, 1000, 0),
    (32, 64, 8, 3, 1, 32769, 0), (128, 128, 128, 2, 0, 257, 0), (32, 128, 16, 2, 0, 40000, 1), (32, 32, 16, 9, 0, 100, 0),
    (96, 32, 32, 2, 1, 65, 0), (16, 64, 64, 3, 0, 31, 1)])
def test_launchers_forward_and_backward(i, h, o, n, act, N, shift):
    """shift: every buffer starts that many elements off its allocation."""
    print(f"[mlp shapes] {i}-{h}-{o} x {n} act={act} N={N} shift={shift}", flush=True)
    P = pkg()
    W, B = make(i, h, o, n, 3)
    rng = np.random.default_rng(4)
    x = rng.standard_normal((N, i)).astype(np.float16)
    dy = (rng.standard_normal((N, o)) * 0.05).astype(np.float16)

    def dev(a):
        t = torch.zeros(a.size + shift, dtype=torch.from_numpy(a[:0]).dtype, device="cuda")
        t[shift:] = torch.from_numpy(a.reshape(-1)).cuda()
        return t[shift:]

    w16 = [w.astype(np.float16) for w in W]
    dW16, dB = [dev(w) for w in w16], [dev(b) for b in B]
    acts = [dev(x)] + [dev(np.zeros((N, h), np.float16)) for _ in range(n - 1)]
    gW, gB = [dev(np.full_like(w, 0.5)) for w in W], [dev(np.full_like(b, 0.25)) for b in B]
    y, y2 = dev(np.zeros((N, o), np.float32)), dev(np.zeros((N, o), np.float32))
    dx = dev(np.zeros((N, i), np.float16))
    d_dy = dev(dy)
    arrays = [pointers(t) for t in (acts, dW16, dB, gW, gB)]
    opt = P.MLPOption(inputDim=i, hiddenDim=h, outputDim=o, numLayers=n, activationType=0, outputActivation=act)
    P.launch("launchNetworkFusionGradKernel", C.byref(opt), acts[0], arrays[0], arrays[1], arrays[2], y, N, None)
    P.launch("launchNetworkFusionKernel", C.byref(opt), acts[0], arrays[1], arrays[2], y2, N, None)
    backward = o < 128  # 128 wide throughout: the backward is refused (LDS)
    if backward:
        P.launch("launchNetworkFusionBackwardKernel", C.byref(opt), d_dy, arrays[1], arrays[2], arrays[0], arrays[3],
                 arrays[4], dx, N, None)
    torch.cuda.synchronize()
    y_ref, a_ref = orc.mlp_forward(x, flat(w16), flat(B), i, h, o, n, out_act=act)
    got = y.cpu().numpy().reshape(N, o)
    assert_close(got, y_ref, what="output")
    np.testing.assert_array_equal(got, y2.cpu().numpy().reshape(N, o))
    a = np.stack([t.cpu().numpy().reshape(N, h) for t in acts[1:]])
    assert_close(a, a_ref, what="activations")
    if not backward:
        return
    rW, rB, rdx = orc.mlp_backward(dy, x, a, flat(w16), i, h, o, n)
    assert_close(flat([t.cpu().numpy() for t in gW]) - 0.5, rW, atol=2e-3 * max(1.0, np.abs(rW).max()), what="dW")
    assert_close(flat([t.cpu().numpy() for t in gB]) - 0.25, rB, atol=2e-3 * max(1.0, np.abs(rB).max()), what="db")
    assert_close(dx.cpu().numpy().reshape(N, i), rdx, what="dx")


@pytest.mark.parametrize("grid", [False, True])
@pytest.mark.parametrize("h,o,n,N", [(32, 64, 2, 40), (32, 128, 3, 32769), (64, 128, 4, 17), (64, 96, 2, 1),
                                     (32, 36, 2, 40), (64, 48, 2, 32769), (128, 80, 3, 33), (64, 112, 4, 17),
                                     (32, 100, 3, 257), (128, 112, 2, 1), (64, 40, 3, 100)])
def test_output_widths(h, o, n, N, grid):
    """Outputs wider than the hidden layers, and widths whose last pair of 16-row blocks is one of padding: both forward launchers of each net."""
    print(f"[mlp outputs] {h}-{o} x {n} N={N} grid={grid}", flush=True)
    P = pkg()
    W, B = make(32, h, o, n, 5)
    rng = np.random.default_rng(6)
    w16 = [w.astype(np.float16) for w in W]
    dW16, dB = [torch.from_numpy(w).cuda() for w in w16], [torch.from_numpy(b).cuda() for b in B]
    acts = [torch.zeros(N, 32 if l == 0 else h, dtype=torch.float16, device="cuda") for l in range(n)]
    y, y2 = torch.zeros(N, o, device="cuda"), torch.zeros(N, o, device="cuda")
    pa, pw, pb = pointers(acts), pointers(dW16), pointers(dB)
    if grid:
        T_, L, b = 1 << 12, 16, 1.3
        table = rng.uniform(-1, 1, L * T_ * 2).astype(np.float16)
        pos = np.zeros((N, 4), np.float32)
        pos[:, :3] = rng.random((N, 3))
        d_tab, d_pos = torch.from_numpy(table).cuda(), torch.from_numpy(pos).cuda()
        opt = P.MLPGridOptions(vectorDim=4, hiddenDim=h, outputDim=o, numLayers=n, activationType=0, tableSize=T_,
                               numLevels=L, b=b, lowestSize=16, featuresLevel=2)
        P.launch("launchNetworkFusionHashTableGradKernel", C.byref(opt), d_tab, d_pos, pa, pw, pb, y, N, None)
        P.launch("launchNetworkFusionHashTableKernel", C.byref(opt), d_tab, d_pos, pw, pb, y2, N, None)
        x = orc.hash_encode(pos, table, T_, L, 16, b)
    else:
        x = rng.standard_normal((N, 32)).astype(np.float16)
        acts[0].copy_(torch.from_numpy(x))
        opt = P.MLPOption(inputDim=32, hiddenDim=h, outputDim=o, numLayers=n, activationType=0, outputActivation=0)
        P.launch("launchNetworkFusionGradKernel", C.byref(opt), acts[0], pa, pw, pb, y, N, None)
        P.launch("launchNetworkFusionKernel", C.byref(opt), acts[0], pw, pb, y2, N, None)
    torch.cuda.synchronize()
    y_ref, a_ref = orc.mlp_forward(x, flat(w16), flat(B), 32, h, o, n)
    assert_close(y.cpu().numpy(), y_ref, what="output")
    np.testing.assert_array_equal(y.cpu().numpy(), y2.cpu().numpy())
    assert_close(np.stack([t.cpu().numpy() for t in acts[1:]]), a_ref, what="activations")


def test_net_with_outputs_wider_than_its_hidden_layers():
    """The class: forward, inference and a gradient from outside, 32 wide with 64 outputs."""
    P = pkg()
    N = 300
    net = P.Net(P.MLPOption(inputDim=32, hiddenDim=32, outputDim=64, numLayers=3, activationType=0, outputActivation=0),
                N, seed=2)
    W, B = make(32, 32, 64, 3, 8)
    net.load_weights(flat(W), flat(B))
    rng = np.random.default_rng(2)
    x, dy = rng.standard_normal((N, 32)).astype(np.float16), (rng.standard_normal((N, 64)) * 0.05).astype(np.float16)
    out, inf = torch.zeros(N, 64, device="cuda"), torch.zeros(N, 64, device="cuda")
    dx = torch.zeros(N, 32, dtype=torch.float16, device="cuda")
    d_x = torch.from_numpy(x).cuda()
    net.zero_grad()
    net.forward(d_x, out, N)
    net.backward(N, custom_grad=torch.from_numpy(dy).cuda(), dx_out=dx)
    net.inference(d_x, inf, N)
    torch.cuda.synchronize()
    w16 = flat([w.astype(np.float16) for w in W])
    y_ref, a_ref = orc.mlp_forward(x, w16, flat(B), 32, 32, 64, 3)
    assert_close(out.cpu().numpy(), y_ref, what="output")
    np.testing.assert_array_equal(out.cpu().numpy(), inf.cpu().numpy())
    rdx = orc.mlp_backward(dy, x, a_ref, w16, 32, 32, 64, 3)[2]
    # one fp16 rounding of a hidden unit moves a gradient by a weight times dL/dy: 2e-3 covers it
    assert_close(dx.cpu().numpy(), rdx, what="dx")


@pytest.mark.parametrize("N", [1, 40, 32769])
def test_padded_ends_match_the_padded_net(N):
    """3 -> 8 inputs and 5 -> 8 outputs padded inside the kernel: activation 0, padded and caller's outputs."""
    P = pkg()
    net = P.Net(P.MLPOption(inputDim=3, hiddenDim=64, outputDim=5, numLayers=3, activationType=0, outputActivation=1),
                N, seed=2)
    x = np.random.default_rng(1).standard_normal((N, 3)).astype(np.float16)
    W, B = make(8, 64, 8, 3, 6)
    net.load_weights(flat(W), flat(B))
    out, inf = torch.zeros(N, 5, device="cuda"), torch.zeros(N, 5, device="cuda")
    d_x = torch.from_numpy(x).cuda()
    net.forward(d_x, out, N)
    net.inference(d_x, inf, N)
    torch.cuda.synchronize()
    xp = np.zeros((N, 8), np.float16)
    xp[:, :3] = x
    y_ref, _ = orc.mlp_forward(xp, flat([w.astype(np.float16) for w in W]), flat(B), 8, 64, 8, 3, out_act=1)
    assert_close(out.cpu().numpy(), y_ref[:, :5], what="output")
    np.testing.assert_array_equal(out.cpu().numpy(), inf.cpu().numpy())


@pytest.mark.parametrize("N,vec,out", [((1 << 15) - 1, 3, 16), (1 << 15, 3, 16), (40001, 4, 3)])
def test_grid_forward_on_both_sides_of_the_separate_encode(N, vec, out):
    """Batches encoded in the net's kernel and in a launch of their own: same encodings and outputs."""
    P = pkg()
    T_, L = 1 << 14, 16
    g = P.HashGrid(P.MLPGridOptions(vectorDim=vec, hiddenDim=64, outputDim=out, numLayers=2, activationType=0,
                                    tableSize=T_, numLevels=L, b=1.4, lowestSize=16, featuresLevel=2), N, seed=3)
    table = np.zeros(L * T_ * 2, np.float32)
    g.save_hashgrid(table)
    o = 8 if out < 8 else 16
    W, B = make(32, 64, o, 2, 9)
    g.load_weights(flat(W), flat(B))
    pos = np.random.default_rng(5).random((N, vec), dtype=np.float32)
    y, z = torch.zeros(N, out, device="cuda"), torch.zeros(N, out, device="cuda")
    d_pos = torch.from_numpy(pos).cuda()
    g.forward(d_pos, y, N)
    g.inference(d_pos, z, N)
    torch.cuda.synchronize()
    p4 = np.zeros((N, 4), np.float32)
    p4[:, :3] = pos[:, :3]
    enc = orc.hash_encode(p4, table.astype(np.float16), T_, L, 16, 1.4)
    y_ref, _ = orc.mlp_forward(enc, flat([w.astype(np.float16) for w in W]), flat(B), 32, 64, o, 2)
    assert_close(y.cpu().numpy(), y_ref[:, :out], what="output")
    np.testing.assert_array_equal(y.cpu().numpy(), z.cpu().numpy())
