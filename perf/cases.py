"""The work a user of this framework has it do, as cases that can be timed and compared.

Kinds:
  train      InstantNerf.trainWithRaysHit on one ray chunk (Nerf.train): march, compaction, encode, both heads
             forward and backward, compositing, gradients, table scatter and Adam, occupancy refresh every 16 steps
  render     InstantNerf.renderImageHit (Nerf.render): held-out views and viewer frames
  grid_step  one training step of the hash grid + MLP (HashGrid: zero_grad, forward, MSE, backward, Adam)
  grid_infer hash grid + MLP inference (HashGrid.inference)
  net_step   one training step of a plain fused MLP (Net: zero_grad, forward, MSE, backward, Adam)
  net_block  a fused MLP inside a larger model (Net: zero_grad, forward, backward from a given dL/dy, with dL/dx)
  net_infer  fused MLP inference (Net.inference)
  encode     the hash encoding as a layer: encode launcher and the gradient scatter launcher
  march      ray setup, DDA march and compaction launchers

Sizes are those of the repository's configurations, tests and benchmark (the trainer's model, the benchmark's
model, the class defaults; batches of 2^12 to 2^20; tables of 2^14 to 2^19; 800 x 800 views).  Everything is
made from the seed with torch generators; the references of exact() are plain torch in 64 bits.
"""
from __future__ import annotations

import ctypes as C
import importlib
import math

import numpy as np
import torch

DEV = "cuda"
LEVELS = 16
RES = 128        # occupancy grid cells per side
MIPS = 4
AABB = 1.5
WHITE = 1.0


def _pkg():
    return importlib.import_module("3dmaker_amd")


def _scenes():
    return importlib.import_module("3dmaker_amd.scenes")


def listed():
    return [
        # The smallest training step anyone runs: an image- or SDF-sized hash grid (T = 2^14), 4,096 points.  Launches
        # and latency count.
        dict(name="grid_step_4k", kind="grid_step", n=4096, table=14, growth=1.447, vec=4, hidden=64, layers=2, out=16),
        # The published benchmark's training row: positions of three floats, T = 2^19, 2^18 points.
        dict(name="grid_step_256k", kind="grid_step", n=1 << 18, table=19, growth=1.38, vec=3, hidden=64, layers=2,
             out=16),
        # Its inference row at the largest batch: density queries over a volume (mesh export, baking).
        dict(name="grid_infer_1m", kind="grid_infer", n=1 << 20, table=19, growth=1.38, vec=3, hidden=64, layers=2,
             out=16),
        # The published plain-MLP training row, 64 wide and 4 layers deep.
        dict(name="net_step_256k", kind="net_step", n=1 << 18, inp=64, hidden=64, layers=4, out=64, act=0),
        # A colour head inside a caller's own model: sigmoid output, gradient from outside, dL/dx to pass on; ragged.
        dict(name="net_block_65537", kind="net_block", n=65537, inp=32, hidden=64, layers=3, out=3, act=1),
        # A small coordinate network asked for a few points: one call's latency; padded input and output.
        dict(name="net_infer_1003", kind="net_infer", n=1003, inp=3, hidden=128, layers=4, out=1, act=0),
        # The encoding as a layer of a caller's own model: forward and table gradient on ray-ordered samples.
        dict(name="encode_256k", kind="encode", n=1 << 18, table=19, growth=1.3819),
        # March and compaction of a whole view batch through five cascades.
        dict(name="march_256k_5", kind="march", n=1 << 18, cascades=5, batch=1 << 18),
        # The trainer's own model (colour head 32 x 3) on one of its chunks: four or five optimizer steps.
        dict(name="train_trainer", kind="train", rays=1 << 16, batch=1 << 18, color_hidden=32, color_layers=3, cascades=1),
        # The benchmark's model (colour head 64 x 3) on the same chunk size.
        dict(name="train_bench", kind="train", rays=1 << 16, batch=1 << 18, color_hidden=64, color_layers=3, cascades=1),
        # A held-out view of 800 x 800 with the class's default model (colour head 64 x 2).
        dict(name="render_800", kind="render", width=800, height=800, batch=1 << 21, color_hidden=64, color_layers=2),
        # A viewer's preview frame with the trainer's model.
        dict(name="render_preview", kind="render", width=201, height=151, batch=1 << 18, color_hidden=32, color_layers=3),
    ]


def _size(rng, lo, hi):
    """Log-uniform, odd as often as not."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n | 1 if rng.random() < 0.5 else n & ~15 or n))


COLOR_HEADS = ((32, 3), (64, 3), (64, 2))


def draw(rng):
    kind = rng.choice(["train", "render", "grid_step", "grid_infer", "net_step", "net_block", "net_infer", "encode",
                       "march"])
    if kind == "train":
        h, l = rng.choice(COLOR_HEADS)
        batch = rng.choice([1 << 16, 1 << 17, 1 << 18])
        return dict(kind=kind, rays=_size(rng, batch // 16, batch // 4), batch=batch, color_hidden=h, color_layers=l,
                    cascades=rng.choice([1, 1, 1, 3]))
    if kind == "render":
        h, l = rng.choice(COLOR_HEADS)
        w = _size(rng, 120, 800)
        return dict(kind=kind, width=w, height=max(90, w * 3 // 4), batch=rng.choice([1 << 18, 1 << 21]),
                    color_hidden=h, color_layers=l)
    if kind in ("grid_step", "grid_infer"):
        hidden = rng.choice([32, 64, 64, 128])  # training 128 wide is two layers deep at most
        return dict(kind=kind, n=_size(rng, 1000, 1 << (18 if kind == "grid_step" else 20)),
                    table=rng.choice([14, 16, 19]), growth=rng.choice([1.38, 1.447]), vec=rng.choice([3, 4]),
                    hidden=hidden, layers=2 if hidden == 128 else rng.choice([2, 2, 4]), out=rng.choice([16, 16, 3, 1]))
    if kind in ("net_step", "net_block", "net_infer"):
        hidden = rng.choice([32, 64, 64, 128])
        small = hidden == 128 and kind != "net_infer"
        wide = rng.random() < 0.4 and not small
        return dict(kind=kind, n=_size(rng, 1000, 1 << (18 if hidden < 128 else 17)),
                    inp=hidden if wide else rng.choice([3, 16, 32]), hidden=hidden, layers=2 if small else rng.choice([2, 3, 4]),
                    out=hidden if wide else rng.choice([1, 3, 8, 16]), act=0 if wide else rng.choice([0, 1]))
    if kind == "encode":
        return dict(kind=kind, n=_size(rng, 1000, 1 << 18), table=rng.choice([14, 16, 19]),
                    growth=rng.choice([1.3819, 1.447]))
    return dict(kind=kind, n=_size(rng, 1 << 12, 1 << 18), cascades=rng.choice([1, 2, 3, 5]), batch=1 << 18)


# ---------------------------------------------------------------------------
# helpers
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _Buffer:
    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner  # the handle lives as long as a view of its memory
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr, "version": 2}


def _view(owner, ptr, shape, typestr="<f4"):
    """A library-owned device buffer as a tensor."""
    return torch.as_tensor(_Buffer(ptr, shape, typestr, owner), device=DEV)


def _layers(owner, ptr_array, shapes):
    """The per-layer buffers behind a device array of device pointers."""
    torch.cuda.synchronize()
    return [_view(owner, p, s) for p, s in zip(_view(owner, ptr_array, (len(shapes),), "<i8").tolist(), shapes)]


def _pow2(d):
    """Padded width of a layer end: the next power of two, at least 8."""
    return max(8, 1 << (d - 1).bit_length())


def _dims(inp, hidden, layers, out):
    """(rows, columns) of every layer's weight matrix."""
    return [(out if l == layers - 1 else hidden, inp if l == 0 else hidden) for l in range(layers)]


def _weights(g, dims):
    """Uniform LeCun weights and small biases, as [out][in] per layer."""
    W = [(torch.rand(o, i, generator=g, device=DEV) * 2 - 1) / math.sqrt(i) for o, i in dims]
    return W, [(torch.rand(o, generator=g, device=DEV) - 0.5) * 0.1 for o, _ in dims]


def _flat(ts):
    return torch.cat([t.reshape(-1) for t in ts]).float().cpu().numpy()


def _forward64(x, W, B):
    """Activations of every layer's input, and the last layer's pre-activation, with the 16-bit weights."""
    acts = [x]
    for l, (w, b) in enumerate(zip(W, B)):
        y = acts[-1] @ w.half().double().T + b.double()
        if l < len(W) - 1:
            acts.append(y.clamp_min(0))
    return acts, y


def _backward64(acts, W, dy, dx0):
    """dW, db per layer, and dL/dx of the input when dx0."""
    dW, dB = [], []
    for l in range(len(W) - 1, -1, -1):
        dW.append(dy.T @ acts[l])
        dB.append(dy.sum(0))
        if l or dx0:
            dy = dy @ W[l].half().double()
            if l:
                dy = dy * (acts[l] > 0)
    return dW[::-1], dB[::-1], dy


# ---------------------------------------------------------------------------
# the hash grid
# ---------------------------------------------------------------------------

def _grid_meta(table, growth):
    """(level scales, resolutions, first hashed level)."""
    T = 1 << table
    scale = [float(np.float32(16.0 * float(np.float32(growth)) ** l)) for l in range(LEVELS)]
    res = [int(math.floor(s)) for s in scale]
    inner = (T ** (1.0 / 3.0) - 1.0) / 16.0
    dense = max(0, min(int(math.floor(math.log2(inner) / math.log2(growth))) + 1, LEVELS))
    return scale, res, dense


def _corners64(pos, level, table, growth, backward):
    """Entry indices [8, n] and weights [8, n] of a level."""
    scale, res, dense = _grid_meta(table, growth)
    N = res[level]
    x = pos[:, :3].double() * scale[level]
    f = x.floor()
    i0 = f.long().clamp(0, N - 1 if backward else N)
    i1 = (i0 + 1).clamp_max(N)
    u = x - f
    idx, w = [], []
    for c in range(8):
        pick = [(c >> k) & 1 for k in range(3)]
        q = [i1[:, k] if pick[k] else i0[:, k] for k in range(3)]
        if level < dense:
            e = q[0] + q[1] * (N + 1) + q[2] * (N + 1) ** 2
        else:
            e = (q[0] ^ (q[1] * 2654435761 & 0xffffffff) ^ (q[2] * 805459861 & 0xffffffff)) & ((1 << table) - 1)
        idx.append(e)
        w.append(torch.stack([u[:, k] if pick[k] else 1 - u[:, k] for k in range(3)]).prod(0))
    return torch.stack(idx), torch.stack(w)


def _encode64(pos, tab16, table, growth):
    """tab16: [LEVELS, T, 2] 16-bit table -> [n, 2 * LEVELS]."""
    out = torch.empty(pos.shape[0], 2 * LEVELS, dtype=torch.float64, device=DEV)
    for l in range(LEVELS):
        idx, w = _corners64(pos, l, table, growth, False)
        out[:, 2 * l:2 * l + 2] = (tab16[l][idx].double() * w[..., None]).sum(0)
    return out


def _grid_inputs(case, seed):
    g = _gen(seed)
    n, T = case["n"], 1 << case["table"]
    pos = torch.rand(n, case["vec"], generator=g, device=DEV)
    tab = (torch.rand(LEVELS, T, 2, generator=g, device=DEV) * 2 - 1) * 0.1
    W, B = _weights(g, _dims(2 * LEVELS, case["hidden"], case["layers"], _pow2(case["out"])))
    tgt = torch.rand(n, case["out"], generator=g, device=DEV).half()
    return pos, tab, W, B, tgt


def _prepare_grid(case, seed):
    P = _pkg()
    pos, tab, W, B, tgt = _grid_inputs(case, seed)
    opt = P.MLPGridOptions(vectorDim=case["vec"], hiddenDim=case["hidden"], outputDim=case["out"],
                           numLayers=case["layers"], activationType=0, tableSize=1 << case["table"], numLevels=LEVELS,
                           b=case["growth"], lowestSize=16, featuresLevel=2)
    train = case["kind"] == "grid_step"
    net = P.HashGrid(opt, case["n"], seed=int(seed) & 0x7fffffff, training=train)
    net.load_hashgrid(tab.reshape(-1).cpu().numpy())
    net.load_weights(_flat(W), _flat(B))
    s = dict(net=net, n=case["n"], x=pos, tgt=tgt, stream=_stream(),
             out=torch.zeros(case["n"], case["out"], device=DEV))
    if train:
        b = net.buffers()
        s["state"] = dict(wg=_layers(net, b.w_grad, [w.shape for w in W]), bg=_layers(net, b.b_grad, [v.shape for v in B]),
                          w=_layers(net, b.master_weights, [w.shape for w in W]), table=_view(net, b.master_hashtable, tab.shape))
    return s


LOSS_SCALE = 65536.0  # of the published benchmark


def _run_step(s):
    """zero_grad, forward, MSE, backward and Adam (HashGrid and Net alike)."""
    net, n, st = s["net"], s["n"], s["stream"]
    net.zero_grad(stream=st)
    net.forward(s["x"], s["out"], n, stream=st)
    net.calculate_loss_and_grad(s["tgt"], n, LOSS_SCALE, stream=st)
    net.backward(n, stream=st)
    net.step(1e-2, 0.9, 0.99, 1e-15, LOSS_SCALE, stream=st)
    return dict(s["state"], out=s["out"])


def _step64(x, W, B, tgt, act):
    """Outputs and gradients of _run_step's first pass (widths of W are the padded ones)."""
    acts, y = _forward64(x, W, B)
    valid = tgt.shape[1]
    p = torch.sigmoid(y) if act else y
    dy = torch.zeros_like(y)
    dy[:, :valid] = (p[:, :valid] - tgt.double()) * (2.0 * LOSS_SCALE / (tgt.shape[0] * valid))
    if act:
        dy = dy * p * (1 - p)
    dW, dB, _ = _backward64(acts, W, dy, False)
    none = [None] * len(W)
    return dict(out=p[:, :valid], wg=dW, bg=dB, w=none, table=None)


def _exact_grid(case, seed):
    pos, tab, W, B, tgt = _grid_inputs(case, seed)
    enc = _encode64(pos, tab.half(), case["table"], case["growth"])
    if case["kind"] == "grid_infer":
        return _forward64(enc, W, B)[1][:, :case["out"]]
    return _step64(enc, W, B, tgt, 0)


# ---------------------------------------------------------------------------
# plain MLPs
# ---------------------------------------------------------------------------

def _net_inputs(case, seed):
    g = _gen(seed)
    n, dims = case["n"], _dims(_pow2(case["inp"]), case["hidden"], case["layers"], _pow2(case["out"]))
    x = torch.randn(n, case["inp"], generator=g, device=DEV).half()
    W, B = _weights(g, dims)
    tgt = torch.rand(n, case["out"], generator=g, device=DEV).half()
    dy = (torch.randn(n, case["out"], generator=g, device=DEV) * 0.05).half()
    return x, W, B, tgt, dy


def _prepare_net(case, seed):
    P = _pkg()
    x, W, B, tgt, dy = _net_inputs(case, seed)
    opt = P.MLPOption(inputDim=case["inp"], hiddenDim=case["hidden"], outputDim=case["out"], numLayers=case["layers"],
                      activationType=0, outputActivation=case["act"])
    train = case["kind"] != "net_infer"
    net = P.Net(opt, case["n"], seed=int(seed) & 0x7fffffff, training=train)
    net.load_weights(_flat(W), _flat(B))
    s = dict(net=net, n=case["n"], x=x, tgt=tgt, dy=dy, stream=_stream(),
             out=torch.zeros(case["n"], case["out"], device=DEV))
    if train:
        b = net.buffers()
        s["state"] = dict(wg=_layers(net, b.w_grad, [w.shape for w in W]), bg=_layers(net, b.b_grad, [v.shape for v in B]))
        if case["kind"] == "net_step":
            s["state"]["w"] = _layers(net, b.master_weights, [w.shape for w in W])
        else:
            s["dx"] = torch.zeros(case["n"], W[0].shape[1], dtype=torch.float16, device=DEV)
    return s


def _exact_net(case, seed):
    x, W, B, tgt, dy = _net_inputs(case, seed)
    xp = torch.zeros(case["n"], W[0].shape[1], dtype=torch.float64, device=DEV)
    xp[:, :case["inp"]] = x.double()
    if case["kind"] == "net_step":
        return {k: v for k, v in _step64(xp, W, B, tgt, case["act"]).items() if k != "table"}
    acts, y = _forward64(xp, W, B)
    out = (torch.sigmoid(y) if case["act"] else y)[:, :case["out"]]
    if case["kind"] == "net_infer":
        return out
    d = torch.zeros_like(y)
    d[:, :case["out"]] = dy.double()
    dW, dB, dx = _backward64(acts, W, d, True)
    return dict(out=out, wg=dW, bg=dB, dx=dx)


# ---------------------------------------------------------------------------
# the encoding as a layer
# ---------------------------------------------------------------------------

def _encode_inputs(case, seed):
    """Samples in ray order inside the uncontracted half of the grid, 32 to a ray; the upstream gradient of the
    far half of every ray is zero (the ray is saturated there)."""
    g = _gen(seed)
    n, T = case["n"], 1 << case["table"]
    rays = -(-n // 32)
    o = torch.rand(rays, 1, 3, generator=g, device=DEV) * 0.4 + 0.3
    d = torch.randn(rays, 1, 3, generator=g, device=DEV)
    d = d / d.norm(dim=-1, keepdim=True)
    t = (torch.arange(32, device=DEV).view(1, 32, 1) - 16) * 0.003
    pos = torch.zeros(n, 4, device=DEV)
    pos[:, :3] = (o + t * d).reshape(-1, 3)[:n]
    tab = (torch.rand(LEVELS, T, 2, generator=g, device=DEV) * 2 - 1) * 0.1
    denc = torch.randn(rays * 32, 2 * LEVELS, generator=g, device=DEV) * 0.02
    denc = denc.view(rays, 32, -1) * (torch.arange(32, device=DEV) < 16).view(1, 32, 1)
    return pos, tab, denc.reshape(rays * 32, -1)[:n].half().contiguous()


def _prepare_encode(case, seed):
    P = _pkg()
    pos, tab, denc = _encode_inputs(case, seed)
    opt = P.MLPGridOptions(vectorDim=4, hiddenDim=64, outputDim=16, numLayers=2, activationType=0,
                           tableSize=1 << case["table"], numLevels=LEVELS, b=case["growth"], lowestSize=16,
                           featuresLevel=2)
    return dict(P=P, opt=opt, n=case["n"], T=1 << case["table"], growth=case["growth"], pos=pos, tab=tab.half(),
                denc=denc, enc=torch.zeros(case["n"], 2 * LEVELS, dtype=torch.float16, device=DEV),
                grads=torch.zeros_like(tab), stream=_stream())


def _run_encode(s):
    s["P"].launch("launchHashEncodeKernel", C.byref(s["opt"]), s["tab"], s["pos"], 4, s["enc"], s["n"], s["stream"])
    s["P"].launch("launchHashTableBackwardKernel", s["denc"], s["pos"], s["grads"], s["n"], s["T"], LEVELS, s["growth"],
                  16, 2, s["stream"])
    return dict(enc=s["enc"], grads=s["grads"])


def _exact_encode(case, seed):
    pos, tab, denc = _encode_inputs(case, seed)
    grads = torch.zeros(tab.shape, dtype=torch.float64, device=DEV)
    for l in range(LEVELS):
        idx, w = _corners64(pos, l, case["table"], case["growth"], True)
        for c in range(8):
            grads[l].index_add_(0, idx[c], denc[:, 2 * l:2 * l + 2].double() * w[c][:, None])
    return dict(enc=_encode64(pos, tab.half(), case["table"], case["growth"]), grads=grads)


# ---------------------------------------------------------------------------
# march
# ---------------------------------------------------------------------------

def _prepare_march(case, seed):
    P, sc = _pkg(), _scenes()
    n = case["n"]
    o, d = sc.rays_c4(n, n_cams=100, seed=int(seed) & 0x7fffffff)
    bits = sc.occupancy_c4(RES, case["cascades"], MIPS, 0.1, 0.3, AABB, seed=int(seed) & 0x7fffffff)
    f = lambda *s: torch.zeros(*s, device=DEV)  # noqa: E731
    i = lambda *s: torch.zeros(*s, dtype=torch.int32, device=DEV)  # noqa: E731
    return dict(P=P, n=n, batch=case["batch"], cascades=case["cascades"], o=torch.from_numpy(o).to(DEV),
                d=torch.from_numpy(d).to(DEV), bits=torch.from_numpy(bits).to(DEV), inv=f(n, 3), near=f(n), far=f(n),
                counts=i(n), offsets=i(n), pos=f(case["batch"], 4), ray=i(case["batch"]), t=f(case["batch"]), active=i(1),
                stream=_stream())


def _run_march(s):
    P, total = s["P"], C.c_uint32(0)
    lo, hi = P.Float3(-AABB, -AABB, -AABB), P.Float3(AABB, AABB, AABB)
    P.launch("launchComputeRayAabbInv", s["n"], s["o"], s["d"], lo, hi, s["cascades"], s["inv"], s["near"], s["far"],
             s["stream"])
    P.launch("processRaysHitLinear", s["n"], s["o"], s["d"], s["inv"], s["near"], s["far"], s["bits"],
             P.Uint3(RES, RES, RES), lo, hi, s["cascades"], MIPS, 1, s["batch"], C.byref(total), s["active"],
             s["counts"], s["offsets"], s["pos"], s["ray"], s["t"], None, s["stream"])
    return dict({k: s[k] for k in ("inv", "near", "far", "counts", "offsets", "pos", "ray", "t", "active")},
                total=int(total.value))


# ---------------------------------------------------------------------------
# the radiance field
# ---------------------------------------------------------------------------

NERF_TABLE, NERF_GROWTH, NERF_DENSE = 19, 1.3819, 4   # NERF_DENSE: the finest level that is not hashed


def _scene(seed):
    """Three solid spheres: centres and radii."""
    r = np.random.default_rng(int(seed))
    c, q = r.uniform(-0.6, 0.6, (3, 3)), r.uniform(0.25, 0.45, 3)
    return torch.from_numpy(c).to(DEV), torch.from_numpy(q).to(DEV)


def _sdf(scene, p):
    return ((p[..., None, :] - scene[0]).norm(dim=-1) - scene[1]).min(-1).values


def _field(case, seed):
    """A field as training leaves it: the spheres' signed distance in feature 0 of the finest dense level, read by
    the first two hidden units into the density logit (about +5 inside, -5 outside), random colours and features
    of the untrained size everywhere else."""
    g = _gen(seed)
    scene = _scene(seed)
    T = 1 << NERF_TABLE
    tab = torch.randn(LEVELS, T, 2, generator=g, device=DEV) * 0.1
    scale, res, _ = _grid_meta(NERF_TABLE, NERF_GROWTH)
    side = res[NERF_DENSE] + 1
    ax = torch.arange(side, device=DEV, dtype=torch.float64) / scale[NERF_DENSE]
    w = ((ax * 4 - 2) * AABB)  # the box fills [0.25, 0.75] of the encoded space
    p = torch.stack(torch.meshgrid(w, w, w, indexing="ij"), -1).flip(-1)  # entry x + y side + z side^2
    tab[NERF_DENSE, :side ** 3, 0] = (-_sdf(scene, p.reshape(-1, 3)) / 0.1).clamp(-1, 1).float()
    dW, dB = _weights(g, _dims(2 * LEVELS, 64, 2, 16))
    dW[0][:2] = 0
    dW[0][0, 2 * NERF_DENSE], dW[0][1, 2 * NERF_DENSE] = 1, -1
    dW[1][0] *= 0.2
    dW[1][0, :2] = torch.tensor([5.0, -5.0], device=DEV)
    for b in dB:
        b.zero_()
    cW, cB = _weights(g, _dims(2 * LEVELS, case["color_hidden"], case["color_layers"], 8))
    return scene, tab, (dW, dB), (cW, cB)


def _prepare_nerf(case, seed):
    P, sc = _pkg(), _scenes()
    train = case["kind"] == "train"
    scene, tab, (dW, dB), (cW, cB) = _field(case, seed)
    o = P.Nerf.default_options()
    o.gridResolution[:] = [RES] * 3
    o.aabbMin[:], o.aabbMax[:] = [-AABB] * 3, [AABB] * 3
    o.levelsMipmap, o.samplesPerVoxel, o.numCascades = MIPS, 1, case.get("cascades", 1)
    o.densityHiddenDim, o.densityNumLayers = 64, 2
    o.colorHiddenDim, o.colorNumLayers = case["color_hidden"], case["color_layers"]
    o.hashTableSize, o.numLevels, o.growthFactor, o.baseResolution = 1 << NERF_TABLE, LEVELS, NERF_GROWTH, 16
    o.batchSize = case["batch"] if train else 1 << 18
    o.rayChunkSize = o.batchSize // 4
    o.renderBatchSize = 1 << 18 if train else case["batch"]
    o.lambdaDist, o.lambdaDepth, o.lossScale, o.densityBias = 0.1, 0.0, 128.0, 0.0
    o.beta1, o.beta2, o.epsilon = 0.9, 0.999, 1e-8
    nerf = P.Nerf(o)
    nerf.density.load_hashgrid(tab.reshape(-1).cpu().numpy())
    nerf.density.load_weights(_flat(dW), _flat(dB))
    nerf.color.load_weights(_flat(cW), _flat(cB))
    st = _stream()
    s = dict(nerf=nerf, stream=st)
    if not train:
        nerf.set_occupancy(np.packbits(_occupied(scene), bitorder="little"))
        nerf.set_memory_mode(True)
        ro, rd = _view_rays(case, seed)
        return dict(s, o=ro, d=rd, n=ro.shape[0], rgb=torch.zeros(ro.shape[0], 3, device=DEV))
    # a grid that has followed the field for a while, as in the middle of a training
    for _ in range(80):
        nerf.update_occupancy(stream=st)
    n = case["rays"]
    ro, rd = (torch.from_numpy(a).to(DEV) for a in sc.rays_c4(n, n_cams=100, seed=int(seed) & 0x7fffffff))
    # ground truth: what the field renders, off by a few per cent
    truth = torch.zeros(n, 3, device=DEV)
    nerf.render(ro, rd, n, truth, stream=st)
    truth = (truth + torch.randn(n, 3, generator=_gen(seed + 1), device=DEV) * 0.03).clamp(0, 1)
    nerf.set_learning_rate(1e-3)
    b, c = nerf.density.buffers(), nerf.color.buffers()
    state = dict(table=_view(nerf, b.master_hashtable, tab.shape), dw=_layers(nerf, b.master_weights, [w.shape for w in dW]),
                 cw=_layers(nerf, c.master_weights, [w.shape for w in cW]))
    return dict(s, o=ro, d=rd, n=n, truth=truth, rgb=torch.zeros(n, 3, device=DEV), state=state)


def _run_train(s):
    _, hits = s["nerf"].train(s["o"], s["d"], s["truth"], s["n"], rgb_out=s["rgb"], stream=s["stream"])
    return dict(s["state"], rgb=s["rgb"])


def _run_render(s):
    s["nerf"].render(s["o"], s["d"], s["n"], s["rgb"], stream=s["stream"])
    return s["rgb"]


def _occupied(scene):
    """The occupancy pyramid's bits: cells within a cell and a half of a sphere."""
    c = ((torch.arange(RES, device=DEV, dtype=torch.float64) + 0.5) / RES * 2 - 1) * AABB
    p = torch.stack(torch.meshgrid(c, c, c, indexing="ij"), -1).flip(-1)  # indexed [z, y, x]
    cur = _sdf(scene, p) < 1.5 * 2 * AABB / RES
    bits = []
    for _ in range(MIPS):
        bits.append(cur.reshape(-1))
        r = cur.shape[0] // 2
        if r:
            cur = cur.view(r, 2, r, 2, r, 2).any(5).any(3).any(1)
    return torch.cat(bits).cpu().numpy()


def _view_rays(case, seed):
    sc = _scenes()
    w, h = case["width"], case["height"]
    cams = sc.cameras(8, AABB, int(seed) & 0x7fffffff)
    py, px = np.meshgrid(np.arange(h, dtype=np.float64), np.arange(w, dtype=np.float64), indexing="ij")
    o, d = sc.camera_rays(cams, np.full(w * h, 3), px.reshape(-1), py.reshape(-1), w, h, sc.focal_from_fov(w, 50.0))
    return torch.from_numpy(o).to(DEV), torch.from_numpy(d).to(DEV)


def _march64(scene, o, d):
    """Sample t of every ray [n, most], padded with inf: one sample in the middle of each occupied cell's span."""
    grid = torch.from_numpy(_occupied(scene)).to(DEV)
    n = o.shape[0]
    o, d = o.double(), d.double()
    inv = 1 / torch.where(d.abs() < 1e-8, torch.full_like(d, 1e-8), d)
    a, b = (-AABB - o) * inv, (AABB - o) * inv
    near, far = torch.minimum(a, b).max(1).values, torch.maximum(a, b).min(1).values
    alive = (near <= far) & (far >= 0)
    t, far = torch.where(alive, near.clamp_min(0), torch.zeros_like(near)), torch.where(alive, far, torch.zeros_like(far))
    fwd = (d >= 0).double()
    off, base = [], 0
    for l in range(MIPS):
        off.append(base)
        base += (RES >> l) ** 3
    found = []
    while bool((t < far).any()):
        go = t < far
        cell0 = (((o + t[:, None] * d + AABB) / (2 * AABB)) * RES).floor().clamp(0, RES - 1).long()
        level, done = torch.zeros(n, dtype=torch.long, device=DEV), torch.zeros(n, dtype=torch.bool, device=DEV)
        occ = torch.zeros_like(done)
        for l in range(MIPS - 1, -1, -1):
            c, r = cell0 >> l, RES >> l
            bit = grid[off[l] + (c[:, 2] * r + c[:, 1]) * r + c[:, 0]] != 0
            level = torch.where(done, level, torch.full_like(level, l))
            occ = torch.where(done, occ, bit)
            done = done | ~bit
        c = (cell0 >> level[:, None]).double()
        edge = (c + fwd) * (2 * AABB / RES * (2.0 ** level.double())[:, None]) - AABB
        nxt = ((edge - o) * inv).min(1).values
        found.append(torch.where(go & occ, t + 0.5 * (nxt - t), torch.full_like(t, math.inf)))
        t = torch.where(go, torch.maximum(t + 1e-5, nxt + 1e-6), t)
    return torch.stack(found, 1).sort(1).values


def _sh64(d):
    x, y, z = d.double().unbind(1)
    k = (0.28209479, 0.48860251, 1.09254843, 0.31539156, 0.54627421, 0.59004359, 2.89061144, 0.45704580, 0.37317633,
         1.44530572)
    return torch.stack([
        torch.full_like(x, k[0]), -k[1] * y, k[1] * z, -k[1] * x, k[2] * x * y, -k[2] * y * z, k[3] * (3 * z * z - 1),
        -k[2] * x * z, k[4] * (x * x - y * y), -k[5] * y * (3 * x * x - y * y), k[6] * x * y * z,
        -k[7] * y * (5 * z * z - 1), k[8] * z * (5 * z * z - 3), -k[7] * x * (5 * z * z - 1),
        k[9] * z * (x * x - y * y), -k[5] * x * (x * x - 3 * y * y)], 1)


def _exact_render(case, seed):
    scene, tab, (dW, dB), (cW, cB) = _field(case, seed)
    tab16 = tab.half()
    ro, rd = _view_rays(case, seed)
    out = []
    for k in range(0, ro.shape[0], 1 << 15):
        o, d = ro[k:k + (1 << 15)], rd[k:k + (1 << 15)]
        t = _march64(scene, o, d)
        ray, col = torch.nonzero(torch.isfinite(t), as_tuple=True)
        sig, rgb = torch.zeros_like(t), torch.zeros(*t.shape, 3, dtype=torch.float64, device=DEV)
        p = o[ray].double() + t[ray, col][:, None] * d[ray].double()
        enc = _encode64((p / AABB + 2) * 0.25, tab16, NERF_TABLE, NERF_GROWTH)
        logit = _forward64(enc, dW, dB)[1].clamp(-64, 64)
        sig[ray, col] = logit[:, 0].clamp_max(8).exp()
        rgb[ray, col] = torch.sigmoid(_forward64(torch.cat([logit, _sh64(d)[ray]], 1), cW, cB)[1][:, :3])
        nxt = torch.cat([t[:, 1:], torch.full_like(t[:, :1], math.inf)], 1)
        delta = torch.where(torch.isfinite(nxt), nxt - t, torch.full_like(t, 1e-3))
        alpha = torch.where(torch.isfinite(t), 1 - torch.exp(-sig * delta.nan_to_num(0)), torch.zeros_like(t))
        left = torch.cumprod(1 - alpha, 1)
        before = torch.cat([torch.ones_like(left[:, :1]), left[:, :-1]], 1)
        w = torch.where(before < 1e-4, torch.zeros_like(alpha), alpha * before)
        # a ray stops behind the first sample that leaves less than 1e-4
        last = torch.where(before < 1e-4, torch.ones_like(left), left).min(1).values
        out.append((w[..., None] * rgb).sum(1) + last[:, None] * WHITE)
    return torch.cat(out)


# ---------------------------------------------------------------------------

_PREPARE = dict(train=_prepare_nerf, render=_prepare_nerf, grid_step=_prepare_grid, grid_infer=_prepare_grid,
                net_step=_prepare_net, net_block=_prepare_net, net_infer=_prepare_net, encode=_prepare_encode,
                march=_prepare_march)


def _run_infer(s):
    s["net"].inference(s["x"], s["out"], s["n"], stream=s["stream"])
    return s["out"]


def _run_block(s):
    net, n, st = s["net"], s["n"], s["stream"]
    net.zero_grad(stream=st)
    net.forward(s["x"], s["out"], n, stream=st)
    net.backward(n, custom_grad=s["dy"], dx_out=s["dx"], stream=st)
    return dict(s["state"], out=s["out"], dx=s["dx"])


_RUN = dict(train=_run_train, render=_run_render, grid_step=_run_step, grid_infer=_run_infer, net_step=_run_step,
            net_block=_run_block, net_infer=_run_infer, encode=_run_encode, march=_run_march)


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, int(seed)), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("grid_step", "grid_infer"):
        return _exact_grid(case, seed)
    if kind in ("net_step", "net_block", "net_infer"):
        return _exact_net(case, seed)
    if kind == "encode":
        return _exact_encode(case, seed)
    if kind == "render":
        return _exact_render(case, seed)
    return None


def _reached(n, table, growth):
    """Table entries that n samples can reach, over all levels."""
    _, res, _ = _grid_meta(table, growth)
    return sum(min(8 * n, 1 << table, (r + 1) ** 3) for r in res)


SAMPLES_PER_RAY = 15   # of the sphere field's rays, all pixels together


def work(case):
    """Each input read once, each output and each updated parameter written once; matrix products of the true widths."""
    kind = case["kind"]
    if kind in ("grid_step", "grid_infer"):
        n, reach = case["n"], _reached(case["n"], case["table"], case["growth"])
        mac = sum(a * b for a, b in _dims(2 * LEVELS, case["hidden"], case["layers"], case["out"]))
        io = n * (4 * case["vec"] + 4 * case["out"]) + 4 * reach + 2 * mac
        if kind == "grid_infer":
            return dict(bytes=io, flops=2 * n * mac)
        # targets, and w, m, v read and written and the 16-bit copy written per reached parameter
        return dict(bytes=io + 2 * n * case["out"] + 26 * (2 * reach + mac), flops=6 * n * mac)
    if kind in ("net_step", "net_block", "net_infer"):
        n = case["n"]
        dims = _dims(case["inp"], case["hidden"], case["layers"], case["out"])
        mac = sum(a * b for a, b in dims)
        io = n * (2 * case["inp"] + 4 * case["out"]) + 2 * mac
        if kind == "net_infer":
            return dict(bytes=io, flops=2 * n * mac)
        if kind == "net_block":
            return dict(bytes=io + n * 2 * (case["out"] + case["inp"]) + 4 * mac, flops=6 * n * mac)
        return dict(bytes=io + 2 * n * case["out"] + 30 * mac, flops=6 * n * mac - 2 * n * dims[0][0] * dims[0][1])
    if kind == "encode":
        reach = _reached(case["n"], case["table"], case["growth"])
        return dict(bytes=case["n"] * (16 + 64 + 64) + 4 * reach + 16 * reach, flops=case["n"] * LEVELS * 8 * 4)
    if kind == "march":
        return dict(bytes=case["n"] * (24 + 12 + 8 + 8) + case["batch"] // 4 * 24, flops=case["n"] * 60 * 40)
    cw = sum(a * b for a, b in _dims(32, case["color_hidden"], case["color_layers"], 3))
    mac = cw + 32 * 64 + 64 * 16
    if kind == "render":
        rays = case["width"] * case["height"]
        n = rays * SAMPLES_PER_RAY
        return dict(bytes=rays * (24 + 12) + 4 * _reached(n, NERF_TABLE, NERF_GROWTH), flops=2 * n * mac)
    n = case["rays"] * SAMPLES_PER_RAY
    per = min(n, case["batch"])
    steps = max(1, round(n / case["batch"]))
    reach = _reached(per, NERF_TABLE, NERF_GROWTH)
    return dict(bytes=case["rays"] * (24 + 12 + 12) + steps * (4 * reach + 52 * reach), flops=6 * n * mac)


def tolerance(case):
    """About four times what a second implementation with the same roundings and another order of sums showed (the
    layers in torch with 32-bit products; the training step and the render with their other kernels)."""
    kind = case["kind"]
    if kind == "march":
        return "exact"  # cells, counts and the sample t are the reference's operations one by one
    if kind in ("grid_infer", "net_infer", "encode"):
        return {"rel": 4e-4, "max": 0.01}
    if kind == "render":
        return {"rel": 2e-4, "max": 0.01}
    if kind == "train":
        return {"rel": 2e-3, "max": 0.05}
    # A hidden unit that rounds to zero on one side only gains or loses its whole gradient; a first Adam step turns a
    # tiny gradient's sign into a whole step.
    return {"rel": 0.025 if kind == "grid_step" else 0.01, "max": 0.99}
