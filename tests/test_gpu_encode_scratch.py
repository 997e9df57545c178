"""The scratch for level-major encodings: batches of several pieces, how much stays allocated whatever the batch and
the number of streams, streams under capture (no scratch), and streams and threads that share one grid.  The
encodings and outputs are those of small batches, which need no scratch, bit for bit."""
import ctypes as C
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import pkg  # noqa: E402

pytestmark = pytest.mark.gpu

L, T, B = 16, 1 << 12, 1.3
PIECE = 1 << 20          # samples of one piece
SMALL = (1 << 15) - 16   # no scratch below 2^15
KEPT = PIECE * L * 4     # bytes of one stream's scratch
SLACK = 24 << 20         # allocation granularity, code objects, streams


def options(P, hidden=64, out=16, layers=2):
    return P.MLPGridOptions(vectorDim=4, hiddenDim=hidden, outputDim=out, numLayers=layers, activationType=0,
                            tableSize=T, numLevels=L, b=B, lowestSize=16, featuresLevel=2)


def positions(n, seed):
    return torch.rand(n, 4, generator=torch.Generator("cuda").manual_seed(seed), device="cuda")


def table(seed=1):
    g = torch.Generator("cuda").manual_seed(seed)
    return (torch.rand(L * T * 2, generator=g, device="cuda") * 2 - 1).half()


def encode(P, tab, pos, out, stream=None):
    P.launch("launchHashEncodeKernel", C.byref(options(P)), tab, pos, 4, out, pos.shape[0], stream)


def small_batches(P, tab, pos):
    out = torch.zeros(pos.shape[0], 2 * L, dtype=torch.float16, device="cuda")
    for k in range(0, pos.shape[0], SMALL):
        encode(P, tab, pos[k:k + SMALL], out[k:k + SMALL])
    return out


def used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def same(a, b):
    return bool(torch.equal(a.view(torch.int16) if a.dtype == torch.float16 else a.view(torch.int32),
                            b.view(torch.int16) if b.dtype == torch.float16 else b.view(torch.int32)))


def test_encode_in_pieces_keeps_one_piece():
    P = pkg()
    N = 3 * PIECE + 12345
    tab, pos = table(), positions(N, 2)
    out = torch.zeros(N, 2 * L, dtype=torch.float16, device="cuda")
    want = small_batches(P, tab, pos)
    before = used()
    encode(P, tab, pos, out)
    encode(P, tab, pos, out)
    assert used() - before <= KEPT + SLACK
    assert same(out, want)


def test_many_streams_keep_few_workspaces():
    P = pkg()
    N = PIECE
    tab, pos = table(), positions(N, 3)
    want = small_batches(P, tab, pos)
    streams = [torch.cuda.Stream() for _ in range(12)]
    outs = [torch.zeros(N, 2 * L, dtype=torch.float16, device="cuda") for _ in range(3)]
    for s in streams:                  # their own queues, before the count
        with torch.cuda.stream(s):
            outs[0].add_(0)
    before = used()
    for turn in range(3):
        for k, s in enumerate(streams):
            encode(P, tab, pos, outs[k % 3], s.cuda_stream)
            s.synchronize()
            assert same(outs[k % 3], want)
            outs[k % 3].zero_()
            torch.cuda.synchronize()
    assert used() - before <= 4 * KEPT + SLACK
    # streams that are gone give theirs back: one stream alone gets its own in time and keeps the right values
    late = torch.cuda.Stream()
    for _ in range(70):
        encode(P, tab, pos, outs[0], late.cuda_stream)
    late.synchronize()
    assert same(outs[0], want)
    assert used() - before <= 4 * KEPT + SLACK


def test_forward_with_saved_activations_in_pieces():
    """The gradient launcher over several pieces: saved encodings, hidden activations and outputs."""
    P = pkg()
    N, hid, out = 3 * PIECE + 777, 32, 16
    tab, pos = table(), positions(N, 4)
    g = torch.Generator("cuda").manual_seed(5)
    dims = [(hid, 2 * L), (hid, hid), (out, hid)]
    W = [((torch.rand(*d, generator=g, device="cuda") * 2 - 1) / d[1] ** 0.5).half() for d in dims]
    bias = [(torch.rand(d[0], generator=g, device="cuda") - 0.5) * 0.1 for d in dims]
    ptr = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device="cuda")  # noqa: E731
    opt = options(P, hid, out, 3)

    def run(pos, acts, y):
        pa, pw, pb = ptr(acts), ptr(W), ptr(bias)
        P.launch("launchNetworkFusionHashTableGradKernel", C.byref(opt), tab, pos, pa, pw, pb, y, pos.shape[0], None)
        torch.cuda.synchronize()

    def buffers():
        return [torch.zeros(N, 2 * L if l == 0 else hid, dtype=torch.float16, device="cuda") for l in range(3)], \
            torch.zeros(N, out, device="cuda")

    acts, y = buffers()
    before = used()
    run(pos, acts, y)
    assert used() - before <= KEPT + SLACK
    a2, y2 = buffers()
    for k in range(0, N, SMALL):
        run(pos[k:k + SMALL], [a[k:k + SMALL] for a in a2], y2[k:k + SMALL])
    for a, b in zip(acts, a2):
        assert same(a, b)
    assert same(y, y2)
    y3 = torch.zeros_like(y)
    P.launch("launchNetworkFusionHashTableKernel", C.byref(opt), tab, pos, ptr(W), ptr(bias), y3, N, None)
    torch.cuda.synchronize()
    assert same(y, y3)


def grid(P, n):
    net = P.HashGrid(options(P), n, seed=3, training=False)
    net.load_hashgrid(table().float().cpu().numpy())
    return net


def test_under_capture():
    """Captured encodes and inferences take the route without scratch; every replay gives the eager values."""
    P = pkg()
    N = 40000
    tab, pos = table(), positions(N, 6)
    net = grid(P, N)
    enc, y = torch.zeros(N, 2 * L, dtype=torch.float16, device="cuda"), torch.zeros(N, 16, device="cuda")
    want_enc, want_y = torch.zeros_like(enc), torch.zeros_like(y)
    encode(P, tab, pos, want_enc)
    net.inference(pos, want_y, N)
    torch.cuda.synchronize()
    other = positions(N, 7)
    other_enc, other_y = torch.zeros_like(enc), torch.zeros_like(y)
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side):
        encode(P, tab, pos, enc, side.cuda_stream)
        net.inference(pos, y, N, stream=side.cuda_stream)
    keep = pos.clone()
    for turn in range(4):
        pos.copy_(keep if turn % 2 == 0 else other)
        enc.zero_()
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        encode(P, tab, pos, other_enc)       # the program's own work between the replays
        net.inference(pos, other_y, N)
        torch.cuda.synchronize()
        assert same(enc, other_enc) and same(y, other_y)
        if turn % 2 == 0:
            assert same(enc, want_enc) and same(y, want_y)
    net.close()


def test_streams_and_threads_share_a_grid():
    P = pkg()
    N = 1 << 16
    net = grid(P, N)
    ins = [positions(N, 10 + k) for k in range(4)]
    want = [torch.zeros(N, 16, device="cuda") for _ in ins]
    for p, w in zip(ins, want):
        net.inference(p, w, N)
    torch.cuda.synchronize()
    got = [torch.zeros(N, 16, device="cuda") for _ in ins]
    shared = torch.cuda.Stream()
    streams = [torch.cuda.Stream(), torch.cuda.Stream(), shared, shared]   # the last two threads on one stream
    failed = []

    def work(k):
        try:
            for _ in range(20):
                net.inference(ins[k], got[k], N, stream=streams[k].cuda_stream)
            streams[k].synchronize()
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    for g, w in zip(got, want):
        assert same(g, w)
    net.close()
