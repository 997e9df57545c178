"""The encode launcher where its path changes: below and above the size from which rows are made from
level-major encodings, ragged tails, level counts that are not a multiple of four or eight, position strides
and unaligned outputs; bit-exact against the oracle."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import pyoracle as orc  # noqa: E402

from helpers import pkg, positions  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,stride,shift", [(255, 16, 4, 0), (257, 9, 3, 0), ((1 << 15) - 1, 16, 4, 0),
                                              (1 << 15, 16, 3, 0), (40001, 7, 4, 0), (33333, 17, 3, 2),
                                              (65537, 8, 5, 2)])
def test_encode_rows_bit_exact(N, L, stride, shift):
    P = pkg()
    print(f"[encode rows] N={N} L={L} stride={stride} shift={shift}", flush=True)
    T_, b = 1 << 14, 1.3
    pos = np.zeros((N, stride), np.float32)
    pos[:, :3] = positions(N, 5)[:, :3]
    k = min(N, 256)
    pos[:k, :3] = np.random.default_rng(6).choice(np.float32([0, 1, 0.5, np.nextafter(np.float32(1), 0)]), (k, 3))
    table = np.random.default_rng(7).uniform(-1, 1, L * T_ * 2).astype(np.float16)
    opt = P.MLPGridOptions(vectorDim=4, hiddenDim=64, outputDim=16, numLayers=2, activationType=0, tableSize=T_,
                           numLevels=L, b=b, lowestSize=16, featuresLevel=2)
    out = torch.zeros(N * 2 * L + shift, dtype=torch.float16, device="cuda")  # shift halves off 16-byte alignment
    for _ in range(2):
        P.launch("launchHashEncodeKernel", C.byref(opt), torch.from_numpy(table).cuda(), torch.from_numpy(pos).cuda(),
                 stride, out.data_ptr() + 2 * shift, N, None)
    torch.cuda.synchronize()
    p4 = np.zeros((N, 4), np.float32)
    p4[:, :3] = pos[:, :3]
    want = orc.hash_encode(p4, table, T_, L, 16, b).view(np.uint16)
    got = out[shift:].cpu().numpy().view(np.uint16).reshape(N, 2 * L)
    np.testing.assert_array_equal(got, want)
