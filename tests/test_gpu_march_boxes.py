"""The march over boxes of every kind against the oracle: cubes around the origin, whose quotients
come from a reciprocal and whose cascades from comparisons, and boxes off centre or of unequal
sides, which divide.  Bar: bit-exact (both forms give the correctly rounded quotient and the same
cascade).  The quotient itself is checked in double precision, where the residuals are exact."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as orc
from helpers import pkg

torch = pytest.importorskip("torch")

BELOW_ONE = float(np.nextafter(np.float32(1), np.float32(0)))
BOXES = [([-1.5] * 3, [1.5] * 3), ([-0.7] * 3, [0.7] * 3), ([-1.3] * 3, [1.3] * 3), ([-11.9] * 3, [11.9] * 3),
         ([-0.9999999] * 3, [0.9999999] * 3),
         ([-1.3, -1.3, -1.3], [1.3, 1.3, 1.4]), ([-1.0, -1.2, -1.1], [1.1, 1.0, 1.2]),
         ([-BELOW_ONE] * 3, [BELOW_ONE] * 3)]             # an extent with an all-ones significand: divides


def test_the_last_box_has_an_all_ones_extent():
    mn, mx = (np.float32(v[0]) for v in BOXES[-1])
    assert (mx - mn).view(np.uint32) & 0x7fffff == 0x7fffff


def fma32(a, b, c):
    """fmaf on float32: the product of two floats is exact in double, and np.longdouble (64-bit
    significand) rounds the sum once more than fmaf only for ties that need over 64 bits."""
    return (a.astype(np.longdouble) * b.astype(np.longdouble) + c.astype(np.longdouble)).astype(np.float32)


@pytest.mark.parametrize("ext", [3.0, 1.4, 2.6, 23.8, 1.0, 1.9999997, 0.0011, 7e5])
def test_two_corrections_give_the_quotient(ext):
    """a r, corrected twice by its residual, is a / b for r = 1 / b, at every scale of a."""
    b = np.float32(ext)
    r = np.float32(1) / b
    rng = np.random.default_rng(3)
    a = np.concatenate([(rng.uniform(-2, 2, 200000) * ext), 10.0 ** rng.uniform(-20, 20, 100000),
                        np.nextafter(np.float32(ext) * np.float32(2.0) ** np.arange(-12, 13, dtype=np.float32),
                                     np.float32(np.inf))]).astype(np.float32)
    B, Rr = np.full_like(a, b), np.full_like(a, r)
    q = a * Rr
    for _ in range(2):
        q = fma32(fma32(-q, B, a), Rr, q)
    np.testing.assert_array_equal(q.view(np.uint32), (a / b).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("Cc,L,K", [(1, 4, 1), (2, 3, 2), (5, 4, 1), (8, 2, 1), (3, 6, 1), (34, 2, 1)])
@pytest.mark.parametrize("box", range(len(BOXES)))
def test_march_boxes_bit_exact(box, Cc, L, K):
    print(f"[march box] {BOXES[box]} C={Cc} L={L} K={K}", flush=True)
    P = pkg()
    dev = torch.device("cuda:0")
    res, R = 32, 1200
    mn, mx = (np.float32(v) for v in BOXES[box])
    rng = np.random.default_rng(100 * Cc + box)
    cells = Cc * sum((res >> l) ** 3 for l in range(L))
    bits = np.packbits((rng.random(cells + (-cells) % 8) < 0.75).astype(np.uint8), bitorder="little")
    o = (rng.uniform(-1.2, 1.2, (R, 3)) * mx[2] * 2.0 ** rng.integers(0, min(Cc, 8), (R, 1))).astype(np.float32)
    d = rng.normal(size=(R, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o[:4] = np.float32([[0, 0, 0], mx, mn, mx * np.float32(2)])  # on the boxes' own corners
    d[:3] = np.float32([[1, 0, 0], [0, -1, 0], [0, 0, 1]])
    if Cc == 34:                                                 # far beyond where quotients overflow
        o[4:8] = np.float32([[2e30, 0, 0], [0, -3e38, 0], [3e38, 3e38, 3e38], [0, 0, 1e31]])
        d[4:8] = np.float32([[-1, 0, 0], [0, 1, 0], [-1, -1, -1], [0, 0, -1]])
    di, nr, fr = orc.ray_aabb_inv(o, d, mn, mx, Cc)
    fr = np.where(np.arange(R) % 97 == 5, fr * np.float32(1.5), fr).astype(np.float32)  # on past the box
    want = orc.march_hits(o, d, di, nr, fr, bits, [res] * 3, mn, mx, Cc, L, K, 1 << 30)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    keep = [T(a) for a in (o, d, di, nr, fr, bits)]
    cap = max(want["total"], 1) + 1
    cnt, off, ridx, act = (torch.zeros(n, dtype=torch.int32, device=dev) for n in (R, R, cap, 1))
    pos, ts = torch.zeros((cap, 4), device=dev), torch.zeros(cap, device=dev)
    total = C.c_uint32(0)
    u3, f3 = P.Uint3(res, res, res), lambda v: P.Float3(float(v[0]), float(v[1]), float(v[2]))
    got = P.lib().processRaysHitLinear(R, *[k.data_ptr() for k in keep], u3, f3(mn), f3(mx), Cc, L, K, cap,
                                       C.byref(total), act.data_ptr(), cnt.data_ptr(), off.data_ptr(),
                                       pos.data_ptr(), ridx.data_ptr(), ts.data_ptr(), None, None)
    P.check()
    torch.cuda.synchronize()
    n = total.value
    assert got == R and n == want["total"] and n > 0
    np.testing.assert_array_equal(cnt.cpu().numpy().view(np.uint32), want["counts"])
    np.testing.assert_array_equal(ridx.cpu().numpy().view(np.uint32)[:n], want["ray_idx"])
    np.testing.assert_array_equal(ts.cpu().numpy()[:n].view(np.uint32), want["t"].view(np.uint32))
    np.testing.assert_array_equal(pos.cpu().numpy()[:n].view(np.uint32), want["pos"].view(np.uint32))
