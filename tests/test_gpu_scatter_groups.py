"""The table-gradient scatter where its launches change: level groups per batch size (one level per workgroup
for the smallest, 4 at 85 rounds of 512 samples, 8 from 86 to 128, all levels from 129 on), the largest batch without a second accumulate
launch and the next one, level counts that leave a short last group, and gradients off 16-byte alignment; within
the per-word bound of the oracle's fp64 sums."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import pyoracle as orc  # noqa: E402

from helpers import assert_scatter_close, pkg, positions, scatter_bound, scatter_quantum  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,shift,spread", [(1, 16, 0, 1.0), (511, 7, 0, 1.0), (513, 17, 2, 1.0), (4096, 16, 0, 1e-3),
                                              (6144, 16, 0, 1e-3), (6145, 16, 2, 1e-3), (8192, 5, 0, 1e-3),
                                              (8193, 16, 0, 1e-3), (33333, 12, 2, 1.0), (85 * 512, 16, 0, 0.1),
                                              (85 * 512 + 1, 16, 0, 0.1), (65536, 16, 2, 0.1), (65537, 16, 0, 0.1),
                                              (65536, 20, 0, 1.0), (65537, 9, 0, 0.1),
                                              (130560, 16, 2, 1.0), (130561, 16, 0, 0.1)])
def test_scatter_groups_match_oracle(N, L, shift, spread):
    P = pkg()
    print(f"[scatter groups] N={N} L={L} shift={shift} spread={spread}", flush=True)
    T_, b = 1 << 14, 1.3
    rng = np.random.default_rng(N)
    pos = positions(N, 3)
    pos[:, :3] = (0.4 + spread * (pos[:, :3] - 0.5)).clip(0, 1)
    denc = rng.normal(0, 1, (N, 2 * L)).astype(np.float16)
    denc[::7] = 0  # samples without records
    d_denc = torch.zeros(N * 2 * L + shift, dtype=torch.float16, device="cuda")
    d_denc[shift:] = torch.from_numpy(denc).cuda().reshape(-1)
    grads = torch.full((L * T_ * 2,), 0.5, dtype=torch.float32, device="cuda")
    P.launch("launchHashTableBackwardKernel", d_denc.data_ptr() + 2 * shift, torch.from_numpy(pos).cuda(), grads, N, T_,
             L, b, 16, 2, None)
    torch.cuda.synchronize()
    g, gabs, cnt = orc.hash_scatter_stats(pos, denc, T_, L, 16, b)
    bound = scatter_bound(g, gabs, cnt, scatter_quantum(denc, L, T_))
    assert_scatter_close(grads.cpu().numpy(), g + np.float32(0.5), bound, base=0.5, what="hash grads")
