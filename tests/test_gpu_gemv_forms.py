"""The decode GEMV has a wide and a narrow form of some kernels, taken by the number of rows and the row length: both give a
row the same bits, on either side of every line of the rule (256, 512 and 768 workgroups of 8 rows; rows of 8192 values).
One call of 64 rows is checked against the oracle (test_gpu_gemv.py's bound); every longer call repeats those rows."""
import numpy as np
import pytest
import torch

import qwengine_amd.ops as ops
from test_gpu_gemv import FMTS, NAMES, act
from wutil import random_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", FMTS, ids=lambda f: NAMES[f])
@pytest.mark.parametrize("K", [8192, 8448, 17408])
def test_forms_agree(gpu, oracle, fmt, K):
    print(f"gemv forms {NAMES[fmt]} K={K}", flush=True)
    Wn = random_rows(fmt, 64, K, 400 + fmt)
    rb = Wn.shape[1]
    base = torch.from_numpy(Wn).cuda()
    a = act(torch.randn((4, K), generator=torch.Generator("cuda").manual_seed(K), device="cuda"))
    idx = torch.arange(6145, device="cuda") * 37 % 64
    W = base[idx].contiguous()
    q, d = a.q.cpu().numpy().reshape(4, K), a.d.cpu().numpy().reshape(4, K // 32)
    ref = oracle.gemv_ref(fmt, Wn, K, 64, q, d)
    Wf = np.abs(oracle.w_dequant(fmt, Wn, K).astype(np.float64))
    for nb in (1, 2, 3, 4):
        want = torch.empty((nb, 64), device="cuda")
        ops.gemv_q8n(fmt, base, rb, K, 64, a, nb, K, want, 64)
        for c in range(nb):
            mag = Wf @ np.abs(np.repeat(d[c].astype(np.float64), 32) * q[c])
            assert (np.abs(want[c].cpu().numpy().astype(np.float64) - ref[c]) / mag).max() < 2e-6
        for N in (2048, 2049, 4096, 4097, 6144, 6145):
            y = torch.full((nb, N + 3), 7.0, device="cuda")
            ops.gemv_q8n(fmt, W, rb, K, N, a, nb, K, y, N + 3)
            assert torch.equal(y[:, :N], want[:, idx[:N]]), (nb, N)
            assert (y[:, N:] == 7.0).all()
