"""Gated DeltaNet prefill at the edges of its 16-token chunks (whole and ragged last chunks, every remainder of the three
chunks that the recurrence keeps in flight), against the oracle with the bounds of test_gpu_deltanet.py: outputs within
half an fp16 ulp of the rounded oracle plus the fp32 kernel's error, state within rel 2e-4, conv window exact.  The
scratch is a guard from the last float of the layout on: 14400 floats per token of the padded chunks (12288 of v, q, k and
transposed k, 2112 of coefficients), which dn_work_bytes(B) covers."""
import numpy as np
import pytest
import torch

import qwengine_amd.ops as ops
from test_gpu_deltanet import EPS, RTOL, VD, VH, Layer, gpu_state, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [3, 15, 16, 31, 33, 48, 49, 64, 80, 95, 97, 145])
@pytest.mark.parametrize("strong_decay", [False, True])
def test_rows_chunk_edges(gpu, oracle, B, strong_decay):
    print(f"deltanet_rows B={B} strong_decay={strong_decay}", flush=True)
    L = Layer(200 + B, 0.1, 0.5)
    qkv, z, b, a = L.tokens(B)
    if strong_decay:
        a[::3, :VH] += 60.0  # decays that underflow to 0 within a chunk
        b[1::4, :VH] = -40.0  # tokens that write almost nothing
    p = L.device(0)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    n, stated = (B + 15) // 16 * 16 * 14400, ops.dn_work_bytes(B) // 4
    assert stated >= n
    work = torch.full((stated + 1024,), float("nan"), device="cuda")
    core = torch.empty((B, VD), device="cuda")
    o16 = torch.empty((B, VD), dtype=torch.float16, device="cuda")
    ops.deltanet_rows(p, dev(qkv), dev(z), dev(b[:, :VH]), dev(a[:, :VH]), B, 0, EPS, work, core, o16)
    torch.cuda.synchronize()
    assert torch.isnan(work[n:]).all()
    o = o16.float().cpu().numpy()
    o_ref, cs_ref, S_ref = L.oracle(oracle, qkv, z, b[:, :VH], a[:, :VH])
    assert rel_l2(o, o_ref) < 1e-3
    assert np.all(np.abs(o - o_ref) <= 2e-3 + 2.0 ** -11 * np.abs(o_ref))
    assert rel_l2(gpu_state(p), S_ref) < RTOL
    assert np.array_equal(p.conv_state[1].cpu().numpy(), cs_ref)
