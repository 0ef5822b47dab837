"""attn_prep_rows takes one kernel on 16-byte aligned buffers and another on any others: both give the same bits, for every
cache format, on rows of ordinary values and on rows with ties, zeros, infinities and NaN."""
import pytest
import torch

import qwengine_amd.ops as ops
from kvutil import KVTS, KV_NAMES, seeded_normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kvt", KVTS, ids=lambda k: KV_NAMES[k])
@pytest.mark.parametrize("B,p0", [(1, 0), (2, 31), (3, 0), (7, 100), (64, 5), (203, 17)])
def test_aligned_and_general_kernels_agree(gpu, kvt, B, p0):
    qg, k, v = (seeded_normal(s, 40 + i) for i, s in enumerate(((B, 24, 512), (B, 4, 256), (B, 4, 256))))
    k[0, 1] = 0.0
    v[0, 0] = 0.0
    v[0, 1] = torch.tensor([3.0, -3.0], device="cuda").repeat(128)
    v[0, 2, 5] = float("inf")
    v[0, 3, 40] = float("nan")
    qg[0, 3, 7] = float("nan")
    qg[0, 4, 300] = float("inf")
    qn, kn = (0.5 + torch.rand(256, device="cuda") for _ in range(2))
    rope = torch.empty((B, 64), device="cuda")
    ops.rope_table(p0, B, 1e7, rope)
    got = []
    for off in (0, 1):  # floats by which q_out misses 16-byte alignment
        kv = ops.KVLayer.allocate(kvt, p0 + B + 3)
        q = torch.full((B * 6144 + 8,), 7.0, device="cuda")
        gate = torch.full((B * 6144,), 7.0, device="cuda")
        ops.attn_prep_rows(qg, k, v, qn, kn, B, p0, rope, 1e-6, kvt, kv, q[off:off + B * 6144], gate)
        torch.cuda.synchronize()
        assert (q[:off] == 7.0).all() and (q[off + B * 6144:] == 7.0).all()
        got.append([q[off:off + B * 6144].clone(), gate, kv.k, kv.v] + ([] if kv.ks is None else [kv.ks, kv.vs]))
    for a, b in zip(*got):
        as_int = lambda t: t.view(torch.int32) if t.dtype == torch.float32 else t
        assert torch.equal(as_int(a), as_int(b))
