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


BUFFERS = ["qg", "k", "v", "qn", "kn", "rope", "q", "gate", "kv.k", "kv.v", "kv.ks", "kv.vs"]


@pytest.mark.parametrize("kvt", KVTS, ids=lambda k: KV_NAMES[k])
def test_any_misaligned_buffer_takes_the_general_kernel(gpu, kvt):
    """Every buffer in turn 4 bytes (a cache buffer 2 bytes) off: the same bits as with all of them aligned."""
    B, p0, cap = 19, 3, 24
    data = {n: seeded_normal((s,), 70 + i) for i, (n, s) in enumerate((("qg", B * 12288), ("k", B * 1024), ("v", B * 1024),
                                                                      ("qn", 256), ("kn", 256)))}
    data["rope"] = torch.empty(B * 64, device="cuda")
    ops.rope_table(p0, B, 1e7, data["rope"])

    def placed(name, numel, dtype, init=None):
        """numel elements, shifted by 4 bytes (2 in the cache) if this is the buffer that `off` names"""
        size = torch.empty((), dtype=dtype).element_size()
        shift = ((2 if name.startswith("kv.") else 4) if name == off else 0) // size
        t = torch.full((numel + 16,), 7, dtype=dtype, device="cuda")[shift:shift + numel]
        if init is not None:
            t.copy_(init)
        assert (t.data_ptr() % 16 != 0) == (name == off)
        return t

    want = None
    for off in [None] + BUFFERS:
        if kvt == ops.F16 and off in ("kv.ks", "kv.vs"):
            continue
        print(f"prep rows {KV_NAMES[kvt]} misaligned: {off}", flush=True)
        a = {n: placed(n, t.numel(), t.dtype, t) for n, t in data.items()}
        q, gate = (placed(n, B * 6144, torch.float32) for n in ("q", "gate"))
        vb = ops.kv_value_bytes(kvt)
        kv = ops.KVLayer(kvt, cap, *(placed(n, 4 * cap * vb, torch.uint8).view(4, cap, vb) for n in ("kv.k", "kv.v")),
                         *(None if kvt == ops.F16 else placed(n, 4 * cap * 8, torch.int16).view(4, cap, 8)
                           for n in ("kv.ks", "kv.vs")))
        ops.attn_prep_rows(a["qg"], a["k"], a["v"], a["qn"], a["kn"], B, p0, a["rope"], 1e-6, kvt, kv, q, gate)
        torch.cuda.synchronize()
        got = [t.clone() for t in (q, gate, kv.k, kv.v, kv.ks, kv.vs) if t is not None]
        want = want or got
        assert all(torch.equal(x, y) for x, y in zip(got, want)), off
