"""Prefill passes of few 256-row blocks (up to 512 tokens): the split count follows the key range and the row blocks,
up to 64, and the shortest passes convert their raw tiles in the loop instead of through fp16 images.  Both sides of
every boundary (row blocks: 42 / 43 / 85 / 128 / 170 / 213 / 512 tokens; key ranges of one tile, of fewer tiles than
splits, and long), every row against the oracle at the path's tolerance (kvutil: max-abs 2e-3, rel-L2 1e-3: fp16 keys,
queries, probabilities and output)."""
import pytest
import torch

import qwengine_amd.ops as ops
from kvutil import KVTS, KV_NAMES, assert_close, dequant_cache, make_cache, seeded_normal

pytestmark = pytest.mark.gpu

N_POS = 6100


@pytest.fixture(scope="module", params=KVTS, ids=lambda k: KV_NAMES[k])
def cache(request, gpu):
    kv, _, _ = make_cache(request.param, N_POS, N_POS, seed=900 + request.param)
    return kv, dequant_cache(kv, N_POS)


@pytest.mark.parametrize("B,p0", [(1, 0), (1, 6099), (3, 30), (21, 0), (42, 6058), (43, 31), (43, 5000), (85, 6000),
                                  (86, 1), (128, 4000), (129, 2500), (170, 33), (171, 5900), (213, 700), (512, 64),
                                  (513, 64)])
def test_short_pass_vs_oracle(gpu, oracle, cache, B, p0):
    kv, (Kd, Vd) = cache
    print(f"short prefill {KV_NAMES[kv.kvt]} B={B} p0={p0}", flush=True)
    q, gate = seeded_normal((B, 24, 256), 910 + B), seeded_normal((B, 24, 256), 911 + B)
    out = torch.full((B, 24, 256), float("nan"), dtype=torch.float16, device="cuda")
    # a caller-owned workspace of exactly the stated size, filled with NaN: nothing outside what the call writes counts
    work = torch.full((ops.attn_prefill_work_bytes(B, p0 + B) // 4,), float("nan"), device="cuda")
    ops.attn_prefill_ws(q, gate, kv, kv.kvt, B, p0, out, work)
    torch.cuda.synchronize()
    ref = oracle.attention(q.cpu().numpy(), gate.cpu().numpy(), Kd, Vd, p0, B)
    assert_close(out.float().cpu().numpy(), ref, f"B={B} p0={p0}")


@pytest.mark.parametrize("B,p0", [(86, 139), (86, 170), (299, 0), (320, 41), (341, 5700)])
def test_short_pass_of_eight_splits(gpu, oracle, cache, B, p0):
    """8 splits, by the row blocks (299 to 341 tokens) or by the tiles (keys that end at 225 to 256): not the kernel of the
    1024-token passes, which have as many."""
    test_short_pass_vs_oracle(gpu, oracle, cache, B, p0)


# either side of every line between raw tiles and images: tokens, and positions for 1, 2, 3, 4 row blocks
ROUTES = {ops.F16: [(36, 900), (37, 900), (42, 2559), (42, 2560), (85, 4095), (85, 4096), (128, 6143), (128, 6144),
                    (170, 16383), (170, 16384), (171, 16384)],
          ops.Q8_0: [(20, 900), (21, 900), (42, 16383), (42, 16384), (43, 16384)],
          ops.Q4_0: [(36, 900), (37, 900), (42, 4607), (42, 4608), (85, 18431), (85, 18432), (86, 18432)]}


@pytest.mark.parametrize("kvt", KVTS, ids=lambda k: KV_NAMES[k])
def test_both_forms_at_the_lines_between_them(gpu, oracle, kvt):
    kv, _, _ = make_cache(kvt, 18432, 18432, seed=930 + kvt)
    Kd, Vd = dequant_cache(kv, 18432)
    for B, n in ROUTES[kvt]:
        print(f"prefill form {KV_NAMES[kvt]} B={B} n={n}", flush=True)
        q, gate = seeded_normal((B, 24, 256), 940 + B), seeded_normal((B, 24, 256), 941 + B)
        out = torch.full((B, 24, 256), float("nan"), dtype=torch.float16, device="cuda")
        work = torch.full((ops.attn_prefill_work_bytes(B, n) // 4,), float("nan"), device="cuda")
        ops.attn_prefill_ws(q, gate, kv, kvt, B, n - B, out, work)
        torch.cuda.synchronize()
        # the oracle on the first, a middle and the last tokens
        for t in (0, B // 2, B - 3):
            ref = oracle.attention(q[t:t + 3].cpu().numpy(), gate[t:t + 3].cpu().numpy(), Kd, Vd, n - B + t, 3)
            assert_close(out[t:t + 3].float().cpu().numpy(), ref, f"B={B} n={n} t={t}")


def test_work_bytes_never_decrease(gpu):
    """A workspace for a longer chunk or context covers every shorter call."""
    for n in (1, 33, 5000, 262144):
        sizes = [ops.attn_prefill_work_bytes(B, max(n, B)) for B in range(1, 1400)]
        assert sizes == sorted(sizes)
