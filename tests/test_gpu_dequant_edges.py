"""Prefill dequantizer at the edges of its work split (waves of 64 sub-blocks, workgroups of 256, or of two runs of 256 in
large IQ2_S calls; rows shorter and longer than a wave's span, row strides wider than the row): bit-exact with the oracle's fp32 value rounded to fp16
(nearest-even), and nothing written behind the output."""
import numpy as np
import pytest
import torch

import qwengine_amd.ops as ops
from wutil import random_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [ops.W_Q4_K, ops.W_Q6_K, ops.W_IQ2_S, ops.W_IQ3_S])
@pytest.mark.parametrize("K,rows,pad", [(256, 1, 0), (256, 7, 0), (256, 9, 16), (2048, 3, 0), (2304, 5, 0), (5120, 7, 32),
                                        (17408, 2, 0), (8192, 4, 0), (8448, 4, 0), (256, 1025, 0)])
def test_dequant_edges_bit_exact(gpu, oracle, fmt, K, rows, pad):
    Wn = random_rows(fmt, rows, K, 300 + fmt)
    rb = Wn.shape[1]
    W = torch.zeros((rows, rb + pad), dtype=torch.uint8, device="cuda")
    W[:, :rb] = torch.from_numpy(Wn).cuda()
    out = torch.full((rows * K + 4096,), float("nan"), dtype=torch.float16, device="cuda")
    ops.dequant_rows_f16(fmt, W, rb + pad, K, rows, out)
    torch.cuda.synchronize()
    want = oracle.w_dequant(fmt, Wn, K).astype(np.float16).reshape(-1)
    assert np.array_equal(out[:rows * K].cpu().numpy().view(np.uint16), want.view(np.uint16))
    assert torch.isnan(out[rows * K:]).all()


@pytest.mark.parametrize("K,rows", [(256, 32767), (256, 32768), (256, 32801), (256, 32833), (2304, 3641)])
def test_dequant_iq2_s_paired_runs(gpu, oracle, K, rows):
    """IQ2_S from 262144 sub-blocks on: two runs a workgroup; the last workgroup full, ending in its first run, in its
    second one, and across rows."""
    test_dequant_edges_bit_exact(gpu, oracle, ops.W_IQ2_S, K, rows, 0)
