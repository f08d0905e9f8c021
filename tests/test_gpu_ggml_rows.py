"""ggml hook, two to eight fp32 rows: rounded to fp16 inside the LDS kernel, bit
for bit bf_gemm on the rounded rows, with no workspace (run on an MI355X)."""
import numpy as np
import pytest
import torch

import busfill as bf
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt,gt", [(O.Q4_0, bf.GGML_Q4_0), (O.Q4_K, bf.GGML_Q4_K)], ids=["q4_0", "q4_k"])
# step rings (17408 x 5120: batch 2-8), the activation rings that are staged (8192: tests/test_plans.py)
@pytest.mark.parametrize("N,K", [(1, 1024), (77, 2048), (5120, 5120), (17408, 1024), (17408, 5120), (300, 8192),
                                 (3000, 8192)])
def test_fp32_rows_equal_gemm_on_rounded_rows(qt, gt, N, K):
    w = O.gen_weights(qt, N, K, seed=N + K)
    W = torch.from_numpy(w.W).cuda()
    g = torch.Generator().manual_seed(N + K)
    for M in range(2, 9):
        for pad in (0, 4):
            x = torch.randn(M, K + pad, generator=g).cuda()
            x[:, K:] = float("nan")                      # row padding: never read
            y, want = (torch.full((M, N), -7.0, device="cuda") for _ in range(2))
            views = bf.ggml_view(W, gt), bf.ggml_view(x[:, :K]), bf.ggml_view(y)
            staged = K == 8192 and M >= {(300, O.Q4_K): 8, (3000, O.Q4_0): 8, (3000, O.Q4_K): 7}.get((N, qt), 9)
            assert (bf.ggml_mul_mat_workspace_bytes(*views) > 0) == staged
            bf.ggml_mul_mat(*views)
            half = x[:, :K].half().contiguous()
            bf.gemm(qt, W, None, half, want, M, N, K)
            assert (y == want).all(), (M, pad)
