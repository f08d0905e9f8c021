"""The tile kernel (bf_gemm above 128 batch rows) on the GPU: against the dense
kernel's 128-row launches on the same inputs, and against the oracle.

Both kernels multiply the same fp16 weights and accumulate in fp32, each output
over K terms in an order of its own, so an output of either is within
K * 2^-24 * sum_k |a w| of the exact sum and the two differ by at most twice
that (fp16 outputs: plus the rounding, 2^-11 of the value)."""
import numpy as np
import pytest
import torch

import busfill as bf
import oracle as O

pytestmark = pytest.mark.gpu

QTS = [O.Q4_0_PLANES, O.Q4_0, O.Q4_K]
QT_NAME = {O.Q4_0_PLANES: "planes", O.Q4_0: "q4_0", O.Q4_K: "q4_k"}


def to_dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()


def operands(qt, M, N, K, seed):
    w = O.gen_weights(qt, N, K, seed=seed)
    A = O.gen_act(M, K, seed=seed + 1)
    return w, to_dev(w.W), (to_dev(w.W_aux) if w.W_aux is not None else None), A, to_dev(A)


def magnitudes(qt, Wd, aux, Ad, N, K):
    """sum_k |a w| over the fp16 weights, fp32 (its own rounding is far below the bound's slack)."""
    deq = torch.empty((N, K), dtype=torch.int16, device="cuda")
    bf.dequant_f16(qt, Wd, aux, deq, N, K)
    return Ad.view(torch.float16).float().abs() @ deq.view(torch.float16).float().abs().t().contiguous()


# one k step range, ragged rows and columns, every tile shape (64, 128 and 256
# wide), tiles cut along K (the remainder of a round) and several m bands
SHAPES = [(129, 1, 256), (129, 128, 512), (192, 127, 768), (257, 300, 1280), (300, 1024, 1024), (640, 129, 2304),
          (193, 5120, 512), (1000, 1000, 1024), (2000, 17408, 512)]


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tile_matches_dense_slices(qt, M, N, K):
    w, Wd, aux, A, Ad = operands(qt, M, N, K, seed=M + N + K)
    C, D = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
    print(f"tile {QT_NAME[qt]} M={M} N={N} K={K}", flush=True)
    bf.gemm(qt, Wd, aux, Ad, C, M, N, K)
    bf.gemm(qt, Wd, aux, Ad, D, M, N, K, algo=bf.ALGO_DENSE)
    bound = 2 * K * 2.0 ** -24 * magnitudes(qt, Wd, aux, Ad, N, K) + 1e-30
    assert ((C - D).abs() <= bound).all()
    H = torch.empty((M, N), dtype=torch.float16, device="cuda")
    bf.gemm(qt, Wd, aux, Ad, H, M, N, K, otype=bf.OUT_F16)
    assert (H == C.half()).all()
    again = torch.empty_like(C)
    bf.gemm(qt, Wd, aux, Ad, again, M, N, K)
    assert (again == C).all()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", [(130, 70, 512), (300, 200, 1024)])
def test_tile_against_oracle_and_entry_points(qt, M, N, K):
    """The oracle's gate; strided rows and untouched columns; the
    caller-owned workspace, the no-allocation entry and the batched call give
    the same bits."""
    w, Wd, aux, A, Ad = operands(qt, M, N, K, seed=5 * M + N)
    lda, ldc = K + 8, N + 3
    Ax = torch.zeros((M, lda), dtype=torch.int16, device="cuda")
    Ax[:, :K] = Ad
    C = torch.full((M, ldc), -7.0, device="cuda")
    bf.gemm(qt, Wd, aux, Ax, C, M, N, K, lda=lda, ldc=ldc)
    assert (C[:, N:] == -7.0).all()
    ok, mae, rfe, nf = O.gate(C[:, :N].cpu().numpy(), O.gemm_f64(w, A))
    assert ok, (mae, rfe, nf)
    ref = C[:, :N].contiguous()
    nb = bf.gemm_workspace_bytes(qt, M, N, K)
    ws = torch.empty(max(nb, 256), dtype=torch.uint8, device="cuda")
    D = torch.empty((M, N), device="cuda")
    bf.gemm_ws(qt, Wd, aux, Ad, D, M, N, K, ws if nb else None, nb)
    assert (D == ref).all()
    D.fill_(0)
    bf.gemm_noalloc(qt, Wd, aux, Ad, D, M, N, K)
    assert (D == ref).all()
    E = torch.empty((M, N), device="cuda")
    bf.gemm_batched(qt, [(Wd, aux, Ad, D.fill_(0), M, N, K), (Wd, aux, Ad, E, M, N, K)])
    assert (D == ref).all() and (E == ref).all()
