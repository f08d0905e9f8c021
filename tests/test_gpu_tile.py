"""The tile kernel (bf_gemm above 128 batch rows) on the GPU: against the dense
kernel's 128-row launches on the same inputs, and against the oracle; and the
batches that stay with 128-row launches.

Both kernels multiply the same fp16 weights and accumulate in fp32, each output
over K terms in an order of its own, so an output of either is within
K * 2^-24 * sum_k |a w| of the exact sum and the two differ by at most twice
that (fp16 outputs: plus the rounding, 2^-11 of the value)."""
import threading

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


# (M, N, K): (TA, NB, whole rounds of tiles, S), the form of the kernel it runs (tiles of 64 TA x 128 NB,
# the tiles past the whole rounds cut in S ranges of K); tests/test_plans.py holds the plans to it on the CPU.
# One super-group to dozens per range, ragged rows and columns, several bands of tiles; the last three are
# prefill calls at their full size.
FORMS = {
    (129, 1, 256): (2, 1, 0, 1), (129, 128, 512): (2, 1, 0, 1), (192, 127, 768): (2, 1, 0, 3),
    (257, 300, 1280): (2, 1, 0, 3), (300, 1024, 1024): (2, 1, 0, 2), (640, 129, 2304): (2, 1, 0, 3),
    (193, 5120, 512): (2, 1, 0, 1), (1000, 1000, 1024): (2, 1, 0, 1), (2000, 17408, 512): (4, 2, 2, 1),
    (129, 130, 4096): (3, 1, 0, 16), (700, 2000, 3072): (3, 1, 0, 4), (1000, 4097, 768): (3, 1, 0, 1),
    (513, 12000, 2048): (3, 1, 1, 4), (193, 4097, 4096): (4, 1, 0, 4), (1025, 16500, 1536): (4, 1, 2, 1),
    (1500, 6000, 4096): (4, 1, 1, 8), (257, 16500, 768): (4, 2, 0, 1), (2000, 8200, 512): (4, 2, 1, 2),
    (1500, 12000, 3072): (4, 2, 1, 4),
    (512, 17408, 5120): (4, 1, 1, 10), (2000, 17408, 5120): (4, 2, 2, 4), (2000, 5120, 17408): (4, 1, 1, 4),
}


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", FORMS)
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


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", [(129, 128, 512), (700, 2000, 3072), (193, 4097, 4096), (1500, 12000, 3072)])
def test_tile_weights_equal_dense(qt, M, N, K):
    """Rows of A with a single one read the weights out: in every tile shape the
    dense kernel's, bit for bit."""
    w, Wd, aux, A, Ad = operands(qt, M, N, K, seed=M + K)
    k = torch.randperm(max(M, K), generator=torch.Generator().manual_seed(M))[:M] % K
    Ad.zero_()
    Ad.view(torch.float16)[torch.arange(M), k] = 1.0
    C, D = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
    bf.gemm(qt, Wd, aux, Ad, C, M, N, K)
    bf.gemm(qt, Wd, aux, Ad, D, M, N, K, algo=bf.ALGO_DENSE)
    assert (C == D).all() and (C != 0).any()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", [(132, 2048, 8192), (129, 17408, 5120)])
def test_sliced_batches_equal_their_launches(qt, M, N, K):
    """Up to 256 rows of some matrices stay with launches of 128 rows: the same
    bits as a call for each slice."""
    w, Wd, aux, A, Ad = operands(qt, M, N, K, seed=M + N)
    C, D = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
    bf.gemm(qt, Wd, aux, Ad, C, M, N, K)
    bf.gemm(qt, Wd, aux, Ad, D, 128, N, K)
    bf.gemm(qt, Wd, aux, Ad[128:], D[128:], M - 128, N, K)
    assert (C == D).all()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", [(300, 200, 1024), (193, 4097, 4096), (2000, 8200, 512)])
def test_tile_non_finite(qt, M, N, K):
    """Infinite and NaN activations and scales reach the outputs they reach in
    the dense kernel, with its infinities and NaN, and no others."""
    w, Wd, aux, A, Ad = operands(qt, M, N, K, seed=3 * M)
    x = Ad.view(torch.float16)
    x[5, 7], x[60, 100], x[M - 1, K - 1], x[128, 0] = float("inf"), float("nan"), -float("inf"), float("inf")
    x[128, K - 1] = -float("inf")
    bits = {3: 0x7C00, 9: 0xFC00, N - 1: 0x7E00}
    for n, h in bits.items():
        if aux is not None:
            aux.view(N, K // 32)[n, n % (K // 32)] = h - (1 << 16) if h > 0x7FFF else h
        else:
            blk = Wd.view(N, -1, 144 if qt == O.Q4_K else 18)
            blk[n, n % blk.shape[1], 0], blk[n, n % blk.shape[1], 1] = h & 255, h >> 8
    C, D = (torch.full((M, N), 7.0, device="cuda") for _ in range(2))
    bf.gemm(qt, Wd, aux, Ad, C, M, N, K)
    bf.gemm(qt, Wd, aux, Ad, D, M, N, K, algo=bf.ALGO_DENSE)
    odd = ~D.isfinite()
    assert (odd == ~C.isfinite()).all() and (C.isnan() == D.isnan()).all()
    assert (C[D.isinf()] == D[D.isinf()]).all()
    assert odd[[5, 60, 128, M - 1]].all() and odd[:, list(bits)].all()
    odd[[5, 60, 128, M - 1]] = False
    odd[:, list(bits)] = False
    assert not odd.any()


def test_threads_share_a_stream_and_its_partials():
    """Two host threads issue calls whose cut tiles are summed by a second launch
    from the stream's workspace, on one stream: each gets its own bits."""
    s = torch.cuda.Stream()
    qt, M, N, K = O.Q4_K, 300, 1024, 2048              # two ranges of K and more
    ops = [operands(qt, M, N, K, seed=70 + t) for t in range(2)]
    assert bf.gemm_workspace_bytes(qt, M, N, K) > 0
    torch.cuda.synchronize()

    def call(t, C):
        bf.gemm(qt, ops[t][1], None, ops[t][4], C, M, N, K, stream=s)

    want = [torch.empty((M, N), device="cuda") for _ in range(2)]
    outs = [[torch.full((M, N), float("nan"), device="cuda") for _ in range(24)] for _ in range(2)]
    torch.cuda.synchronize()
    errors = []

    def run(t):
        try:
            for C in outs[t]:
                call(t, C)
        except Exception as e:          # noqa: BLE001 -- reported by the main thread
            errors.append(e)

    for t in range(2):
        call(t, want[t])
    s.synchronize()
    ts = [threading.Thread(target=run, args=(t,)) for t in range(2)]
    for th in ts:
        th.start()
    for th in ts:
        th.join()
    s.synchronize()
    assert not errors, errors
    assert not (want[0] == want[1]).all()
    for t in range(2):
        for C in outs[t]:
            assert (C == want[t]).all()
