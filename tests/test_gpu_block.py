"""The block-wise GEMM (bf_gemm for Q4_0 formats with K % 256 != 0 or operands
off their 16-byte boundaries) against the one-thread-per-output kernel on the
same inputs (run on an MI355X).

Neither rounds a weight and both accumulate in fp32, over at most K + 8 terms
in orders of their own, so the two differ by at most 2 (K + 8) * 2^-24 *
sum_k |a w| (fp16 outputs: plus the rounding)."""
import numpy as np
import pytest
import torch

import busfill as bf
import oracle as O

pytestmark = pytest.mark.gpu

QTS = [O.Q4_0_PLANES, O.Q4_0]
QT_NAME = {O.Q4_0_PLANES: "planes", O.Q4_0: "q4_0"}


# (M, N, K): (MT, NT, NW), the form of the kernel it runs (16 MT batch rows x 16 NT weight rows; NT = 0: activations
# through LDS, NW of the eight waves over weight rows); tests/test_plans.py holds the plans to it on the CPU.
FORMS = {
    (1, 1, 32): (1, 1, 8), (16, 15, 96): (1, 1, 8), (17, 33, 288): (2, 1, 8), (48, 300, 160): (3, 1, 8),
    (64, 17, 1184): (4, 1, 8), (65, 100, 2336): (4, 1, 8), (1, 4900, 416): (1, 2, 8), (129, 1700, 96): (4, 2, 8),
    (5, 70, 512): (1, 1, 8), (140, 64, 1024): (4, 1, 8), (20, 5000, 416): (2, 2, 8), (40, 4900, 416): (3, 2, 8),
    (129, 2800, 1184): (3, 0, 4), (80, 4200, 1056): (3, 0, 4), (260, 2600, 416): (4, 0, 4), (300, 2600, 32): (4, 0, 4),
    (300, 3301, 96): (4, 0, 8), (300, 3301, 1120): (4, 0, 8), (129, 6000, 1120): (3, 0, 8),
}


def to_dev(a, shift=0):
    """On the device, `shift` elements into a buffer of its own."""
    t = torch.from_numpy(np.ascontiguousarray(a).view(np.int16 if a.dtype == np.uint16 else a.dtype))
    buf = torch.zeros(t.numel() + 16, dtype=t.dtype, device="cuda")
    buf[shift:shift + t.numel()] = t.reshape(-1).cuda()
    return buf[shift:]


def run(qt, w, A, M, N, K, *, algo=bf.ALGO_AUTO, a_shift=0, w_shift=0, pad=0, otype=bf.OUT_F32):
    lda = K + pad
    Ax = np.zeros((M, lda), np.uint16)
    Ax[:, :K] = A
    C = torch.full((M, N + pad), -7.0, device="cuda", dtype=torch.float32 if otype == bf.OUT_F32 else torch.float16)
    bf.gemm(qt, to_dev(w.W, w_shift), to_dev(w.W_aux, w_shift // 2) if w.W_aux is not None else None,
            to_dev(Ax, a_shift), C, M, N, K, lda=lda, ldc=N + pad, algo=algo, otype=otype)
    assert (C[:, N:] == -7.0).all()
    return C[:, :N].cpu().numpy()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K,a_shift,w_shift,pad", [
    (1, 1, 32, 0, 0, 0), (16, 15, 96, 0, 0, 0), (17, 33, 288, 0, 0, 3), (48, 300, 160, 1, 0, 0), (64, 17, 1184, 0, 0, 5),
    (65, 100, 2336, 3, 2, 1), (1, 4900, 416, 0, 0, 0), (129, 1700, 96, 0, 0, 0), (5, 70, 512, 1, 0, 1),
    (140, 64, 1024, 0, 2, 0), (20, 5000, 416, 0, 0, 0), (40, 4900, 416, 0, 0, 1)])
def test_block_matches_simple(qt, M, N, K, a_shift, w_shift, pad):
    w = O.gen_weights(qt, N, K, seed=N + K)
    A = O.gen_act(M, K, seed=M + K)
    kw = dict(a_shift=a_shift, w_shift=w_shift, pad=pad)
    C = run(qt, w, A, M, N, K, **kw)
    D = run(qt, w, A, M, N, K, algo=bf.ALGO_SIMPLE, **kw)
    mag = np.abs(O.f16_bits_to_f32(A)).astype(np.float64) @ np.abs(O.dequant_f32(w)).astype(np.float64).T
    assert (np.abs(C.astype(np.float64) - D) <= 2 * (K + 8) * 2.0 ** -24 * mag).all()
    assert (run(qt, w, A, M, N, K, **kw) == C).all()
    assert (run(qt, w, A, M, N, K, otype=bf.OUT_F16, **kw) == C.astype(np.float16)).all()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
def test_block_non_finite_rows(qt):
    """An infinite or NaN activation, and an infinite scale, reach the same
    outputs as in the one-thread-per-output kernel and no others."""
    M, N, K = 20, 40, 352
    w = O.gen_weights(qt, N, K, seed=9)
    scales = w.W_aux if qt == O.Q4_0_PLANES else w.W.reshape(N, K // 32, 18)[:, :, :2].view(np.uint16)[..., 0]
    scales[3, 5] = 0x7C00
    A = O.gen_act(M, K, seed=10)
    A[2, 7], A[11, 100], A[19, 351] = 0x7C00, 0x7E00, 0xFC00
    C, D = run(qt, w, A, M, N, K), run(qt, w, A, M, N, K, algo=bf.ALGO_SIMPLE)
    assert (np.isfinite(C) == np.isfinite(D)).all()
    assert not np.isfinite(C[[2, 11, 19]]).any() and not np.isfinite(C[:, 3]).any()
    assert np.isfinite(np.delete(np.delete(C, [2, 11, 19], 0), 3, 1)).all()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K,a_shift,w_shift,pad", [
    (129, 2800, 1184, 1, 2, 1), (80, 4200, 1056, 0, 0, 0), (260, 2600, 416, 0, 0, 5), (300, 2600, 32, 0, 0, 0),
    (300, 3301, 96, 0, 0, 3), (300, 3301, 1120, 3, 2, 1), (129, 6000, 1120, 0, 0, 0)])
def test_block_staged_matches_simple(qt, M, N, K, a_shift, w_shift, pad):
    """The form with the activations in LDS: three and four row tiles, K whole
    and in two halves, block counts off its steps of four, one block."""
    test_block_matches_simple(qt, M, N, K, a_shift, w_shift, pad)


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", [(129, 2800, 1056), (300, 3301, 352)])
def test_block_staged_non_finite_rows(qt, M, N, K):
    """Infinite and NaN activations in a row's first and last block, which the
    steps past the end read again, stay in their rows; an infinite last scale in
    its column."""
    w = O.gen_weights(qt, N, K, seed=9)
    scales = w.W_aux if qt == O.Q4_0_PLANES else w.W.reshape(N, K // 32, 18)[:, :, :2].view(np.uint16)[..., 0]
    scales[3, K // 32 - 1] = 0x7C00
    A = O.gen_act(M, K, seed=10)
    A[2, 7], A[11, 100], A[19, K - 1] = 0x7C00, 0x7E00, 0xFC00
    C, D = run(qt, w, A, M, N, K), run(qt, w, A, M, N, K, algo=bf.ALGO_SIMPLE)
    assert np.array_equal(np.isfinite(C), np.isfinite(D))
    assert np.isfinite(np.delete(np.delete(C, [2, 11, 19], 0), 3, 1)).all()


@pytest.mark.parametrize("qt", QTS, ids=lambda q: QT_NAME[q])
@pytest.mark.parametrize("M,N,K", [(1, 40, 352), (20, 4900, 352), (129, 2800, 1056), (300, 3301, 352)])
def test_block_infinite_scales(qt, M, N, K):
    """Weights of infinite scale give what they give one by one: NaN where a code
    is 8 or the signs differ, an infinity of the right sign where they agree."""
    w = O.gen_weights(qt, N, K, seed=11)
    blocks = K // 32
    planes = qt == O.Q4_0_PLANES
    scales = w.W_aux.reshape(N, blocks) if planes else w.W.reshape(N, blocks, 18)[:, :, :2].view(np.uint16)[..., 0]
    codes = w.W.reshape(N, blocks, 16) if planes else w.W.reshape(N, blocks, 18)[:, :, 2:]
    A = O.gen_act(M, K, seed=12)
    A[0] &= 0x7FFF
    A[0] |= 0x2000                                     # row 0: all positive, none zero
    scales[3, blocks - 1], scales[5, 0], scales[7, 1], scales[9, blocks // 2] = 0x7C00, 0xFC00, 0x7E00, 0x7C00
    codes[5, 0] = 0x99                                 # q - 8 = 1 throughout: -inf times a positive row
    codes[9, blocks // 2] = 0x77                       # -1 throughout
    for otype in (bf.OUT_F32, bf.OUT_F16):
        C, D = (run(qt, w, A, M, N, K, algo=a, otype=otype) for a in (bf.ALGO_AUTO, bf.ALGO_SIMPLE))
        odd = ~np.isfinite(D)
        assert (odd == ~np.isfinite(C)).all() and odd[:, [3, 5, 7, 9]].all() and odd.sum() == 4 * M
        assert np.array_equal(C[odd], D[odd], equal_nan=True)
        assert C[0, 5] == -np.inf and C[0, 9] == -np.inf and np.isnan(C[0, [3, 7]]).all()
