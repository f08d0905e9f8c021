"""bf_dequant_f16's wide kernel (aligned weights and output) and its general one
(anything else) give the oracle's bits (run on an MI355X)."""
import numpy as np
import pytest
import torch

import busfill as bf
import oracle as O

pytestmark = pytest.mark.gpu


def to_dev(a):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()


@pytest.mark.parametrize("qt", [O.Q4_0_PLANES, O.Q4_0, O.Q4_K], ids=["planes", "q4_0", "q4_k"])
@pytest.mark.parametrize("N,blocks", [(1, 1), (3, 5), (65, 7), (129, 9)])
def test_wide_and_general_dequant(qt, N, blocks):
    K = blocks * (256 if qt == O.Q4_K else 32)
    w = O.gen_weights(qt, N, K, seed=N + K)
    Wd, aux = to_dev(w.W), (to_dev(w.W_aux) if w.W_aux is not None else None)
    want = O.dequant_f16(w)
    for shift in (0, 1):                         # fp16 elements off the 16-byte boundary
        out = torch.full((N * K + 16,), -1, dtype=torch.int16, device="cuda")
        bf.dequant_f16(qt, Wd, aux, out[shift:], N, K)
        got = out.cpu().numpy().view(np.uint16)
        assert (got[shift:shift + N * K].reshape(N, K) == want).all()
        assert (got[shift + N * K:] == 0xFFFF).all() and (got[:shift] == 0xFFFF).all()
