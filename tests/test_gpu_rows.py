"""GPU parity of the row stream kernel (automatic calls on row-major weights, 2 <= M <= 16) against the oracle's
tolerance rule, where it can go wrong: channel counts around the 16-row tile, one k-step, an odd number of k-steps, as
many pairs as wavefronts, the most pairs a wavefront holds and one more (a K split, or the general kernel), runs of
uneven length, weight rows further apart than K, and every K split the workspace allows."""
import numpy as np
import pytest
import torch

import qwen_fastpath as qf
from qwen_fastpath import _lib as L
from helpers import bf16_bits, dev_inputs

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.mark.parametrize("N,K", [(1, 64), (15, 128), (17, 192), (100, 1024), (1000, 1088), (4100, 960), (272, 10240),
                                 (256, 10304), (300, 17408), (5000, 2112), (12300, 320), (70000, 64)])
def test_row_stream_shapes(oracle, N, K):
    for M in (2, 5, 11, 16) if N * K < 3000000 else (3, 16):
        inp = oracle.gen_inputs(M, N, K, seed=M + N + K)
        x, w, s = dev_inputs(inp, DEV)
        for _ in range(2):  # a K split's arrival counters are back at zero for the next call
            y = bf16_bits(qf.w8a16_mm(x, w, s, None, torch.bfloat16))
            rep = oracle.check_w8a16(y, inp.x, inp.w, inp.s)
            assert rep.ok, (M, N, K, rep)
        y32 = qf.w8a16_mm(x, w, s, None, torch.float32).cpu()
        assert np.array_equal(bf16_bits(y32.to(torch.bfloat16)), y), (M, N, K)  # the same sums before the rounding


@pytest.mark.parametrize("N,K,Ms", [(333, 1984, (2, 16)), (700, 10304, (5, 16)), (9000, 1472, (3, 12)), (9000, 3136, (5,)),
                                    (12300, 320, (11,)), (40000, 320, (2, 16)), (6000, 2112, (7,))])
def test_row_stream_half_lines(oracle, N, K, Ms):
    """Rows that start in the middle of a cache line, on the shapes that the row stream kernel keeps (rows_plan): one
    tile and up to ten a run, one pair and several, with and without a K split."""
    for M in Ms:
        assert L.rows_plan(M, N, K) is not None, (M, N, K)
        inp = oracle.gen_inputs(M, N, K, seed=M + N + K)
        x, w, s = dev_inputs(inp, DEV)
        for _ in range(2):
            rep = oracle.check_w8a16(bf16_bits(qf.w8a16_mm(x, w, s, None, torch.bfloat16)), inp.x, inp.w, inp.s)
            assert rep.ok, (M, N, K, rep)


def test_row_stream_strided_weights(oracle):
    """Rows 48 bytes further apart than K, NaN-free garbage between them, the last row ending the allocation."""
    M, N, K = 7, 333, 1984
    inp = oracle.gen_inputs(M, N, K, seed=5)
    x, _, s = dev_inputs(inp, DEV)
    buf = torch.full((N * (K + 48),), 99, dtype=torch.int8, device=DEV)
    w = buf.as_strided((N, K), (K + 48, 1))
    w.copy_(torch.from_numpy(inp.w))
    rep = oracle.check_w8a16(bf16_bits(qf.w8a16_mm(x, w.t(), s, None, torch.bfloat16)), inp.x, inp.w, inp.s)
    assert rep.ok, rep
