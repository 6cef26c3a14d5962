"""bf16 products at every way of reading the operands (quads of k, pairs of rows,
element by element), at the edges of their tiles and on both sides of the
length from which the sum is cut over waves.

Tolerance: the products of bf16 numbers are exact in FP32, and any order of
summing K of them is within K 2^-24 of the sum of their magnitudes.
"""
import numpy as np
import pytest
import torch

from oracle import proposal_oracle as PO
from partgs_amd import proposal as SP

pytestmark = pytest.mark.gpu


def _operand(x, rows_first, offset):
    """The operand's bits with k (or the rows) contiguous, `offset` elements into its buffer."""
    bits = PO.bf16_bits(np.ascontiguousarray(x if rows_first else x.T)).view(np.int16).reshape(-1)
    t = torch.from_numpy(np.concatenate([np.zeros(offset, np.int16), bits])).cuda()[offset:]
    return t, ((x.shape[1], 1) if rows_first else (1, x.shape[0]))


@pytest.mark.parametrize("M,N,K", [(31, 33, 511), (32, 32, 512), (34, 66, 514), (64, 2, 516), (128, 64, 2048),
                                   (1, 1, 700), (66, 130, 17), (63, 64, 260), (96, 34, 8)])
@pytest.mark.parametrize("a_k,b_k,offset", [(True, True, 0), (True, False, 0), (False, True, 0), (False, False, 0),
                                            (True, True, 2), (False, False, 1)])
def test_layouts(M, N, K, a_k, b_k, offset):
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    A, B = (PO.bf16_round(rng.normal(size=(n, K)).astype(np.float32)) for n in (M, N))
    bias = rng.normal(size=N).astype(np.float32)
    (At, sa), (Bt, sb) = _operand(A, a_k, offset), _operand(B, b_k, offset)
    exact = A.astype(np.float64) @ B.astype(np.float64).T
    tol = (K + 4) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T + np.abs(bias) + 1)
    got = SP.gemm(At, Bt, M=M, N=N, K=K, a_strides=sa, b_strides=sb, bias=torch.from_numpy(bias).cuda())
    assert (np.abs(got.cpu().numpy() - (exact + bias)) <= tol).all()
    out = torch.full((M, N), 2.0, device="cuda")
    got, bits = SP.gemm(At, Bt, M=M, N=N, K=K, a_strides=sa, b_strides=sb, relu=True, alpha=-0.5, out=out,
                        accumulate=True, want_bf16=True)
    assert (np.abs(got.cpu().numpy() - (np.maximum(-0.5 * exact, 0) + 2)) <= tol + 2.0 ** -22).all()
    assert np.array_equal(bits.cpu().numpy().view(np.uint16), PO.bf16_bits(got.cpu().numpy()))
