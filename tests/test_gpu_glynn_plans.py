"""Glynn permanents of n >= 14 across the chunk plan: matrices of one workgroup and of several,
the paired walk and, in the same batch, matrices that it does not take.

Full matrices are u_i v_j with entries of modulus 1, perm = n! prod u prod v; block matrices have
two such blocks (their zeros leave no row to divide by), perm the product of the blocks'. Walking
n = 26 the terms' magnitudes add up to about 10^5 permanents, each term rounded n times, so FP64
is held to 1e-9; FP32 column sums at n = 23 to 10^4 of them times 23 half units of 2^-24, over
2^22 terms of random sign well below 5e-3."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from theboss_amd import _lib

    _lib.load()
    return torch


def _rank_one(rng, n):
    u, v = np.exp(2j * np.pi * rng.random((2, n)))
    return np.outer(u, v), math.factorial(n) * np.prod(u) * np.prod(v)


def _matrix(rng, n, full):
    if full:
        return _rank_one(rng, n)
    a, pa = _rank_one(rng, n // 2)
    b, pb = _rank_one(rng, n - n // 2)
    M = np.zeros((n, n), dtype=complex)
    M[:n // 2, :n // 2], M[n // 2:, n // 2:] = a, b
    return M, pa * pb


@pytest.mark.parametrize("precision", ["TB_PREC_FP64", "TB_PREC_FP32_COLSUM"])
@pytest.mark.parametrize("n,batch", [(14, 1), (14, 300), (15, 7), (16, 2), (17, 2), (17, 120),
                                     (19, 33), (20, 3), (21, 5), (22, 9), (23, 2), (25, 2), (26, 2)])
def test_plans_and_paths(T, n, batch, precision):
    from theboss_amd import _lib, ops

    rng = np.random.default_rng(n * 1000 + batch)
    pairs = [_matrix(rng, n, (i + n) % 3 != 0) for i in range(batch)]
    want = np.array([p for _, p in pairs])
    A = T.from_numpy(np.stack([m for m, _ in pairs])).cuda()
    got = ops.glynn_batch(A, getattr(_lib, precision)).cpu().numpy()
    fp32 = precision != "TB_PREC_FP64" and n <= _lib.TB_FP32_COLSUM_MAX_N
    assert np.max(np.abs(got - want) / np.abs(want)) <= (5e-3 if fp32 else 1e-9)
    # the same through the entry point that uses no workspace of the caller
    out = T.empty(batch, dtype=T.complex128, device="cuda")
    _lib.check(_lib.load().tb_glynn_batch_noalloc(
        A.data_ptr(), n, batch, n * n, getattr(_lib, precision), out.data_ptr(),
        T.cuda.current_stream().cuda_stream))
    assert np.array_equal(out.cpu().numpy(), got)
