"""The one-launch Glynn kernel of small matrices at the edges of its split: one lane per
matrix up to a whole workgroup, batches that leave lane groups idle, rows from LDS (n <= 6,
FP32) and in broadcast form (n = 7..13), every chunk the tuning table can ask for, padded
strides and matrices with zeros."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# relative to the sum of the Glynn terms' magnitudes, 2^(n-1) terms of n - 1 complex multiplies
# and at most 2^9 row updates each: well under 1e-12 in FP64; FP32 sums and products 5e-5
BOUND = {0: 1e-12, 1: 5e-5}


@pytest.fixture(scope="module")
def T():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from theboss_amd import _lib

    _lib.load()
    return torch


def glynn_terms(A):
    """(perm, mean magnitude of the terms) of each n x n matrix, by Glynn's formula in numpy."""
    n = A.shape[-1]
    d = 1.0 - 2.0 * ((np.arange(2 ** (n - 1))[:, None] >> np.arange(n)) & 1)
    t = np.prod(np.einsum("ti,bij->btj", d, A), axis=2)
    return (t * np.prod(d, axis=1)).sum(1) / 2 ** (n - 1), np.abs(t).mean(1)


@pytest.mark.parametrize("n", range(2, 14))
@pytest.mark.parametrize("precision", [0, 1])
def test_every_split(T, oracle, n, precision):
    from theboss_amd import autotune, ops

    base = np.stack([oracle.haar_unitary(2 * n, 31 * n + b)[:n, :n] for b in range(7)])
    base[5] = np.eye(n)
    base[6, n // 2] = 0.0
    ref, scale = glynn_terms(base)
    for B in (1, 3, 67, 1501):
        A = T.from_numpy(np.ascontiguousarray(base[np.arange(B) % 7])).cuda()
        try:
            for c in (0, 1, 2, 3, 5, 8, 12) if B == 67 else (0,):
                autotune.set_entry("glynn", n, c, B)
                got = ops.glynn_batch(A, precision).cpu().numpy()
                err = np.abs(got - ref[np.arange(B) % 7])
                assert np.all(err <= BOUND[precision] * scale[np.arange(B) % 7]), (B, c)
        finally:
            autotune.set_entry("glynn", n, 0, B)


@pytest.mark.parametrize("n", [3, 7, 13])
def test_padded_matrix_stride(T, oracle, n):
    from theboss_amd import _device as D
    from theboss_amd import _lib as L
    from theboss_amd import ops

    B, stride = 9, n * n + 5
    As = np.stack([oracle.haar_unitary(2 * n, n + b)[:n, :n] for b in range(B)])
    flat = np.full((B, stride), np.nan, dtype=np.complex128)
    flat[:, :n * n] = As.reshape(B, -1)
    Ad = T.from_numpy(flat).cuda()
    out = T.empty(B, dtype=T.complex128, device="cuda")
    L.check(L.load().tb_glynn_batch(D.ptr(Ad), n, B, stride, 0, D.ptr(out), None, 0,
                                    D.stream_ptr(Ad.device)))
    assert T.equal(out, ops.glynn_batch(T.from_numpy(As).cuda()))
