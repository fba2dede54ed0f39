"""Gradient of a matrix with an infinite or NaN entry: the minors that leave its row out do not depend
on it and are those of the matrix with that row put to 0; the ones that have it are not finite, and
no other matrix of the batch is touched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [
    (n, 7) for n in (2, 3, 5, 6, 7, 8, 9, 12, 13, 14, 17, 18, 19, 20)] + [
    (n, 4100) for n in (2, 3, 5, 6, 7, 8, 9, 12, 13, 14)])  # several workgroups a matrix, and one
def test_rows_without_the_entry_are_finite(oracle, n, batch):
    import torch as T

    from theboss_amd import ops

    rng = np.random.default_rng(n)
    A = np.stack([oracle.haar_unitary(2 * n, 3 + b)[:n, :n] for b in range(7)])
    A = np.tile(A, (-(-batch // 7), 1, 1))[:batch]
    zeroed, where = A.copy(), {}
    for b, bad in ((0, np.nan), (1, np.inf), (3, complex(0, -np.inf)), (batch - 2, complex(np.nan, 1))):
        i, j = (0, n - 1) if b == 0 else (n - 1, 0) if b == 1 else rng.integers(0, n, 2)
        A[b, i, j], where[b] = bad, (i, j)
        zeroed[b, i] = 0
    if n > 2:
        A[4, 0, 1] = A[4, 2, 0] = np.nan  # two rows: nothing of the matrix is left
    perm, G = (x.cpu().numpy() for x in ops.perm_grad_batch(T.from_numpy(A).cuda()))
    p0, G0 = (x.cpu().numpy() for x in ops.perm_grad_batch(T.from_numpy(zeroed).cuda()))
    for b in range(batch):
        if b == 4 and n > 2:
            assert not np.isfinite(perm[b])
            assert not np.isfinite(G[b][[r for r in range(n) if r not in (0, 2)]]).all() or n == 3
            assert n < 6 or not np.isfinite(G[b]).any()
        elif b in where:
            i, j = where[b]
            assert not np.isfinite(perm[b])
            scale = np.max(np.abs(G0[b][i]))
            assert np.max(np.abs(G[b][i] - G0[b][i])) <= 1e-12 * scale
            rest = np.delete(np.delete(G[b], i, 0), j, 1)
            assert not np.isfinite(rest).any()
        else:
            assert np.array_equal(G[b], G0[b]) and perm[b] == p0[b]
