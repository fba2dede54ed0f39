"""The gradient's partial sums: bounded however many matrices a call has, and the same minors where
the bound makes a workgroup walk several chunks."""
import numpy as np
import pytest

from theboss_amd import _lib as L


def test_workspace_stays_below_two_to_the_16_workgroups():
    lib = L.load()
    for n in range(2, L.TB_SWEEP_MAX_K + 1):
        for B in (1, 3, 16, 64, 1000, 4096, 10000, 65536, 100000):
            assert lib.tb_perm_grad_workspace_size(n, B) <= max(1 << 16, B) * n * n * 16, (n, B)


@pytest.mark.gpu
@pytest.mark.parametrize("n,B", [(19, 33000), (20, 17000), (21, 8500)])
def test_minors_of_a_batch_at_the_bound(oracle, n, B):
    """Against the same matrices in a batch of three; both sum the same chunks in another order."""
    import torch as T

    from theboss_amd import ops

    few = 3
    g = T.Generator(device="cuda").manual_seed(n)
    A = T.randn(B, n, n, 2, generator=g, device="cuda", dtype=T.float64)
    A = T.view_as_complex(A) * (0.5 / np.sqrt(n))
    for conj in (False, True):
        perm, G = ops.perm_grad_batch(A, conj=conj)
        for at in (0, B // 2, B - few):
            p, g3 = ops.perm_grad_batch(A[at:at + few].contiguous(), conj=conj)
            assert T.max(T.abs(G[at:at + few] - g3)) <= 1e-12 * T.max(T.abs(g3))
            assert T.max(T.abs(perm[at:at + few] - p)) <= 1e-12 * T.max(T.abs(g3))
