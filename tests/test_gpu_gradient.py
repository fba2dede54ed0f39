"""The gradient sweep at the edges of its layouts: the direct expansion (n <= 5), 4 and 2 lanes
per code, columns padded to a multiple of the lanes, one workgroup per matrix and several,
workgroups with fewer waves (n > 28), fewer static bits (n > 32), padded matrix strides, and
the conjugated form the backward pass keeps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL = 1e-10  # the FP64 bar against the oracle, as for the other FP64 kernels


@pytest.fixture(scope="module")
def T():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from theboss_amd import _lib

    _lib.load()
    return torch


def dev_c(T, a):
    return T.from_numpy(np.ascontiguousarray(a, dtype=np.complex128)).cuda()


@pytest.mark.parametrize("n,B", [(2, 1), (3, 257), (4, 64), (5, 300), (6, 1), (7, 5), (8, 700),
                                 (9, 2), (11, 1), (13, 40), (16, 1), (17, 3), (18, 1), (19, 2),
                                 (20, 1)])
def test_minors_and_conjugates_vs_oracle(T, oracle, n, B):
    from theboss_amd import ops

    As = np.stack([oracle.haar_unitary(2 * n, 70 * n + b % 8)[:n, :n] * (1 + b % 3) for b in range(B)])
    A = dev_c(T, As)
    perm, G = (x.cpu().numpy() for x in ops.perm_grad_batch(A))
    permc, Gc = (x.cpu().numpy() for x in ops.perm_grad_batch(A, conj=True))
    assert np.array_equal(perm, permc) and np.array_equal(Gc, G.conj())
    for b in sorted({0, B // 2, B - 1}):
        ref = oracle.perm_minors(As[b])
        assert np.max(np.abs(G[b] - ref)) <= REL * np.max(np.abs(ref)), (n, b)
        p = oracle.perm_glynn_matrix(As[b], 1)
        assert abs(perm[b] - p) <= REL * abs(p), (n, b)


@pytest.mark.parametrize("n", [28, 29, 33])
def test_laplace_expansions_past_the_oracle(T, oracle, n):
    """Every row's and every column's expansion equals the Glynn kernel's permanent."""
    from theboss_amd import ops

    As = oracle.haar_unitary(2 * n, 3 * n)[:n, :n][None]
    A = dev_c(T, As)
    _, G = ops.perm_grad_batch(A)
    G = G.cpu().numpy()[0]
    p = ops.glynn_batch(A).cpu().numpy()[0]
    for axis in (0, 1):
        # n products of relative error REL each, their sum of absolute values beside |perm|
        bound = REL * np.sum(np.abs(As[0] * G), axis=axis)
        assert np.all(np.abs(np.sum(As[0] * G, axis=axis) - p) <= bound + REL * abs(p)), (n, axis)


@pytest.mark.parametrize("n,B", [(4, 3), (8, 3), (15, 3)])
def test_padded_matrix_stride(T, oracle, n, B):
    from theboss_amd import _device as D
    from theboss_amd import _lib as L
    from theboss_amd import ops

    As = np.stack([oracle.haar_unitary(2 * n, n + b)[:n, :n] for b in range(B)])
    stride = n * n + 3
    flat = np.full((B, stride), np.nan, dtype=np.complex128)
    flat[:, :n * n] = As.reshape(B, -1)
    Ad = dev_c(T, flat)
    perm = T.empty(B, dtype=T.complex128, device="cuda")
    G = T.empty((B, n, n), dtype=T.complex128, device="cuda")
    lib = L.load()
    need = lib.tb_perm_grad_workspace_size(n, B)
    ws = D.workspace(max(need, 1))
    L.check(lib.tb_perm_grad_batch(D.ptr(Ad), n, B, stride, D.ptr(perm), D.ptr(G), D.ptr(ws), need,
                                   D.stream_ptr(Ad.device)))
    p0, G0 = ops.perm_grad_batch(dev_c(T, As))
    assert T.equal(perm, p0) and T.equal(G, G0)
