"""Which calls the Glynn entry without a workspace refuses: those whose flags and partial sums exceed
its static array. The FP32 column sums need no more than the FP64 ones: no copy of the matrices."""
import ctypes

import numpy as np
import pytest

from theboss_amd import _lib as L


def partial_bytes(lib, n, B):
    return lib.tb_glynn_workspace_size(n, B, L.TB_PREC_FP64)  # no copy in it


@pytest.mark.parametrize("prec", [L.TB_PREC_FP64, L.TB_PREC_FP32_COLSUM,
                                  L.TB_PREC_FP32_COLSUM_ANY_N])
def test_limit_is_that_of_the_partial_sums(prec):
    """Valid arguments but for the pointer to the matrices, which is looked at after the size: a call
    is refused for its size (TB_ERANGE) or for that or the missing GPU."""
    lib = L.load()
    for n in (14, 17, 21, 22, 23, 30, 40):
        lo, hi = 1, 1 << 24  # the batch sizes around the limit
        while hi - lo > 1:
            mid = (lo + hi) // 2
            lo, hi = (mid, hi) if partial_bytes(lib, n, mid) <= L.TB_GLYNN_NOALLOC_SCRATCH_BYTES \
                else (lo, mid)
        for B in (1, 4544, lo, hi, 2 * hi):
            rc = lib.tb_glynn_batch_noalloc(None, n, B, n * n, prec, ctypes.c_void_p(256), None)
            too_large = partial_bytes(lib, n, B) > L.TB_GLYNN_NOALLOC_SCRATCH_BYTES
            assert (rc == L.TB_ERANGE) == too_large, (n, B)
            assert rc != L.TB_OK


@pytest.mark.gpu
def test_fp32_batch_near_the_limit(oracle):
    import torch as T

    from theboss_amd import _device as D
    from theboss_amd import ops

    n, B = 21, 4500
    U = oracle.haar_unitary(2 * n, 7)
    rng = np.random.default_rng(2)
    rows = np.sort(np.argsort(rng.random((B, 2 * n)), axis=1)[:, :n], axis=1)
    A = T.from_numpy(U[rows][:, :, :n].copy()).cuda()
    out = T.full((B,), np.nan, dtype=T.complex128, device="cuda")
    L.check(L.load().tb_glynn_batch_noalloc(D.ptr(A), n, B, n * n, L.TB_PREC_FP32_COLSUM,
                                            D.ptr(out), D.stream_ptr(A.device)))
    assert T.equal(out, ops.glynn_batch(A, L.TB_PREC_FP32_COLSUM))
