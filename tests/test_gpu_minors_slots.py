"""Minors by input slot where one wave sweeps an item and writes them without a second pass: those of
an item that holds fewer particles than the call says are 0 (a column of each is), the other items
the same as with a slot to spare, which takes the second pass."""
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


@pytest.mark.parametrize("k,batch", [(2, 1), (2, 300), (3, 64), (5, 1000), (7, 4), (12, 500),
                                     (13, 2000), (14, 2000)])
def test_items_with_empty_slots(T, oracle, k, batch):
    from theboss_amd import ops

    rng = np.random.default_rng(k)
    m = 2 * k + 2
    U = T.from_numpy(oracle.haar_unitary(m, 8)).cuda()
    i32 = lambda a: T.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()  # noqa: E731
    ins = np.sort(np.argsort(rng.random((batch, m)), axis=1)[:, :k], axis=1)
    outs = np.sort(np.argsort(rng.random((batch, m)), axis=1)[:, :k - 1], axis=1)
    mult = np.ones((batch, k), dtype=np.int32)
    short = np.arange(batch) % 3 == 0
    mult[short, rng.integers(0, k, short.sum())] = 0
    mult[3::9, :2] = 0
    pad = np.zeros((batch, 1), dtype=np.int32)
    out = [i32(outs), i32(np.ones_like(outs))]
    got = ops.cc_submatrices_batch(U, *out, i32(ins), i32(mult), k, True).cpu().numpy()
    want = ops.cc_submatrices_batch(U, *out, i32(np.hstack([ins, pad])),
                                    i32(np.hstack([mult, pad])), k, True).cpu().numpy()
    assert not want[:, k].any()
    full = mult.all(axis=1)
    assert not got[~full].any() and not want[~full].any()
    assert got[full].all()
    assert np.array_equal(got[full], want[full, :k])
