"""The minors sweep across its chunk plan and task split, against Glynn permanents of the same
matrices without one row: one wave per item (the minors written directly) and several, batches
that the XCDs do not divide, items without a particle to pair, and empty slots in between. Both
sides are FP64 walks of at most 2^17 codes whose errors are below 1e-13 of an item's largest
minor for these matrices (condition below 10^3), so they agree to 1e-11."""
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


def _reference(T, V):
    from theboss_amd import ops

    B, k, _ = V.shape
    rows = T.tensor([[r for r in range(k) if r != d] for d in range(k)], device="cuda")
    M = V[:, rows, :].reshape(B * k, k - 1, k - 1).contiguous()
    return ops.glynn_batch(M).reshape(B, k)


@pytest.mark.parametrize("k,items", [(2, 5), (4, 1), (7, 9), (8, 12), (11, 300), (12, 1), (12, 500),
                                     (12, 1027), (13, 37), (14, 3), (14, 67), (15, 1), (16, 9),
                                     (16, 17), (17, 2), (18, 1), (18, 3)])
def test_plans_and_tasks(T, k, items):
    from theboss_amd import ops

    rng = np.random.default_rng(100 * k + items)
    m = k + 3
    U = rng.normal(size=(m, m)) + 1j * rng.normal(size=(m, m))
    U[2, 0] = 0.0  # a zero in every column set: items holding mode 0 pair with another
    if items % 2:
        U[0] = np.where(np.arange(m) % 2, U[0], 0.0)
    U = U / np.sqrt(m)
    # item b: input modes of k, output rows of k - 1, both random
    ins = np.array([np.sort(rng.permutation(m)[:k]) for _ in range(items)], dtype=np.int32)
    outs = np.array([np.sort(rng.permutation(m)[:k - 1]) for _ in range(items)], dtype=np.int32)
    V = np.stack([U[np.ix_(o, i)].T for o, i in zip(outs, ins)])
    Vd = T.from_numpy(np.ascontiguousarray(V)).cuda()
    ref = _reference(T, Vd) if k > 2 else Vd.flip(1)[:, :, 0]
    scale = ref.abs().amax(dim=1, keepdim=True)

    def close(got):
        assert bool(((got - ref).abs() <= 1e-11 * scale).all())

    close(ops.sweep_minors_batch(Vd, k))
    dev = lambda a: T.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()  # noqa: E731
    Ud, ones = T.from_numpy(U).cuda(), np.ones((items, k), dtype=np.int32)
    om, ou = dev(outs), dev(np.ones_like(outs))
    close(ops.cc_submatrices_batch(Ud, om, ou, dev(ins), dev(ones), k, True))
    # the same particles with an empty slot in front: placed behind it, a zero in it
    wide_m, wide_u = np.zeros((items, k + 1)), np.zeros((items, k + 1))
    wide_m[:, 1:], wide_u[:, 1:] = ins, 1
    got = ops.cc_submatrices_batch(Ud, om, ou, dev(wide_m), dev(wide_u), k, True)
    assert not got[:, 0].abs().any()
    close(got[:, 1:])


# waves that walk several chunks: one wave per item (written directly) and several, with the wide
# reduction too, and batches just past a round of waves
@pytest.mark.parametrize("k,items", [(13, 1025), (14, 1501), (16, 301), (18, 70), (20, 17)])
def test_several_chunks_per_wave(T, k, items):
    test_plans_and_tasks(T, k, items)
