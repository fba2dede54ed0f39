"""The minors sweep that gathers its items while staging: slot lists longer than a wave, empty
and negative slots, padding at either end, the reductions of few and of many partial sums and
sizes whose sums need two values per lane, against the oracle or the compact form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL = 1e-10  # the FP64 bar against the oracle


@pytest.fixture(scope="module")
def T():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from theboss_amd import _lib

    _lib.load()
    return torch


def i32(T, a):
    return T.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()


@pytest.mark.parametrize("k,B,in_max,out_max", [(2, 5, 3, 1), (5, 7, 130, 70), (7, 3, 7, 66),
                                                (9, 40, 64, 8), (13, 2, 65, 200)])
def test_scattered_slots_equal_compact_ones(T, oracle, k, B, in_max, out_max):
    """Slots in any place of the lists, the rest empty or negative: the compact call's minors at
    the occupied slots (bit for bit: the same item is swept) and 0 elsewhere."""
    from theboss_amd import ops

    m = 24
    rng = np.random.default_rng(k)
    U = T.from_numpy(oracle.haar_unitary(m, k)).cuda()
    cols = np.sort(np.argsort(rng.random((B, m)), axis=1)[:, :k], axis=1)
    rows = np.sort(rng.integers(0, m, (B, k - 1)), axis=1)
    place = np.sort(np.argsort(rng.random((B, in_max)), axis=1)[:, :k], axis=1)
    im, iu = rng.integers(0, m, (B, in_max)), -rng.integers(0, 3, (B, in_max))
    om, ou = rng.integers(0, m, (B, out_max)), np.zeros((B, out_max), dtype=int)
    cm, cu = np.zeros((B, k - 1), dtype=int), np.zeros((B, k - 1), dtype=int)
    for b in range(B):
        im[b, place[b]], iu[b, place[b]] = cols[b], 1
        modes, mult = np.unique(rows[b], return_counts=True)
        at = np.sort(rng.permutation(out_max)[:len(modes)])
        if len(at) < len(modes):  # out_max 1, k = 2
            at = np.arange(len(modes))
        om[b, at], ou[b, at] = modes, mult
        cm[b, :len(modes)], cu[b, :len(modes)] = modes, mult
    got = ops.cc_submatrices_batch(U, i32(T, om), i32(T, ou), i32(T, im), i32(T, iu), k, True).cpu().numpy()
    ref = ops.cc_submatrices_batch(U, i32(T, cm), i32(T, cu), i32(T, cols), i32(T, np.ones((B, k))), k,
                                   True).cpu().numpy()
    for b in range(B):
        assert np.array_equal(got[b, place[b]], ref[b])
        empty = np.ones(in_max, dtype=bool)
        empty[place[b]] = False
        assert np.all(got[b, empty] == 0.0)


@pytest.mark.parametrize("k,B", [(3, 1), (8, 1), (12, 70), (16, 1), (20, 1), (20, 130)])
def test_minors_vs_oracle_for_few_and_many_partials(T, oracle, k, B):
    from theboss_amd import ops

    m = 2 * k
    Uh = oracle.haar_unitary(m, 7 * k)
    U = T.from_numpy(Uh).cuda()
    cols = np.tile(np.arange(k), (B, 1))
    rows = np.tile(np.arange(k - 1) + 1, (B, 1))
    one = np.ones((B, k))
    got = ops.cc_submatrices_batch(U, i32(T, rows), i32(T, one[:, 1:]), i32(T, cols), i32(T, one), k,
                                   True).cpu().numpy()
    ref = oracle.perm_minors(np.vstack([np.ones(k), Uh[1:k, :k]]))[0]  # row 0 deleted
    assert np.max(np.abs(got - ref[None])) <= REL * np.max(np.abs(ref))


def test_two_values_per_lane(T, oracle):
    """k = 33: 66 minor components on 64 lanes. The Laplace expansion along a further row equals
    the Glynn kernel's permanent."""
    from theboss_amd import ops

    k = 33
    A = oracle.haar_unitary(2 * k, 3)[:k, :k]
    Vt = T.from_numpy(np.ascontiguousarray(A[:k - 1].T)[None]).cuda()
    minors = ops.sweep_minors_batch(Vt, k).cpu().numpy()[0]
    p = ops.glynn_batch(T.from_numpy(A[None].copy()).cuda()).cpu().numpy()[0]
    bound = REL * (np.sum(np.abs(A[k - 1] * minors)) + abs(p))
    assert abs(np.sum(A[k - 1] * minors) - p) <= bound
