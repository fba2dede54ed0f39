"""GCC-A layers that take the recurrence inside the layer call, and histograms of every partition
size: each case first asserts, by the workspace asked for, that it goes the way it is meant to."""
import itertools

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


# one particle per mode and collisions; a workgroup and a wave per output row; the lattice's limit
@pytest.mark.parametrize("top,k,m,P", [
    ((1,) * 8, 5, 20, 60), ((2, 1, 2, 1, 1, 1), 5, 20, 120), ((2, 1, 2, 1, 1, 1), 4, 24, 300),
    ((7, 7, 7, 7), 8, 12, 70), ((1,) * 12, 6, 13, 40)])
@pytest.mark.parametrize("formula", [0, 1])
def test_layer_by_recurrence_equals_the_walk(T, oracle, top, k, m, P, formula):
    """The sums are of at most 924 positive terms of permanents of at most 8 particles."""
    from theboss_amd import _lib, ops
    from theboss_amd.states import compact_batch, has_small_common_state

    rng = np.random.default_rng(m + P)
    U = T.from_numpy(oracle.haar_unitary(m, 4)).cuda()
    rows = [s for s in itertools.product(*[range(c + 1) for c in top]) if sum(s) == k]
    S = np.zeros((len(rows), m), dtype=np.int64)
    S[:, :len(top)] = rows
    assert has_small_common_state(S)
    modes, mult = (T.from_numpy(a).cuda() for a in compact_batch(S))
    Pf = np.array([np.bincount(rng.integers(0, m, k - 1), minlength=m) for _ in range(P)])
    w = T.from_numpy(rng.random(len(S))).cuda()
    size = [_lib.load().tb_gcca_layer_workspace_size(m, P, k - 1, modes.shape[1], len(S), common)
            for common in (0, 1)]
    assert 0 < size[0] < size[1]
    got = ops.gcca_layer_pmfs(U, T.from_numpy(Pf.astype(np.int32)).cuda(), k - 1, modes, mult, w,
                              formula, True).cpu().numpy()
    outs = (Pf[:, None, :] + np.eye(m, dtype=np.int64)[None]).reshape(-1, m)
    perms = ops.guan_perm_outer(U, *(T.from_numpy(a).cuda() for a in compact_batch(outs)), modes,
                                mult, formula, common=False)
    want = (T.view_as_real(perms).square().sum(-1) @ w).reshape(P, m).cpu().numpy()
    assert np.max(np.abs(got - want)) <= 1e-11 * np.max(want)


# four, eight and sixteen rows per thread; one sample over and under the next size; odd and even modes
@pytest.mark.parametrize("m,n,losses,S", [
    (20, 6, False, 1 << 19), (19, 6, False, 1 << 20), (20, 6, False, (1 << 20) + 1),
    (18, 7, True, 1 << 21), (20, 6, False, (1 << 21) + 1), (17, 7, False, (1 << 21) + 4097),
    (33, 5, True, (1 << 21) + 12345)])
def test_partition_equals_atomics(T, m, n, losses, S):
    from theboss_amd import _lib, ops

    lib = _lib.load()
    assert lib.tb_outcome_histogram64_workspace_size(S, m, n, int(losses)) > 0
    gen = T.Generator(device="cuda").manual_seed(S)
    smp = T.zeros((S, m), dtype=T.int32, device="cuda")
    smp.scatter_add_(1, T.randint(0, m, (S, n), generator=gen, device="cuda"),
                     (T.rand((S, n), generator=gen, device="cuda") < (0.7 if losses else 2)).int())
    smp[::1013, 0] -= 3
    counts, outside = ops.outcome_histogram(smp, n, losses=losses)
    ref = T.zeros(ops.outcome_count(n, m, losses), dtype=T.int32, device="cuda")
    out = T.zeros(1, dtype=T.int32, device="cuda")
    _lib.check(lib.tb_outcome_histogram(smp.data_ptr(), m, S, m, n, int(losses), ref.data_ptr(),
                                        out.data_ptr(), T.cuda.current_stream().cuda_stream))
    assert T.equal(counts, ref.to(T.int64)) and outside == int(out)
    assert int(counts.sum()) + outside == S


def test_counters_that_fit_lds_need_no_workspace(T):
    from theboss_amd import _lib

    lib = _lib.load()
    assert lib.tb_outcome_histogram64_workspace_size((1 << 21) + 513, 11, 7, 1) == 0
    assert lib.tb_outcome_histogram64_workspace_size(1 << 22, 4, 3, 0) == 0
