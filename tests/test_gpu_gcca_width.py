"""GCC-A layer sums of prefixes that occupy more modes than the call says: NaN, not the sums of a
prefix without its last modes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n_in,P,common", [(12, 5, 40, 30, False), (12, 5, 60, 120, True)])
def test_too_narrow_a_width_is_nan(oracle, m, k, n_in, P, common):
    import torch as T

    from theboss_amd import ops
    from theboss_amd.states import compact_batch

    rng = np.random.default_rng(k + P)
    dev = lambda a: T.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    U = dev(oracle.haar_unitary(m, 4))
    S = np.array([np.bincount(rng.permutation(9)[:k], minlength=m) for _ in range(n_in)])
    Pf = np.array([np.bincount(rng.integers(0, m, k - 1), minlength=m) for _ in range(P)])
    modes, mult = (dev(a) for a in compact_batch(S))
    w = dev(rng.random(n_in))
    occupied = np.count_nonzero(Pf, axis=1)
    assert occupied.max() == k - 1 and occupied.min() < k - 1
    Pd = dev(Pf.astype(np.int32))
    want = ops.gcca_layer_pmfs(U, Pd, k - 1, modes, mult, w, 0, common).cpu().numpy()
    assert not np.isnan(want).any()
    for width in range(1, k - 1):
        got = ops.gcca_layer_pmfs(U, Pd, width, modes, mult, w, 0, common).cpu().numpy()
        fits = occupied <= width
        assert np.isnan(got[~fits]).all()
        assert np.allclose(got[fits], want[fits], rtol=1e-12, atol=0)
