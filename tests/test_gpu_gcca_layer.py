"""GCC-A's layer sums on the device against the same sums over compute_permanent_outer's
permanents of rows formed densely. Both add at most a few hundred positive terms of permanents
with at most 2^9 codes, so they agree to 1e-12 of a layer's largest entry."""
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


# one mode; empty prefixes; collisions; rows with a small common state (substates of a state),
# and without; more input rows than a wave, and a number of rows no workgroup divides
@pytest.mark.parametrize("m,k,n_in,P,common", [
    (1, 1, 1, 1, True), (1, 4, 1, 1, True), (7, 1, 5, 3, True), (9, 3, 12, 7, False),
    (20, 5, 70, 11, True), (30, 4, 65, 5, False), (6, 9, 40, 6, False)])
@pytest.mark.parametrize("name", ["GPURyserPermanentCalculator", "GPUChinHuhPermanentCalculator"])
def test_layer_sums_equal_outer(T, oracle, m, k, n_in, P, common, name):
    from theboss_amd import permanent_calculators

    rng = np.random.default_rng(m * 10 + k)
    U = oracle.haar_unitary(m, 4)
    pool = min(m, 8) if common else m
    S = np.array([np.bincount(rng.permutation(pool)[:k] if common and k <= pool
                              else rng.integers(0, m, k), minlength=m) for _ in range(n_in)])
    Pf = np.array([np.bincount(rng.integers(0, m, k - 1), minlength=m) for _ in range(P)])
    w = rng.random(n_in)
    calc = getattr(permanent_calculators, name)(U)
    got = calc.compute_layer_pmfs(calc.layer_inputs(S, w), Pf).cpu().numpy()
    rows = (Pf[:, None, :] + np.eye(m, dtype=np.int64)[None]).reshape(-1, m)
    perms = calc.compute_permanent_outer(S, rows).cpu().numpy()
    want = ((perms.real ** 2 + perms.imag ** 2) @ w).reshape(P, m)
    assert got.shape == (P, m)
    assert np.max(np.abs(got - want)) <= 1e-12 * np.max(want)


def test_layer_sums_refuse_what_does_not_fit(T, oracle):
    """Rows past the Guan kernels' limits and mismatched prefixes are left to the caller; wrong
    sizes raise."""
    from theboss_amd import ops
    from theboss_amd.permanent_calculators import GPURyserPermanentCalculator

    m = 80
    calc = GPURyserPermanentCalculator(oracle.haar_unitary(m, 2))
    wide = np.ones((1, m), dtype=np.int64)
    assert calc.layer_inputs(wide, np.ones(1)) is None
    one = np.eye(m, dtype=np.int64)[:2]
    inputs = calc.layer_inputs(one, np.ones(2))
    assert calc.compute_layer_pmfs(inputs, one) is None
    with pytest.raises(ValueError):
        ops.gcca_layer_pmfs(T.zeros((4, 4), dtype=T.complex128, device="cuda"),
                            T.zeros((2, 5), dtype=T.int32, device="cuda"), 1, inputs[1], inputs[2],
                            inputs[3])
