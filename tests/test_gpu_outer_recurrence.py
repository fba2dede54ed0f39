"""The all-pairs subset recurrence against the pair-by-pair walk (the same entry without a
workspace) and the oracle: common states with and without collisions, the edges of the lattice
(12 modes, 4096 substates, 13 modes, 12 and 13 particles), wide levels, few and many output
rows, repeated slots, output rows of another particle number and calls it does not take."""
import itertools
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL = 1e-10  # the FP64 bar; the walk's own cancellation at 12 photons is ~1e-12


@pytest.fixture(scope="module")
def T():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from theboss_amd import _lib

    _lib.load()
    return torch


def substates(top, k):
    return np.array([s for s in itertools.product(*[range(c + 1) for c in top]) if sum(s) == k],
                    dtype=np.int64).reshape(-1, len(top))


def random_rows(rng, n, m, k):
    rows = np.zeros((n, m), dtype=np.int64)
    np.add.at(rows, (np.repeat(np.arange(n), k), rng.integers(0, m, n * k)), 1)
    return rows


def rows_to_device(T, states):
    from theboss_amd.states import compact_batch

    return [T.from_numpy(a).cuda() for a in compact_batch(states)]


def both(T, U, outs, ins):
    """(recurrence or fallback, walk) of the same rows; attempts whatever the size."""
    from theboss_amd import _device as D
    from theboss_amd import _lib as L

    lib = L.load()
    n_out, n_in = outs[0].shape[0], ins[0].shape[0]
    res = []
    ws = T.full((4 * n_out + 256,), 255, dtype=T.uint8, device="cuda")
    for w in (ws, None):
        o = T.full((n_out, n_in), np.nan, dtype=T.complex128, device="cuda")
        L.check(lib.tb_guan_perm_outer_ws(
            D.ptr(U), U.shape[1], D.ptr(outs[0]), D.ptr(outs[1]), outs[0].shape[1], n_out,
            D.ptr(ins[0]), D.ptr(ins[1]), ins[0].shape[1], n_in, 0, D.ptr(o),
            D.ptr(w) if w is not None else None, ws.numel() if w is not None else 0,
            D.stream_ptr(U.device)))
        res.append(o.cpu().numpy())
    return res


def close(a, b):
    return np.max(np.abs(a - b)) <= REL * np.max(np.abs(b))


@pytest.mark.parametrize("top,k,n_out", [
    ((1,) * 10, 5, 2100),        # a wave per output row
    ((1,) * 10, 5, 1000),        # a workgroup per output row
    ((1,) * 10, 1, 60000),
    ((1,) * 10, 10, 1100),       # one input row, every level
    ((1,) * 11, 6, 300),         # levels too wide for a wave
    ((1,) * 12, 6, 100),         # 12 modes, 4096 substates
    ((1,) * 12, 12, 300),
    ((1,) * 13, 6, 100),         # one mode too many: walked
    ((3, 2, 2, 1, 1), 5, 2500),  # collisions
    ((7, 7, 7, 7), 6, 600),      # 4096 substates
    ((8, 7, 7, 7), 6, 600),      # more than 4096: walked
    ((12,), 12, 530000), ((13,), 13, 530000),  # one input row of one mode
])
def test_recurrence_equals_walk(T, oracle, top, k, n_out):
    rng = np.random.default_rng(k + n_out)
    m = 16
    Uh = oracle.haar_unitary(m, 5)
    ins = np.zeros((len(substates(top, k)), m), dtype=np.int64)
    ins[:, 2:2 + len(top)] = substates(top, k)
    outs = random_rows(rng, n_out, m, k)
    U = T.from_numpy(Uh).cuda()
    got, walk = both(T, U, rows_to_device(T, outs), rows_to_device(T, ins))
    if top == (12,):
        # One mode holds all particles: 12! prod_l U[t_l][mode]. The walk's alternating sum
        # cancels from 12^12 down to 12! here, so it is no reference to 1e-10.
        walk = math.factorial(12) * np.prod(Uh[:, 2][None, :] ** outs, axis=1)[:, None]
    assert close(got, walk)
    s, t = ins[-1], outs[n_out // 2]
    A = Uh[np.ix_(np.repeat(np.arange(m), t), np.repeat(np.arange(m), s))]
    ref = oracle.perm_glynn_matrix(A, 1) if k > 1 else A[0, 0]
    assert abs(got[n_out // 2, -1] - ref) <= REL * np.max(np.abs(walk))


def test_repeated_slots_other_particle_numbers_and_padding(T, oracle):
    """An input mode split over two slots counts with its sum; an output row with another
    particle number is left to the walk; the rows around it are not."""
    rng = np.random.default_rng(0)
    U = T.from_numpy(oracle.haar_unitary(12, 9)).cuda()
    i32 = lambda a: T.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()  # noqa: E731
    in_modes = np.array([[4, 7, 4, 0], [1, 4, 7, 9], [7, 7, 1, 0]])
    in_mult = np.array([[1, 2, 1, 0], [1, 1, 1, 1], [1, 1, 2, -3]])
    n_out = 90000
    out_modes = rng.integers(0, 12, (n_out, 4))
    out_mult = np.ones((n_out, 4), dtype=np.int64)
    out_mult[5] = [1, 1, 1, 0]
    out_mult[6] = [4, 0, 0, 0]
    out_mult[7] = [2, 2, 1, 1]
    got, walk = both(T, U, [i32(out_modes), i32(out_mult)], [i32(in_modes), i32(in_mult)])
    fine = np.ones(n_out, dtype=bool)
    fine[[5, 7]] = False
    assert close(got[fine], walk[fine])
    assert np.array_equal(got[~fine], walk[~fine])  # the walk's own values, whatever they mean


def test_op_takes_both_routes_and_the_calculator_says_which(T, oracle):
    from theboss_amd import ops
    from theboss_amd.states import has_small_common_state

    m, k = 14, 4
    U = T.from_numpy(oracle.haar_unitary(m, 3)).cuda()
    top = np.array([1] * 8 + [0] * 6)
    ins = substates(top, k)
    assert has_small_common_state(ins) and not has_small_common_state(np.eye(13, dtype=np.int64))
    outs = random_rows(np.random.default_rng(1), 3000, m, k)
    o, i = rows_to_device(T, outs), rows_to_device(T, ins)
    walk = ops.guan_perm_outer(U, *o, *i, common=False).cpu().numpy()
    for how in (True, None):
        for formula in (0, 1):
            assert close(ops.guan_perm_outer(U, *o, *i, formula, how).cpu().numpy(), walk)


def test_walk_of_the_rows_left_in_a_large_call(T, oracle):
    """More than 64 turns of the walk that follows the recurrence; rows left to it here and there."""
    n_out, m = 120001, 12
    U = T.from_numpy(oracle.haar_unitary(m, 4)).cuda()
    ins = np.zeros((36, m), dtype=np.int64)
    ins[:, :9] = substates((1,) * 9, 2)
    rng = np.random.default_rng(8)
    modes = rng.integers(0, m, (n_out, 2)).astype(np.int32)
    mult = np.ones((n_out, 2), dtype=np.int32)
    left = np.array([0, 3000, 3001, 60000, n_out - 1])
    mult[left] = 2
    outs = [T.from_numpy(modes).cuda(), T.from_numpy(mult).cuda()]
    got, walk = both(T, U, outs, rows_to_device(T, ins))
    assert np.array_equal(got[left], walk[left])
    assert close(np.delete(got, left, 0), np.delete(walk, left, 0))
