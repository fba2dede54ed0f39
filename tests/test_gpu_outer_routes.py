"""Which way an all-pairs call goes, read from the flags it leaves in its workspace: the recurrence
up to the lattice's 4096 substates and 12 modes, the walk of every pair beyond, with as many turns
as its blocks take from their counters and with the smallest workspace; and the op that leaves the
choice to the device."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL = 1e-10  # the FP64 bar


@pytest.fixture(scope="module")
def T():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from theboss_amd import _lib

    _lib.load()
    return torch


def substates(top, k, m):
    rows = [s for s in itertools.product(*[range(c + 1) for c in top]) if sum(s) == k]
    S = np.zeros((len(rows), m), dtype=np.int64)
    S[:, 1:1 + len(top)] = rows
    return S


def random_rows(rng, n, m, k):
    rows = np.zeros((n, m), dtype=np.int64)
    np.add.at(rows, (np.repeat(np.arange(n), k), rng.integers(0, m, n * k)), 1)
    return rows


def on_device(T, states):
    from theboss_amd.states import compact_batch

    return [T.from_numpy(a).cuda() for a in compact_batch(states)]


def outer(T, U, outs, ins, nbytes):
    """(result, flags of the output rows) with a workspace of nbytes; 0: the walk, no flags."""
    from theboss_amd import _device as D
    from theboss_amd import _lib as L

    n_out, n_in = outs[0].shape[0], ins[0].shape[0]
    out = T.full((n_out, n_in), np.nan, dtype=T.complex128, device="cuda")
    ws = T.full((max(nbytes, 4),), 85, dtype=T.uint8, device="cuda")
    L.check(L.load().tb_guan_perm_outer_ws(
        D.ptr(U), U.shape[1], D.ptr(outs[0]), D.ptr(outs[1]), outs[0].shape[1], n_out,
        D.ptr(ins[0]), D.ptr(ins[1]), ins[0].shape[1], n_in, 0, D.ptr(out),
        D.ptr(ws) if nbytes else None, nbytes, D.stream_ptr(U.device)))
    return out.cpu().numpy(), ws[:4 * n_out].view(T.int32).cpu().numpy() if nbytes else None


def sizes(outs, ins, m):
    """The workspace asked for, and the least one: a flag per output row."""
    from theboss_amd import _lib as L

    n_out = outs[0].shape[0]
    asked = L.load().tb_guan_outer_workspace_size(m, outs[0].shape[1], n_out, ins[0].shape[1],
                                                  ins[0].shape[0])
    assert asked > 0  # the call is large enough for the recurrence
    return asked, -(-4 * n_out // 256) * 256


@pytest.mark.parametrize("top,k,n_out", [
    ((7, 7, 7, 7), 8, 800),          # 4096 substates, collisions, a workgroup per row
    ((7, 7, 7, 7), 8, 2500),         # a wave per row
    ((3, 3, 3, 3, 3, 3), 8, 400),    # 4096 substates of six modes
    ((1, 2, 1, 2, 1, 2, 1, 2), 6, 300),
    ((1,) * 12, 6, 40),
])
def test_recurrence_does_every_row(T, oracle, top, k, n_out):
    m = 14
    U = T.from_numpy(oracle.haar_unitary(m, 6)).cuda()
    ins = on_device(T, substates(top, k, m))
    outs = on_device(T, random_rows(np.random.default_rng(k), n_out, m, k))
    walk, _ = outer(T, U, outs, ins, 0)
    for nbytes in sizes(outs, ins, m):
        got, flags = outer(T, U, outs, ins, nbytes)
        assert np.array_equal(flags, np.ones(n_out))
        assert np.max(np.abs(got - walk)) <= REL * np.max(np.abs(walk))


@pytest.mark.parametrize("top,k,n_out", [
    ((8, 7, 7, 7), 8, 900),          # more than 4096 substates
    ((8, 7, 7, 7), 8, 40000),        # several turns a block
    ((1,) * 13, 2, 13500),           # a mode too many; turns taken eight items at a time
    ((1,) * 13, 1, 530000),
    ((1,) * 13, 3, 460),
    ((1,) * 13, 11, 27),             # few items, the least number of blocks and of counters
    ((1,) * 13, 10, 400),
    ((1,) * 13, 12, 3000),
])
def test_refused_rows_are_all_walked(T, oracle, top, k, n_out):
    """The walk's own values, whatever the workspace held before and how many counters it has."""
    m = 15
    U = T.from_numpy(oracle.haar_unitary(m, 2)).cuda()
    ins = on_device(T, substates(top, k, m))
    outs = on_device(T, random_rows(np.random.default_rng(n_out), n_out, m, k))
    walk, _ = outer(T, U, outs, ins, 0)
    assert not np.isnan(walk).any()
    for nbytes in sizes(outs, ins, m):
        got, flags = outer(T, U, outs, ins, nbytes)
        assert flags[0] < 0
        assert np.array_equal(got, walk)


def test_op_leaves_the_choice_to_the_device(T, oracle):
    from theboss_amd import ops

    m, k, n_out = 14, 4, 4200
    U = T.from_numpy(oracle.haar_unitary(m, 3)).cuda()
    outs = on_device(T, random_rows(np.random.default_rng(1), n_out, m, k))
    for top in ((1,) * 8, (1,) * 13):
        ins = on_device(T, substates(top, k, m))
        assert (n_out * ins[0].shape[0]) << ins[0].shape[1] >= ops._OUTER_TRY_CODES
        walk = ops.guan_perm_outer(U, *outs, *ins, common=False).cpu().numpy()
        for formula in (0, 1):
            got = ops.guan_perm_outer(U, *outs, *ins, formula).cpu().numpy()
            assert np.max(np.abs(got - walk)) <= REL * np.max(np.abs(walk))
        same = np.array_equal(ops.guan_perm_outer(U, *outs, *ins).cpu().numpy(), walk)
        assert same == (len(top) == 13)  # the walk's values exactly, or the recurrence's


@pytest.mark.parametrize("modes", [8, 13])
def test_op_shares_no_scratch_between_calls(T, oracle, monkeypatch, modes):
    """The scratch of a call is its own: threads share a stream, and a graph outlives the call."""
    from theboss_amd import _device as D
    from theboss_amd import ops

    m, k = 14, 4
    U = T.from_numpy(oracle.haar_unitary(m, 3)).cuda()
    outs = on_device(T, random_rows(np.random.default_rng(1), 4200, m, k))
    ins = on_device(T, substates((1,) * modes, k, m))
    walk = ops.guan_perm_outer(U, *outs, *ins, common=False)
    monkeypatch.setattr(D, "workspace", lambda *a: pytest.fail("the stream's workspace"))
    want = ops.guan_perm_outer(U, *outs, *ins)
    assert T.max(T.abs(want - walk)) <= REL * T.max(T.abs(walk))
    side = T.cuda.Stream()
    side.wait_stream(T.cuda.current_stream())
    with T.cuda.stream(side):
        ops.guan_perm_outer(U, *outs, *ins)
        T.cuda.synchronize()
        graph = T.cuda.CUDAGraph()
        with T.cuda.graph(graph, stream=side):
            got = ops.guan_perm_outer(U, *outs, *ins)
    T.cuda.current_stream().wait_stream(side)
    more = on_device(T, random_rows(np.random.default_rng(2), 9000, m, k))
    for _ in range(3):
        got.zero_()
        ops.guan_perm_outer(U, *more, *ins)
        graph.replay()
        ops.guan_perm_outer(U, *more, *ins)
        T.cuda.synchronize()
        assert T.equal(got, want)
