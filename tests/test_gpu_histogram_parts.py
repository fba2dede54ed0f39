"""Every way the outcome histogram counts, against a plain count of host ranks. All are whole
numbers, so equality is exact."""
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


def _host_counts(smp, n, losses, count):
    """Counts by the documented rank, vectorised over the samples."""
    from math import comb

    S, m = smp.shape
    keep = (smp >= 0).all(axis=1)
    total = smp.astype(np.int64).sum(axis=1)
    keep &= (total <= n) if losses else (total == n)
    good = smp[keep].astype(np.int64)
    total = total[keep]
    term = np.array([[comb(r - 1 + y, y) if r else 0 for r in range(n + 1)] for y in range(m + 1)],
                    dtype=object).astype(np.float64).astype(np.int64)
    rank = term[m][total] if losses else np.zeros(len(good), dtype=np.int64)
    after = np.zeros(len(good), dtype=np.int64)
    for i in range(m - 1, -1, -1):
        rank = rank + term[m - 1 - i][after]
        after = after + good[:, i]
    return np.bincount(rank, minlength=count), S - len(good)


def _samples(rng, S, m, n, lossy):
    """Uniform placements with rows that are in no list, and a stretch of equal rows (one
    counter, so one long run)."""
    smp = np.zeros((S, m), dtype=np.int32)
    for _ in range(n):
        on = np.arange(S) if not lossy else np.nonzero(rng.random(S) < 0.8)[0]
        np.add.at(smp, (on, rng.integers(0, m, len(on))), 1)
    smp[::97, 0] += n + 1
    smp[5::101, -1] = -1
    smp[7::1009, 0] = 2**30  # four of these wrap a 32-bit sum
    smp[S // 3: S // 2] = smp[S // 3]
    return smp


# counters in LDS (few, or many enough for the narrower workgroup), straight into memory, and
# by partition: one, two and four rows per thread more than a chunk; odd, even and single modes
@pytest.mark.parametrize("m,n,losses,S", [
    (1, 4, False, 1000), (2, 64, True, 9001), (3, 3, True, 257), (8, 4, False, 70001),
    (14, 6, False, 120001), (64, 3, False, 1023), (20, 10, False, 1000), (9, 10, True, 300001),
    (9, 10, True, (1 << 19) - 1), (9, 10, True, 1 << 19), (18, 6, False, (1 << 20) + 1),
    (11, 7, True, (1 << 21) + 513), (20, 10, False, 600001)])
def test_histogram_routes(T, m, n, losses, S):
    from theboss_amd import _lib, ops

    smp = _samples(np.random.default_rng(m + n), S, m, n, losses)
    dev = T.from_numpy(smp).cuda()
    count = ops.outcome_count(n, m, losses)
    counts, outside = ops.outcome_histogram(dev, n, losses=losses)
    ref, ref_out = _host_counts(smp, n, losses, count)
    assert counts.dtype == T.int64 and np.array_equal(counts.cpu().numpy(), ref)
    assert outside == ref_out
    # rows with a gap, an unaligned start, no workspace; and the 32-bit counters, which add
    lib = _lib.load()
    wide = T.full((S, m + 3), 7, dtype=T.int32, device="cuda")
    wide[:, 1:m + 1] = dev
    stream = T.cuda.current_stream().cuda_stream
    c64 = T.full((count,), 5, dtype=T.int64, device="cuda")
    o64 = T.full((1,), 5, dtype=T.int64, device="cuda")
    need = lib.tb_outcome_histogram64_workspace_size(S, m, n, int(losses))
    ws = T.empty(max(need, 1), dtype=T.uint8, device="cuda")
    for p, room in ((ws.data_ptr(), need), (ws.data_ptr(), max(need - 1, 0)), (None, 0)):
        _lib.check(lib.tb_outcome_histogram64(wide.data_ptr() + 4, m + 3, S, m, n, int(losses),
                                              c64.data_ptr(), o64.data_ptr(), p, room, stream))
        assert np.array_equal(c64.cpu().numpy(), ref) and int(o64) == ref_out
        c64.fill_(3)
    c32 = T.ones(count, dtype=T.int32, device="cuda")
    _lib.check(lib.tb_outcome_histogram(dev.data_ptr(), m, S, m, n, int(losses), c32.data_ptr(),
                                        None, stream))
    assert np.array_equal(c32.cpu().numpy(), ref + 1)


def test_histogram_of_nothing_clears(T):
    from theboss_amd import ops

    counts, outside = ops.outcome_histogram(T.empty((0, 5), dtype=T.int32, device="cuda"), 3)
    assert counts.shape == (35,) and not counts.any() and outside == 0


def test_histogram_in_several_slabs(T):
    """More samples than the workspace holds ranks for: the second slab adds to the first."""
    from theboss_amd import _lib, ops

    S, m, n = (1 << 24) + 777, 9, 10
    smp = T.zeros((S, m), dtype=T.int32, device="cuda")
    gen = T.Generator(device="cuda").manual_seed(5)
    one = T.ones((S, 1), dtype=T.int32, device="cuda")
    for _ in range(n - 1):
        smp.scatter_add_(1, T.randint(0, m, (S, 1), generator=gen, device="cuda"), one)
    counts, outside = ops.outcome_histogram(smp, n, losses=True)
    ref = T.zeros(ops.outcome_count(n, m, True), dtype=T.int32, device="cuda")
    lib = _lib.load()
    _lib.check(lib.tb_outcome_histogram(smp.data_ptr(), m, S, m, n, 1, ref.data_ptr(), None,
                                        T.cuda.current_stream().cuda_stream))
    assert outside == 0 and int(counts.sum()) == S and T.equal(counts, ref.to(T.int64))


# the partition's tiles: as many modes as are loaded ahead, one fewer and one more; a last tile
# whose values are no multiple of four; and tiles smaller than a chunk's sorted offsets
@pytest.mark.parametrize("m,n,S", [(31, 4, (1 << 19) + 3), (32, 4, (1 << 20) + 1),
                                   (33, 4, (1 << 20) + 513), (5, 40, (1 << 21) + 77)])
def test_histogram_partition_tiles(T, m, n, S):
    from theboss_amd import _lib, ops

    assert _lib.load().tb_outcome_histogram64_workspace_size(S, m, n, 0) > 0
    smp = _samples(np.random.default_rng(m), S, m, n, False)
    counts, outside = ops.outcome_histogram(T.from_numpy(smp).cuda(), n)
    ref, ref_out = _host_counts(smp, n, False, ops.outcome_count(n, m, False))
    assert np.array_equal(counts.cpu().numpy(), ref) and outside == ref_out
