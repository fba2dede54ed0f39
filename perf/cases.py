"""Performance cases: what programs ask of theboss_amd, over the sizes they ask it for.

Kinds of case (one public entry point each):
  perm     permanents of a batch of n x n blocks of a Haar unitary, `ops.glynn_batch`
           (FP64, or the FP32 column sums): one permanent to check a probability, a batch of
           output probabilities, a few large permanents.
  grad     `autograd.permanent` forward and backward: permanents and the gradient of every
           entry, as likelihood fits and interferometer derivatives need them.
  sampler  `ops.gccb_sample`: batched GCC-B sampling, lossless or with uniform losses.
  gcca     `GeneralizedCliffordsSimulationStrategy.simulate` with the Ryser calculator: the
           whole GCC-A call from Python, its host work included.
  pairs    `ops.guan_perm_outer`: every (output row, input row) permanent of a GCC-A layer or
           of one particle number of an exact distribution.
  minors   `ops.cc_submatrices_batch`: all input-deleted minors, one item (a step of the
           plain GCC-B sampler) or a batch, with and without input collisions.
  counts   `ops.outcome_histogram`: samples counted over the outcome list.
"""
import math
from itertools import combinations

import numpy as np
import torch

from theboss_amd import ops
from theboss_amd._lib import TB_PREC_FP32_COLSUM, TB_PREC_FP64
from theboss_amd.autograd import permanent
from theboss_amd.permanent_calculators import GPURyserPermanentCalculator
from theboss_amd.simulation_strategies import GeneralizedCliffordsSimulationStrategy


def listed():
    return [
        # One 10 x 10 permanent: the check of a single output probability. Latency only.
        {"name": "perm_n10_b1", "kind": "perm", "n": 10, "batch": 1, "fp32": False},
        # 16 single large permanents of Haar blocks, two of the three sizes.
        {"name": "perm_n24_b16", "kind": "perm", "n": 24, "batch": 16, "fp32": False},
        {"name": "perm_n28_b16", "kind": "perm", "n": 28, "batch": 16, "fp32": False},
        # The opt-in FP32 column sums on a batch of mid-size blocks.
        {"name": "perm_fp32_n20_b1024", "kind": "perm", "n": 20, "batch": 1024, "fp32": True},
        # Permanents and all minors of 64 n = 20 blocks, through autograd.
        {"name": "grad_n20_b64", "kind": "grad", "n": 20, "batch": 64, "collisions": False},
        # The likelihood step of an interferometer fit: 10000 samples of 8 photons, output
        # collisions included.
        {"name": "fit_n8_s10000", "kind": "grad", "n": 8, "batch": 10000, "collisions": True},
        # Headline sampler: 20 photons in 400 modes, 4096 samples in flight.
        {"name": "gccb_m400_n20_s4096", "kind": "sampler", "m": 400, "n": 20, "samples": 4096,
         "eta": 1.0},
        # Uniform losses: 40 photons in 80 modes at transmissivity 1/2, uneven samples.
        {"name": "lossy_m80_n40_s1024", "kind": "sampler", "m": 80, "n": 40, "samples": 1024,
         "eta": 0.5},
        # The plain GCC-A method end to end: 200 samples of 10 photons in 20 modes.
        {"name": "gcca_m20_n10_s200", "kind": "gcca", "m": 20, "n": 10, "samples": 200},
        # One GCC-A layer of it as the op sees it: 200 prefixes x 20 outputs x C(10, 5) inputs.
        {"name": "pairs_m20_n10_k5_p200", "kind": "pairs", "m": 20, "n": 10, "k": 5,
         "prefixes": 200, "chin_huh": False},
        # One step of the plain GCC-B sampler: all 20 minors of one item.
        {"name": "minors_k20_b1", "kind": "minors", "m": 40, "k": 20, "batch": 1,
         "collisions": False},
        # Sample-based distribution: 4M samples of 10 particles in 20 modes.
        {"name": "counts_m20_n10_s4m", "kind": "counts", "m": 20, "n": 10, "samples": 1 << 22,
         "losses": False},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["perm", "perm", "grad", "grad", "sampler", "gcca", "pairs", "minors",
                       "counts"])
    if kind == "perm":
        fp32 = rng.random() < 0.3
        n = rng.randint(4, 23) if fp32 else rng.randint(4, 28)
        most = min(20000, max(1, int(16 * 28 * 2.0 ** 28 / (n * 2.0 ** n))))
        return {"kind": kind, "n": n, "batch": _log_int(rng, 1, most), "fp32": fp32}
    if kind == "grad":
        n = rng.randint(2, 25)
        most = min(20000, max(1, int(1024 * 400 * 2.0 ** 20 / (n * n * 2.0 ** n))))
        return {"kind": kind, "n": n, "batch": _log_int(rng, 1, most),
                "collisions": rng.random() < 0.5}
    if kind == "sampler":
        n = rng.randint(2, 20)
        eta = 1.0 if rng.random() < 0.5 else round(rng.uniform(0.4, 0.95), 2)
        return {"kind": kind, "m": _log_int(rng, max(n, 8), 400), "n": n,
                "samples": _log_int(rng, 16, 4096), "eta": eta}
    if kind == "gcca":
        n = rng.randint(3, 10)
        return {"kind": kind, "m": rng.randint(n, 24), "n": n, "samples": rng.randint(10, 200)}
    if kind == "pairs":
        n = rng.randint(3, 12)
        k = rng.randint(1, n)
        m = rng.randint(n, 24)
        most = max(1, min(400, 1500000 // (math.comb(n, k) * m)))
        return {"kind": kind, "m": m, "n": n, "k": k, "prefixes": _log_int(rng, 1, most),
                "chin_huh": rng.random() < 0.5}
    if kind == "minors":
        k = rng.randint(2, 22)
        most = min(2000, max(1, int(2.0 ** 26 / 2.0 ** k)))
        return {"kind": kind, "m": rng.randint(2 * k, 4 * k), "k": k,
                "batch": _log_int(rng, 1, most), "collisions": k >= 3 and rng.random() < 0.4}
    m = rng.randint(4, 20)
    n = rng.randint(2, 10)
    return {"kind": "counts", "m": m, "n": n, "samples": _log_int(rng, 1000, 1 << 22),
            "losses": rng.random() < 0.5}


# ------------------------------------------------------------------------------ inputs

def _haar(m, rng):
    """Haar-random m x m unitary (QR of a complex Gaussian with the phase fix)."""
    z = (rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))) / math.sqrt(2.0)
    q, r = np.linalg.qr(z)
    d = np.diagonal(r)
    return q * (d / np.abs(d))


def _blocks(n, batch, rng, collisions=False):
    """batch n x n blocks of one 2n-mode Haar unitary: input modes 0..n-1 for repeated
    outputs (the samples of one experiment), else random input and output modes."""
    U = torch.from_numpy(_haar(2 * n, rng)).cuda()
    if collisions:
        rows = np.sort(rng.integers(0, 2 * n, (batch, n)), axis=1)
        cols = np.tile(np.arange(n), (batch, 1))
    else:
        rows = np.sort(np.argsort(rng.random((batch, 2 * n)), axis=1)[:, :n], axis=1)
        cols = np.sort(np.argsort(rng.random((batch, 2 * n)), axis=1)[:, :n], axis=1)
    rows, cols = torch.from_numpy(rows).cuda(), torch.from_numpy(cols).cuda()
    return U[rows[:, :, None], cols[:, None, :]].contiguous()


def _compact(modes):
    """Sorted mode lists (B x k) as compact occupations: (modes, multiplicities), B x W."""
    B, k = modes.shape
    new = np.ones((B, k), dtype=bool)
    new[:, 1:] = modes[:, 1:] != modes[:, :-1]
    slot = np.cumsum(new, axis=1) - 1
    W = int(slot.max()) + 1
    out = np.zeros((2, B, W), dtype=np.int32)
    b = np.repeat(np.arange(B), k)
    out[0, b, slot.ravel()] = modes.ravel()
    np.add.at(out[1], (b, slot.ravel()), 1)
    return out


def _pairs_rows(case, rng):
    """Sorted mode lists of a layer: outputs prefix + e_o, and every k-subset of the inputs."""
    m, n, k = case["m"], case["n"], case["k"]
    pre = rng.integers(0, m, (case["prefixes"], k - 1))
    out = np.concatenate([np.repeat(pre, m, axis=0),
                          np.tile(np.arange(m), case["prefixes"])[:, None]], axis=1)
    return np.sort(out, axis=1), np.asarray(list(combinations(range(n), k)), dtype=np.int64)


def _minors_rows(case, rng):
    """Sorted mode lists: k input particles (one mode doubled, with collisions) and k - 1
    output particles with repeats."""
    m, k, B = case["m"], case["k"], case["batch"]
    ins = np.argsort(rng.random((B, m)), axis=1)[:, :k]
    if case["collisions"]:
        ins[:, 1] = ins[:, 0]
    return np.sort(rng.integers(0, m, (B, k - 1)), axis=1), np.sort(ins, axis=1)


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()


def prepare(case, seed):
    rng = np.random.default_rng([seed, 7])
    kind = case["kind"]
    s = {"case": dict(case)}
    if kind == "perm":
        s["A"] = _blocks(case["n"], case["batch"], rng)
    elif kind == "grad":
        s["A"] = _blocks(case["n"], case["batch"], rng, case["collisions"]).requires_grad_(True)
        g = rng.standard_normal((2, case["batch"]))
        s["g"] = torch.from_numpy(g[0] + 1j * g[1]).cuda()
    elif kind == "sampler":
        s["U"] = torch.from_numpy(_haar(case["m"], rng)).cuda()
        s["particles"] = torch.arange(case["n"], dtype=torch.int32, device="cuda")
        s["seed"] = int(rng.integers(1 << 60))
    elif kind == "gcca":
        s["U"] = _haar(case["m"], rng)
        s["seed"] = int(rng.integers(1 << 60))
    elif kind == "pairs":
        out, ins = _pairs_rows(case, rng)
        s["U"] = torch.from_numpy(_haar(case["m"], rng)).cuda()
        s["rows"] = [_i32(a) for a in (*_compact(out), *_compact(ins))]
    elif kind == "minors":
        out, ins = _minors_rows(case, rng)
        s["U"] = torch.from_numpy(_haar(case["m"], rng)).cuda()
        s["rows"] = [_i32(a) for a in (*_compact(out), *_compact(ins))]
    else:
        # each particle leaves through a mode of its own drawing; with losses it survives
        # with probability 0.7
        g = torch.Generator(device="cuda").manual_seed(int(rng.integers(1 << 60)))
        m, n, S = case["m"], case["n"], case["samples"]
        modes = torch.randint(m, (S, n), generator=g, device="cuda")
        kept = torch.ones((S, n), dtype=torch.int32, device="cuda")
        if case["losses"]:
            kept = (torch.rand((S, n), generator=g, device="cuda") < 0.7).to(torch.int32)
        s["samples"] = torch.zeros((S, m), dtype=torch.int32, device="cuda").scatter_add_(
            1, modes, kept)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "perm":
        return ops.glynn_batch(state["A"], TB_PREC_FP32_COLSUM if case["fp32"] else TB_PREC_FP64)
    if kind == "grad":
        p = permanent(state["A"])
        (dA,) = torch.autograd.grad(p, state["A"], state["g"])
        return {"perm": p.detach(), "grad": dA}
    if kind == "sampler":
        return ops.gccb_sample(state["U"], state["particles"], case["samples"], state["seed"],
                               case["eta"])[0]
    if kind == "gcca":
        strategy = GeneralizedCliffordsSimulationStrategy(
            GPURyserPermanentCalculator(state["U"]), np.random.default_rng(state["seed"]))
        photons = [1] * case["n"] + [0] * (case["m"] - case["n"])
        return np.asarray(strategy.simulate(photons, case["samples"]))
    if kind == "pairs":
        return ops.guan_perm_outer(state["U"], *state["rows"], 1 if case["chin_huh"] else 0)
    if kind == "minors":
        return ops.cc_submatrices_batch(state["U"], *state["rows"], case["k"],
                                        not case["collisions"])
    counts, outside = ops.outcome_histogram(state["samples"], case["n"], case["losses"])
    return {"counts": counts, "outside": outside}


# ---------------------------------------------------------------- what a pass cannot do without

def _subset_terms(n, k):
    """Complex multiply-adds of the subset recurrence up to k rows of n columns."""
    return sum(math.comb(n, l) * l for l in range(1, k + 1))


def work(case):
    kind = case["kind"]
    if kind == "perm":
        n, b = case["n"], case["batch"]
        return {"bytes": 16 * b * (n * n + 1), "flops": b * (8 * n - 4) * 2.0 ** (n - 1)}
    if kind == "grad":
        # per Gray step: the row flip (2n), the n leave-one-out products (3n complex
        # multiplies), one running sum and one corrector per column
        n, b = case["n"], case["batch"]
        return {"bytes": 16 * b * (2 * n * n + 2), "flops": b * 2.0 ** (n - 1) * 26 * n}
    if kind == "sampler":
        m, n, S, eta = case["m"], case["n"], case["samples"], case["eta"]
        f = 0.0
        for k in range(1, n + 1):  # steps of photon number k, and how many samples reach them
            reach = sum(math.comb(n, l) * eta ** l * (1 - eta) ** (n - l) for l in range(k, n + 1))
            f += reach * ((2.0 ** (k - 1) * (10 * k - 12) if k > 1 else 0) + 8 * m * k)
        return {"bytes": 16 * m * n + 4 * S * m, "flops": S * f}
    if kind == "gcca":
        # every sample its own prefix: the subset recurrence along it and the m amplitudes of
        # every substate of each layer
        m, n, S = case["m"], case["n"], case["samples"]
        f = 8 * (_subset_terms(n, n) + m * sum(math.comb(n, k) * k for k in range(1, n + 1)))
        return {"bytes": 16 * m * m + 8 * S * m, "flops": S * f}
    if kind == "pairs":
        n, k = case["n"], case["k"]
        rows = case["prefixes"] * case["m"]
        pairs = rows * math.comb(n, k)
        return {"bytes": 16 * pairs + 8 * k * (rows + math.comb(n, k)),
                "flops": 8 * (case["prefixes"] * _subset_terms(n, k - 1) + pairs * k)}
    if kind == "minors":
        k, b = case["k"], case["batch"]
        return {"bytes": 16 * b * k * k, "flops": b * 2.0 ** (k - 1) * max(10 * k - 12, 4)}
    top = case["n"] + case["m"] - (0 if case["losses"] else 1)
    states = math.comb(top, case["m"] if case["losses"] else case["m"] - 1)
    return {"bytes": 4 * case["samples"] * case["m"] + 8 * states,
            "flops": case["samples"] * case["m"]}


# ---------------------------------------------------------------------- the same in 64 bits

def _levels(n, device):
    """The n-bit subsets sorted by size, and where each size begins."""
    t = torch.arange(1 << n, dtype=torch.int32 if n < 31 else torch.int64, device=device)
    size = torch.zeros(1 << n, dtype=torch.uint8, device=device)
    for d in range(n):
        size += ((t >> d) & 1).to(torch.uint8)
    return torch.argsort(size, stable=True), np.concatenate(
        [[0], np.cumsum([math.comb(n, l) for l in range(n + 1)])])


def _subset_perms(A, levels):
    """F[b, T] = perm of the first |T| rows of A[b] (r x n) on the columns T, |T| <= r, by
    expansion along the last row: sums of products with no cancelling signs."""
    B, r, n = A.shape
    order, at = levels
    F = torch.zeros((B, 1 << n), dtype=torch.complex128, device=A.device)
    F[:, 0] = 1.0
    for l in range(1, r + 1):
        T = order[at[l]:at[l + 1]]
        v = torch.zeros((B, len(T)), dtype=torch.complex128, device=A.device)
        for d in range(n):
            has = torch.nonzero((T >> d) & 1).ravel()
            v[:, has] += A[:, l - 1, d, None] * F[:, T[has] ^ (1 << d)]
        F[:, T] = v
    return F


def _chunked(A, most, f):
    """f over slices of the batch that hold at most `most` subset values, concatenated."""
    step = max(1, int(most) >> A.shape[-1])
    parts = [f(A[b:b + step]) for b in range(0, len(A), step)]
    return [torch.cat(p) for p in zip(*parts)]


def _perm_and_minors(A, levels):
    n = A.shape[-1]
    F = _subset_perms(A, levels)
    R = _subset_perms(A.flip(1), levels)  # R[T]: the last |T| rows on the columns T
    order, at = levels
    G = torch.zeros_like(A)
    full = (1 << n) - 1
    for i in range(n):
        T = order[at[i]:at[i + 1]]
        for j in range(n):
            t = T[((T >> j) & 1) == 0]
            G[:, i, j] = (F[:, t] * R[:, full ^ t ^ (1 << j)]).sum(1)
    return F[:, full].clone(), G


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sampler", "gcca", "counts"):
        return None  # whole numbers
    rng = np.random.default_rng([seed, 7])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "perm":
        n, b = case["n"], case["batch"]
        if n > 25 or n * b * 2.0 ** n > 2.0 ** 35:
            return None
        A, levels = _blocks(n, b, rng), _levels(n, dev)
        return _chunked(A, 1 << 26, lambda a: (_subset_perms(a, levels)[:, -1].clone(),))[0]
    if kind == "grad":
        n, b = case["n"], case["batch"]
        if n > 22 or n * n * b * 2.0 ** n > 2.0 ** 35.5:
            return None
        A = _blocks(n, b, rng, case["collisions"])
        g = rng.standard_normal((2, b))
        g = torch.from_numpy(g[0] + 1j * g[1]).to(A.device)
        levels = _levels(n, dev)
        p, G = _chunked(A, 1 << 25, lambda a: _perm_and_minors(a, levels))
        return {"perm": p, "grad": g[:, None, None] * G.conj()}
    if kind == "pairs":
        out, ins = _pairs_rows(case, rng)
        U = torch.from_numpy(_haar(case["m"], rng)).to(dev)
        A = U[torch.from_numpy(out).to(dev)][:, :, :case["n"]].contiguous()
        levels = _levels(case["n"], dev)
        at = torch.from_numpy((1 << ins).sum(axis=1)).to(dev)
        return _chunked(A, 1 << 25, lambda a: (_subset_perms(a, levels)[:, at],))[0]
    # minors: the k particles are the columns; minor of particle i is on all but column i
    k = case["k"]
    out, ins = _minors_rows(case, rng)
    U = torch.from_numpy(_haar(case["m"], rng)).to(dev)
    A = U[torch.from_numpy(out).to(dev)[:, :, None], torch.from_numpy(ins).to(dev)[:, None, :]]
    levels = _levels(k, dev)
    without = ((1 << k) - 1) ^ (1 << torch.arange(k, device=A.device))
    M = _chunked(A.reshape(len(ins), k - 1, k), 1 << 25,
                 lambda a: (_subset_perms(a, levels)[:, without],))[0]
    new = np.ones(ins.shape, dtype=bool)  # a doubled mode's particles share one slot
    new[:, 1:] = ins[:, 1:] != ins[:, :-1]
    return M[torch.from_numpy(new).to(M.device)].reshape(len(ins), -1)
