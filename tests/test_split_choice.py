"""CPU tests of the chunk length a split-KV plan takes (fa_fwd_plan).

Two rules offer one: chunks about the average load of a workgroup slot, or the
shortest with which every item runs at once.  Each is the slower one on a part
of the shapes (measured on MI355X: the second lost 14 % at causal fp16 D = 64
B1 H5 N12000, the first 20 % at causal bf16 D = 128 B1 H2 N8192), so the plan
must take the one whose launch is modelled shorter, and without a search that
costs the host more than the launch."""
from __future__ import annotations

import ctypes
import time

import pytest

import abi_ctypes as A
from test_abi import contiguous
from test_split_plan import check_plan, plan, tiles

CUS = 256
SCRATCH = A.FA_SCRATCH_BYTES


@pytest.fixture(scope="module")
def lib():
    return A.load()


class Split:
    """The plan with chunks of at most S tiles, and its modelled cost."""

    def __init__(self, bh, N, D, BM, causal, S):
        nq = (N + BM - 1) // BM
        self.lens, self.slots = [], 0
        for qb in range(nq):
            T = tiles(qb, N, BM, causal)
            n = min(255, -(-T // S))
            self.lens += [(c + 1) * T // n - c * T // n for c in range(n)]
            self.slots += n if n > 1 else 0
        self.lens.sort(reverse=True)
        self.items = bh * len(self.lens)
        self.bytes = bh * self.slots * BM * (4 * D + 16)
        chunks = -(-tiles(nq - 1, N, BM, causal) // S)
        self.cost = self._load(BM) + 10.0 * self.slots * bh / CUS + 0.75 * ((chunks + 3) // 4)

    def _load(self, BM):
        """The last CU's load: each XCD hands its run of items to its 32 CUs,
        the least loaded next; two 4-wave workgroups of a CU share it at 1.1
        times the rate of one."""
        if self.items <= CUS:
            return self.lens[0]
        worst, first = 0, 0
        for x in range(8):
            count = self.items // 8 + (x < self.items % 8)
            load = [0] * (CUS // 8)
            for i in range(first, first + count):
                k = load.index(min(load))
                load[k] += self.lens[i % len(self.lens)]
            first += count
            worst = max(worst, *load)
        return max(self.lens[0], worst / (1.1 if BM == 128 else 1.0))


def candidates(bh, N, D, BM, causal):
    """(average-load plan, one-round plan or None)."""
    nq = (N + BM - 1) // BM
    slots = CUS * (2 if BM == 128 else 1)
    t = [tiles(qb, N, BM, causal) for qb in range(nq)]
    avg = -(-sum(t) * bh // slots)
    S = max(8, avg)
    while len(Split(bh, N, D, BM, causal, S).lens) > A.FA_PLAN_MAX_ITEMS:
        S *= 2
    first = Split(bh, N, D, BM, causal, S)
    if first.bytes > SCRATCH:
        return first, None
    for S in range(max(4, avg), max(t)):
        p = Split(bh, N, D, BM, causal, S)
        if len(p.lens) <= A.FA_PLAN_MAX_ITEMS and p.items <= slots and p.bytes <= SCRATCH:
            return first, p
    return first, None


# Shapes either rule loses: (H, N, D, dtype, longest item at most).  The bounds
# are between the two rules' longest items.
@pytest.mark.parametrize("H,N,D,dtype,longest", [
    (6, 10000, 64, A.FA_DTYPE_F16, 100), (7, 8192, 64, A.FA_DTYPE_F16, 80),
    (5, 12000, 64, A.FA_DTYPE_F16, 120), (4, 14000, 64, A.FA_DTYPE_F16, 130),
    (3, 16384, 64, A.FA_DTYPE_F16, 130), (3, 20000, 64, A.FA_DTYPE_F16, 200),
    (2, 8192, 128, A.FA_DTYPE_BF16, 20), (1, 16384, 128, A.FA_DTYPE_F16, 90),
])
def test_longest_item(lib, H, N, D, dtype, longest):
    pl = plan(lib, contiguous(B=1, H=H, N=N, D=D, dtype=dtype, causal=1))
    check_plan(pl, 1, H, N, D, 1)
    assert max(pl.tile_end[i] - pl.tile_begin[i] for i in range(pl.n_items)) <= longest


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("D", [64, 128])
def test_shorter_launch_is_taken(lib, D, causal):
    """Over the shapes that split: the plan is one of the two rules', and the
    other's modelled cost is no lower."""
    took = set()
    for N in (513, 768, 1000, 1280, 1537, 2048, 2500, 3000, 4096, 6000, 8192, 9000, 12000, 16384,
              20000, 24000, 32512):
        for H in (1, 2, 3, 4, 5, 7, 10, 12, 16, 20):
            for dtype in (A.FA_DTYPE_F16, A.FA_DTYPE_BF16):
                pl = plan(lib, contiguous(B=1, H=H, N=N, D=D, dtype=dtype, causal=causal), CUS)
                if pl.n_merge == 0:
                    continue
                lens = [pl.tile_end[i] - pl.tile_begin[i] for i in range(pl.n_items)]
                first, second = candidates(H, N, D, pl.block_rows, causal)
                mine, other = (first, second) if lens == first.lens else (second, first)
                assert mine is not None and lens == mine.lens and pl.n_slots == mine.slots, (H, N)
                assert first.slots > 0, (H, N)  # a problem the first rule leaves whole is not split
                if other is not None and other.lens != mine.lens:
                    assert mine.cost <= other.cost, (H, N, mine.cost, other.cost)
                    took.add(mine is first)
    assert took == {True, False} or not causal


@pytest.mark.parametrize("H,N,D,split", [
    (3, 7000, 64, True), (3, 7168, 64, True),    # two groups 3...9 % slower than the split
    (2, 9032, 64, True), (2, 9032, 128, True),
    (4, 5341, 64, False), (2, 14000, 64, False), (5, 4147, 64, False),  # the split the slower one
])
@pytest.mark.parametrize("dtype", [A.FA_DTYPE_F16, A.FA_DTYPE_BF16])
def test_split_or_two_key_groups(lib, H, N, D, split, dtype):
    """Non-causal grids of at most one 128-row q-tile per CU run two key groups
    unless a split's modelled time is clearly lower."""
    pl = plan(lib, contiguous(B=1, H=H, N=N, D=D, dtype=dtype, causal=0))
    if split:
        check_plan(pl, 1, H, N, D, 0)
        assert pl.workspace_bytes <= SCRATCH
    else:
        assert pl.n_items == 0 and pl.block_rows == 128 and pl.workspace_bytes == 0


@pytest.mark.parametrize("H,N,D,causal", [
    (1, 32512, 128, 1), (1, 28000, 64, 1), (1, 24000, 128, 1), (2, 24000, 64, 1), (4, 16384, 64, 1),
    (1, 16384, 128, 1), (7, 2500, 128, 1), (8, 2048, 64, 1), (1, 16384, 128, 0),
])
def test_plan_time(lib, H, N, D, causal):
    """The plan is made two or three times a call: about 10 us at most where
    one without a split takes 1 (a search over every length took 27 to 130 us
    for most of these shapes).  Timed against that one, best of many; the
    bound leaves twice the largest ratio seen."""
    def best(p):
        out, t_min = A.FaFwdPlan(), float("inf")
        for _ in range(300):
            t = time.perf_counter()
            lib.fa_fwd_plan(ctypes.byref(p), CUS, ctypes.byref(out))
            t_min = min(t_min, time.perf_counter() - t)
        return t_min

    unsplit = best(contiguous(B=1, H=64, N=4096, D=128, causal=1))
    mine = best(contiguous(B=1, H=H, N=N, D=D, dtype=A.FA_DTYPE_F16, causal=causal))
    assert mine < 20 * unsplit, f"{mine * 1e6:.1f} us, unsplit {unsplit * 1e6:.1f}"
