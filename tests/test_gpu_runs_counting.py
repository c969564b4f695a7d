"""Counts of large inputs that lie in runs of equal ids (csrc/fgl_bucket.hip): sorted ids, hubs over several tiles of 8192, runs
on either side of the limit of six entries, in order and in none, tiles of either kind in turn, tiles in order only at their
beginning or up to their last entries, sorted stretches one after another, also as long as the 64th parts of the input or with ids
beyond those, ids that no counter has -- against torch.bincount; and that ids which recur in runs take no longer."""
import pytest
import torch

from fastgl import ops

pytestmark = pytest.mark.gpu
N, BINS, TILE = 3_000_017, 700_000, 8192
UP = {"fives up": 5, "sixes up": 6, "sevens up": 7, "tens up": 10, "hundreds up": 100, "hundreds down": 100}


def _ids(kind, gen, dev):
    if kind == "sorted":
        return torch.randint(0, BINS, (N,), generator=gen, device=dev).sort()[0]
    if kind == "hub":  # one id over 40 tiles and a bit
        x = torch.randint(0, BINS, (N,), generator=gen, device=dev).sort()[0]
        x[100_001:100_001 + 40 * TILE + 77] = BINS - 1
        return x
    if kind in ("threes", "fours", "fives"):
        k = {"threes": 3, "fours": 4, "fives": 5}[kind]
        return (torch.arange(N, device=dev) // k * 7919) % BINS
    if kind in UP:
        i = torch.arange(N, device=dev) // UP[kind]
        return BINS - 1 - i if kind.endswith("down") else i
    if kind == "beginnings":  # the first eighth of every tile in order, and all but its last few entries in every third
        i = torch.arange(N, device=dev)
        x = torch.randint(0, BINS, (N,), generator=gen, device=dev)
        return torch.where((i % TILE < torch.where(i // TILE % 3 == 0, TILE - 3, TILE // 8)), i // 22 % BINS, x)
    if kind == "mixed":  # tiles in order between tiles in none
        x = torch.randint(0, BINS, (N,), generator=gen, device=dev)
        in_runs = (torch.arange(N, device=dev) // TILE) % 2 == 0
        return torch.where(in_runs, torch.arange(N, device=dev) // 23 % BINS, x)
    if kind.startswith("stretches"):  # sorted ones, of two tiles, of a part of six tiles, of five tiles with a few high ids at their ends
        i = torch.arange(N, device=dev)
        long = {"stretches": 2, "stretches of a part": 6, "stretches beyond": 5}[kind] * TILE
        base = i // long * (long // 16) if kind == "stretches of a part" else 0
        return torch.where((i % long > long - 20) & (kind == "stretches beyond"), BINS - 1, base + i % long // 16)
    x = torch.randint(0, BINS // (8 if kind.startswith("long") else 1), (N,), generator=gen, device=dev).sort()[0]
    if kind == "long sorted":  # (34 a run: counted where their histogram is taken)
        return x
    # "gaps": ids out of range in runs and alone
    x[5_000:30_000] = -1
    x[2_000_000:2_000_999:3] = BINS + 5
    x[N - 10:] = -7
    return x


@pytest.mark.parametrize("kind", ["sorted", "long sorted", "hub", "threes", "fours", "fives", *UP, "stretches", "stretches of a part", "stretches beyond", "beginnings", "mixed", "gaps", "long gaps"])
def test_counts(cuda, kind):
    print("runs", kind, flush=True)
    x = _ids(kind, torch.Generator(device=cuda).manual_seed(7), cuda)
    for part in (x, x[1:], x[:2_600_000], x[3:TILE * 300 + 3]):
        part = part.int().contiguous()
        want = torch.bincount(part[(part >= 0) & (part < BINS)].long(), minlength=BINS).int()
        assert torch.equal(ops.cal_deg(part, BINS), want)


@pytest.mark.parametrize("n,bins,times", [(5_000_000, 2, 10), (5_000_000, 1000, 10), (5_000_000, 2048, 10), (54_000_000, 497, 2), (54_000_000, 600_000, 2)])
def test_ids_that_recur_in_runs(cuda, n, bins, times):
    """An atomic a run in device memory would take hundreds of times as long for the first of these (54 M ids, fives of two ids in
    turn: 122 ms against 0.26), and more than three times as long for the
    last but one, sorted stretches of two tiles (880 us against 260); such that begin anew for each 64th part of the input, the last, pass a look at the parts alone."""
    i = torch.arange(n, device=cuda)
    part = (n // TILE + 64) // 64 * TILE
    runs = (i // part * 8000 + i % (2 * TILE) // 8 if bins == 600_000 else i % (2 * TILE) // 33 if bins == 497 else i % TILE // 4 if bins == 2048 else i // 5 % bins).int()
    no_order = torch.randint(0, bins, (n,), device=cuda, dtype=torch.int32)

    def time(x):
        assert torch.equal(ops.cal_deg(x, bins), torch.bincount(x.long(), minlength=bins).int())
        best = float("inf")
        for _ in range(5):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            ops.cal_deg(x, bins)
            end.record()
            end.synchronize()
            best = min(best, begin.elapsed_time(end))
        return best

    assert time(runs) < times * time(no_order)


@pytest.mark.parametrize("n", [8_886_435, 8_886_272])
def test_sorted_ids_of_few_counters(cuda, n):
    """A last tile that is not full counts as in order too: alone in buckets it kept the launches behind waiting, half as long again."""
    x = torch.randint(0, 176, (n,), device=cuda, dtype=torch.int32).sort()[0]
    for part in (x, x[:-1], x[:-8000], x[5:]):
        part = part.contiguous()
        assert torch.equal(ops.cal_deg(part, 176), torch.bincount(part.long(), minlength=176).int())
    best = []
    for ids in (x, x[:8192 * 1084].contiguous()):
        times = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(20):
                ops.cal_deg(ids, 176)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        best.append(min(times))
    assert best[0] < 1.25 * best[1]
