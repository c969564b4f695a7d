"""Counts of large inputs that lie in runs of equal ids (csrc/fgl_bucket.hip): sorted ids, hubs over several tiles of 8192, runs on either side of the limit of four
entries, tiles of either kind in turn, ids that no counter has, and a count on the device -- against torch.bincount."""
import pytest
import torch

from fastgl import ops

pytestmark = pytest.mark.gpu
N, BINS, TILE = 3_000_017, 700_000, 8192


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
    if kind == "mixed":  # tiles in order between tiles in none
        x = torch.randint(0, BINS, (N,), generator=gen, device=dev)
        in_runs = (torch.arange(N, device=dev) // TILE) % 2 == 0
        return torch.where(in_runs, torch.arange(N, device=dev) // 13 % BINS, x)
    x = torch.randint(0, BINS, (N,), generator=gen, device=dev).sort()[0]  # "gaps": ids out of range in runs and alone
    x[5_000:30_000] = -1
    x[2_000_000:2_000_999:3] = BINS + 5
    x[N - 10:] = -7
    return x


@pytest.mark.parametrize("kind", ["sorted", "hub", "threes", "fours", "fives", "mixed", "gaps"])
def test_counts(cuda, kind):
    print("runs", kind, flush=True)
    x = _ids(kind, torch.Generator(device=cuda).manual_seed(7), cuda)
    for part in (x, x[1:], x[:2_600_000], x[3:TILE * 300 + 3]):
        part = part.int().contiguous()
        want = torch.bincount(part[(part >= 0) & (part < BINS)].long(), minlength=BINS).int()
        assert torch.equal(ops.cal_deg(part, BINS), want)
