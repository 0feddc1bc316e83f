"""The merge launch on its own: list lengths around its batches of eight rows and around the fourteen a record
holds, with few requests (a list's parts merged over the waves of a block) and with many; lists over 64 entries."""

import pytest
import torch

from fasttree_hip.decode import fasttree_decode_stage2

LENGTHS = [0, 1, 7, 8, 9, 14, 15, 16, 17, 33, 70]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim,heads", [(16, 6), (32, 5), (64, 24), (128, 9), (256, 3)])
@pytest.mark.parametrize("copies", [1, 40])
def test_merge_of_lists_of_every_length(head_dim, heads, copies, dtype, device):
    print(f"\n[gpu case] merge {head_dim} x {heads}, {copies} copies, {dtype}", flush=True)
    _check_merge(LENGTHS, copies, head_dim, heads, dtype, device)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim,heads", [(16, 6), (32, 5), (64, 24), (128, 9), (256, 3)])
@pytest.mark.parametrize("lengths", [[65], [64, 63], [513, 0, 3], [66, 127, 128, 129, 15, 100], [1000, 20, 64] * 9], ids=len)
def test_merge_of_long_lists(head_dim, heads, lengths, dtype, device):
    """Lists of more than 64 entries, of which few requests' are cut for groups of lanes, beside shorter ones."""
    print(f"\n[gpu case] merge {head_dim} x {heads}, {lengths[:6]}, {dtype}", flush=True)
    _check_merge(lengths, 1, head_dim, heads, dtype, device)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,heads", [(16, 6), (32, 5), (64, 24), (128, 9), (256, 3)])
@pytest.mark.parametrize("copies", [1, 40])
def test_rows_without_weight_are_not_looked_at(head_dim, heads, copies, device):
    """Every count of rows up to one past the sixteen that a row of lanes holds, the rows of log-sum-exp -inf (and those
    so far below the rest that their weight is 0) holding NaN and infinities."""
    print(f"\n[gpu case] merge without weight {head_dim} x {heads}, {copies} copies", flush=True)
    _check_merge(list(range(1, 18)), copies, head_dim, heads, torch.float16, device, unseen=True)


def _check_merge(lengths, copies, head_dim, heads, dtype, device, unseen=False):
    gen = torch.Generator().manual_seed(head_dim + copies)
    lens = torch.tensor(lengths * copies, dtype=torch.int32)
    rows = int(lens.sum())
    entries = torch.randperm(rows, generator=gen).to(torch.int32)
    offs = (torch.cumsum(lens, 0) - lens).to(torch.int32)
    mid_o = torch.randn(rows, heads, head_dim, generator=gen)
    mid_lse = 6 * torch.randn(rows, heads, generator=gen)
    # rows that attended nothing: output 0, log-sum-exp -inf; for one request all of them
    mid_lse[torch.rand(rows, heads, generator=gen) < 0.1] = float("-inf")
    nothing = max(len(lengths) - 2, 0)
    mid_lse[entries[offs[nothing]: offs[nothing] + lens[nothing]].long()] = float("-inf")
    mid_o[mid_lse == float("-inf")] = 0
    given_o, given_lse = mid_o, mid_lse
    if unseen:
        # (exp of less than -104 is 0 in fp32, subnormal numbers included)
        given_lse, given_o = mid_lse.clone(), mid_o.clone()
        given_lse[(mid_lse == float("-inf")) & (torch.rand(rows, heads, generator=gen) < 0.3)] = -1e4
        odd = torch.tensor([float("nan"), float("inf"), float("-inf")])
        given_o[mid_lse == float("-inf")] = odd[torch.randint(3, given_o.shape, generator=gen)][mid_lse == float("-inf")]
        alone = given_lse.clone()
        for off, n in zip(offs.tolist(), lens.tolist()):        # where no row of a list has weight they would be the maximum
            at = entries[off: off + n].long()
            none = (mid_lse[at] == float("-inf")).all(0)
            alone[at] = torch.where(none, float("-inf"), given_lse[at])
        given_lse = alone
    o = torch.full((len(lens), heads, head_dim), float("nan"), dtype=dtype, device=device)
    fasttree_decode_stage2(entries.to(device), offs.to(device), lens.to(device), given_o.to(device), given_lse.to(device), o)
    o = o.cpu().double()
    # rounding to a significand of 11 (fp16) or 8 (bf16) bits is off by at most 2^-11 or 2^-8 of the value; the weights
    # are good to 1e-5; fp16's smallest step is 2^-24
    rounding = 2.0 ** (-11 if dtype is torch.float16 else -8)
    for r, (off, n) in enumerate(zip(offs.tolist(), lens.tolist())):
        at = entries[off: off + n].long()
        lse, x = mid_lse[at].double(), mid_o[at].double()
        top = lse.max(0).values if n else torch.full((heads,), float("-inf"), dtype=torch.float64)
        w = torch.where(lse == float("-inf"), 0.0, torch.exp(lse - top))
        total = w.sum(0)
        want = torch.where(total > 0, 1 / total, 0.0)[:, None] * (w[:, :, None] * x).sum(0)
        bound = rounding * want.abs() + 1e-5 * (x.abs().amax() if n else 0.0) + 2.0 ** -25
        assert bool(((o[r] - want).abs() <= bound).all()), (r, n, float(((o[r] - want).abs() - bound).max()))
