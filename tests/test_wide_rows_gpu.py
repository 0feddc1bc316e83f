"""Row groups, token groups and tile remainders of the wide and narrow passes: the numbers of query rows
and tokens at which a block changes how its waves share them (16-row groups, three or two of them per
wave, one, two or four token groups, 64-token super tiles with a ring of two), in both list orders and from
lists made by hand."""
import math

import pytest
import torch

from cases import build_tree
from fasttree_hip.decode import fasttree_decode, fasttree_decode_stage1, gathered_decode
from fasttree_hip.inputs import make_decode_inputs
from fasttree_hip.planner import FastTreeParams, fasttree_preparation
from test_decode_gpu import _dense_check

pytestmark = pytest.mark.gpu

# requests of one KV head each: rows of the shared run
ROWS = [16, 17, 33, 48, 49, 64, 65, 96, 97, 128, 129, 144, 191, 192, 193, 385]
# tokens of the shared run: within a tile, at the edges of a tile, of a super tile and of the ring
TOKENS = [1, 31, 33, 64, 65, 129, 321]


def _run(device, rows, tokens, group, heads, d, dtype, launch_order):
    print("\n[gpu case] wide rows", rows, tokens, group, heads, d, dtype, launch_order, flush=True)
    requests = -(-rows // group)
    tree, ptrs, batch = build_tree({"kind": "regular", "sizes": [1, requests], "lens": [tokens, 5]})
    inp = make_decode_inputs(tree, group * heads, heads, d, device=device, dtype=dtype, seed=rows + tokens, shuffle_slots=True)
    params = FastTreeParams()
    # (no merging: the shared run stays one of `rows` query rows)
    params.set_values(0.66, 0.33, 0.1)
    params.set_q_tile_sizes([max(1, 512 // group), max(1, 16 // group)])
    params.set_kv_tile_sizes([32, 32])
    params.set_kv_group_num(group)
    aux, _ = fasttree_preparation(tree, inp.KV_ptrs, batch, group * heads, heads, d, [4096, 4096], [1, 1], [1, 1], params,
                                  device=device, kv_slot_map=inp.slot_map, launch_order=launch_order)
    o = torch.full_like(inp.Q, float("nan"))
    fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, o, *aux, list(params.TSQs), list(params.TSKs), 1.0 / math.sqrt(d))
    torch.cuda.synchronize()
    _dense_check(tree, inp, o, f"{rows} rows, {tokens} tokens", dtype=dtype)


@pytest.mark.parametrize("launch_order", [False, True], ids=["planner_order", "launch_order"])
@pytest.mark.parametrize("rows", ROWS)
def test_row_groups(rows, launch_order, device):
    _run(device, rows, 200, 1, 8, 128, torch.float16, launch_order)


@pytest.mark.parametrize("launch_order", [False, True], ids=["planner_order", "launch_order"])
@pytest.mark.parametrize("tokens", TOKENS)
@pytest.mark.parametrize("rows", [40, 80, 180])
def test_token_remainders(rows, tokens, launch_order, device):
    _run(device, rows, tokens, 4, 2, 64, torch.bfloat16, launch_order)


@pytest.mark.parametrize("d", [32, 256])
@pytest.mark.parametrize("rows", [33, 64, 97, 128, 129, 200])
def test_row_groups_of_other_head_sizes(rows, d, device):
    _run(device, rows, 97, 3, 2, d, torch.float16, True)


@pytest.mark.parametrize("d,dtype", [(128, torch.float16), (64, torch.bfloat16), (32, torch.float16)])
@pytest.mark.parametrize("rows", [33, 48, 64, 80, 96])
def test_token_groups_round_their_own_probabilities(rows, d, dtype, device):
    """33 to 96 rows are two token groups, each with a soft-max reference of its own: where each half of a run has one
    token that counts, both have the probability 1, which 16 bits hold exactly, and the partial result is as good as
    its fp32 sums.  (With one group for both, the lesser token's probability would be rounded to 16 bits.)"""
    print("\n[gpu case] token groups", rows, d, dtype, flush=True)
    tokens, group, heads = 64, 4, 2
    requests = -(-rows // group)
    tree, ptrs, batch = build_tree({"kind": "regular", "sizes": [1, requests], "lens": [tokens, 5]})
    inp = make_decode_inputs(tree, group * heads, heads, d, device=device, dtype=dtype, seed=0, shuffle_slots=False)
    params = FastTreeParams()
    params.set_values(0.66, 0.33, 0.1)
    params.set_q_tile_sizes([512 // group, 16 // group])
    params.set_kv_tile_sizes([32, 32])
    params.set_kv_group_num(group)
    aux, _ = fasttree_preparation(tree, inp.KV_ptrs, batch, group * heads, heads, d, [4096, 4096], [1, 1], [1, 1], params,
                                  device=device, launch_order=False)
    assert aux[11][0] == 1 and aux[2][0] == tokens and aux[5][0] == requests
    # a score below the first by s: of the candidates the one whose probability is worst to hold in 16 bits
    scale = 1.0 / math.sqrt(d)
    steps = torch.arange(1, 64, dtype=torch.float64) / 64
    p = torch.exp(-scale * steps)
    off = (p.to(dtype).double() - p).abs()
    step = float(steps[off.argmax()])
    w = math.exp(-scale * step)
    assert float(off.max()) > 2.0 ** -13
    inp.Q.zero_()
    inp.Q[..., 0] = 1
    slots = aux[0][:tokens].long()
    inp.K_pool.zero_()
    inp.K_pool[slots, :, 0] = -8192.0                      # (probability 0)
    inp.K_pool[slots[5], :, 0] = 0
    inp.K_pool[slots[32 + 7], :, 0] = -step
    inp.V_pool[slots[5]] = 1
    inp.V_pool[slots[32 + 7]] = -1
    mid_o, mid_lse = aux[9], aux[10]
    mid_o.fill_(float("nan"))
    fasttree_decode_stage1(inp.Q, inp.K_pool, inp.V_pool, *aux[:6], scale, mid_o, mid_lse, aux[11], aux[12],
                           list(params.TSQs), list(params.TSKs))
    first = int(aux[4][0])
    got = mid_o[first: first + requests].double().cpu()
    # w and the sums are good to a few 2^-24 each; w rounded to 16 bits would be off by more than 2^-13, the result by
    # 2 / (1 + w)^2, at least half, of that
    assert float((got - (1 - w) / (1 + w)).abs().max()) < 2.0 ** -18


@pytest.mark.parametrize("d,dtype", [(128, torch.float16), (64, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("rows", [5, 16, 17, 32, 48, 80])
def test_partials_of_one_wide_vnode(rows, d, dtype, device):
    """A wide phase of one vnode, from lists made by hand (the planner gives runs this short or narrow to other
    phases): two token groups, at head_dim 256 four up to 16 rows, two up to 32, then one; at these lengths some of
    them get no tile."""
    print("\n[gpu case] one wide vnode", rows, d, dtype, flush=True)
    heads = 2
    gen = torch.Generator().manual_seed(rows)
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32, device=device)  # noqa: E731
    scale = 1.0 / math.sqrt(d)
    for tokens in TOKENS:
        q = torch.randn(rows, heads, d, generator=gen).to(dtype)
        k, v = (torch.randn(400, heads, d, generator=gen).to(dtype) for _ in range(2))
        slots = torch.randperm(400, generator=gen)[:tokens]
        mid_o = torch.full((rows, heads, d), float("nan"), device=device)
        mid_lse = torch.full((rows, heads), float("nan"), device=device)
        fasttree_decode_stage1(q.to(device), k.to(device), v.to(device), i32(slots), i32([0]), i32([tokens]), i32(range(rows)), i32([0]),
                               i32([rows]), scale, mid_o, mid_lse, [1, 0], [0, 1], [512, 16], [32, 32])
        s = torch.einsum("rhd,thd->rht", q.double(), k[slots].double()) * scale
        p = torch.softmax(s, -1)
        want = torch.einsum("rht,thd->rhd", p, v[slots].double())
        # a probability is rounded to 16 bits once: off by 2^-11 (2^-8) of itself, fp16's small ones by 2^-25 of the largest
        spread = torch.einsum("rht,thd->rhd", p, v[slots].double().abs())
        bound = 2.0 ** (-11 if dtype is torch.float16 else -8) * spread + 2.0 ** -25 * tokens * float(v.abs().max()) + 1e-5
        assert bool(((mid_o.cpu().double() - want).abs() <= bound).all()), tokens
        assert float((mid_lse.cpu().double() - torch.logsumexp(s, -1)).abs().max()) < 1e-4, tokens


@pytest.mark.parametrize("d,dtype", [(128, torch.float16), (64, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("group", [17, 32, 33, 48, 64])
def test_gathered_decode_of_large_groups(group, d, dtype, device):
    """Gathered caches with more than 16 query heads per KV head, which are wide vnodes there: two token groups with a row
    group per wave and with two, whole runs and splits of 8 tokens, most of them empty, whose lists of 88 entries the
    merge cuts for groups of lanes."""
    print("\n[gpu case] gathered, large groups", group, d, dtype, flush=True)
    heads, lens = 2, [700, 1, 131]
    gen = torch.Generator().manual_seed(group)
    scale = 1.0 / math.sqrt(d)
    q = torch.randn(len(lens), group * heads, d, generator=gen).to(dtype)
    k, v = (torch.randn(len(lens), max(lens), heads, d, generator=gen).to(dtype) for _ in range(2))
    for kv_split in (8, 700):
        o = torch.full_like(q, float("nan"), device=device)
        gathered_decode(q.to(device), k.to(device), v.to(device), torch.tensor(lens, dtype=torch.int32, device=device), o, scale,
                        kv_split=kv_split)
        got = o.cpu().double()
        for r, n in enumerate(lens):
            kr, vr = (x[r, :n].double().repeat_interleave(group, dim=1) for x in (k, v))
            p = torch.softmax(torch.einsum("hd,thd->ht", q[r].double(), kr) * scale, -1)
            want = torch.einsum("ht,thd->hd", p, vr)
            # a probability is rounded to 16 bits once, as in the test above, and so is the result
            eps = 2.0 ** (-11 if dtype is torch.float16 else -8)
            bound = eps * (torch.einsum("ht,thd->hd", p, vr.abs()) + want.abs()) + 2.0 ** -25 * n * float(vr.abs().max()) + 1e-5
            assert bool(((got[r] - want).abs() <= bound).all()), (kv_split, r)
