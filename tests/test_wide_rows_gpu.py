"""Row groups, token groups and tile remainders of the wide and narrow passes: the numbers of query rows
and tokens at which a block changes how its waves share them (16-row groups, three or two of them per
wave, one, two or four token groups, 64-token super tiles with a ring of two), in both list orders."""
import math

import pytest
import torch

from cases import build_tree
from fasttree_hip.decode import fasttree_decode, fasttree_decode_stage1
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
