"""Plans of whole paths (a request's path is one vnode, the call one launch): path lengths at the edges of tiles and of
the rounds of tiles that a block's waves take, every head size, one and two groups of 16 query rows."""
import math

import pytest
import torch

from fasttree_hip.decode import fasttree_decode, fasttree_decode_stage1, fasttree_decode_stage2, fasttree_decode_static
from fasttree_hip.inputs import make_decode_inputs
from fasttree_hip.kv_tree import generate_tree, nodes_from_rows
from fasttree_hip.planner import FastTreeParams, PlanBuffers, fasttree_preparation
from test_decode_gpu import _dense_check


def _plan(sizes, lens, group, heads, d, dtype, device, buffers=None, num_cus=None, seed=0):
    tree = nodes_from_rows(generate_tree(sizes, lens))
    inp = make_decode_inputs(tree, group * heads, heads, d, device=device, dtype=dtype, seed=seed, shuffle_slots=True)
    params = FastTreeParams()
    params.set_q_tile_sizes([max(1, 64 // group), max(1, 16 // group)])
    params.set_kv_tile_sizes([32, 32])
    params.set_kv_group_num(group)
    aux, _ = fasttree_preparation(tree, inp.KV_ptrs, inp.batch_size, group * heads, heads, d, [1024, 256], [256, 1024], [256, 256], params,
                                  device=device, kv_slot_map=inp.slot_map, launch_order=True, buffers=buffers, num_cus=num_cus)
    return tree, inp, aux, (list(params.TSQs), list(params.TSKs), 1.0 / math.sqrt(d))


@pytest.mark.gpu
@pytest.mark.parametrize("d,group,heads,dtype", [(128, 4, 8, torch.float16), (128, 16, 1, torch.bfloat16), (128, 32, 2, torch.float16),
                                                 (64, 3, 8, torch.bfloat16), (64, 20, 2, torch.float16), (32, 1, 4, torch.float16),
                                                 (256, 16, 1, torch.bfloat16), (256, 24, 2, torch.float16)])
@pytest.mark.parametrize("lens", [[1, 1], [20, 11], [20, 12], [20, 13], [120, 8], [121, 8], [250, 6], [250, 7], [400, 9], [507, 6]],
                         ids=lambda x: str(sum(x)))
def test_path_lengths(lens, d, group, heads, dtype, device):
    if dtype is torch.bfloat16 and sum(lens) == 2:
        # (outputs of two tokens are 0.7 in the mean and the output's rounding, up to 2^-9 of a value, takes half of the bar
        # of 1e-3 by itself, that of the two probabilities as much)
        lens = [5, 4]
    print(f"\n[gpu case] whole paths of {sum(lens)} tokens, {group * heads}/{heads} heads of {d}, {dtype}", flush=True)
    tree, inp, aux, rest = _plan([1, 3], lens, group, heads, d, dtype, device, seed=sum(lens))
    if aux[11].wave_records is None:
        assert d == 256 and sum(lens) > 128, "a launch of paths this short is one of whole paths"
        pytest.skip("long paths of wide rows are laid out in pieces")
    assert list(aux[11]) == [0, 3] and aux[3].numel() == 3
    o = torch.full_like(inp.Q, float("nan"))
    fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, o, *aux, *rest)
    _dense_check(tree, inp, o, f"whole paths of {sum(lens)} tokens", dtype=dtype)
    # the partial results are those of a plan as any other, and so is the plan in two launches
    mid_o, mid_lse, two = aux[9].clone(), aux[10].clone(), torch.empty_like(o)
    fasttree_decode_stage1(inp.Q, inp.K_pool, inp.V_pool, *aux[:6], rest[2], aux[9], aux[10], aux[11], aux[12], *rest[:2])
    assert torch.allclose(mid_lse, aux[10], rtol=0, atol=1e-3) and torch.allclose(mid_o, aux[9], rtol=0, atol=4e-3 if dtype is torch.float16 else 3e-2)
    fasttree_decode_stage2(*aux[6:9], mid_o, mid_lse, two)
    assert torch.equal(two, o), "the merge of one partial result is the rounded result"


@pytest.mark.gpu
def test_paths_of_unequal_length_in_other_entry_points(device):
    """A plan in buffers made beforehand, with o in rows of another pitch; the entry point that keeps its scratch to
    itself; a captured call, replayed between others."""
    print("\n[gpu case] whole paths in buffers, static, captured", flush=True)
    buffers = PlanBuffers(32, 128, 8192, 256, 256, 64)
    tree, inp, aux, rest = _plan([1, 2, 9], [190, 70, 33], 4, 8, 128, torch.float16, device, buffers=buffers, seed=5)
    assert aux[11].wave_records is not None and aux[11].wave_records.data_ptr() == buffers.wave_records.data_ptr()
    want = torch.full_like(inp.Q, float("nan"))
    fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, want, *aux, *rest)
    _dense_check(tree, inp, want, "whole paths in buffers")
    pitched = torch.full((inp.batch_size, 40, 160), float("nan"), dtype=torch.float16, device=device)
    fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, pitched[:, 4:36, 16:144], *aux, *rest)
    assert torch.equal(pitched[:, 4:36, 16:144], want) and bool(torch.isnan(pitched[:, :4]).all()) and bool(torch.isnan(pitched[..., 144:]).all())
    o = torch.full_like(want, float("nan"))
    fasttree_decode_static(inp.Q, inp.K_pool, inp.V_pool, o, *aux[:9], aux[11], aux[12], rest[2])
    assert torch.equal(o, want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    q = inp.Q.clone()
    with torch.cuda.stream(side):
        fasttree_decode(q, inp.K_pool, inp.V_pool, o, *aux, *rest)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        fasttree_decode(q, inp.K_pool, inp.V_pool, o, *aux, *rest)
    for turn in range(3):
        q.copy_(inp.Q * (turn + 1))
        fasttree_decode(q, inp.K_pool, inp.V_pool, want, *aux, *rest)
        o.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want), turn


def test_which_trees_are_laid_out_as_whole_paths():
    """Short paths with less than a block per unit; not long ones, not more of them."""
    def whole(sizes, lens, group, heads, d=128, cus=256):
        tree = nodes_from_rows(generate_tree(sizes, lens))
        from fasttree_hip.kv_tree import assign_requests, kv_prefix_sums
        batch, ptrs = assign_requests(tree), kv_prefix_sums(tree)
        params = FastTreeParams()
        params.set_q_tile_sizes([max(1, 64 // group), max(1, 16 // group)])
        params.set_kv_tile_sizes([32, 32])
        params.set_kv_group_num(group)
        aux, assigned = fasttree_preparation(tree, ptrs, batch, group * heads, heads, d, [1024, 256], [256, 1024], [256, 256], params, device="cpu",
                                             launch_order=True, num_cus=cus)
        if aux[11].wave_records is None:
            return False
        assert assigned == [0] + [1] * (len(tree) - 1) and list(aux[11]) == [0, batch] and aux[11].num_programs == 0
        waves = 8 if d <= 128 else 4
        rec = aux[11].wave_records.view(batch, waves, 64)
        for v in range(batch):
            off, n = int(aux[1][v]), int(aux[2][v])
            for w in range(waves):
                assert rec[v, w, :4].tolist() == [off, n, int(aux[4][v]), 1] and int(rec[v, w, 4]) == int(aux[3][aux[4][v]])
                at = [min(32 * w + t, n - 1) for t in range(32)]
                assert rec[v, w, 20:52].tolist() == aux[0][[off + t for t in at]].tolist()
        return True

    assert whole([1, 4], [384, 24], 4, 8) and whole([1, 31], [200, 100], 4, 8) and whole([1, 4], [384, 24], 4, 8, d=64)
    assert whole([1, 200], [300, 30], 16, 1, d=256)
    assert not whole([1, 4], [3000, 24], 4, 8) and not whole([1, 32], [200, 100], 4, 8) and not whole([1, 31], [200, 100], 4, 8, cus=128)


@pytest.mark.parametrize("short_by", [0, 1])
def test_whole_paths_need_room_in_the_slot_list(short_by):
    """A plan of whole paths lists a token once per leaf; buffers that have no room for that hold the plan that lists it once."""
    paths = 4 * (384 + 24) + 32
    buffers = PlanBuffers(32, 128, paths - short_by, 256, 256, 64, device="cpu")
    tree = nodes_from_rows(generate_tree([1, 4], [384, 24]))
    from fasttree_hip.kv_tree import assign_requests, kv_prefix_sums
    params = FastTreeParams()
    params.set_q_tile_sizes([16, 4])
    params.set_kv_tile_sizes([32, 32])
    params.set_kv_group_num(4)
    aux, assigned = fasttree_preparation(tree, kv_prefix_sums(tree), assign_requests(tree), 32, 8, 128, [1024, 256], [256, 1024], [256, 256], params,
                                         device="cpu", launch_order=True, num_cus=256, buffers=buffers)
    assert (aux[11].wave_records is None) == bool(short_by)
    assert aux[0].numel() == (384 + 4 * 24 + 32 if short_by else paths) and aux[11].modelled_us is not None


def test_wave_records_go_with_the_records_they_repeat():
    """A caller that edits the lists in place drops or replaces ``narrow_table``: the plan is then one in two launches."""
    from fasttree_hip import _lib
    from fasttree_hip.decode import _narrow_in_programs
    from fasttree_hip.launch_schedule import LaunchPhases
    for value in (None, torch.zeros(64, dtype=torch.int32)):
        phases = LaunchPhases([0, 4])
        phases.narrow_table, phases.wave_records = torch.zeros(64, dtype=torch.int32), torch.zeros(512, dtype=torch.int32)
        assert _narrow_in_programs(phases) == _lib.FT_WHOLE_PATHS
        phases.narrow_table = value
        assert phases.wave_records is None and _narrow_in_programs(phases) == 0 and phases.narrow_table is value


def _infinite_values(v, slots, d):
    """A copy of ``v`` with infinities in single dims of the tokens at ``slots``: dim 1 of the first +inf, dim 2 of the second -inf, dim
    d - 1 both; and those dims."""
    v = v.clone()
    v[slots[0], :, 1] = v[slots[0], :, d - 1] = float("inf")
    v[slots[1], :, 2] = v[slots[1], :, d - 1] = float("-inf")
    return v, [1, 2, d - 1]


@pytest.mark.gpu
@pytest.mark.parametrize("d,group,heads,dtype", [(128, 4, 8, torch.float16), (128, 20, 2, torch.bfloat16), (64, 3, 8, torch.float16),
                                                 (32, 1, 4, torch.bfloat16), (256, 16, 1, torch.float16)])
@pytest.mark.parametrize("at", [(0, 1), (40, 3), (70, 95)])
def test_infinite_values_stay_infinite(at, d, group, heads, dtype, device):
    """An infinity among the values of a prompt's tokens is one in the outputs of that dim (and of two of either sign, NaN); the other
    dims are what they are without it."""
    print(f"\n[gpu case] whole paths with infinite values at {at}, {group * heads}/{heads} heads of {d}, {dtype}", flush=True)
    tree, inp, aux, rest = _plan([1, 3], [100, 28], group, heads, d, dtype, device, seed=d)
    assert aux[11].wave_records is not None
    o = torch.full_like(inp.Q, float("nan"))
    v, dims = _infinite_values(inp.V_pool, [int(inp.slot_map[i]) for i in at], d)
    fasttree_decode(inp.Q, inp.K_pool, v, o, *aux, *rest)
    assert bool((o[..., 1] == float("inf")).all()) and bool((o[..., 2] == float("-inf")).all()) and bool(torch.isnan(o[..., d - 1]).all())
    o[..., dims] = 0
    v[:, :, dims] = 0
    plain = inp.V_pool
    inp.V_pool = v
    _dense_check(tree, inp, o, "the other dims", dtype=dtype)
    inp.V_pool = plain


@pytest.mark.parametrize("inference", [False, True])
@pytest.mark.parametrize("in_buffers", [False, True])
def test_written_records_are_two_launches(in_buffers, inference):
    """A caller that writes into the narrow vnodes' records has the waves' records left alone from there on; one that decodes rows of
    another size than the plan was made for, for that call."""
    from fasttree_hip import _lib
    from fasttree_hip.decode import _narrow_in_programs
    from fasttree_hip.kv_tree import assign_requests, kv_prefix_sums
    with torch.inference_mode(inference):
        buffers = PlanBuffers(32, 128, 8192, 256, 256, 64, device="cpu") if in_buffers else None
        tree = nodes_from_rows(generate_tree([1, 4], [384, 24]))
        params = FastTreeParams()
        params.set_q_tile_sizes([16, 4])
        params.set_kv_tile_sizes([32, 32])
        params.set_kv_group_num(4)
        aux, _ = fasttree_preparation(tree, kv_prefix_sums(tree), assign_requests(tree), 32, 8, 128, [1024, 256], [256, 1024], [256, 256], params,
                                      device="cpu", launch_order=True, num_cus=256, buffers=buffers)
        assert [_narrow_in_programs(aux[11], d) for d in (32, 64, 128, 256)] == [_lib.FT_WHOLE_PATHS] * 3 + [0]
        aux[11].narrow_table.view(-1, 64)[:, 1] -= 1
        assert _narrow_in_programs(aux[11], 128) == 0 and _narrow_in_programs(aux[11]) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("in_buffers", [False, True])
def test_shortened_runs_are_decoded_as_they_are(in_buffers, static, device):
    """Lists and narrow vnodes' records rewritten in place: the last two tokens of every path are not attended any more."""
    print(f"\n[gpu case] whole paths shortened in place, buffers {in_buffers}, static {static}", flush=True)
    buffers = PlanBuffers(32, 128, 8192, 256, 256, 64) if in_buffers else None
    tree, inp, aux, rest = _plan([1, 3], [100, 28], 4, 8, 128, torch.float16, device, buffers=buffers)

    def decode():
        o = torch.full_like(inp.Q, float("nan"))
        if static:
            fasttree_decode_static(inp.Q, inp.K_pool, inp.V_pool, o, *aux[:9], aux[11], aux[12], rest[2])
        else:
            fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, o, *aux, *rest)
        return o

    assert aux[11].wave_records is not None
    _dense_check(tree, inp, decode(), "as planned")
    aux[2].sub_(2)
    aux[11].narrow_table.view(-1, 64)[:, 1] -= 2
    inp.path_tokens = [p[:-2] for p in inp.path_tokens]
    _dense_check(tree, inp, decode(), "shortened")


@pytest.mark.gpu
@pytest.mark.parametrize("planned,decoded", [(256, 128), (256, 32), (64, 256), (128, 64)])
def test_plans_made_for_another_head_size(planned, decoded, device):
    """A model with two head sizes decodes both on one plan (the waves' records are laid out for one number of waves a block)."""
    print(f"\n[gpu case] plan for head_dim {planned}, call of {decoded}", flush=True)
    tree, plain, aux, rest = _plan([1, 6], [70, 20], 4, 4, planned, torch.float16, device)
    assert aux[11].wave_records is not None
    inp = make_decode_inputs(tree, 16, 4, decoded, device=device, dtype=torch.float16, seed=4, shuffle_slots=True)
    order = torch.as_tensor(plain.slot_map).argsort()      # the plan's slots -> positions -> these pools' rows
    k, v = (x[torch.as_tensor(inp.slot_map)[order].to(device)].contiguous() for x in (inp.K_pool, inp.V_pool))
    width = max(planned, decoded)
    mid_o, mid_lse = torch.empty(aux[3].numel(), 16, width, device=device), torch.empty(aux[3].numel(), 16, device=device)
    o = torch.full_like(inp.Q, float("nan"))
    fasttree_decode(inp.Q, k, v, o, *aux[:9], mid_o, mid_lse, *aux[11:], *rest[:2], 1.0 / math.sqrt(decoded))
    _dense_check(tree, inp, o, f"head_dim {decoded} on a plan for {planned}")


def _several_a_leaf(per_leaf, lens, group, planned_group, heads, d, dtype, device):
    """A prompt of lens[0] tokens and leaves of lens[1] that per_leaf[i] requests end at (numbered across the leaves in turn), planned for
    ``planned_group`` query heads per KV head and to be decoded with ``group``."""
    from types import SimpleNamespace

    tree = nodes_from_rows(generate_tree([1, len(per_leaf)], lens))
    inp = make_decode_inputs(tree, group * heads, heads, d, device=device, dtype=dtype, seed=len(per_leaf) + d, shuffle_slots=True)
    left, of_leaf, batch = list(per_leaf), [[] for _ in per_leaf], sum(per_leaf)
    paths = []
    while any(left):
        for i, n in enumerate(left):
            if n > 0:
                of_leaf[i].append(len(paths))
                paths.append(inp.path_tokens[i])
                left[i] -= 1
    tree[0].requests = list(range(batch))
    for node, requests in zip(tree[1:], of_leaf):
        node.requests = requests
    q = torch.randn(batch, group * heads, d, generator=torch.Generator().manual_seed(d)).to(dtype).to(device)
    inp = SimpleNamespace(Q=q, K_pool=inp.K_pool, V_pool=inp.V_pool, KV_ptrs=inp.KV_ptrs, slot_map=inp.slot_map, path_tokens=paths, batch_size=batch)
    params = FastTreeParams()
    params.set_q_tile_sizes([max(1, 64 // planned_group), max(1, 16 // planned_group)])
    params.set_kv_tile_sizes([32, 32])
    params.set_kv_group_num(planned_group)
    aux, _ = fasttree_preparation(tree, inp.KV_ptrs, batch, planned_group * heads, heads, d, [1024, 256], [256, 1024], [256, 256], params,
                                  device=device, kv_slot_map=inp.slot_map, launch_order=True, num_cus=256)
    return tree, inp, aux, (list(params.TSQs), list(params.TSKs), 1.0 / math.sqrt(d))


@pytest.mark.gpu
@pytest.mark.parametrize("per_leaf,planned_group,group", [([3, 1, 2], 4, 4), ([16, 2], 1, 1), ([17, 16], 1, 1), ([32, 5], 1, 1), ([8, 3], 4, 4),
                                                          ([8, 7], 4, 16), ([32, 17], 1, 3)])
@pytest.mark.parametrize("d,heads", [(128, 4), (64, 3), (256, 2)])
def test_leaves_of_several_requests(per_leaf, planned_group, group, d, heads, device):
    """Every request of a leaf gets its own output: a few, as many as a record names and more, one and two row groups; and, on a plan made
    for fewer query heads per KV head, more rows than the two groups of a pass."""
    print(f"\n[gpu case] leaves of {per_leaf} requests, group {group} on a plan for {planned_group}, head_dim {d}", flush=True)
    tree, inp, aux, rest = _several_a_leaf(per_leaf, [90, 45], group, planned_group, heads, d, torch.float16, device)
    assert aux[11].wave_records is not None and list(aux[11]) == [0, len(per_leaf)] and sorted(aux[5].tolist()) == sorted(per_leaf)
    rows = inp.batch_size
    mid_o, mid_lse = torch.empty(rows, group * heads, d, device=device), torch.empty(rows, group * heads, device=device)
    o = torch.full_like(inp.Q, float("nan"))
    fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, o, *aux[:9], mid_o, mid_lse, *aux[11:], *rest)
    _dense_check(tree, inp, o, f"leaves of {per_leaf} requests")
    two = torch.empty_like(o)
    fasttree_decode_stage2(*aux[6:9], mid_o, mid_lse, two)
    assert torch.equal(two, o), "the merge of one partial result is the rounded result"


@pytest.mark.gpu
@pytest.mark.parametrize("d,group,heads", [(128, 16, 1), (64, 3, 8), (256, 16, 1)])
def test_paths_of_two_tokens_in_bf16(d, group, heads, device):
    """What rounding the probabilities leaves over is contracted too, so only the output's rounding is left: 2^-8 of a value that has 8
    significant bits.  The remainders are rounded likewise (2^-8 of 2^-8 of a probability), the rest is fp32."""
    print(f"\n[gpu case] whole paths of two tokens, {group * heads}/{heads} heads of {d}, bf16", flush=True)
    tree, inp, aux, rest = _plan([1, 3], [1, 1], group, heads, d, torch.bfloat16, device, seed=2)
    assert aux[11].wave_records is not None
    o = torch.full_like(inp.Q, float("nan"))
    fasttree_decode(inp.Q, inp.K_pool, inp.V_pool, o, *aux, *rest)
    for r, path in enumerate(inp.path_tokens):
        k, v = (x[torch.as_tensor(path).to(device)].double().cpu() for x in (inp.K_pool, inp.V_pool))
        q = inp.Q[r].double().cpu().view(heads, group, d)
        p = torch.softmax(torch.einsum("hgd,thd->hgt", q, k) * rest[2], -1)
        want, most = torch.einsum("hgt,thd->hgd", p, v), torch.einsum("hgt,thd->hgd", p, v.abs())
        error = (o[r].double().cpu().view(heads, group, d) - want).abs()
        assert bool((error <= want.abs() * 2 ** -8 + most * 2 ** -16 + 1e-5).all()), (r, error.max())
