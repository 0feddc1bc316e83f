"""The native launch schedule (csrc/fasttree_schedule.cpp) on the CPU: from the planner's lists and from
a tree, for several devices and head layouts, every request attends every token of its path exactly
once, the program table covers the wide vnodes, and the records say what the lists say."""

import numpy as np
import pytest

from cases import PLANNER_CASES, build_tree
from fasttree_hip import _plan_lib
from fasttree_hip import launch_schedule as ls
from helpers import run_planner

NAMES = ["kat1", "c1", "c3", "c5_seed0", "shape07_h16_1_gamma10", "rand03", "rand17", "rand41"]
# (query heads per KV head, KV heads, head_dim, compute units)
LAYOUTS = [(4, 8, 128, 256), (1, 32, 64, 256), (16, 1, 256, 256), (3, 8, 128, 304), (8, 8, 32, 38), (200, 2, 128, 256)]
ROWS_PER_BLOCK = {32: 192, 64: 192, 128: 192, 256: 128}


def _arrays(plan):
    return {name: t.numpy() for name, t in plan.part.items()}


def _attended(a, batch, entries):
    """For each request: the slots its listed scratch rows attend."""
    qo, ql = a["q_offs"].astype(np.int64), a["q_lens"].astype(np.int64)
    assert ql.sum() == len(a["q_entries"])
    row_vnode = np.full(len(a["q_entries"]), -1)
    for v in range(len(qo)):
        assert (row_vnode[qo[v]: qo[v] + ql[v]] == -1).all(), "a scratch row belongs to one vnode"
        row_vnode[qo[v]: qo[v] + ql[v]] = v
    out = []
    for r in range(batch):
        rows = a["req_entries"][a["req_offs"][r]: a["req_offs"][r] + a["req_lens"][r]]
        assert (np.diff(rows) > 0).all() and (a["q_entries"][rows] == r).all()
        parts = [entries[a["kv_offs"][v]: a["kv_offs"][v] + a["kv_lens"][v]] for v in row_vnode[rows]]
        out.append(np.sort(np.concatenate(parts)) if parts else np.zeros(0, np.int32))
    assert a["req_lens"].sum() == len(a["q_entries"])
    return out


def _check_tables(plan, a, group, head_dim, entries):
    table = a["prog_table"].reshape(-1, 4)
    assert len(table) == plan.num_programs and plan.narrow_in_programs == 0
    assert plan.n_wide + plan.n_narrow == len(a["kv_offs"])
    if len(table):
        assert table[0, 0] == 0 and table[-1, 1] == plan.n_wide
        assert (table[1:, 0] == table[:-1, 1]).all() and (table[:, 1] > table[:, 0]).all() and (table[:, 2:] == 0).all()
    # (a request with more query heads per KV head than a pass holds takes several passes)
    rows = a["q_lens"][: plan.n_wide].astype(np.int64) * group
    assert (rows <= max(ROWS_PER_BLOCK[head_dim], group)).all()
    assert a["req_entries"][-32:].tolist() == [-1] * 32
    lists = (a["kv_offs"], a["kv_lens"], a["q_offs"], a["q_lens"], a["q_entries"])
    want = ls.narrow_records(entries, *lists, plan.n_wide, plan.n_narrow)
    assert np.array_equal(a["narrow_table"].reshape(-1, 64), want)
    assert np.array_equal(a["req_table"].reshape(-1, 16), ls.request_records(a["req_entries"], a["req_offs"], a["req_lens"]))
    records = a["prog_records"].reshape(-1, 256)
    assert len(records) == len(table)
    for rec, (v, *_) in zip(records, table):
        n, k = int(a["q_lens"][v]), int(a["kv_lens"][v])
        assert rec[:4].tolist() == [a["kv_offs"][v], k, a["q_offs"][v], n]
        assert rec[4] == int(1 <= n <= 128 and n * group <= ROWS_PER_BLOCK[head_dim])
        if rec[4]:
            reqs = a["q_entries"][a["q_offs"][v]: a["q_offs"][v] + n]
            assert np.array_equal(rec[8:136], reqs[np.minimum(np.arange(128), n - 1)])
            slots = entries[a["kv_offs"][v]: a["kv_offs"][v] + k]
            assert np.array_equal(rec[136:200], slots[np.minimum(np.arange(64), k - 1)])


@pytest.mark.parametrize("layout", LAYOUTS, ids=lambda x: "g%d_h%d_d%d_cu%d" % x)
@pytest.mark.parametrize("name", NAMES)
def test_lists_and_tree_attend_every_path_once(name, layout):
    group, heads, d, cus = layout
    tree, ptrs, batch, plan, _, _ = run_planner(next(c for c in PLANNER_CASES if c["name"] == name))
    slot_map = np.random.default_rng(1).permutation(int(ptrs[-1])).astype(np.int32)
    paths = []
    for node in tree:
        for r in node.requests:
            paths.append((r, np.arange(ptrs[node.id], ptrs[node.id + 1])))
    want = [np.sort(np.concatenate([p for r, p in paths if r == i])) for i in range(batch)]
    lists = (plan.vnode_to_kv_offs, plan.vnode_to_kv_lens, plan.vnode_to_q_offs, plan.vnode_to_q_lens, plan.vnode_to_q_entries)
    entries = np.asarray(plan.vnode_to_kv_entries, dtype=np.int32)
    arranged = ls.arrange(*lists, batch, group, heads, kv_entries=entries, head_dim=d, num_cus=cus)
    a = _arrays(arranged)
    for got, path in zip(_attended(a, batch, entries), want):
        assert np.array_equal(got, path)
    _check_tables(arranged, a, group, d, entries)
    arranged = ls.arrange_tree(_plan_lib.TreeArrays(tree, ptrs), batch, group, heads, head_dim=d, num_cus=cus, kv_slot_map=slot_map)
    a = _arrays(arranged)
    assert a["kv_entries"][-32:].tolist() == [-1] * 32
    for got, path in zip(_attended(a, batch, a["kv_entries"]), want):
        assert np.array_equal(got, np.sort(slot_map[path]))
    _check_tables(arranged, a, group, d, a["kv_entries"])


def test_runs_without_tokens_and_without_requests():
    """An empty run shared by many requests gets scratch rows; an empty launch is an empty schedule."""
    reqs = 40
    s = ls.arrange([0, 0], [0, 300], [0, reqs], [reqs, reqs], list(range(reqs)) * 2, reqs, 4, 8,
                   kv_entries=np.arange(300, dtype=np.int32), num_cus=256)
    a = _arrays(s)
    assert all(np.array_equal(x, np.arange(300)) for x in _attended(a, reqs, np.arange(300)))
    s = ls.arrange([], [], [], [], [], 0, 4, 8, kv_entries=np.zeros(0, np.int32), num_cus=256)
    assert (s.n_wide, s.n_narrow, s.num_programs, s.num_rows) == (0, 0, 0, 0)


@pytest.mark.parametrize("change", [dict(q_entries=[0, 5]), dict(q_entries=[-1, 0]), dict(q_lens=[3]), dict(kv_lens=[11]), dict(kv_offs=[-1])])
def test_lists_out_of_range_are_refused(change):
    lists = dict(kv_offs=[0], kv_lens=[10], q_offs=[0], q_lens=[2], q_entries=[0, 1])
    lists.update(change)
    with pytest.raises(_plan_lib.FastTreePlannerError):
        ls.arrange(*lists.values(), 2, 4, 8, kv_entries=np.arange(10, dtype=np.int32), num_cus=256)
