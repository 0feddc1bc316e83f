"""Host-side planner of FastTree decode attention: cost model, greedy tree splitter,
adaptive parallelism loop and the virtual-node ("vnode") metadata builder.

The planner decides, for every radix-tree node, whether its KV is attended together
with its parent's KV by the node's own requests only (``assignment 1``: the child
absorbs the ancestor KV, a "Q split") or whether the parent keeps one shared pass
for all of its requests and the child adds a separate partial (``assignment 0``: a
"K split" whose price is one more partial to merge).  It then cuts every resulting
(query set, KV run) pair into vnodes of at most ``Q_TILE`` queries and
``KV_SPLIT`` tokens and emits the index arrays the two device kernels walk.

Every list this module produces is element-for-element identical to what the
reference planner produces for the same arguments, including its mutation of the
``FastTreeParams`` object and the lines it prints.

Reference: kernel_bench/fasttree.py:7-27 (parameters), :30-61 (cost model),
:64-96 (greedy splitter), :99-296 (adaptive loop and metadata builder).
"""

from __future__ import annotations

import os
from collections import deque
from dataclasses import dataclass, field
from typing import List, Optional, Sequence, Tuple

import numpy as np

from . import _plan_lib

#: The reference prints its parallelism estimates, final tile/split sizes and the
#: per-phase vnode counts on every call.  Set to False to silence the planner.
VERBOSE = True

#: Which implementation ``fasttree_plan`` runs: "native" (libfasttree_plan.so, the C++ planner
#: behind include/fasttree_plan.h), "python" (this module), or "auto": native when the library is
#: built and the arguments fit its 32-bit interface.  Both produce identical plans.  Plans in launch
#: order are arranged accordingly, by the library's schedule or by ``launch_schedule.block_programs``:
#: the same computation either way, cut and ordered differently.
BACKEND = os.environ.get("FASTTREE_PLANNER", "auto")

#: Number of -1 entries appended to the two entry arrays (kernel_bench/fasttree.py:261-262).
ENTRY_PADDING = 32


class FastTreeParams:
    """Mutable hyper-parameters of the cost model (kernel_bench/fasttree.py:7-27).

    ``fasttree_preparation`` may replace ``TSQs``/``TSKs`` through the setters while
    it adapts the tile sizes; callers that reuse one object across trees see that.
    """

    alpha = 0.66
    beta = 0.33
    gamma = 0.1
    TSQs = [64, 16]
    TSKs = [32, 128]
    kv_group_num = 1

    def set_values(self, alpha, beta, gamma):
        self.alpha, self.beta, self.gamma = alpha, beta, gamma

    def set_kv_group_num(self, kv_group_num):
        self.kv_group_num = kv_group_num

    def set_q_tile_sizes(self, TSQs):
        self.TSQs = TSQs

    def set_kv_tile_sizes(self, TSKs):
        self.TSKs = TSKs


# --------------------------------------------------------------------------------------
# Cost model.  All arithmetic is Python int / IEEE double evaluated left to right,
# exactly as in the reference, so that near-tie decisions come out the same.
# --------------------------------------------------------------------------------------

def _CpadQ(TS, N):
    """Query rows wasted when N queries are tiled by TS (kernel_bench/fasttree.py:30-31).
    Python's floor modulo makes N == 0 cost nothing: (-1) % TS == TS - 1."""
    return TS - ((N - 1) % TS + 1)


def _CpadK(TS, N):
    """KV columns wasted when fewer than one tile of keys exists (fasttree.py:34-35)."""
    return max(0, TS - N)


def _Cmm(nQ, nK, params: FastTreeParams):
    """Padding cost of one (nQ queries x nK keys) contraction (fasttree.py:38-45)."""
    phase = 0 if nQ > params.TSQs[1] else 1
    tsq, tsk = params.TSQs[phase], params.TSKs[phase]
    q_waste = params.alpha * _CpadQ(tsq, nQ) * params.kv_group_num * nK
    k_waste = params.beta * _CpadK(tsk, nK) * nQ * params.kv_group_num
    return q_waste + k_waste


def _Cred(nQl, params: FastTreeParams, lenl, lenv):
    """Cost of merging one more partial per query (fasttree.py:48-49)."""
    return params.gamma * nQl


def _SplitQCost(nQcurr, nQl, lenv, lenl, params: FastTreeParams):
    """Child l leaves with its queries and a private copy of the parent's run
    (fasttree.py:52-53)."""
    return _Cmm(nQcurr - nQl, lenv, params) + _Cmm(nQl, lenl + lenv, params)


def _SplitKCost(nQcurr, nQl, lenl, lenv, params: FastTreeParams):
    """Parent run stays shared; child l is a separate partial (fasttree.py:56-61)."""
    return _Cmm(nQcurr, lenv, params) + _Cmm(nQl, lenl, params) + _Cred(nQl, params, lenl, lenv)


def _tree_heuristic(tree_info, params: FastTreeParams) -> List[int]:
    """Greedy top-down split decision per node (kernel_bench/fasttree.py:64-96).

    Nodes are visited breadth first from node 0, children in ascending id.  While a
    node's children are scanned, the number of queries still attached to the node
    shrinks by every child that took the Q split, and a child that took it carries the
    accumulated run length down to its own children.
    """
    count = len(tree_info)
    children: List[List[int]] = [[] for _ in range(count)]
    for nid in range(1, count):
        children[tree_info[nid].parent].append(nid)
    run_len = [tree_info[nid].seqlen for nid in range(count)]

    assignment = [0] * count
    pending = deque([0])
    while pending:
        v = pending.popleft()
        attached = len(tree_info[v].requests)
        lenv = run_len[v]
        for l in children[v]:
            nQl = len(tree_info[l].requests)
            lenl = run_len[l]
            keep_shared = _SplitKCost(attached, nQl, lenl, lenv, params)
            go_private = _SplitQCost(attached, nQl, lenv, lenl, params)
            if keep_shared > go_private:
                assignment[l] = 1
                attached -= nQl
                run_len[l] = lenl + lenv
            pending.append(l)
    return assignment


# --------------------------------------------------------------------------------------
# Plan: the pure-host result of the planner (python lists / numpy arrays only).
# --------------------------------------------------------------------------------------

@dataclass
class FastTreePlan:
    """Everything ``fasttree_preparation`` computes before it touches a device."""

    vnode_to_kv_entries: np.ndarray          # int32, padded with ENTRY_PADDING x -1
    vnode_to_kv_offs: List[int]
    vnode_to_kv_lens: List[int]
    vnode_to_q_entries: List[int]
    vnode_to_q_offs: List[int]
    vnode_to_q_lens: List[int]
    req_to_vnode_entries: List[int]          # padded with ENTRY_PADDING x -1
    req_to_vnode_offs: List[int]
    req_to_vnode_lens: List[int]
    phase_node_nums: List[int]
    phase_node_offsets: List[int]
    node_assignments: List[int]
    q_tile_sizes: List[int]                  # final Q_TILE_SIZE_PER_PHASE
    kv_split_sizes: List[int]                # final KV_SPLIT_SIZE_PER_PHASE
    parallelisms: List[List[int]] = field(default_factory=list)  # one entry per loop pass

    @property
    def num_rows(self) -> int:
        """Rows of the partial-result scratch (``mid_o.shape[0]``)."""
        return len(self.vnode_to_q_entries)

    @property
    def num_vnodes(self) -> int:
        return len(self.vnode_to_q_lens)


def _say(*args):
    if VERBOSE:
        print(*args)


def _requests_per_node(tree_info, assignment) -> List[List[int]]:
    """Which requests each node's own vnodes serve (fasttree.py:126-141).

    Leaves start with their own request list.  Nodes are then retired in a FIFO order
    (all leaves in ascending id first, a parent as soon as its last child retires); a
    retiring node that did not take the Q split hands *all* requests below it to its
    parent, in retirement order.  The root's parent is -1, which Python resolves to
    the last list element; the reference does the same and nothing depends on it.
    """
    count = len(tree_info)
    served: List[List[int]] = [[] for _ in range(count)]
    fifo = deque()
    for nid in range(count):
        if tree_info[nid].num_children == 0:
            fifo.append(nid)
            served[nid] = list(tree_info[nid].requests)
    waiting = [tree_info[nid].num_children for nid in range(count)]
    while fifo:
        nid = fifo.popleft()
        up = tree_info[nid].parent
        if assignment[nid] == 0 and nid != 0:
            served[up] += tree_info[nid].requests
        waiting[up] -= 1
        if waiting[up] == 0:
            fifo.append(up)
    return served


def _run_chain(tree_info, assignment, nid) -> Tuple[List[int], int]:
    """Nodes whose KV the vnodes of ``nid`` attend, ancestors first, and the run length
    (fasttree.py:149-153, :202-210)."""
    chain = [nid]
    total = tree_info[nid].seqlen
    walk = nid
    while assignment[walk] == 1:
        walk = tree_info[walk].parent
        chain.append(walk)
        total += tree_info[walk].seqlen
    chain.reverse()
    return chain, total


def _estimate_parallelism(tree_info, assignment, served, q_tiles, kv_splits, num_kv_heads):
    """Thread-block count per phase the current plan would launch (fasttree.py:143-159)."""
    blocks = [0, 0]
    for nid, reqs in enumerate(served):
        n = len(reqs)
        if n == 0:
            continue
        _, kv_len = _run_chain(tree_info, assignment, nid)
        phase = 0 if n > q_tiles[1] else 1
        blocks[phase] += ((kv_len - 1) // kv_splits[phase] + 1) * ((n - 1) // q_tiles[phase] + 1)
    return [b * num_kv_heads for b in blocks]


def _fits_native(KV_ptrs, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params) -> bool:
    """The native planner takes tile sizes, split sizes, thresholds and token positions as int32."""
    limit = 2 ** 31 - 1 - ENTRY_PADDING
    small = [*KV_SPLIT_SIZES[:2], *para_threshs1[:2], *para_threshs2[:2], *params.TSQs[:2], *params.TSKs[:2],
             params.kv_group_num]
    return (all(isinstance(x, (int, np.integer)) and 1 <= x <= limit for x in small[:2] + small[6:])
            and all(isinstance(x, (int, np.integer)) and -limit <= x <= limit for x in small[2:6])
            and len(KV_ptrs) > 0 and int(KV_ptrs[-1]) <= limit)


def _native_arrays(tree_info, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1, para_threshs2,
                   params: FastTreeParams, kv_slot_map, arrays=None):
    """The arrays of libfasttree_plan.so."""
    return _plan_lib.plan(tree_info, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1, para_threshs2,
                          params.alpha, params.beta, params.gamma, params.TSQs, params.TSKs, params.kv_group_num,
                          kv_slot_map=kv_slot_map, arrays=arrays)


def _report(r, params: FastTreeParams):
    """Prints the planner's lines and replaces ``params.TSQs`` / ``params.TSKs`` when the second adaptation
    pass fired."""
    L = _plan_lib
    for para in r[L.PARALLELISMS].reshape(-1, 2).tolist():
        _say("parallelisms:", para)
    q_tiles = r[L.Q_TILE_SIZES].tolist()
    if int(r[L.TILES_REPLACED][0]):
        params.set_q_tile_sizes(q_tiles)
        params.set_kv_tile_sizes(r[L.KV_TILE_SIZES].tolist())
    _say(q_tiles)
    _say(r[L.KV_SPLIT_SIZES].tolist())
    nums = r[L.PHASE_NODE_NUMS].tolist()
    _say("Above threshold: ", nums[0])
    _say("Below threshold: ", nums[1])


def _plan_native(tree_info, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1, para_threshs2,
                 params: FastTreeParams, kv_slot_map) -> FastTreePlan:
    """``fasttree_plan`` through libfasttree_plan.so: same result, same printed lines, same
    replacement of ``params.TSQs`` / ``params.TSKs`` when the second adaptation pass fires."""
    L = _plan_lib
    r = _native_arrays(tree_info, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params, kv_slot_map)
    _report(r, params)
    q_tiles, kv_splits, nums = r[L.Q_TILE_SIZES].tolist(), r[L.KV_SPLIT_SIZES].tolist(), r[L.PHASE_NODE_NUMS].tolist()
    return FastTreePlan(
        vnode_to_kv_entries=r[L.KV_ENTRIES],
        vnode_to_kv_offs=r[L.KV_OFFS].tolist(),
        vnode_to_kv_lens=r[L.KV_LENS].tolist(),
        vnode_to_q_entries=r[L.Q_ENTRIES].tolist(),
        vnode_to_q_offs=r[L.Q_OFFS].tolist(),
        vnode_to_q_lens=r[L.Q_LENS].tolist(),
        req_to_vnode_entries=r[L.REQ_ENTRIES].tolist(),
        req_to_vnode_offs=r[L.REQ_OFFS].tolist(),
        req_to_vnode_lens=r[L.REQ_LENS].tolist(),
        phase_node_nums=nums,
        phase_node_offsets=r[L.PHASE_NODE_OFFSETS].tolist(),
        node_assignments=r[L.NODE_ASSIGNMENTS].tolist(),
        q_tile_sizes=list(q_tiles),
        kv_split_sizes=kv_splits,
        parallelisms=r[L.PARALLELISMS].reshape(-1, 2).tolist(),
    )


def _native_chosen(backend, KV_ptrs, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params) -> bool:
    choice = backend or BACKEND
    return choice == "native" or (choice == "auto" and _plan_lib.available() and _fits_native(
        KV_ptrs, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params))


def fasttree_plan(
    tree_info,
    KV_ptrs: Sequence[int],
    batch_size: int,
    num_kv_heads: int,
    KV_SPLIT_SIZES: Sequence[int],
    para_threshs1: Sequence[int],
    para_threshs2: Sequence[int],
    params: FastTreeParams,
    kv_slot_map: Optional[np.ndarray] = None,
    backend: Optional[str] = None,
) -> FastTreePlan:
    """Run the planner and return host-side lists (kernel_bench/fasttree.py:111-262).

    ``backend`` overrides the module's ``BACKEND`` for this call.

    ``kv_slot_map`` (optional, length ``KV_ptrs[-1]``) maps the logical token position
    ``KV_ptrs[node] + t`` to the slot of the KV pool that holds it; without it the pool
    is node-major and the entries are the logical positions themselves, as in the
    reference's bench.
    """
    if _native_chosen(backend, KV_ptrs, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params):
        return _plan_native(tree_info, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1,
                            para_threshs2, params, kv_slot_map)

    count = len(tree_info)
    q_tiles = params.TSQs                       # alias on purpose, as in the reference
    kv_splits = [KV_SPLIT_SIZES[0], KV_SPLIT_SIZES[0]]
    history: List[List[int]] = []

    # Up to three passes: (0) shrink KV splits of under-parallel phases, (1) collapse
    # both phases onto one tile shape if still under-parallel, (2) re-plan with those.
    for attempt in range(3):
        assignment = _tree_heuristic(tree_info, params)
        served = _requests_per_node(tree_info, assignment)
        para = _estimate_parallelism(tree_info, assignment, served, q_tiles, kv_splits, num_kv_heads)
        history.append(para)
        _say("parallelisms:", para)
        if attempt == 0:
            starved = [ph for ph in range(2) if 0 < para[ph] < para_threshs1[ph]]
            for ph in starved:
                kv_splits[ph] = KV_SPLIT_SIZES[1]
            if not starved:
                break
        elif attempt == 1:
            if 0 < para[0] < para_threshs2[0]:
                keep = 1
            elif 0 < para[1] < para_threshs2[1]:
                keep = 0
            else:
                break
            q_tiles = [q_tiles[keep], q_tiles[keep]]
            params.set_q_tile_sizes(q_tiles)
            params.set_kv_tile_sizes([params.TSKs[keep], params.TSKs[keep]])

    _say(q_tiles)
    _say(kv_splits)

    ptrs = np.asarray(KV_ptrs, dtype=np.int64)
    kv_runs: List[np.ndarray] = []
    kv_total = 0
    kv_offs: List[int] = []
    kv_lens: List[int] = []
    q_entries: List[int] = []
    q_offs: List[int] = []
    q_lens: List[int] = []

    q_tile = q_tiles[0]                         # phase-0 tile for every node (fasttree.py:194)
    for nid in range(count):
        reqs = served[nid]
        n = len(reqs)
        if n == 0:
            continue
        kv_split = kv_splits[0 if n > q_tiles[1] else 1]
        chain, kv_len = _run_chain(tree_info, assignment, nid)
        run_base = kv_total
        for member in chain:
            kv_runs.append(np.arange(ptrs[member], ptrs[member + 1], dtype=np.int64))
        kv_total += kv_len

        for kv_lo in range(0, kv_len, kv_split):
            row_base = len(q_entries)
            q_entries.extend(reqs)              # one scratch row per (request, kv split)
            span = min(kv_lo + kv_split, kv_len) - kv_lo
            for q_lo in range(0, n, q_tile):
                kv_offs.append(run_base + kv_lo)
                kv_lens.append(span)
                q_offs.append(row_base + q_lo)
                q_lens.append(min(q_lo + q_tile, n) - q_lo)

    rows_of_req: List[List[int]] = [[] for _ in range(batch_size)]
    for row, req in enumerate(q_entries):
        rows_of_req[req].append(row)
    req_offs: List[int] = []
    req_lens: List[int] = []
    req_entries: List[int] = []
    for rows in rows_of_req:
        req_offs.append(len(req_entries))
        req_lens.append(len(rows))
        req_entries.extend(rows)

    # Stable partition: vnodes wider than the small tile run first (phase 0).
    small = q_tiles[1]
    wide = [v for v, n in enumerate(q_lens) if n > small]
    narrow = [v for v, n in enumerate(q_lens) if n <= small]
    _say("Above threshold: ", len(wide))
    _say("Below threshold: ", len(narrow))
    order = wide + narrow

    logical = np.concatenate(kv_runs) if kv_runs else np.zeros(0, dtype=np.int64)
    if kv_slot_map is not None:
        logical = np.asarray(kv_slot_map)[logical]
    padded = np.concatenate([logical, np.full(ENTRY_PADDING, -1, dtype=np.int64)]).astype(np.int32)

    return FastTreePlan(
        vnode_to_kv_entries=padded,
        vnode_to_kv_offs=[kv_offs[v] for v in order],
        vnode_to_kv_lens=[kv_lens[v] for v in order],
        vnode_to_q_entries=q_entries,
        vnode_to_q_offs=[q_offs[v] for v in order],
        vnode_to_q_lens=[q_lens[v] for v in order],
        req_to_vnode_entries=req_entries + [-1] * ENTRY_PADDING,
        req_to_vnode_offs=req_offs,
        req_to_vnode_lens=req_lens,
        phase_node_nums=[len(wide), len(narrow)],
        phase_node_offsets=[0, len(wide)],
        node_assignments=assignment,
        q_tile_sizes=list(q_tiles),
        kv_split_sizes=kv_splits,
        parallelisms=history,
    )


class PlanBuffers:
    """Device buffers for :func:`fasttree_preparation`, allocated once at stated maxima and
    filled in place by every call that is given them: a serving loop re-plans whenever its batch
    changes, and neither the nine index arrays nor the fp32 scratch should be allocated anew each
    time (the reference says so of its own bench code, kernel_bench/fasttree.py:264, and
    pre-allocates in its plugin, metadata.py:40-58).

    ``max_kv_entries`` bounds the flat KV index list (unique tokens plus what merged chains
    replicate, plus the 32 padding entries), ``max_rows`` the scratch rows (one per request and
    KV split), ``max_vnodes`` the vnodes, ``max_batch_size`` the requests.

    Launch-order plans cut long runs finer than the KV splits, into pieces of at least 128 tokens: for
    any of them ``sum(tokens of the path // 128 + nodes of the path)`` over the requests is enough for
    ``max_rows`` and for ``max_vnodes``, and the sum of the paths' tokens plus 32 for
    ``max_kv_entries``.  In smaller buffers the plan is made from the planner's own lists, cut only where the
    buffers hold it: slower to make and to decode with, but the same computation.
    """

    def __init__(self, num_qo_heads, head_dim, max_kv_entries, max_rows, max_vnodes, max_batch_size, device="cuda"):
        import torch

        def ints(n):
            with torch.inference_mode(False):   # (tensors whose writes are counted: launch_schedule.times_written)
                return torch.empty(int(n), dtype=torch.int32, device=device)

        self.device = device
        self.vnode_to_kv_entries = ints(max_kv_entries)
        self.vnode_to_kv_offs, self.vnode_to_kv_lens = ints(max_vnodes), ints(max_vnodes)
        self.vnode_to_q_entries = ints(max_rows)
        self.vnode_to_q_offs, self.vnode_to_q_lens = ints(max_vnodes), ints(max_vnodes)
        self.req_to_vnode_entries = ints(max_rows + 32)
        self.req_to_vnode_offs, self.req_to_vnode_lens = ints(max_batch_size), ints(max_batch_size)
        self.prog_table = ints(4 * max_vnodes)
        self.narrow_table = ints(64 * max_vnodes)     # (launch_schedule.NARROW_RECORD entries per narrow vnode)
        self.req_table = ints(16 * max_batch_size)    # (launch_schedule.REQUEST_RECORD entries per request)
        self.prog_records = ints(256 * max_vnodes)    # (launch_schedule.PROGRAM_RECORD entries per program)
        self.wave_records = ints(64 * 8 * min(int(max_vnodes), 512))   # (of plans of whole paths: a vnode per unit at most)
        self.mid_o = torch.empty((int(max_rows), num_qo_heads, head_dim), dtype=torch.float32, device=device)
        self.mid_lse = torch.empty((int(max_rows), num_qo_heads), dtype=torch.float32, device=device)

    def fill(self, name, values):
        """Copies ``values`` into the front of buffer ``name`` and returns that part of it."""
        import torch

        host = values if isinstance(values, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(np.asarray(values, dtype=np.int32)))
        dst = getattr(self, name)
        if host.numel() > dst.numel():
            raise ValueError(f"{name}: {host.numel()} entries do not fit the {dst.numel()} that were allocated")
        part = dst[: host.numel()]
        # (tensors handed in lie in pinned memory: their copies are queued, and :func:`wait_for_copies` waits for all of them)
        part.copy_(host, non_blocking=host is values)
        return part


def wait_for_copies(device):
    """Waits for the copies of a plan that were queued on the current stream: a plan may be used on any
    stream once the call that made it has returned."""
    import torch

    if _on_gpu(device):
        torch.cuda.current_stream(device).synchronize()


def place_plan(kv_entries, vnodes, q_entries, per_request, phase_nums, phase_offs,
               batch_size, num_qo_heads, num_kv_heads, head_dim, *,
               device="cuda", launch_order=False, buffers=None, num_cus=None):
    """The 13 arguments ``fasttree_decode`` takes after the output tensor, from vnode lists on the
    host: ``kv_entries`` (flat pool slots), ``vnodes = (kv_offs, kv_lens, q_offs, q_lens)``,
    ``q_entries`` (request of every scratch row), ``per_request = (entries, offs, lens)`` (scratch
    rows of every request; ignored with ``launch_order``, which derives its own), the two phase
    lists.  Places the nine int32 arrays and the two fp32 partial-result buffers on ``device`` (into
    ``buffers`` if given).  With ``launch_order`` the lists are first arranged as block programs
    (:func:`launch_schedule.block_programs`) for ``num_cus`` compute units, and ``phase_node_nums``
    comes back as a list that also carries the program table and the host-written records."""
    import torch

    names = ("vnode_to_kv_entries", "vnode_to_kv_offs", "vnode_to_kv_lens", "vnode_to_q_entries", "vnode_to_q_offs",
             "vnode_to_q_lens", "req_to_vnode_entries", "req_to_vnode_offs", "req_to_vnode_lens")

    def place(name, values):
        if buffers is not None:
            return buffers.fill(name, values)
        host = torch.from_numpy(np.ascontiguousarray(np.asarray(values, dtype=np.int32)))
        return host.to(device)

    if launch_order:
        from . import launch_schedule

        kv_entries = np.ascontiguousarray(np.asarray(kv_entries, dtype=np.int32))
        if num_cus is None:
            num_cus = launch_schedule.compute_units(device)
        lists = (*vnodes, q_entries, batch_size, max(1, num_qo_heads // num_kv_heads), num_kv_heads)
        kw = dict(kv_entries=kv_entries, head_dim=head_dim, num_cus=num_cus, pin=_on_gpu(device))
        plan = launch_schedule.arrange(*lists, **kw) if buffers is None else launch_schedule.arrange_within(
            buffers.mid_o.shape[0], buffers.vnode_to_kv_offs.numel(), *lists, **kw)
        return _place_arranged(plan, place("vnode_to_kv_entries", kv_entries), num_qo_heads, head_dim, device, buffers)
    rows = int(len(np.asarray(q_entries).reshape(-1)))
    placed = [place(name, values) for name, values in zip(names, (kv_entries, vnodes[0], vnodes[1], q_entries, vnodes[2], vnodes[3],
                                                                 *per_request))]
    return (*placed, *_scratch(rows, num_qo_heads, head_dim, device, buffers), phase_nums, phase_offs)


def _on_gpu(device):
    import torch

    return torch.device(device).type == "cuda"


def _scratch(rows, num_qo_heads, head_dim, device, buffers):
    """The two fp32 partial-result buffers of a plan."""
    import torch

    if buffers is not None:
        if rows > buffers.mid_o.shape[0] or buffers.mid_o.shape[1:] != (num_qo_heads, head_dim):
            raise ValueError(f"the scratch of the buffers ({tuple(buffers.mid_o.shape)}) does not hold "
                             f"{rows} rows of {num_qo_heads} x {head_dim}")
        return buffers.mid_o[:rows], buffers.mid_lse[:rows]
    return (torch.empty((rows, num_qo_heads, head_dim), dtype=torch.float32, device=device),
            torch.empty((rows, num_qo_heads), dtype=torch.float32, device=device))


def _place_arranged(plan, kv_entries, num_qo_heads, head_dim, device, buffers):
    """The decode call's arguments for a :class:`launch_schedule.Arranged` plan; ``kv_entries``: the flat
    slot list on the device, or None where it is part of the plan."""
    import torch

    from . import launch_schedule
    from .launch_schedule import LaunchPhases

    if buffers is not None:
        part = {name: buffers.fill(full, plan.part[name]) for name, full in _BUFFER_OF.items()
                if name in plan.part and (name != "wave_records" or plan.where[name][1] > 0)}
        wait_for_copies(buffers.device)
    else:
        # one copy for the whole plan; the arrays are views of it
        with torch.inference_mode(False):
            whole = plan.packed.to(device)
        part = {name: whole[lo: lo + n] for name, (lo, n) in plan.where.items()}
    nums = LaunchPhases([plan.n_wide, plan.n_narrow])
    nums.modelled_us, nums.num_cus, nums.block_slots = plan.modelled_us, plan.num_cus, plan.block_slots
    if plan.num_programs > 0:
        nums.prog_table = part["prog_table"]
        nums.num_programs = plan.num_programs
        nums.narrow_in_programs = plan.narrow_in_programs
        if head_dim >= 32 and launch_schedule.USE_PROGRAM_RECORDS:
            nums.prog_records = part["prog_records"]
    if plan.n_narrow > 0 and head_dim >= 32 and launch_schedule.USE_NARROW_RECORDS:
        nums.narrow_table = part["narrow_table"]
    if head_dim >= 32 and launch_schedule.USE_REQUEST_RECORDS:
        nums.req_table = part["req_table"]
    if plan.where.get("wave_records", (0, 0))[1] > 0 and launch_schedule.USE_NARROW_RECORDS:
        nums.wave_records = part["wave_records"]
    return (part["kv_entries"] if kv_entries is None else kv_entries, part["kv_offs"], part["kv_lens"], part["q_entries"], part["q_offs"],
            part["q_lens"], part["req_entries"], part["req_offs"], part["req_lens"],
            *_scratch(plan.num_rows, num_qo_heads, head_dim, device, buffers), nums, [0, plan.n_wide])


#: The buffer of :class:`PlanBuffers` each array of an arranged plan goes to.
_BUFFER_OF = {
    "kv_entries": "vnode_to_kv_entries", "kv_offs": "vnode_to_kv_offs", "kv_lens": "vnode_to_kv_lens", "q_entries": "vnode_to_q_entries", "q_offs": "vnode_to_q_offs",
    "q_lens": "vnode_to_q_lens", "req_entries": "req_to_vnode_entries", "req_offs": "req_to_vnode_offs", "req_lens": "req_to_vnode_lens",
    "prog_table": "prog_table", "narrow_table": "narrow_table", "prog_records": "prog_records", "req_table": "req_table",
    "wave_records": "wave_records",
}


#: The cost model's parameters as :class:`FastTreeParams` and the reference's benchmark have them.
_STOCK = (FastTreeParams.alpha, FastTreeParams.beta, FastTreeParams.gamma)


def fasttree_preparation(
    tree_info,
    KV_ptrs,
    batch_size,
    num_qo_heads,
    num_kv_heads,
    head_dim,
    KV_SPLIT_SIZES,
    para_threshs1,
    para_threshs2,
    params: FastTreeParams,
    *,
    device="cuda",
    kv_slot_map=None,
    launch_order=False,
    buffers=None,
    num_cus=None,
):
    """Drop-in for kernel_bench/fasttree.py:99-296: plan on the host, then place the nine
    int32 index arrays and the two fp32 partial-result buffers on ``device``.

    Returns ``((vnode_to_kv_entries, vnode_to_kv_offs, vnode_to_kv_lens,
    vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, req_to_vnode_entries,
    req_to_vnode_offs, req_to_vnode_lens, mid_o, mid_lse, phase_node_nums,
    phase_node_offsets), node_assignments)``: element for element the reference's lists.

    The keyword-only arguments do not exist in the reference: ``device`` defaults to the
    reference's hard-wired "cuda"; ``kv_slot_map`` is described in :func:`fasttree_plan`; with
    ``buffers`` (a :class:`PlanBuffers`) nothing is allocated on the device: the arrays are
    written into its buffers and the returned tensors are their leading parts.  With
    ``launch_order=True`` the lists come back arranged for an MI355X instead
    (:func:`launch_schedule.block_programs`: the same computation as block programs,
    with scratch rows and per-request lists of its own); ``phase_node_nums`` is then a list that
    also carries the program table, which ``fasttree_decode`` picks up; the programs are laid out
    for ``num_cus`` compute units (None: those ``device`` reports, 256 where it is not a GPU).  With the
    cost model's parameters as :class:`FastTreeParams` has them, which nodes attend their ancestors' tokens
    with their own is then decided by what it makes this device move, or by the reference's padding costs
    where that launch is modelled clearly shorter (include/fasttree_schedule.h); parameters set to
    anything else are obeyed.  The assignments returned are those of the plan returned.
    """
    from . import launch_schedule

    if (launch_order and (params.alpha, params.beta, params.gamma) == _STOCK
            and _native_chosen(None, KV_ptrs, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params)):
        L = _plan_lib
        tree = L.TreeArrays(tree_info, KV_ptrs)
        r = _native_arrays(tree, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1, para_threshs2, params, kv_slot_map,
                           arrays=(L.NODE_ASSIGNMENTS, L.PARALLELISMS, L.PHASE_NODE_NUMS, L.Q_TILE_SIZES, L.KV_SPLIT_SIZES,
                                   L.KV_TILE_SIZES, L.TILES_REPLACED))
        arranged = launch_schedule.arrange_tree(
            tree, batch_size, max(1, num_qo_heads // num_kv_heads), num_kv_heads, head_dim=head_dim,
            num_cus=launch_schedule.compute_units(device) if num_cus is None else num_cus, kv_slot_map=kv_slot_map, pin=_on_gpu(device),
            decided=r[L.NODE_ASSIGNMENTS], most_kv_entries=None if buffers is None else buffers.vnode_to_kv_entries.numel())
        # (buffers sized for the planner's own lists may not hold this plan: they get one made from those lists)
        if buffers is None or arranged.fits(
                buffers.mid_o.shape[0], buffers.vnode_to_kv_offs.numel(), buffers.vnode_to_kv_entries.numel(), buffers.wave_records.numel()):
            _report(r, params)
            assignments = arranged.part["node_assignments"].tolist()
            return _place_arranged(arranged, None, num_qo_heads, head_dim, device, buffers), assignments

    plan = fasttree_plan(
        tree_info, KV_ptrs, batch_size, num_kv_heads,
        KV_SPLIT_SIZES, para_threshs1, para_threshs2, params, kv_slot_map=kv_slot_map,
    )

    aux = place_plan(
        plan.vnode_to_kv_entries,
        (plan.vnode_to_kv_offs, plan.vnode_to_kv_lens, plan.vnode_to_q_offs, plan.vnode_to_q_lens),
        plan.vnode_to_q_entries,
        (plan.req_to_vnode_entries, plan.req_to_vnode_offs, plan.req_to_vnode_lens),
        list(plan.phase_node_nums), list(plan.phase_node_offsets),
        batch_size, num_qo_heads, num_kv_heads, head_dim,
        device=device, launch_order=launch_order, buffers=buffers, num_cus=num_cus,
    )
    return aux, plan.node_assignments
