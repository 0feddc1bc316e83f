"""ctypes binding of libfasttree_plan.so: the native host planner (include/fasttree_plan.h) and the
launch schedule (include/fasttree_schedule.h)."""

from __future__ import annotations

import ctypes
import os

import numpy as np

LIB_NAME = "libfasttree_plan.so"
LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)

# order of the result arrays (enum in include/fasttree_plan.h)
(KV_ENTRIES, KV_OFFS, KV_LENS, Q_ENTRIES, Q_OFFS, Q_LENS, REQ_ENTRIES, REQ_OFFS, REQ_LENS, NODE_ASSIGNMENTS,
 PARALLELISMS, PHASE_NODE_NUMS, PHASE_NODE_OFFSETS, Q_TILE_SIZES, KV_SPLIT_SIZES, KV_TILE_SIZES, TILES_REPLACED,
 N_ARRAYS) = range(18)

_ERRORS = {-1: "null pointer", -2: "invalid argument", -3: "out of memory", -4: "incomplete schedule"}

_P32 = ctypes.POINTER(ctypes.c_int32)
_P64 = ctypes.POINTER(ctypes.c_int64)
SIGNATURES = {
    "ft_plan_version": (ctypes.c_char_p, []),
    "ft_plan_create": (ctypes.c_int, [ctypes.c_int, _P32, _P32, _P32, _P64, _P32, _P64, ctypes.c_int, ctypes.c_int,
                                      _P32, _P32, _P32, ctypes.c_double, ctypes.c_double, ctypes.c_double, _P32, _P32,
                                      ctypes.c_int, _P32, ctypes.c_int64, ctypes.POINTER(ctypes.c_void_p)]),
    "ft_plan_size": (ctypes.c_int64, [ctypes.c_void_p, ctypes.c_int]),
    "ft_plan_copy": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, _P32, ctypes.c_int64]),
    "ft_plan_destroy": (None, [ctypes.c_void_p]),
}

# order of a schedule's arrays (enum in include/fasttree_schedule.h)
SCHEDULE_ARRAYS = ("kv_offs", "kv_lens", "q_entries", "q_offs", "q_lens", "req_entries", "req_offs", "req_lens", "prog_table",
                   "narrow_table", "prog_records", "req_table", "counts", "kv_entries", "node_assignments", "wave_records")
SCHEDULE_SIGNATURES = {
    "ft_schedule_create": (ctypes.c_int, [ctypes.c_int64, _P32, _P32, _P32, _P32, ctypes.c_int64, _P32, ctypes.c_int64, _P32]
                           + [ctypes.c_int] * 5 + [ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_void_p)]),
    "ft_schedule_tree": (ctypes.c_int, [ctypes.c_int, _P32, _P32, _P32, _P64, _P32, _P64, _P32, ctypes.c_int64]
                         + [ctypes.c_int] * 5 + [ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_void_p)]),
    "ft_schedule_tree_weighed": (ctypes.c_int, [ctypes.c_int, _P32, _P32, _P32, _P64, _P32, _P64, _P32, ctypes.c_int64, _P32]
                                 + [ctypes.c_int] * 5 + [ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_void_p)]),
    "ft_schedule_tree_within": (ctypes.c_int, [ctypes.c_int, _P32, _P32, _P32, _P64, _P32, _P64, _P32, ctypes.c_int64, _P32, ctypes.c_int64]
                                + [ctypes.c_int] * 5 + [ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_void_p)]),
    "ft_schedule_size": (ctypes.c_int64, [ctypes.c_void_p, ctypes.c_int]),
    "ft_schedule_pack": (ctypes.c_int, [ctypes.c_void_p, _P32, ctypes.c_int64, _P64, _P64]),
    "ft_schedule_destroy": (None, [ctypes.c_void_p]),
}

_lib = None


class FastTreePlannerError(RuntimeError):
    pass


def available() -> bool:
    return os.path.exists(LIB_PATH)


def load():
    global _lib
    if _lib is None:
        if not available():
            raise FastTreePlannerError(
                f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'`")
        lib = ctypes.CDLL(LIB_PATH)
        for name, (restype, argtypes) in [*SIGNATURES.items(), *SCHEDULE_SIGNATURES.items()]:
            fn = getattr(lib, name)
            fn.restype, fn.argtypes = restype, argtypes
        _lib = lib
    return _lib


def _i32(values):
    return np.ascontiguousarray(np.asarray(values, dtype=np.int32))


def _ptr32(a):
    return a.ctypes.data_as(_P32)


class TreeArrays:
    """A tree as the arrays the native entry points take."""

    def __init__(self, tree_info, KV_ptrs):
        self.n = n = len(tree_info)
        self.parent = _i32([t.parent for t in tree_info])
        self.seqlen = _i32([t.seqlen for t in tree_info])
        self.children = _i32([t.num_children for t in tree_info])
        counts = np.fromiter((len(t.requests) for t in tree_info), dtype=np.int64, count=n)
        self.req_offs = np.zeros(n + 1, dtype=np.int64)
        np.cumsum(counts, out=self.req_offs[1:])
        self.req_ids = _i32([r for t in tree_info for r in t.requests]) if self.req_offs[-1] else np.zeros(1, dtype=np.int32)
        self.ptrs = np.ascontiguousarray(np.asarray(KV_ptrs, dtype=np.int64))
        if self.ptrs.shape[0] != n + 1:
            raise FastTreePlannerError("KV_ptrs must have one entry per node plus one")


def plan(tree_info, KV_ptrs, batch_size, num_kv_heads, KV_SPLIT_SIZES, para_threshs1, para_threshs2,
         alpha, beta, gamma, TSQs, TSKs, kv_group_num, kv_slot_map=None, arrays=None):
    """Runs the native planner; returns the list of result arrays (numpy int32), indexed by the
    constants above.  ``tree_info``: the nodes, or a :class:`TreeArrays` made from them; ``arrays``: the
    constants of the arrays wanted (None: all; the others come back as None)."""
    lib = load()
    tree = tree_info if isinstance(tree_info, TreeArrays) else TreeArrays(tree_info, KV_ptrs)
    n, parent, seqlen, children, req_offs, req_ids, ptrs = (
        tree.n, tree.parent, tree.seqlen, tree.children, tree.req_offs, tree.req_ids, tree.ptrs)
    splits, th1, th2 = _i32(list(KV_SPLIT_SIZES)[:2]), _i32(list(para_threshs1)[:2]), _i32(list(para_threshs2)[:2])
    tsq, tsk = _i32(list(TSQs)[:2]), _i32(list(TSKs)[:2])
    slot_map = None if kv_slot_map is None else _i32(kv_slot_map)
    handle = ctypes.c_void_p()
    rc = lib.ft_plan_create(
        n, _ptr32(parent), _ptr32(seqlen), _ptr32(children), req_offs.ctypes.data_as(_P64), _ptr32(req_ids),
        ptrs.ctypes.data_as(_P64), int(batch_size), int(num_kv_heads), _ptr32(splits), _ptr32(th1), _ptr32(th2),
        float(alpha), float(beta), float(gamma), _ptr32(tsq), _ptr32(tsk), int(kv_group_num),
        None if slot_map is None else _ptr32(slot_map), 0 if slot_map is None else slot_map.shape[0],
        ctypes.byref(handle))
    if rc != 0:
        raise FastTreePlannerError(f"ft_plan_create failed: {_ERRORS.get(rc, rc)}")
    try:
        out = []
        for which in range(N_ARRAYS):
            if arrays is not None and which not in arrays:
                out.append(None)
                continue
            size = lib.ft_plan_size(handle, which)
            a = np.empty(max(size, 0), dtype=np.int32)
            rc = lib.ft_plan_copy(handle, which, _ptr32(a) if size else None, size)
            if rc != 0:
                raise FastTreePlannerError(f"ft_plan_copy failed: {_ERRORS.get(rc, rc)}")
            out.append(a)
        return out
    finally:
        lib.ft_plan_destroy(handle)


def schedule(kv_offs, kv_lens, q_offs, q_lens, q_entries, kv_entries, batch_size, group, num_kv_heads, head_dim, num_cus, allocate):
    """Runs the native launch schedule on vnode lists (``kv_entries`` may be None: no records then).
    ``allocate(n)`` gives the int32 numpy array of at least ``n`` entries that the result is packed into.
    Returns ``(packed, {array name: (first entry, entries)}, modelled microseconds)``."""
    lib = load()
    lists = [_i32(x).reshape(-1) for x in (kv_offs, kv_lens, q_offs, q_lens, q_entries)]
    entries = None if kv_entries is None else _i32(kv_entries).reshape(-1)
    us, handle = ctypes.c_double(), ctypes.c_void_p()
    rc = lib.ft_schedule_create(
        lists[0].shape[0], *(_ptr32(x) for x in lists[:4]), lists[4].shape[0], _ptr32(lists[4]),
        0 if entries is None else entries.shape[0], None if entries is None else _ptr32(entries),
        int(batch_size), int(group), int(num_kv_heads), int(head_dim), int(num_cus), ctypes.byref(us), ctypes.byref(handle))
    return _packed(lib, rc, "ft_schedule_create", handle, us, allocate)


def schedule_tree(tree, batch_size, group, num_kv_heads, head_dim, num_cus, kv_slot_map, allocate, decided=None, most_kv_entries=None):
    """The same from a :class:`TreeArrays` (the array "kv_entries" holds the flat slot list, "node_assignments"
    which nodes attend their parents' runs with their own); ``decided``: a second decision on that to weigh; ``most_kv_entries``: entries that the
    caller's slot list has room for (None: any number)."""
    lib = load()
    slot_map = None if kv_slot_map is None else _i32(kv_slot_map)
    us, handle = ctypes.c_double(), ctypes.c_void_p()
    other = None if decided is None else _i32(decided)
    if other is not None and other.shape[0] != tree.n:
        raise FastTreePlannerError("one decision per node")
    rc = lib.ft_schedule_tree_within(
        tree.n, _ptr32(tree.parent), _ptr32(tree.seqlen), _ptr32(tree.children), tree.req_offs.ctypes.data_as(_P64), _ptr32(tree.req_ids),
        tree.ptrs.ctypes.data_as(_P64), None if slot_map is None else _ptr32(slot_map), 0 if slot_map is None else slot_map.shape[0],
        None if other is None else _ptr32(other), -1 if most_kv_entries is None else int(most_kv_entries),
        int(batch_size), int(group), int(num_kv_heads), int(head_dim), int(num_cus), ctypes.byref(us), ctypes.byref(handle))
    return _packed(lib, rc, "ft_schedule_tree", handle, us, allocate)


def _packed(lib, rc, what, handle, us, allocate):
    if rc != 0:
        raise FastTreePlannerError(f"{what} failed: {_ERRORS.get(rc, rc)}")
    try:
        offsets, total = (ctypes.c_int64 * len(SCHEDULE_ARRAYS))(), ctypes.c_int64()
        lib.ft_schedule_pack(handle, None, 0, offsets, ctypes.byref(total))
        packed = allocate(total.value)
        rc = lib.ft_schedule_pack(handle, _ptr32(packed), packed.shape[0], offsets, ctypes.byref(total))
        if rc != 0:
            raise FastTreePlannerError(f"ft_schedule_pack failed: {_ERRORS.get(rc, rc)}")
        where = {name: (offsets[i], lib.ft_schedule_size(handle, i)) for i, name in enumerate(SCHEDULE_ARRAYS)}
        return packed, where, us.value
    finally:
        lib.ft_schedule_destroy(handle)
