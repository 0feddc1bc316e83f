"""What a user of this library has it do: tree decode calls over the sizes, head layouts and types the
library is used with, planning for a tree that changed, and the decode forwards of a serving loop.

Three kinds of case:

* ``decode``: one ``fasttree_decode`` call on a plan that is in hand.  A model runs one such call per
  layer on one plan, so the plan is made by ``prepare``.  ``lists`` is "arranged" for plans made with
  ``fasttree_preparation(launch_order=True)`` and the settings for this part, "reference" for a program
  that only changed its import: default arguments, the reference's settings and list order.
* ``replan``: the tree changed (branches were added or dropped), so ``fasttree_preparation`` runs into
  buffers allocated beforehand and every layer decodes once on the new plan.
* ``serve``: the serving plugin between two plans: ``plan_or_step`` before every forward (one plan over
  the radix cache, in-place steps after it), then in every layer the hook that stores the step's K/V
  rows and decodes.

Trees are level-regular (``sizes`` nodes of ``lens`` tokens per level, each length varied by up to
``spread`` of itself) or irregular (``irregular`` is the generator's seed).  The pool has page size 1 and
shuffled slots, values are N(0, 1).
"""

import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("fasttree-artifact_amd"))

from fasttree_hip import planner  # noqa: E402
from fasttree_hip import PlanBuffers, FastTreeParams, fasttree_decode, fasttree_preparation  # noqa: E402
from fasttree_hip.inputs import make_decode_inputs  # noqa: E402
from fasttree_hip.kv_tree import assign_requests, generate_irregular_tree, generate_tree, nodes_from_rows  # noqa: E402
from fasttree_hip.sglang_plugin import FastTreeMetadata, decode_forward_fasttree, plan_or_step  # noqa: E402

planner.VERBOSE = False

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
#: Planner settings that go with each list order: the reference benchmark's, and the ones for 256 compute units.
SETTINGS = {
    "reference": dict(kv_splits=(1024, 128), thr1=(132, 528), thr2=(132, 132), launch_order=False),
    "arranged": dict(kv_splits=(1024, 256), thr1=(256, 1024), thr2=(256, 256), launch_order=True),
}
#: Forwards the serving loop makes on one plan.
FORWARDS = 10


def _decode(name, sizes, lens, hq, hkv, d=128, dtype="fp16", lists="arranged", spread=0.0, tree_seed=0):
    case = dict(kind="decode", sizes=sizes, lens=lens, hq=hq, hkv=hkv, d=d, dtype=dtype, lists=lists, spread=spread, tree_seed=tree_seed)
    return dict(case, name=name) if name else case


_SERVE = dict(kind="serve", system=2048, groups=8, group_len=512, per_group=16, prompt=128, output=48, layers=16, hq=32, hkv=8, d=128,
              dtype="fp16")


def listed():
    return [
        # a few samples of one short prompt: latency and launches are all there is
        _decode("few_short", "1,4", "384,24", 32, 8),
        # parallel sampling without grouped heads
        _decode("sampling_mha", "1,16", "1024,128", 32, 32),
        # one long document, a few questions on it
        _decode("long_document", "1,8", "32768,512", 64, 8, dtype="bf16"),
        # long shared prefix, medium batch
        _decode("shared_prefix", "1,64", "4096,256", 32, 8),
        # system prompt, examples, questions: the headline tree, in both list orders
        _decode("three_level", "1,10,400", "4000,400,40", 32, 8),
        _decode("three_level_drop_in", "1,10,400", "4000,400,40", 32, 8, lists="reference"),
        # ragged lengths, a group of three query heads, 64-dim heads, bf16
        _decode("ragged_small_heads", "1,7,111", "1531,213,57", 24, 8, d=64, dtype="bf16", spread=0.5, tree_seed=3),
        # one KV head for 16 query heads, large heads
        _decode("multi_query_large_heads", "1,16,64", "1024,256,32", 16, 1, d=256, dtype="bf16", spread=0.25, tree_seed=4),
        # deep irregular tree, several hundred requests
        dict(kind="decode", irregular=0, hq=64, hkv=8, d=128, dtype="fp16", lists="arranged", name="irregular"),
        # short system prompt, a large batch of long private contexts: the largest pool
        _decode("large_batch", "1,2048", "512,1024", 32, 8, dtype="bf16"),
        # the headline tree planned anew before every token of a model of 16 layers
        dict(_decode("", "1,10,400", "4000,400,40", 32, 8), kind="replan", layers=16, name="replan_three_level"),
        # a serving batch between two plans: one system prompt, eight tasks, 128 requests
        dict(_SERVE, name="serve_128_requests"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: Most bytes and operations of a drawn decode case and of a drawn replan case: those of the largest listed ones.
MOST = {"decode": (8.6e9, 1.3e11), "replan": (1.6e9, 4.6e11)}


def _fits(case, bytes_, flops):
    w = work(case)
    return w["bytes"] <= bytes_ and w["flops"] <= flops


def draw(rng):
    kind = rng.choices(["decode", "replan", "serve"], [8, 1, 1])[0]
    if kind == "serve":
        most = work(_SERVE)
        while True:
            case = dict(kind="serve", system=_log_int(rng, 64, 4096), groups=rng.randint(1, 12), group_len=_log_int(rng, 16, 1024),
                        per_group=rng.randint(1, 16), prompt=_log_int(rng, 8, 384), output=_log_int(rng, 1, 96), layers=rng.randint(4, 16),
                        hq=32, hkv=8, d=128, dtype=rng.choice(["fp16", "bf16"]))
            if _serve_tokens(case)[1] <= _serve_tokens(_SERVE)[1] and _fits(case, most["bytes"], most["flops"]):
                return case
    hq, hkv = rng.choice([(32, 8), (32, 8), (64, 8), (32, 32), (16, 1), (24, 8)])
    d = rng.choice([128, 128, 128, 128, 64, 256])
    dtype = rng.choice(["fp16", "bf16"])
    lists = rng.choice(["arranged", "arranged", "reference"])
    if kind == "decode" and rng.random() < 0.15:
        case = dict(kind="decode", irregular=rng.randint(1, 99), hq=hq, hkv=hkv, d=d, dtype=dtype, lists=lists)
        if _fits(case, *MOST["decode"]):
            return case
    depth = rng.randint(2, 4)
    leaves = _log_int(rng, 2, 2048 if kind == "decode" else 400)
    inner = leaves if kind == "decode" else max(1, leaves // 8)
    sizes = sorted([1] + [_log_int(rng, 1, inner) for _ in range(depth - 2)]) + [leaves]
    lens = [_log_int(rng, 32, 16384)] + [_log_int(rng, 8, 1024) for _ in range(depth - 1)]
    spread = round(rng.uniform(0.0, 0.6), 2)
    seed = rng.randint(0, 10**6)
    layers = rng.randint(4, 16)
    while True:
        case = _decode("", ",".join(map(str, sizes)), ",".join(map(str, lens)), hq, hkv, d, dtype, lists, spread, seed)
        if kind == "replan":
            case.update(kind="replan", layers=layers)
        if _fits(case, *MOST[kind]):
            return case
        lens = [max(8, int(0.7 * n)) for n in lens]
        sizes = [max(1, int(0.9 * n)) for n in sizes]


def _tree(case):
    if "irregular" in case:
        rows = generate_irregular_tree(case["irregular"])
    else:
        rows = generate_tree([int(x) for x in case["sizes"].split(",")], [int(x) for x in case["lens"].split(",")])
        rng = random.Random(case["tree_seed"])
        if case["spread"] > 0:
            rows = [[up, i, max(1, int(round(n * rng.uniform(1 - case["spread"], 1 + case["spread"])))), kids] for up, i, n, kids in rows]
    return nodes_from_rows(rows)


# ---- decode and replan ------------------------------------------------------------------

def _plan(case, tree, ptrs, batch, slot_map, buffers=None):
    """The plan as a user's program makes it; returns the decode call's trailing arguments."""
    g = case["hq"] // case["hkv"]
    s = SETTINGS[case["lists"]]
    params = FastTreeParams()
    params.set_values(0.66, 0.33, 0.1)
    params.set_q_tile_sizes([max(1, 64 // g), max(1, 16 // g)])
    params.set_kv_tile_sizes([32, 32])
    params.set_kv_group_num(g)
    aux, _ = fasttree_preparation(tree, ptrs, batch, case["hq"], case["hkv"], case["d"], list(s["kv_splits"]), list(s["thr1"]),
                                  list(s["thr2"]), params, kv_slot_map=slot_map, launch_order=s["launch_order"], buffers=buffers)
    return (*aux, list(params.TSQs), list(params.TSKs), 1.0 / math.sqrt(case["d"]))


def _prepare_decode(case, seed):
    tree = _tree(case)
    layers = case.get("layers", 1)
    first = make_decode_inputs(tree, case["hq"], case["hkv"], case["d"], dtype=DTYPES[case["dtype"]], seed=seed, host_rng=False)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 1)
    more = lambda t: torch.randn(t.shape, device=t.device, dtype=t.dtype, generator=gen)  # noqa: E731
    state = dict(case=case, tree=tree, ptrs=first.KV_ptrs, batch=first.batch_size, slot_map=first.slot_map,
                 q=[first.Q] + [more(first.Q) for _ in range(layers - 1)],
                 k=[first.K_pool] + [more(first.K_pool) for _ in range(layers - 1)],
                 v=[first.V_pool] + [more(first.V_pool) for _ in range(layers - 1)],
                 o=[torch.zeros_like(first.Q) for _ in range(layers)])
    if case["kind"] == "decode":
        state["aux"] = _plan(case, tree, first.KV_ptrs, first.batch_size, first.slot_map)
    else:
        # room for the largest plan of such a tree, as a serving program would allocate it once
        depth = case["sizes"].count(",") + 1
        rows = 2 * sum(len(p) // 128 + depth + 1 for p in first.path_tokens)
        entries = sum(len(p) for p in first.path_tokens) + 64
        state["buffers"] = PlanBuffers(case["hq"], case["d"], entries, rows, rows, first.batch_size)
    return state


def _run_decode(s):
    aux = s["aux"] if "aux" in s else _plan(s["case"], s["tree"], s["ptrs"], s["batch"], s["slot_map"], s["buffers"])
    for q, k, v, o in zip(s["q"], s["k"], s["v"], s["o"]):
        fasttree_decode(q, k, v, o, *aux)
    return s["o"][0] if len(s["o"]) == 1 else s["o"]


# ---- serve: objects with the fields of the serving system's own --------------------------

class _Fields:
    def __init__(self, **kw):
        self.__dict__.update(kw)


class _Node:
    """A node of the radix cache: its tokens, their pool slots, its children by first token."""

    def __init__(self, key=(), value=()):
        self.key, self.value, self.children = list(key), value, {}


class _Pool:
    def __init__(self, keys, values):
        self.keys, self.values = keys, values

    def get_key_buffer(self, layer):
        return self.keys[layer]

    def get_value_buffer(self, layer):
        return self.values[layer]


def _serve_tokens(case):
    """Tokens in the radix cache, requests, tokens per request (prompt path and generated)."""
    requests = case["groups"] * case["per_group"]
    cached = case["system"] + case["groups"] * case["group_len"] + requests * case["prompt"]
    path = case["system"] + case["group_len"] + case["prompt"]
    return cached, requests, path


def _prepare_serve(case, seed):
    cached, n, path = _serve_tokens(case)
    grown = case["output"] + FORWARDS                      # generated tokens after the last forward
    slots = np.random.default_rng(seed).permutation(cached + n * grown)
    at = 0

    def take(count):
        nonlocal at
        at += count
        return slots[at - count: at]

    token = iter(range(1, 1 << 30))
    new_tokens = lambda count: [next(token) for _ in range(count)]  # noqa: E731
    root, reqs = _Node(), []
    table = np.zeros((n, path + grown), dtype=np.int32)
    tail = np.zeros((n, grown), dtype=np.int64)

    def child(up, tokens):
        node = _Node(tokens, take(len(tokens)))
        up.children[tokens[0]] = node
        return node

    system = child(root, new_tokens(case["system"]))
    for _ in range(case["groups"]):
        group = child(system, new_tokens(case["group_len"]))
        for _ in range(case["per_group"]):
            own = child(group, new_tokens(case["prompt"]))
            r = len(reqs)
            tail[r] = take(grown)
            table[r] = np.concatenate([system.value, group.value, own.value, tail[r]])
            reqs.append(_Fields(origin_input_ids=system.key + group.key + own.key, output_ids=new_tokens(case["output"])))

    hq, hkv, d, layers, dtype = case["hq"], case["hkv"], case["d"], case["layers"], DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    randn = lambda *shape: torch.randn(shape, device="cuda", dtype=dtype, generator=gen)  # noqa: E731
    req_to_token = _Fields(req_to_token=torch.from_numpy(table).cuda())
    batch = _Fields(reqs=reqs, tree_cache=_Fields(root_node=root), req_pool_indices=torch.arange(n, device="cuda"),
                    req_to_token_pool=req_to_token)
    meta = FastTreeMetadata(hq, hkv, d, fused_store=True)
    pool = _Pool([randn(len(slots), hkv, d) for _ in range(layers)], [randn(len(slots), hkv, d) for _ in range(layers)])
    hooks = [_Fields(qk_head_dim=d, v_head_dim=d, tp_q_head_num=hq, tp_k_head_num=hkv, scaling=1.0 / math.sqrt(d), logit_cap=-1, layer_id=i)
             for i in range(layers)]
    # forward f decodes the token at position path + output + f of every request
    inputs = [_Fields(token_to_kv_pool=pool, req_to_token_pool=req_to_token, fasttree=meta,
                      out_cache_loc=torch.from_numpy(np.ascontiguousarray(tail[:, case["output"] + f])).cuda()) for f in range(FORWARDS)]
    return dict(case=case, batch=batch, server=_Fields(fasttree_metadata=meta), hooks=hooks, inputs=inputs,
                q=[randn(n, hq * d) for _ in range(layers)], k=[randn(n, hkv * d) for _ in range(layers)],
                v=[randn(n, hkv * d) for _ in range(layers)])


def _run_serve(s):
    out = []
    for inputs in s["inputs"]:
        plan_or_step(s["server"], s["batch"], FORWARDS)
        for hook, q, k, v in zip(s["hooks"], s["q"], s["k"], s["v"]):
            o = decode_forward_fasttree(hook, q, k, v, inputs)
        out.append(o)
    return out


# ---- what perf measurements call ---------------------------------------------------------

def prepare(case, seed):
    return _prepare_serve(case, seed) if case["kind"] == "serve" else _prepare_decode(case, seed)


def run(state):
    return _run_serve(state) if "server" in state else _run_decode(state)


def work(case):
    """K/V rows, slot indices and queries read once, outputs written once; the two contractions."""
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    if case["kind"] == "serve":
        cached, n, path = _serve_tokens(case)
        calls = case["layers"] * FORWARDS
        generated = case["output"] + (FORWARDS + 1) / 2    # per request, over the forwards
        tokens = cached + n * generated
        pairs = n * (path + generated)
        new_rows = 4 * n * hkv * d * 2                     # the step's K and V rows, read and stored
        return {"bytes": calls * (tokens * (4 * hkv * d + 4) + 4 * n * hq * d + new_rows), "flops": calls * 4 * hq * d * pairs}
    tree = _tree(case)
    n = assign_requests(tree)
    layers = case.get("layers", 1)
    tokens = sum(node.seqlen for node in tree)
    pairs = sum(node.seqlen * len(node.requests) for node in tree)
    return {"bytes": layers * (tokens * (4 * hkv * d + 4) + 4 * n * hq * d), "flops": layers * 4 * hq * d * pairs}


def tolerance(case):
    # probabilities are rounded to the storage type before the second contraction, outputs once more; sums are fp32
    return {"rel": 2e-3 if case["dtype"] == "fp16" else 1e-2}
