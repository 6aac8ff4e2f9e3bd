"""What a serving worker has this package do, as measurable cases.

Seven kinds of call, each through the public entry points as a worker calls them:

  step     one scheduler step, eager: the index tensors from the request objects
           (`to_device_one_launch`), a plan for the step, then the rotation fused with
           the K/V write once per layer, Q/K/V read in place from the fused projection
  graph    the same step through fixed-capacity buffers (`KVWriteStep`) and one replay
           of a graph that was recorded beforehand
  dropin   the step in the shape of the code this package replaces: host-built index
           arrays, then `rotary_pos_emb` and `append_paged_kv_cache` per layer
  layers   K and V of every layer at hand at once, one launch, by slot or by page table
  copy     `copy_blocks` from the scheduler's dict (copy-on-write of shared blocks)
  handoff  blocks of one pool gathered into a dense buffer and scattered into another
           pool (prefill to decode on one device)
  swap     `KVWorker`: blocks to the pinned host pool and back into other GPU blocks

Requests share prompt prefixes, as a prefix cache makes them do, so block tables have the
lengths of the stated contexts while the pools stay small enough to be compared whole.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import lmserve_amd as kvc

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BLOCK = 16           # tokens per block, everywhere in this repository's configurations
PREFIXES = 4         # distinct shared prompt prefixes of a step
OWN = 128            # tokens of a request beyond its shared prefix, at most (new ones aside)
ACTIVATIONS = 4      # distinct projection outputs the layers of a step cycle through

# layers, query heads, KV heads, head_dim, rotated lanes of a head
MODELS = {
    "1b": (16, 32, 8, 64, 64),
    "7b": (28, 28, 4, 128, 128),
    "8b": (32, 32, 8, 128, 128),
    "70b": (80, 64, 8, 128, 128),
    "70b/tp8": (80, 8, 1, 128, 128),      # the head slice of one rank of eight
    "partial": (24, 32, 8, 80, 32),       # rotation of a part of an 80-lane head
    "odd": (12, 12, 3, 96, 96),           # rows that are no power of two
}


def listed():
    return [
        # Blocks evicted to host memory and brought back into other GPU blocks (96 blocks of 2 MiB).
        {"name": "swap-8b-96", "kind": "swap", "model": "8b", "dtype": "bf16", "blocks": 96},
        # An interactive session: two requests, one new token each; latency and host work only.
        {"name": "decode-1b-2", "kind": "step", "model": "1b", "dtype": "bf16", "chunks": 0, "tokens": 0,
         "decodes": 2, "context": 2048},
        # The full decode batch of the repository's benchmark, contexts up to 4096 tokens.
        {"name": "decode-8b-256", "kind": "step", "model": "8b", "dtype": "bf16", "chunks": 0, "tokens": 0,
         "decodes": 256, "context": 4096},
        # A middling decode batch replayed from a recorded graph, a new step packed and uploaded each time.
        {"name": "decode-7b-64-graph", "kind": "graph", "model": "7b", "dtype": "bf16", "chunks": 0, "tokens": 0,
         "decodes": 64, "context": 4096},
        # The benchmark's chunked prefill: 2048 tokens of four long prompts.
        {"name": "prefill-7b-2048", "kind": "step", "model": "7b", "dtype": "bf16", "chunks": 4, "tokens": 2048,
         "decodes": 0, "context": 8192},
        # The largest step: 8192 prompt tokens through 80 layers of a model that fits one card whole.
        {"name": "prefill-70b-8192", "kind": "step", "model": "70b", "dtype": "bf16", "chunks": 5, "tokens": 8192,
         "decodes": 0, "context": 4096},
        # Prompts and running requests in one step, fp16, partial rotation, ragged sizes, the drop-in calls.
        {"name": "mixed-partial-fp16", "kind": "dropin", "model": "partial", "dtype": "fp16", "chunks": 2,
         "tokens": 777, "decodes": 61, "context": 3000},
        # The benchmark's headline: the decode batch of every layer in one launch, by slot.
        {"name": "layers-8b-256", "kind": "layers", "model": "8b", "dtype": "bf16", "by": "slots", "chunks": 0,
         "tokens": 0, "decodes": 256, "context": 4096},
        # A tensor-parallel rank's prefill chunk of every layer in one launch, by page table: 256-byte rows.
        {"name": "layers-70b-tp8-3001", "kind": "layers", "model": "70b/tp8", "dtype": "bf16", "by": "pages",
         "chunks": 3, "tokens": 3001, "decodes": 0, "context": 4096},
        # A few sequences forked: six shared blocks, two copies of each.
        {"name": "fork-8b-6x2", "kind": "copy", "model": "8b", "dtype": "bf16", "sources": 6, "copies": 2},
        # A large copy-on-write batch.
        {"name": "copy-8b-2048", "kind": "copy", "model": "8b", "dtype": "bf16", "sources": 2048, "copies": 1},
        # The finished prompts of a prefill worker handed to a decode pool, 256 blocks of 5 MiB.
        {"name": "handoff-70b-256", "kind": "handoff", "model": "70b", "dtype": "bf16", "blocks": 256},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "graph", "dropin", "layers", "layers", "copy", "handoff", "swap"])
    case = {"kind": kind, "model": rng.choice(sorted(MODELS)),
            "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"])}
    if kind == "dropin" and MODELS[case["model"]][0] > 40:
        case["model"] = "8b"                     # its outputs come back layer by layer: 40 at most
    layers, heads, kv_heads, dim, _ = MODELS[case["model"]]
    elem = 4 if case["dtype"] == "fp32" else 2
    block = 2 * BLOCK * kv_heads * dim * elem * layers             # bytes of one block over all layers
    if kind in ("step", "graph", "dropin", "layers"):
        form = rng.choice(["decode", "prefill", "mixed"])
        case["context"] = _log_int(rng, 64, 8192)
        # at most 4 GB of projection outputs over all layers, and as much of block pool, in one step
        most = int(min(8192, 4e9 / (layers * (heads + 2 * kv_heads) * dim * elem)))
        case["decodes"] = 0 if form == "prefill" else _log_int(rng, 1, 256)
        case["tokens"] = 0 if form == "decode" else _log_int(rng, 16, max(16, most - case["decodes"]))
        case["chunks"] = 0 if form == "decode" else rng.randint(1, min(6, case["tokens"]))
        while case["context"] > 64 and _pool_blocks(case) * block > 8e9:
            case["context"] //= 2
        if kind == "layers":
            case["by"] = rng.choice(["slots", "pages"])
    elif kind == "copy":
        case["copies"] = rng.randint(1, 3)
        case["sources"] = _log_int(rng, 1, max(1, int(min(2048, 4e9 / (block * case["copies"])))))
    elif kind == "handoff":
        case["blocks"] = _log_int(rng, 2, int(min(2048, 1.3e9 / block)))
    else:
        case["blocks"] = _log_int(rng, 1, max(1, int(min(512, 96 * 2**21 / block))))
    return case


# ---------------------------------------------------------------------------- inputs
_GONE = []           # KV workers whose state is gone: closed when the next state is made


class State:
    """What the worker process holds, as plain attributes. The host pool of a swap state is an output, which may
    outlive the state, so its KV worker is closed only when the next state is made."""

    worker = None

    def __init__(self, case):
        self.kind = case["kind"]
        self.dtype = DTYPES[case["dtype"]]
        self.layers, self.heads, self.kv_heads, self.dim, self.rotary = MODELS[case["model"]]

    def __del__(self):
        worker, self.worker = self.worker, None
        if worker is not None:
            _GONE.append(worker)


def _new_tokens(case, rng):
    """New tokens of every request, in arrival order."""
    sizes = []
    if case["chunks"]:
        cuts = np.sort(rng.choice(np.arange(1, case["tokens"]), case["chunks"] - 1, replace=False)) \
            if case["chunks"] > 1 else np.empty(0, dtype=np.int64)
        sizes = np.diff(np.concatenate([[0], cuts, [case["tokens"]]])).tolist()
    return [int(n) for n in rng.permutation(np.asarray(sizes + [1] * case["decodes"], dtype=np.int64))]


def _pool_blocks(case):
    """Blocks of a pool that holds any step of the case."""
    own = case["decodes"] * (OWN // BLOCK + 1) + case["chunks"] * (OWN // BLOCK + 2) + case["tokens"] // BLOCK
    return PREFIXES * (case["context"] // BLOCK + 1) + own + 16


def _requests(case, rng):
    """The scheduler's requests of one step: shared prefix blocks, then blocks of their own."""
    blocks = rng.permutation(_pool_blocks(case)).astype(np.int64)
    per_prefix = case["context"] // BLOCK + 1
    prefixes = [blocks[i * per_prefix:(i + 1) * per_prefix] for i in range(PREFIXES)]
    at = PREFIXES * per_prefix
    requests = []
    for i, new in enumerate(_new_tokens(case, rng)):
        shared = int(rng.integers(0, case["context"] // BLOCK + 1))
        own = int(rng.integers(1, OWN + 1))
        need = (own + new + BLOCK - 1) // BLOCK
        table = np.concatenate([prefixes[int(rng.integers(PREFIXES))][:shared], blocks[at:at + need]])
        at += need
        filled = shared * BLOCK + own
        requests.append(kvc.InferInput(seq_id=i, input_ids=[0] * new, input_len=new, filled_token_len=filled,
                                       context_len=filled + new, block_ids=table.tolist()))
    return requests


def _randn(shape, dtype, gen):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)


def _pool(s, blocks, gen=None):
    shape = (s.layers, blocks, 2, BLOCK, s.kv_heads, s.dim)
    return torch.zeros(shape, dtype=s.dtype, device="cuda") if gen is None else _randn(shape, s.dtype, gen)


def _prepare_step(case, s, rng, gen):
    s.requests = _requests(case, rng)
    s.context = case["context"] + OWN + case["tokens"] + 1
    tokens = case["tokens"] + case["decodes"]
    s.pool = _pool(s, _pool_blocks(case))
    s.caches = list(s.pool.unbind(0))
    if s.kind == "layers":
        shape = (s.layers, tokens, s.kv_heads, s.dim)
        s.key, s.value = _randn(shape, s.dtype, gen), _randn(shape, s.dtype, gen)
        s.index = kvc.to_device_one_launch(s.requests, BLOCK)
        s.by_slots = case["by"] == "slots"
        return
    s.table = kvc.make_cos_sin_cache(s.rotary, s.context, 500000.0, dtype=s.dtype, device="cuda")
    q_row, kv_row = s.heads * s.dim, s.kv_heads * s.dim
    projections = [_randn((tokens, q_row + 2 * kv_row), s.dtype, gen).split([q_row, kv_row, kv_row], dim=1)
                   for _ in range(min(ACTIVATIONS, s.layers))]
    s.qkv = [projections[layer % len(projections)] for layer in range(s.layers)]
    if s.kind == "dropin":
        return
    s.query_out = torch.zeros((s.layers, tokens, q_row), dtype=s.dtype, device="cuda")
    s.query_outs = list(s.query_out.unbind(0))
    if s.kind == "graph":
        ids = sum(len(r.block_ids) for r in s.requests)
        s.step = kvc.KVWriteStep(s.kv_heads, s.dim, BLOCK, s.dtype, "cuda", max_requests=len(s.requests),
                                 max_tokens=tokens, max_block_ids=ids, cos_sin_cache=s.table, num_heads=s.heads)
        s.step.set_requests(s.requests)
        q, k, v = zip(*s.qkv)
        s.graph = s.step.capture(k, v, s.caches, queries=q, query_outs=s.query_outs)


def prepare(case, seed):
    while _GONE:
        _GONE.pop().close()
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    s = State(case)
    if s.kind in ("step", "graph", "dropin", "layers"):
        _prepare_step(case, s, rng, gen)
    elif s.kind == "copy":
        n, copies = case["sources"], case["copies"]
        ids = rng.permutation(n * (1 + copies) + 8)
        s.pool = _pool(s, ids.size, gen)
        dst = ids[n:n * (1 + copies)].reshape(n, copies).tolist()
        s.pairs = {int(src): row for src, row in zip(ids[:n], dst)}
    elif s.kind == "handoff":
        n = case["blocks"]
        s.pool, s.other = _pool(s, 2 * n, gen), _pool(s, 2 * n)
        s.ids, s.other_ids = (torch.from_numpy(rng.permutation(2 * n)[:n]).cuda() for _ in range(2))
    else:
        n = case["blocks"]
        s.pool = _pool(s, 2 * n, gen)
        gpu, host = rng.permutation(2 * n).tolist(), rng.permutation(2 * n)[:n].tolist()
        s.worker = kvc.KVWorker(s.pool, 2 * n)
        s.worker.host_kv_caches[...] = 0
        # one mapping per sequence of a few blocks, as the scheduler sends them
        cut = range(0, n, 8)
        s.to_host = [kvc.BlockMapping.from_pairs(zip(gpu[i:min(n, i + 8)], host[i:i + 8])) for i in cut]
        s.to_gpu = [kvc.BlockMapping.from_pairs(zip(host[i:i + 8], gpu[n + i:n + i + 8])) for i in cut]
    return s


# ------------------------------------------------------------------------------ passes
def _run_step(s):
    x = kvc.to_device_one_launch(s.requests, BLOCK)
    plan = kvc.PagedRotaryWritePlan(x.batch_indices, x.positions, x.kv_block_indices, x.kv_block_indptrs,
                                    x.kv_last_block_lens, s.table, s.heads, s.kv_heads, s.dim, BLOCK,
                                    slots=x.slot_mapping)
    for (q, k, v), cache, out in zip(s.qkv, s.caches, s.query_outs):
        plan.run(q, k, v, cache, query_out=out)
    return {"query": s.query_out, "pool": s.pool, "cu_seqlens": x.cu_seqlens_q, "indptr": x.kv_block_indptrs,
            "last": x.kv_last_block_lens, "positions": x.positions,
            "requests": x.batch_indices, "slots": x.slot_mapping}


def _run_graph(s):
    s.step.set_requests(s.requests)
    s.graph.replay()
    return {"query": s.query_out, "pool": s.pool, "indptr": s.step.kv_indptr, "positions": s.step.positions,
            "slots": s.step.slot_mapping}


def _run_dropin(s):
    x = kvc.to_device(kvc.make_kv_index_inputs(s.requests, BLOCK), BLOCK)
    queries = []
    for (q, k, v), cache in zip(s.qkv, s.caches):
        q, k = kvc.rotary_pos_emb(q, k, x.position_ids, s.table, s.dim)
        queries.append(q)
        kvc.append_paged_kv_cache(k.view(-1, s.kv_heads, s.dim), v.view(-1, s.kv_heads, s.dim), x.batch_indices,
                                  x.positions, cache, x.kv_block_indices, x.kv_block_indptrs, x.kv_last_block_lens)
    return {"query": queries, "pool": s.pool, "cu_seqlens": x.cu_seqlens_q, "indptr": x.kv_block_indptrs,
            "last": x.kv_last_block_lens, "positions": x.positions,
            "requests": x.batch_indices, "slots": x.slot_mapping}


def _run_layers(s):
    x = s.index
    if s.by_slots:
        kvc.reshape_and_cache_layers(s.key, s.value, s.pool, x.slot_mapping)
    else:
        kvc.append_paged_kv_cache_layers(s.key, s.value, x.batch_indices, x.positions, s.pool, x.kv_block_indices,
                                         x.kv_block_indptrs, x.kv_last_block_lens)
    return s.pool


def _run_copy(s):
    kvc.copy_blocks(s.pool, s.pairs)
    return s.pool


def _run_handoff(s):
    dense = kvc.gather_blocks(s.pool, s.ids)
    kvc.scatter_blocks(s.other, s.other_ids, dense)
    return {"dense": dense, "pool": s.other}


def _run_swap(s):
    s.worker.copy_kv_sync(s.to_host, kvc.Device.GPU, kvc.Device.Host)
    s.worker.copy_kv_sync(s.to_gpu, kvc.Device.Host, kvc.Device.GPU)
    return {"host": s.worker.host_kv_caches, "pool": s.pool}


RUN = {"step": _run_step, "graph": _run_graph, "dropin": _run_dropin, "layers": _run_layers, "copy": _run_copy,
       "handoff": _run_handoff, "swap": _run_swap}


def run(state):
    return RUN[state.kind](state)


# ------------------------------------------------------------- what a pass has to move
def work(case):
    layers, heads, kv_heads, dim, rotary = MODELS[case["model"]]
    elem = 4 if case["dtype"] == "fp32" else 2
    row = kv_heads * dim * elem
    block = 2 * BLOCK * row * layers
    kind = case["kind"]
    if kind == "copy":
        return {"bytes": (1 + case["copies"]) * case["sources"] * block, "flops": 0}   # a source is read once
    if kind == "handoff":
        return {"bytes": 3 * case["blocks"] * block, "flops": 0}        # read, dense buffer out, pool out
    if kind == "swap":
        return {"bytes": 4 * case["blocks"] * block, "flops": 0}        # out and in, both sides of the link
    tokens, requests = case["tokens"] + case["decodes"], case["chunks"] + case["decodes"]
    index = 4 * requests * (case["context"] // (2 * BLOCK) + 8) + 16 * tokens
    cache = layers * tokens * 4 * row                                   # K and V in, K and V rows out
    if kind == "layers":
        return {"bytes": cache + 8 * tokens, "flops": 0}
    query = layers * tokens * 2 * heads * dim * elem
    key_out = layers * tokens * row if kind == "dropin" else 0
    table = tokens * 2 * rotary * elem
    return {"bytes": cache + query + key_out + table + 2 * index,
            "flops": 3 * layers * tokens * (heads + kv_heads) * rotary}


def tolerance(case):
    # Copies are bytes. The rotation is fp32 arithmetic with one rounding to the storage type. Measured on
    # normal inputs against the same formula in float64, unrounded: rel 1.64e-3, max 3.9e-3 in bf16; 2.07e-4
    # and 4.9e-4 in fp16; 3.6e-8 and 1.7e-7 in fp32 (1.2e-7 rel with a contracted product). Four times that.
    if case["kind"] not in ("step", "graph", "dropin"):
        return "exact"
    return {"bf16": {"rel": 6.6e-3, "max": 1.6e-2}, "fp16": {"rel": 8.3e-4, "max": 2e-3},
            "fp32": {"rel": 5e-7, "max": 2e-6}}[case["dtype"]]
