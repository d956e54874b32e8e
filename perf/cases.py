"""What the LoRA path is timed on: the work that a serving program has it do, through the
package's public classes, over the range of batches, adapter mixes and models that the
repository's own configurations and tests name.

A case is one of three kinds of work:

* ``decode``  -- one decode step of a batch: the per-step object (``LoraUnorderedBatchInfer``),
  ``begin_step`` and, for every layer, the q/k/v and the o projections' LoRA deltas added to
  what the base model computed.
* ``prefill`` -- the same for a batch of prompts laid end to end.
* ``load``    -- adapters that a new batch needs are packed into pages of the pool
  (``InferAdapter.load_adapters``) and dropped again (``offload_adapters``).

All layers have pools, activations and outputs of their own, as in a model, so that no layer
finds its weights in a cache that the one before it filled.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "s-lora_amd")  # the package of the tree that is the working folder
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
HEAD_DIM = 128


# ---------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------
def listed():
    def decode(name, hidden, kv, layers, adapters, ranks, zipf, batch, dtype, fused=True):
        return {"name": name, "kind": "decode", "hidden": hidden, "kv": kv, "layers": layers, "adapters": adapters,
                "ranks": ranks, "zipf": zipf, "batch": batch, "dtype": dtype, "fused": fused}

    def prefill(name, hidden, kv, layers, adapters, ranks, zipf, requests, shortest, longest, tokens, dtype):
        return {"name": name, "kind": "prefill", "hidden": hidden, "kv": kv, "layers": layers, "adapters": adapters,
                "ranks": ranks, "zipf": zipf, "requests": requests, "shortest": shortest, "longest": longest,
                "tokens": tokens, "dtype": dtype, "fused": True}

    return [
        # one user alone on the server: a token through all layers, adapters of rank 8 (the S1 model)
        decode("decode_one_token", 4096, 4096, 32, 8, "8", 0.0, 1, "f16"),
        # a quiet server: a ragged handful of users of the S2 mix of ranks
        decode("decode_23_tokens", 4096, 4096, 32, 100, "64,32,16,8", 1.0, 23, "bf16"),
        # few adapters, many users of each (the reference's runs with 5 adapters)
        decode("decode_five_adapters", 4096, 4096, 32, 5, "8", 0.0, 150, "f16"),
        # the headline workload: S2, batch 256, 200 adapters
        decode("decode_s2", 4096, 4096, 32, 200, "64,32,16,8", 1.0, 256, "f16"),
        # the same models driven by the reference's eight calls per layer
        decode("decode_s2_eight_calls", 4096, 4096, 32, 200, "64,32,16,8", 1.0, 117, "f16", fused=False),
        # S4: the 13B shape, 1000 adapters, batch 512
        decode("decode_s4", 5120, 5120, 8, 1000, "64,32,16", 0.9, 512, "f16"),
        # S6: the 70B shape with grouped-query k and v, nearly every token on an adapter of its own
        decode("decode_s6", 8192, 1024, 2, 2000, "64", 0.0, 1024, "bf16"),
        # prompts of a server whose adapters all have rank 8 (S1)
        prefill("prefill_rank8", 4096, 4096, 8, 100, "8", 1.0, 9, 8, 512, 2311, "f16"),
        # the prefill half of the mixed S4 step: 4 prompts of 256 tokens
        prefill("prefill_s4", 5120, 5120, 8, 1000, "64,32,16", 0.9, 4, 256, 256, 1024, "f16"),
        # 64 prompts of 8..512 tokens (C3)
        prefill("prefill_c3", 4096, 4096, 4, 100, "64,32,16,8", 0.0, 64, 8, 512, 15384, "bf16"),
        # long prompts
        prefill("prefill_long", 4096, 4096, 2, 100, "64,32,16,8", 1.0, 21, 333, 2500, 29001, "f16"),
        # three adapters that are not resident when a batch needs them
        {"name": "load_adapters", "kind": "load", "hidden": 4096, "kv": 4096, "layers": 16, "resident": 20,
         "ranks": "64,32,16,8", "new": "64,16,32", "dtype": "f16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "load"])
    hidden, kv = rng.choice([(4096, 4096), (4096, 4096), (4096, 1024), (5120, 5120), (8192, 1024)])
    ranks = rng.choice(["8", "64,32,16,8", "64,32,16,8", "64,32,16", "64", "16,8"])
    dtype = rng.choice(["f16", "bf16"])
    mean = _mean_rank(ranks)
    if kind == "load":
        new = ",".join(str(rng.choice([int(r) for r in ranks.split(",")])) for _ in range(rng.randint(1, 5)))
        return {"kind": "load", "hidden": hidden, "kv": kv, "layers": rng.randint(4, 16), "resident": rng.randint(1, 40),
                "ranks": ranks, "new": new, "dtype": dtype}
    adapters = _log_int(rng, 1, 1500)
    zipf = rng.choice([0.0, 0.9, 1.0])
    # as many layers as keep a state's pools under 12 GB and a pass under the largest listed one
    pool = _pool_pages(adapters * 4 * mean) * hidden * 2 * 2
    case = {"kind": kind, "hidden": hidden, "kv": kv, "layers": max(1, min(32, int(12e9 / pool))), "adapters": adapters,
            "ranks": ranks, "zipf": zipf}
    if kind == "decode":
        case.update(batch=_log_int(rng, 1, 1100), dtype=dtype, fused=rng.random() < 0.75)
    else:
        requests = _log_int(rng, 1, 90)
        shortest = _log_int(rng, 4, 400)
        longest = max(shortest + 1, _log_int(rng, 40, 2500))
        tokens = min(29000, int(requests * (shortest + (longest - shortest) * rng.uniform(0.35, 0.65))))
        tokens = max(requests * shortest, min(tokens, requests * longest))
        if tokens > 29000:
            requests = 29000 // shortest
            tokens = min(29000, requests * longest)
        case.update(requests=requests, shortest=shortest, longest=longest, tokens=tokens, dtype=dtype, fused=True)
    one = work(dict(case, layers=1))["bytes"]
    case["layers"] = max(1, min(case["layers"], int(5e9 / one)))
    if kind == "prefill":
        # activations and outputs of every layer are held at once
        case["layers"] = max(1, min(case["layers"], int(12e9 / (case["tokens"] * (2 * hidden + 2 * kv + 2 * hidden) * 2))))
    return case


def _mean_rank(ranks):
    r = [int(x) for x in ranks.split(",")]
    return sum(r) / len(r)


def _pool_pages(adapter_pages):
    """Pool size for that many adapter pages: they share it with KV pages, 60 % in use."""
    return int(adapter_pages * 1.7) + 64


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
class _Adapter:
    """What the engine and ``InferAdapter`` ask of an adapter."""

    def __init__(self, lora_dir, r, scaling, lora_A=None, lora_B=None):
        self.lora_dir, self.r, self.scaling = lora_dir, r, scaling
        self.lora_A, self.lora_B = lora_A, lora_B


class State:
    pass


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _tables(s, case, rng, dev, dtype):
    """The pools of all layers with the adapters' pages at random places among KV pages, and the
    adapters' index tables: an ``InferAdapter`` as it is after its adapters have been loaded."""
    from slora_hip.infer_adapter import InferAdapter, MemoryAllocator
    hidden, n = case["hidden"], case["adapters"]
    choices = [int(r) for r in case["ranks"].split(",")]
    ranks = rng.choice(np.asarray(choices), size=n).astype(np.int64)
    ranks[0] = choices[0]
    need = int(4 * ranks.sum())
    pages = _pool_pages(n * 4 * max(_mean_rank(case["ranks"]), ranks.mean()))
    mm = MemoryAllocator(pages, 0, dtype, hidden // HEAD_DIM, HEAD_DIM, case["layers"], device=dev)
    a_loc = torch.from_numpy(rng.permutation(pages)[:need].astype(np.int64)).to(dev)
    std = torch.ones(pages, dtype=dtype, device=dev)  # KV pages: N(0, 1); B^T of a rank-r adapter: N(0, 1/r)
    std[a_loc] = torch.from_numpy(np.repeat(ranks, 4 * ranks) ** -0.5).to(dev, dtype)
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(rng.integers(1 << 40)))
    for kb, vb in zip(mm.key_buffer, mm.value_buffer):
        kb.normal_(0.0, hidden ** -0.5, generator=gen)  # A ~ N(0, 1/hidden)
        vb.normal_(0.0, 1.0, generator=gen)
        vb.mul_(std.view(-1, 1, 1))
    s.gen = gen
    s.adapters = [_Adapter("adapter-%d" % i, int(r), 16.0 / int(r)) for i, r in enumerate(ranks)]
    a_len = 4 * ranks
    a_start = np.concatenate([[0], np.cumsum(a_len)[:-1]])
    s.ia = InferAdapter(
        adapter_dirs=[a.lora_dir for a in s.adapters], a_loc=a_loc,
        a_start=torch.from_numpy(a_start).to(dev), a_len=torch.from_numpy(a_len).to(dev),
        a_scaling=torch.tensor([a.scaling for a in s.adapters], dtype=torch.float16, device=dev), mem_manager=mm,
        idx_map={a.lora_dir: i for i, a in enumerate(s.adapters)}, len_host=[int(v) for v in a_len])


def _popular(rng, case, size):
    p = 1.0 / np.arange(1, case["adapters"] + 1, dtype=np.float64) ** case["zipf"]
    return rng.choice(case["adapters"], size=size, p=p / p.sum())


def _lengths(rng, case):
    """Prompt lengths between the shortest and the longest that sum to the case's tokens."""
    lo, hi, n, total = case["shortest"], case["longest"], case["requests"], case["tokens"]
    lens = rng.integers(lo, hi + 1, size=n)
    while lens.sum() != total:
        step = 1 if lens.sum() < total else -1
        room = np.flatnonzero(lens < hi) if step > 0 else np.flatnonzero(lens > lo)
        take = rng.permutation(room)[: abs(int(total - lens.sum()))]
        lens[take] += step
    return lens.astype(np.int32)


def prepare(case, seed):
    dev, dtype = _device(), DTYPES[case["dtype"]]
    rng = np.random.default_rng([seed, case["hidden"]])
    s = State()
    s.case = case
    if case["kind"] == "load":
        return _prepare_load(s, case, rng, dev, dtype)
    _tables(s, case, rng, dev, dtype)
    if case["kind"] == "decode":
        tokens = case["batch"]
        s.req = [s.adapters[i] for i in _popular(rng, case, tokens)]
        lens = rng.integers(8, 1024, size=tokens).astype(np.int32)
    else:
        tokens = case["tokens"]
        s.req = [s.adapters[i] for i in _popular(rng, case, case["requests"])]
        lens = _lengths(rng, case)
    s.tokens, s.longest = tokens, int(lens.max())
    s.b_seq_len = torch.from_numpy(lens).to(dev)
    s.b_start_loc = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)).to(dev)
    L, H, KV = case["layers"], case["hidden"], case["kv"]

    def normal(width):
        return torch.empty((L, tokens, width), dtype=dtype, device=dev).normal_(0.0, 1.0, generator=s.gen)

    s.x, s.att = normal(H), normal(H)                        # inputs of the q/k/v and of the o projections
    s.q, s.k, s.v, s.o = normal(H), normal(KV), normal(KV), normal(H)  # the base model's projections
    s.views = [tuple(t[l] for t in (s.x, s.att, s.q, s.k, s.v, s.o)) for l in range(L)]
    return s


def _matrices(s, dev, dtype, case, name, r):
    def mat(rows, cols, std):
        return torch.empty((rows, cols), dtype=dtype, device=dev).normal_(0.0, std, generator=s.gen)

    H, KV = case["hidden"], case["kv"]
    A = [[mat(H, r, H ** -0.5) for _ in range(4)] for _ in range(case["layers"])]
    B = [[mat(r, h, r ** -0.5) for h in (H, KV, KV, H)] for _ in range(case["layers"])]
    return _Adapter(name, r, 16.0 / r, A, B)


def _prepare_load(s, case, rng, dev, dtype):
    from slora_hip.infer_adapter import InferAdapter, MemoryAllocator
    choices = [int(r) for r in case["ranks"].split(",")]
    new = [int(r) for r in case["new"].split(",")]
    resident = [choices[i % len(choices)] for i in rng.permutation(case["resident"])]
    need = 4 * (sum(new) + case["resident"] * max(choices))
    s.gen = torch.Generator(device=dev)
    s.gen.manual_seed(int(rng.integers(1 << 40)))
    s.mm = MemoryAllocator(_pool_pages(need), 0, dtype, case["hidden"] // HEAD_DIM, HEAD_DIM, case["layers"], device=dev)
    for b in s.mm.key_buffer + s.mm.value_buffer:
        b.normal_(0.0, 1.0, generator=s.gen)
    # KV pages in use among the free ones
    used = s.mm.alloc(s.mm.tot_size - need)
    s.mm.free(used[torch.from_numpy(np.flatnonzero(rng.random(len(used)) < 0.5)).to(dev)].contiguous())
    s.ia = InferAdapter.init(s.mm, device=dev)
    # adapters that are already there: their tables are what the new ones are appended to
    lens = [4 * r for r in resident]
    s.ia.adapter_dirs = ["resident-%d" % i for i in range(len(resident))]
    s.ia.idx_map = {d: i for i, d in enumerate(s.ia.adapter_dirs)}
    s.ia.len_host = list(lens)
    s.ia.a_loc = s.mm.alloc(sum(lens))
    s.ia.a_len = torch.tensor(lens, dtype=torch.long, device=dev)
    s.ia.a_start = torch.tensor(np.concatenate([[0], np.cumsum(lens)[:-1]]), dtype=torch.long, device=dev)
    s.ia.a_scaling = torch.tensor([16.0 / r for r in resident], dtype=torch.float16, device=dev)
    s.keep = set(s.ia.adapter_dirs)
    s.new = [_matrices(s, dev, dtype, case, "new-%d" % i, r) for i, r in enumerate(new)]
    return s


# ---------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------
def run(s):
    case = s.case
    if case["kind"] == "load":
        s.ia.load_adapters(s.new)
        a_loc, a_start, a_len, a_scaling = s.ia.a_loc, s.ia.a_start, s.ia.a_len, s.ia.a_scaling
        s.ia.offload_adapters(s.keep)
        return s.mm.key_buffer, s.mm.value_buffer, a_loc, a_start, a_len, a_scaling, s.ia.a_loc, s.mm.mem_state
    from slora_hip import LoraUnorderedBatchInfer
    engine = LoraUnorderedBatchInfer(s.ia, s.req, kv_embed_dim=case["kv"], fused=case["fused"])
    engine.begin_step(s.b_start_loc, s.b_seq_len, is_prefill=case["kind"] == "prefill", max_b_seq_len=s.longest,
                      total_token_num=s.tokens)
    for layer, (x, att, q, k, v, o) in enumerate(s.views):
        engine.lora_get_qkv(layer, x, q, k, v)
        engine.lora_get_o(layer, att, o)
    return s.q, s.k, s.v, s.o


# ---------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two right answers may be apart
# ---------------------------------------------------------------------------------------
def work(case):
    H, KV, L = case["hidden"], case["kv"], case["layers"]
    if case["kind"] == "load":
        new = sum(int(r) for r in case["new"].split(","))
        # A and B read, their pages written (a page is as wide as the hidden size, B^T pages included)
        return {"bytes": L * 2 * new * (4 * H + 4 * H + 4 * H + 2 * H + 2 * KV), "flops": 0}
    p = 1.0 / np.arange(1, case["adapters"] + 1, dtype=np.float64) ** case["zipf"]
    p /= p.sum()
    picks, tokens = (case["batch"],) * 2 if case["kind"] == "decode" else (case["requests"], case["tokens"])
    mean = _mean_rank(case["ranks"])
    distinct = float((1.0 - (1.0 - p) ** picks).sum())
    weights = distinct * mean * (4 * H + 2 * H + 2 * KV)
    rows = tokens * (2 * H + 2 * (2 * H + 2 * KV))  # activations read; outputs read and written
    return {"bytes": L * 2 * (weights + rows), "flops": L * 2 * tokens * mean * (4 * H + 2 * H + 2 * KV)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # Sums in 32 bits, delta and outputs each rounded once to the storage type.  Against the same
    # sums in 64 bits (rounded once, at the end) the worst of six cases measures rel 3.9e-4 and
    # max 2.8e-3 in f16, 3.2e-3 and 2.4e-2 in bf16: three times that.
    if case["dtype"] == "f16":
        return {"rel": 1.2e-3, "max": 9e-3}
    return {"rel": 9e-3, "max": 7e-2}
