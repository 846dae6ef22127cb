"""Timed cases of the reselect path: what a user of the library has it do,
through its public calls, from the smallest sizes to the largest.

A case is a dict of plain values; its "kind" says which calls it makes:

  step     kvmem_engine_apply_retrieval: one whole agent step
  score    kvmem_hip_score: the per-token max scorer of a preview
  meank    kvmem_hip_q_accumulate + kvmem_hip_score_meank + kvmem_hip_topk:
           a preview with the mean-K cosine scorer
  keysums  kvmem_hip_meank_sums: key sums of newly stored blocks
  harvest  per layer kvmem_hip_q_window_write and kvmem_hip_meank_add, then
           kvmem_hip_q_window_gather: what a batch of decoded or prefilled
           tokens leaves for the next preview
  stagein  kvmem_hip_stagein_blocks: blocks quantized into the pool, with or
           without RoPE and the Walsh-Hadamard rotation
  spill    kvmem_hip_stageout_blocks + kvmem_hip_stagein_packed_host: packed
           rows to and from pinned host memory

Every handle runs on one stream shared by all states, as a program that owns
a device stream runs them.
"""
from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
PKG_DIR = ROOT / "kvmem-llama.cpp_amd"


def _load_pkg():
    if "kvmem_amd" in sys.modules:
        return sys.modules["kvmem_amd"]
    spec = importlib.util.spec_from_file_location(
        "kvmem_amd", PKG_DIR / "__init__.py", submodule_search_locations=[str(PKG_DIR)])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["kvmem_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


kv = _load_pkg()
from kvmem_amd import host  # noqa: E402

POOL_TYPES = {"q8_0": kv.TYPE_Q8_0, "q5_0": kv.TYPE_Q5_0, "q4_0": kv.TYPE_Q4_0, "f16": kv.TYPE_F16}
FLOATS = {"f32": (kv.TYPE_F32, torch.float32), "f16": (kv.TYPE_F16, torch.float16),
          "bf16": (kv.TYPE_BF16, torch.bfloat16)}
# (query heads, KV heads, head size)
GEOMETRIES = [(24, 4, 256), (8, 2, 128), (32, 8, 128), (16, 4, 256), (16, 2, 128)]


def listed() -> list[dict]:
    return [
        # the headline: a 256K-token workspace, the last 64 query tokens, top 256 of
        # 2048 blocks, about 30 % of them new, q8_0 cache
        dict(name="step_256k", kind="step", layers=16, blocks=2048, block_tokens=128, heads=24, kv_heads=4,
             head_dim=256, q_tokens=64, budget=256, changed=77, type_k="q8_0", type_v="q8_0"),
        # an agent session in its first turns: 32K tokens, a one-line user message,
        # the narrower value cache of the mixed-precision recipe
        dict(name="step_32k", kind="step", layers=16, blocks=256, block_tokens=128, heads=24, kv_heads=4,
             head_dim=256, q_tokens=12, budget=64, changed=19, type_k="q8_0", type_v="q4_0"),
        # the smallest scoring call: a few blocks of a small model's two layers
        dict(name="score_small", kind="score", layers=2, blocks=12, block_tokens=128, last_tokens=0, heads=24,
             kv_heads=4, head_dim=256, q_tokens=8, q_type="bf16"),
        # a short follow-up ("yes, go on") late in a long session
        dict(name="score_short_256k", kind="score", layers=16, blocks=2048, block_tokens=128, last_tokens=0,
             heads=24, kv_heads=4, head_dim=256, q_tokens=14, q_type="bf16"),
        # 32-token blocks, the finer retrieval grain of the published 128K-token runs
        dict(name="score_blocks32_128k", kind="score", layers=16, blocks=4096, block_tokens=32, last_tokens=0,
             heads=24, kv_heads=4, head_dim=256, q_tokens=64, q_type="bf16"),
        # 128-wide heads, a grouping of four, an odd block count and a ragged last block
        dict(name="score_d128", kind="score", layers=16, blocks=1003, block_tokens=128, last_tokens=77,
             heads=32, kv_heads=8, head_dim=128, q_tokens=40, q_type="f16"),
        # the largest: a 1M-token workspace and the longest query window (512 tokens)
        dict(name="score_1m", kind="score", layers=16, blocks=8192, block_tokens=128, last_tokens=0, heads=24,
             kv_heads=4, head_dim=256, q_tokens=512, q_type="bf16"),
        # a preview with the mean-K cosine scorer at 256K tokens
        dict(name="meank_256k", kind="meank", layers=16, blocks=2048, heads=24, kv_heads=4, head_dim=256,
             q_tokens=64, budget=256, q_type="bf16"),
        # the key sums of the blocks one 2048-token prefill batch adds (the last partial)
        dict(name="keysums_append", kind="keysums", layers=16, blocks=512, n=16, block_tokens=128,
             last_tokens=50, kv_heads=4, head_dim=256),
        # the harvest of one 512-token prefill batch over every attention layer
        dict(name="harvest_prefill", kind="harvest", layers=16, tokens=512, block_tokens=128, heads=24,
             kv_heads=4, head_dim=256, k_type="f32", q_type="f32"),
        # blocks restaged from raw keys: partial RoPE and attn_rot before q8_0
        dict(name="stagein_rope", kind="stagein", layers=16, blocks=300, n=24, block_tokens=128, kv_heads=8,
             head_dim=128, n_rot=64, attn_rot=True, type_k="q8_0", type_v="q8_0"),
        # an apply's evicted blocks saved to, and returning ones restored from, host RAM
        dict(name="spill", kind="spill", layers=16, blocks=24, n=8, block_tokens=128, kv_heads=4, head_dim=256,
             type_k="q8_0", type_v="q8_0"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["step", "score", "score", "score", "meank", "keysums", "harvest", "stagein", "stagein",
                       "spill"])
    heads, kv_heads, head_dim = rng.choice(GEOMETRIES)
    geo = dict(heads=heads, kv_heads=kv_heads, head_dim=head_dim)
    layers = rng.choice([1, 2, 4, 8, 16])
    types = rng.choice([("q8_0", "q8_0"), ("q8_0", "q4_0"), ("q5_0", "q5_0"), ("q8_0", "q8_0"), ("f16", "f16")])
    if kind == "step":
        blocks = _log_int(rng, 64, 2048)
        budget = max(8, min(512, blocks // rng.choice([4, 8])))
        return dict(kind=kind, layers=layers, blocks=blocks, block_tokens=rng.choice([128, 128, 64]), **geo,
                    q_tokens=_log_int(rng, 8, 128), budget=budget, changed=max(1, round(0.3 * budget)),
                    type_k=types[0], type_v=types[1])
    if kind == "score":
        T = rng.choice([128, 128, 128, 64, 32])
        tokens = _log_int(rng, 1500, 262144)
        blocks = max(2, tokens // T)
        return dict(kind=kind, layers=layers, blocks=blocks, block_tokens=T,
                    last_tokens=rng.choice([0, rng.randrange(1, T)]), **geo, q_tokens=_log_int(rng, 1, 256),
                    q_type=rng.choice(["bf16", "bf16", "f16"]))
    if kind == "meank":
        blocks = _log_int(rng, 64, 8192)
        return dict(kind=kind, layers=layers, blocks=blocks, **geo, q_tokens=_log_int(rng, 1, 512),
                    budget=max(4, blocks // 8), q_type=rng.choice(["bf16", "f32", "f16"]))
    if kind == "keysums":
        n = _log_int(rng, 1, 512)
        return dict(kind=kind, layers=layers, blocks=n + rng.randrange(0, 200), n=n, block_tokens=128,
                    last_tokens=rng.randrange(1, 129), kv_heads=kv_heads, head_dim=head_dim)
    if kind == "harvest":
        return dict(kind=kind, layers=layers, tokens=_log_int(rng, 1, 512), block_tokens=128, **geo,
                    k_type=rng.choice(["f32", "f32", "f16"]), q_type=rng.choice(["f32", "f32", "bf16"]))
    if kind == "stagein":
        n = _log_int(rng, 1, 200)
        rot = rng.choice([0, 64, head_dim, head_dim])
        return dict(kind=kind, layers=layers, blocks=n + rng.randrange(8, 300), n=n, block_tokens=128,
                    kv_heads=kv_heads, head_dim=head_dim, n_rot=rot,
                    attn_rot=rot > 0 and types[0] != "f16" and rng.random() < 0.7,
                    type_k=types[0], type_v=types[1])
    n = _log_int(rng, 1, 24)
    return dict(kind=kind, layers=layers, blocks=n + rng.randrange(1, 40), n=n, block_tokens=128,
                kv_heads=kv_heads, head_dim=head_dim, type_k=types[0], type_v=types[1])


# ------------------------------------------------------------------ inputs
_shared: dict = {}


def _stream() -> int:
    if "stream" not in _shared:
        _shared["stream"] = torch.cuda.Stream()
    return _shared["stream"].cuda_stream


def _context() -> "kv.Context":
    ctx = kv.Context(torch.cuda.current_device())
    ctx.set_stream(_stream())
    return ctx


def _gen(case: dict, seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + sum(map(ord, case["kind"])))
    return g


def _randn(g, *shape) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _rows(g, L: int, B: int, T: int, E: int, offset: float = 0.3) -> torch.Tensor:
    """F16 history [L][B][T][E]: N(0, 1) plus a per-(block, channel) mean."""
    out = torch.empty((L, B, T, E), dtype=torch.float16, device="cuda")
    step = max(1, (1 << 28) // (T * E))
    for l in range(L):
        for b in range(0, B, step):
            n = min(step, B - b)
            out[l, b:b + n] = _randn(g, n, T, E).add_(_randn(g, n, 1, E) * offset)
    return out


def _query(g, case: dict) -> torch.Tensor:
    return _randn(g, case["layers"], case["q_tokens"], case["heads"], case["head_dim"])


def _relevant(rng: np.random.Generator, case: dict) -> tuple[np.ndarray, np.ndarray]:
    """Two turns' relevant blocks (budget - 1 each beside the sink), `changed`
    of them different."""
    n = case["budget"] - 1
    ids = rng.permutation(np.arange(1, case["blocks"]))
    changed = min(case["changed"], n, len(ids) - n)
    a = ids[:n]
    b = np.concatenate([ids[changed:n], ids[n:n + changed]])
    return np.sort(a), np.sort(b)


def _group_direction(q: torch.Tensor, kv_heads: int) -> torch.Tensor:
    """Unit vector per KV head: the mean of one layer's query rows of its group."""
    Hq, D = q.shape[-2:]
    m = q.float().mean(dim=0).view(kv_heads, Hq // kv_heads, D).mean(dim=1)
    return m / m.norm(dim=-1, keepdim=True)


def _pool(case: dict, n_slots: int, ctx=None, xf=None):
    """Per-layer K and V tensors of the pool, one allocation each."""
    E = case["kv_heads"] * case["head_dim"]
    out, ptrs = [], []
    for t in (case["type_k"], case["type_v"]):
        nbytes = n_slots * case["block_tokens"] * kv.row_size(POOL_TYPES[t], E)
        p = torch.zeros((case["layers"], nbytes // 8), dtype=torch.int64, device="cuda")
        out.append(p)
        ptrs.append([p[l].data_ptr() for l in range(case["layers"])])
    if ctx is None:
        return out, ptrs
    pool = ctx.make_pool(case["layers"], n_slots, case["block_tokens"], E, E, POOL_TYPES[case["type_k"]],
                         POOL_TYPES[case["type_v"]], ptrs[0], ptrs[1], xf)
    return out, pool


# ----------------------------------------------------------------- prepare
def prepare(case: dict, seed: int) -> dict:
    return _KINDS[case["kind"]][0](case, seed)


def run(state: dict):
    return state["run"](state)


def work(case: dict) -> dict:
    return _KINDS[case["kind"]][1](case)


def tolerance(case: dict):
    return _KINDS[case["kind"]][2](case)


def exact(case: dict, seed: int):
    return _KINDS[case["kind"]][3](case, seed)


# -- step
def _step_prepare(case: dict, seed: int) -> dict:
    g = _gen(case, seed)
    L, B, T = case["layers"], case["blocks"], case["block_tokens"]
    Hkv, D = case["kv_heads"], case["head_dim"]
    E = Hkv * D
    k = _rows(g, L, B, T, E)
    v = _rows(g, L, B, T, E, 0.0)
    # two turns' queries; a turn's relevant blocks carry its direction, which
    # lifts them clear of the rest, so the cut of the selection is no near tie
    queries = [_query(g, case).to(torch.bfloat16) for _ in range(2)]
    for q, ids in zip(queries, _relevant(np.random.default_rng(seed), case)):
        at = torch.from_numpy(ids).cuda()
        for l in range(L):
            k[l, at] += (10.0 * _group_direction(q[l], Hkv)).half().view(1, 1, E)
    eng = host.Engine(n_layers=L, block_tokens=T, n_head=case["heads"], n_head_kv=Hkv, head_dim=D,
                      budget_blocks=case["budget"], reserve_blocks=max(4, case["budget"] // 2),
                      type_k=POOL_TYPES[case["type_k"]], type_v=POOL_TYPES[case["type_v"]])
    pool, ptrs = _pool(case, eng.n_slots())
    torch.cuda.synchronize()
    kv.Context.borrow(eng.ctx_handle()).set_stream(_stream())
    eng.set_pool(*ptrs)
    eng.set_device_history(k.data_ptr(), v.data_ptr(), B, B * T)
    # the session so far: the first turn's window is resident
    eng.apply_retrieval(queries[0].data_ptr(), case["q_tokens"])
    return dict(run=_step_run, eng=eng, k=k, v=v, queries=queries, pool=pool, turn=0, tq=case["q_tokens"])


def _step_run(s: dict):
    s["turn"] ^= 1
    st = s["eng"].apply_retrieval(s["queries"][s["turn"]].data_ptr(), s["tq"])
    return {"pool": s["pool"], "staged": st["n_staged"], "moved": st["n_moved"],
            "window_tokens": st["total_window_tokens"]}


def _step_work(case: dict) -> dict:
    E = case["kv_heads"] * case["head_dim"]
    rows = case["layers"] * case["block_tokens"]
    staged = sum(2 * E + kv.row_size(POOL_TYPES[case[t]], E) for t in ("type_k", "type_v"))
    w = _score_work(case)
    return {"bytes": w["bytes"] + case["changed"] * rows * staged, "flops": w["flops"]}


# -- score
def _score_inputs(case: dict, seed: int):
    g = _gen(case, seed)
    k = _rows(g, case["layers"], case["blocks"], case["block_tokens"], case["kv_heads"] * case["head_dim"])
    return k, _query(g, case).to(FLOATS[case["q_type"]][1])


def _score_prepare(case: dict, seed: int) -> dict:
    k, q = _score_inputs(case, seed)
    L, B, T, E = k.shape
    ctx = _context()
    ctx.reserve(n_layers=L, n_blocks=B, n_head=case["heads"], n_head_kv=case["kv_heads"],
                head_dim=case["head_dim"], n_q_tokens=case["q_tokens"])
    hist = ctx.make_history(k.data_ptr(), 0, L, B, T, E, 0, case["last_tokens"])
    scores = torch.zeros(B, dtype=torch.float32, device="cuda")
    layers = torch.zeros((L, B), dtype=torch.float32, device="cuda")
    return dict(run=_score_run, ctx=ctx, hist=hist, k=k, q=q, q_type=FLOATS[case["q_type"]][0], case=case,
                scores=scores, layers=layers)


def _score_run(s: dict):
    c = s["case"]
    s["ctx"].score(s["hist"], s["q"].data_ptr(), s["q_type"], c["q_tokens"], c["heads"], c["kv_heads"],
                   c["head_dim"], s["scores"].data_ptr(), s["layers"].data_ptr())
    return {"scores": s["scores"], "layer_scores": s["layers"]}


def _score_work(case: dict) -> dict:
    keys = case["blocks"] * case["block_tokens"]
    if case.get("last_tokens"):
        keys -= case["block_tokens"] - case["last_tokens"]
    L, Hq, Hkv, D = case["layers"], case["heads"], case["kv_heads"], case["head_dim"]
    q_rows = case["q_tokens"] * Hq
    return {"bytes": 2 * L * D * (keys * Hkv + q_rows) + 4 * (L + 1) * case["blocks"],
            "flops": 2 * L * keys * q_rows * D}


def _score_exact(case: dict, seed: int):
    k, q = _score_inputs(case, seed)
    L, B, T, E = k.shape
    Hkv, D = case["kv_heads"], case["head_dim"]
    R = case["q_tokens"] * (case["heads"] // Hkv)
    layers = torch.full((L, B), -math.inf, dtype=torch.float64, device="cuda")
    step = max(1, min((1 << 27) // (T * R), (1 << 28) // (T * E)))
    for l in range(L):
        ql = q[l].view(case["q_tokens"], Hkv, R // case["q_tokens"], D).transpose(0, 1)
        ql = ql.reshape(Hkv, R, D).double()
        for b in range(0, B, step):
            kb = k[l, b:b + step].view(-1, Hkv, D)
            for h in range(Hkv):
                s = kb[:, h].double() @ ql[h].T
                s = s.view(-1, T, R).amax(dim=2)
                if b + step >= B and case["last_tokens"]:
                    s[-1, case["last_tokens"]:] = -math.inf
                torch.maximum(layers[l, b:b + step], s.amax(dim=1) / math.sqrt(D), out=layers[l, b:b + step])
    return {"scores": layers.mean(dim=0), "layer_scores": layers}


# -- meank
def _meank_inputs(case: dict, seed: int):
    g = _gen(case, seed)
    L, B, Hkv, D = case["layers"], case["blocks"], case["kv_heads"], case["head_dim"]
    q = _query(g, case).to(FLOATS[case["q_type"]][1])
    # key sums of 128-token blocks: 128 times a block mean of N(0, 0.3) per channel
    # plus the sum of 128 N(0, 1); the relevant blocks lean towards the query
    k_sum = torch.empty((L, B, Hkv * D), dtype=torch.float32, device="cuda")
    at = torch.from_numpy(_relevant(np.random.default_rng(seed), dict(case, changed=0))[0]).cuda()
    for l in range(L):
        k_sum[l] = _randn(g, B, Hkv * D) * math.sqrt(128 * 128 * 0.09 + 128)
        k_sum[l, at] += 600.0 * _group_direction(q[l], Hkv).view(1, Hkv * D)
    return q, k_sum


def _meank_prepare(case: dict, seed: int) -> dict:
    q, k_sum = _meank_inputs(case, seed)
    L, B = case["layers"], case["blocks"]
    ctx = _context()
    ctx.reserve(n_layers=L, n_blocks=B, n_head=case["heads"], n_head_kv=case["kv_heads"],
                head_dim=case["head_dim"], n_q_tokens=case["q_tokens"], max_items=64)
    tokens = torch.full((L, B), 128, dtype=torch.int32, device="cuda")
    q_sum = torch.zeros((L, case["heads"] * case["head_dim"]), dtype=torch.float32, device="cuda")
    scores = torch.zeros(B, dtype=torch.float32, device="cuda")
    return dict(run=_meank_run, ctx=ctx, q=q, k_sum=k_sum, tokens=tokens, q_sum=q_sum, scores=scores, case=case,
                counts=[case["q_tokens"]] * L)


def _meank_run(s: dict):
    c, ctx = s["case"], s["ctx"]
    ctx.q_accumulate(s["q"].data_ptr(), FLOATS[c["q_type"]][0], c["layers"], c["q_tokens"],
                     c["heads"] * c["head_dim"], s["q_sum"].data_ptr())
    ctx.score_meank(s["q_sum"].data_ptr(), s["counts"], s["k_sum"].data_ptr(), s["tokens"].data_ptr(),
                    c["layers"], c["blocks"], c["heads"], c["kv_heads"], c["head_dim"], s["scores"].data_ptr())
    sel = ctx.topk(s["scores"].data_ptr(), c["blocks"], c["budget"] - 1, forced=[0])
    return {"q_sum": s["q_sum"], "scores": s["scores"], "selection": np.array(sel, dtype=np.int64)}


def _meank_work(case: dict) -> dict:
    L, B, Hq, Hkv, D = case["layers"], case["blocks"], case["heads"], case["kv_heads"], case["head_dim"]
    esz = FLOATS[case["q_type"]][1].itemsize
    q = L * case["q_tokens"] * Hq * D
    return {"bytes": q * esz + 4 * L * Hq * D + 4 * L * B * (Hkv * D + 1) + 4 * B, "flops": q + 4 * L * B * Hkv * D}


def _meank_exact(case: dict, seed: int):
    q, k_sum = _meank_inputs(case, seed)
    L, B, Hkv, D = case["layers"], case["blocks"], case["kv_heads"], case["head_dim"]
    q_sum = q.double().sum(dim=1).view(L, -1)
    qv = q_sum.view(L, Hkv, -1, D).mean(dim=2) / case["q_tokens"]
    cos = torch.empty((L, B), dtype=torch.float64, device="cuda")
    for l in range(L):
        k = k_sum[l].view(B, Hkv, D).double() / 128
        cos[l] = ((k * qv[l]).sum(-1) / (k.norm(dim=-1) * qv[l].norm(dim=-1) + 1e-6)).mean(-1)
    return {"q_sum": q_sum, "scores": cos.mean(0), "selection": None}


# -- keysums
def _keysums_ids(case: dict) -> list[int]:
    return list(range(case["blocks"] - case["n"], case["blocks"]))


def _keysums_inputs(case: dict, seed: int) -> torch.Tensor:
    return _rows(_gen(case, seed), case["layers"], case["blocks"], case["block_tokens"],
                 case["kv_heads"] * case["head_dim"])


def _keysums_prepare(case: dict, seed: int) -> dict:
    k = _keysums_inputs(case, seed)
    L, B, T, E = k.shape
    ctx = _context()
    ctx.reserve(max_items=case["n"], n_layers=L)
    hist = ctx.make_history(k.data_ptr(), 0, L, B, T, E, 0, case["last_tokens"])
    k_sum = torch.zeros((L, B, E), dtype=torch.float32, device="cuda")
    tokens = torch.zeros((L, B), dtype=torch.int32, device="cuda")
    return dict(run=_keysums_run, ctx=ctx, k=k, hist=hist, k_sum=k_sum, tokens=tokens, ids=_keysums_ids(case))


def _keysums_run(s: dict):
    s["ctx"].meank_sums(s["hist"], s["ids"], s["k_sum"].data_ptr(), s["tokens"].data_ptr())
    return {"k_sum": s["k_sum"], "tokens": s["tokens"]}


def _keysums_work(case: dict) -> dict:
    E = case["kv_heads"] * case["head_dim"]
    rows = case["n"] * case["block_tokens"] - (case["block_tokens"] - case["last_tokens"])
    return {"bytes": case["layers"] * (2 * rows * E + 4 * case["n"] * (E + 1)),
            "flops": case["layers"] * rows * E}


def _keysums_exact(case: dict, seed: int):
    k = _keysums_inputs(case, seed)
    L, B, T, E = k.shape
    out = torch.zeros((L, B, E), dtype=torch.float64, device="cuda")
    for b in _keysums_ids(case):
        nt = case["last_tokens"] if b == B - 1 else T
        out[:, b] = k[:, b, :nt].double().sum(dim=1)
    return {"k_sum": out, "tokens": None}


# -- harvest
def _harvest_inputs(case: dict, seed: int):
    g = _gen(case, seed)
    n, D = case["tokens"], case["head_dim"]
    q = _randn(g, case["layers"], n, case["heads"] * D).to(FLOATS[case["q_type"]][1])
    k = _randn(g, case["layers"], n, case["kv_heads"] * D).to(FLOATS[case["k_type"]][1])
    return q, k


_WINDOW = 512   # rows of the query ring per layer
_LAST = 64      # newest rows a preview takes


def _harvest_parts(case: dict) -> list[tuple[int, int]]:
    T = case["block_tokens"]
    return [(t, min(T, case["tokens"] - t)) for t in range(0, case["tokens"], T)]


def _harvest_prepare(case: dict, seed: int) -> dict:
    q, k = _harvest_inputs(case, seed)
    L, n = case["layers"], case["tokens"]
    Eq, Ek = q.shape[2], k.shape[2]
    ctx = _context()
    ctx.reserve(max_items=max(n, 64), n_layers=L)
    window = torch.zeros((L, _WINDOW, Eq), dtype=torch.float32, device="cuda")
    sums = torch.zeros((L, len(_harvest_parts(case)), Ek), dtype=torch.float32, device="cuda")
    counts = torch.zeros(sums.shape[:2], dtype=torch.int32, device="cuda")
    take = min(n, _LAST)
    out = torch.zeros((L, take, Eq), dtype=torch.bfloat16, device="cuda")
    return dict(run=_harvest_run, ctx=ctx, q=q, k=k, window=window, sums=sums, counts=counts, out=out, case=case,
                parts=_harvest_parts(case), tokens=list(range(n)), last=list(range(n - take, n)))


def _harvest_run(s: dict):
    c, ctx, q, k = s["case"], s["ctx"], s["q"], s["k"]
    D = c["head_dim"]
    (qt, qd), (kt, kd) = FLOATS[c["q_type"]], FLOATS[c["k_type"]]
    qe, ke = qd.itemsize, kd.itemsize
    Eq, Ek = q.shape[2], k.shape[2]
    for l in range(c["layers"]):
        ctx.q_window_write(q[l].data_ptr(), qt, c["heads"], D, qe, D * qe, Eq * qe, s["tokens"], s["tokens"],
                           s["window"][l].data_ptr(), _WINDOW)
        for i, (t, n) in enumerate(s["parts"]):
            ctx.meank_add(k[l].data_ptr(), kt, Ek, D, ke, D * ke, Ek * ke, t, n, s["sums"][l, i].data_ptr(),
                          s["counts"][l, i].data_ptr(), reset=True)
    ctx.q_window_gather(s["window"].data_ptr(), c["layers"], _WINDOW, Eq, s["last"], kv.TYPE_BF16,
                        s["out"].data_ptr())
    return {"window": s["window"], "key_sums": s["sums"], "counts": s["counts"], "query": s["out"]}


def _harvest_work(case: dict) -> dict:
    n, D, L = case["tokens"], case["head_dim"], case["layers"]
    Eq, Ek = case["heads"] * D, case["kv_heads"] * D
    qe, ke = FLOATS[case["q_type"]][1].itemsize, FLOATS[case["k_type"]][1].itemsize
    sums = 4 * (Ek + 1) * len(_harvest_parts(case))
    return {"bytes": L * (n * Eq * (qe + 4) + n * Ek * ke + sums + min(n, _LAST) * Eq * 6),
            "flops": L * n * Ek}


def _harvest_exact(case: dict, seed: int):
    q, k = _harvest_inputs(case, seed)
    window = torch.zeros((case["layers"], _WINDOW, q.shape[2]), dtype=torch.float64, device="cuda")
    window[:, :case["tokens"]] = q.double()
    sums = torch.stack([k[:, t:t + n].double().sum(dim=1) for t, n in _harvest_parts(case)], dim=1)
    take = min(case["tokens"], _LAST)
    return {"window": window, "key_sums": sums, "counts": None, "query": q[:, case["tokens"] - take:].double()}


# -- stagein
def _stagein_prepare(case: dict, seed: int) -> dict:
    g = _gen(case, seed)
    L, B, T, D = case["layers"], case["blocks"], case["block_tokens"], case["head_dim"]
    E = case["kv_heads"] * D
    k, v = _rows(g, L, B, T, E), _rows(g, L, B, T, E, 0.0)
    # a few channels of every head an order larger, as trained keys have them
    rng = np.random.default_rng(seed)
    ch = torch.from_numpy(np.concatenate([h * D + rng.choice(D, 4, replace=False)
                                          for h in range(case["kv_heads"])])).cuda()
    k[..., ch] *= 20.0
    ctx = _context()
    ctx.reserve(max_items=case["n"], n_layers=L)
    xf = None
    if case["n_rot"] or case["attn_rot"]:
        theta = 1e6 ** (-2.0 * np.arange(case["n_rot"] // 2) / max(1, case["n_rot"]))
        width = (D if case["attn_rot"] else 0, 64 if case["attn_rot"] else 0)
        xf = ctx.make_transform(D, case["n_rot"], theta.astype(np.float32), *width)
    n_slots = case["n"] + max(4, case["n"] // 2)
    pool, desc = _pool(case, n_slots, ctx, xf)
    ids = np.sort(rng.choice(B, case["n"], replace=False)).tolist()
    slots = rng.choice(n_slots, case["n"], replace=False).tolist()
    hist = ctx.make_history(k.data_ptr(), v.data_ptr(), L, B, T, E, E)
    return dict(run=_stagein_run, ctx=ctx, hist=hist, k=k, v=v, pool=pool, desc=desc, ids=ids, slots=slots)


def _stagein_run(s: dict):
    s["ctx"].stagein_blocks(s["hist"], s["desc"], s["ids"], s["slots"])
    return s["pool"]


def _stagein_work(case: dict) -> dict:
    E = case["kv_heads"] * case["head_dim"]
    rows = case["n"] * case["layers"] * case["block_tokens"]
    per = sum(2 * E + kv.row_size(POOL_TYPES[case[t]], E) for t in ("type_k", "type_v"))
    return {"bytes": rows * per, "flops": 0}


# -- spill
def _spill_prepare(case: dict, seed: int) -> dict:
    g = _gen(case, seed)
    rng = np.random.default_rng(seed)
    L, T, B, n = case["layers"], case["block_tokens"], case["blocks"], case["n"]
    E = case["kv_heads"] * case["head_dim"]
    ctx = _context()
    n_slots = 2 * n + 2
    pool, desc = _pool(case, n_slots, ctx)
    for p in pool:  # rows as a cache holds them: packed bytes
        p.random_(generator=g)
    per = sum(kv.row_size(POOL_TYPES[case[t]], E) for t in ("type_k", "type_v"))
    store = torch.zeros((B, L * T * per // 8), dtype=torch.int64, pin_memory=True)
    ctx.reserve(max_items=n, n_layers=L)
    packed = kv.PackedHost(store.data_ptr(), L, B, T)
    ids = rng.choice(B, n, replace=False)
    slots = rng.choice(n_slots, 2 * n, replace=False)
    return dict(run=_spill_run, ctx=ctx, pool=pool, desc=desc, store=store, packed=packed,
                blocks=ids.tolist(), out=slots[:n].tolist(), into=slots[n:].tolist(), tokens=[T] * n)


def _spill_run(s: dict):
    s["ctx"].stageout_blocks(s["desc"], s["packed"], s["blocks"], s["out"], s["tokens"])
    s["ctx"].stagein_packed_host(s["packed"], s["desc"], s["blocks"], s["into"], s["tokens"])
    return {"pool": s["pool"], "store": s["store"]}


def _spill_work(case: dict) -> dict:
    E = case["kv_heads"] * case["head_dim"]
    per = sum(kv.row_size(POOL_TYPES[case[t]], E) for t in ("type_k", "type_v"))
    # out: pool rows read, host rows written; back: the same
    return {"bytes": 4 * case["n"] * case["layers"] * case["block_tokens"] * per, "flops": 0}


def _whole(case: dict):
    return "exact"


def _no_exact(case: dict, seed: int):
    return None


# kind -> (prepare, work, tolerance, exact).  Pool and packed bytes, key sums
# (a fixed order of 32-bit additions), copies and counts are the same bit for
# bit.  Scores are maxima of 32-bit accumulated dot products, 0.9e-7 (2-norm)
# from their 64-bit values; mean cosines are 0.3e-7 from theirs over 16
# layers, and more over one layer of blocks the query has nothing to do with.
_KINDS = {
    "step": (_step_prepare, _step_work, _whole, _no_exact),
    "score": (_score_prepare, _score_work, lambda c: {"rel": 4e-7, "max": 4e-6}, _score_exact),
    "meank": (_meank_prepare, _meank_work, lambda c: {"rel": 1e-6, "max": 1e-5, "differ": 0.005}, _meank_exact),
    "keysums": (_keysums_prepare, _keysums_work, _whole, _keysums_exact),
    "harvest": (_harvest_prepare, _harvest_work, _whole, _harvest_exact),
    "stagein": (_stagein_prepare, _stagein_work, _whole, _no_exact),
    "spill": (_spill_prepare, _spill_work, _whole, _no_exact),
}
