"""Performance cases of the paged decode path: what a serving program has this
framework do, through the entry points such a program calls.

A case is a dict of plain values. Its "kind" names the call:

  decode  paged_mqa_decode over device-resident tables: one query per
          sequence against a paged K/V pool (16/32-bit or fp8 pools)
  step    paged_attention_append_meta for every layer of a ragged step: the
          new K/V rows appended and attended to (decode rows, prefill chunks
          or both)
  block   one decoder layer of PagedTransformer (norm, q/k/v + RoPE, append +
          attention, out projection, norm, SwiGLU MLP, both residual adds)
  head    final norm, vocabulary projection and the token choice (sampled with
          temperature / top-k / top-p, or greedy)
  append  KVPool.write of prompt rows by slot mapping
  model   PagedTransformer: a whole step from host lists (forward_batch) or a
          greedy decode step replayed from its HIP graph (DecodeStepGraph)

Context lengths come from the case itself ("shape" seeds them), values, block
tables and weights from the seed handed to prepare().
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

# the package folder's name is no Python identifier, so its path is added;
# the working folder is the repository's root
sys.path.insert(0, os.path.join(os.getcwd(), "tiny-transformer-inference-engine_amd"))

from serving import fused_ops  # noqa: E402
from serving.batch import BatchStep  # noqa: E402
from serving.fake_paged_attn import paged_attention_append_meta, paged_mqa_decode  # noqa: E402
from serving.graph_step import DecodeStepGraph  # noqa: E402
from serving.kv_pool import KVPool  # noqa: E402
from serving.layers import ModelConfig, RMSNorm  # noqa: E402
from serving.paged_meta import pack_batch_meta  # noqa: E402
from serving.paged_model import PagedBlock, PagedTransformer  # noqa: E402

DEV = "cuda:0"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
ESIZE = {"fp32": 4, "bf16": 2, "fp16": 2}
EPS = 1e-5  # RMSNorm's


def listed():
    return [
        # the smallest attention call: a small fp32 model's decode batch, where
        # the launch and the call itself count
        dict(name="decode_op_small_fp32", kind="decode", batch=32, hq=8, hkv=1, d=32, bs=16,
             dtype="fp32", kv="same", dist="uniform", lo=64, hi=256, shape=0),
        # four layers of a batch-128 decode step of a 1024-wide, 16-head model
        dict(name="step_decode_b128", kind="step", layers=4, decodes=128, hq=16, hkv=1, d=64,
             bs=16, dtype="bf16", dist="uniform", lo=256, hi=2048, prompts=0, plo=0, phi=0,
             past=0, shape=0),
        # long-context decode batch with heavy-tailed lengths, 32 heads of 128
        dict(name="decode_long_b256", kind="decode", batch=256, hq=32, hkv=1, d=128, bs=16,
             dtype="bf16", kv="same", dist="lognormal", lo=1024, hi=8192, shape=0),
        # the same batch served from an fp8 KV cache
        dict(name="decode_long_b256_fp8", kind="decode", batch=256, hq=32, hkv=1, d=128, bs=16,
             dtype="bf16", kv="fp8", dist="lognormal", lo=1024, hi=8192, shape=0),
        # a continuous-batching step: 256 running sequences and four new
        # prompts' 512-token chunks
        dict(name="step_mixed_b256", kind="step", layers=1, decodes=256, hq=32, hkv=1, d=128,
             bs=16, dtype="bf16", dist="lognormal", lo=1024, hi=8192, prompts=4, plo=512,
             phi=512, past=0, shape=0),
        # prompts of the default configuration's attention (fp32, 8 heads of 64)
        dict(name="step_prefill_fp32", kind="step", layers=1, decodes=0, hq=8, hkv=1, d=64,
             bs=16, dtype="fp32", dist="uniform", lo=1, hi=1, prompts=16, plo=32, phi=511,
             past=0, shape=0),
        # long prompts of a 32-head model, partly behind an earlier chunk
        dict(name="step_prefill_long", kind="step", layers=1, decodes=0, hq=32, hkv=1, d=128,
             bs=16, dtype="bf16", dist="uniform", lo=1, hi=1, prompts=4, plo=1024, phi=4096,
             past=2048, shape=0),
        # one decoder layer of the batch-128 step
        dict(name="block_decode_b128", kind="block", decodes=128, prompts=0, plo=0, phi=0,
             d_model=1024, hq=16, hkv=1, bs=16, dtype="bf16", lo=256, hi=2048, shape=0),
        # the step's end: 128 rows to the GPT-2 vocabulary and a draw from each
        dict(name="head_sample_b128", kind="head", rows=128, d_model=1024, vocab=50257,
             dtype="bf16", pick="sample", top_k=32, top_p=0.9, temperature=0.8),
        # 64 prompts' rows into the pool
        dict(name="append_prompts", kind="append", rows=8192, hkv=1, d=64, bs=16, dtype="bf16"),
        # the whole greedy decode step of the 12-layer model, from its graph
        dict(name="model_decode_graph_b128", kind="model", mode="graph", layers=12,
             d_model=1024, hq=16, hkv=1, vocab=50257, max_seq=4096, bs=16, dtype="bf16",
             decodes=128, lo=256, hi=2048, prompts=0, plo=0, phi=0, shape=0),
        # the default model (34 layers, 512 wide, fp32) taking in eight prompts
        dict(name="model_prefill_default", kind="model", mode="batch", layers=34, d_model=512,
             hq=8, hkv=1, vocab=50257, max_seq=512, bs=16, dtype="fp32", decodes=0, lo=1, hi=1,
             prompts=8, plo=32, phi=511, shape=0),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "step_decode", "step_prefill", "step_prefill",
                       "step_mixed", "block", "head", "append", "model"])
    shape = rng.randrange(1 << 20)
    bs = rng.choice([8, 16, 16, 32])
    if kind == "decode":
        if rng.random() < 0.5:  # small groups, every float type
            hq, hkv, d = rng.choice([(4, 1, 32), (8, 1, 32), (8, 1, 64), (8, 2, 64), (8, 1, 128)])
            dtype, kv = rng.choice(["fp32", "bf16", "fp16"]), "same"
            hi = _logint(rng, 64, 2048)
        else:
            hq, hkv, d = rng.choice([(16, 1, 64), (32, 1, 128), (32, 2, 64), (32, 1, 64)])
            dtype, kv = rng.choice(["bf16", "bf16", "fp16"]), rng.choice(["same", "same", "fp8"])
            hi = _logint(rng, 256, 8192)
        batch = _logint(rng, 1, 256)
        dist = rng.choice(["uniform", "lognormal"])
        lo = max(1, hi // 8)
        return dict(kind="decode", batch=batch, hq=hq, hkv=hkv, d=d, bs=bs, dtype=dtype, kv=kv,
                    dist=dist, lo=lo, hi=hi, shape=shape)
    if kind.startswith("step"):
        small = rng.random() < 0.4
        if small:
            hq, hkv, d = rng.choice([(4, 1, 32), (8, 1, 32), (8, 1, 64), (8, 2, 64)])
            dtype = rng.choice(["fp32", "fp32", "bf16", "fp16"])
            cap = 512
        else:
            hq, hkv, d = rng.choice([(16, 1, 64), (32, 1, 128), (32, 2, 64)])
            dtype = rng.choice(["bf16", "bf16", "fp16"])
            cap = 2048
        decodes = 0 if kind == "step_prefill" else _logint(rng, 1, 256)
        prompts = 0 if kind == "step_decode" else rng.randint(1, 8)
        phi = _logint(rng, 9, cap) if prompts else 0
        past = rng.choice([0, 0, rng.randint(1, cap)]) if prompts else 0
        hi = _logint(rng, 64, 2 * cap)
        return dict(kind="step", layers=rng.randint(1, 2), decodes=decodes, hq=hq, hkv=hkv, d=d,
                    bs=bs, dtype=dtype, dist=rng.choice(["uniform", "lognormal"]),
                    lo=max(1, hi // 8), hi=hi, prompts=prompts, plo=max(2, phi // 4) if phi else 0,
                    phi=phi, past=past, shape=shape)
    if kind == "block":
        d_model, hq, hkv, dtype = rng.choice([(512, 8, 1, "fp32"), (512, 8, 1, "bf16"),
                                              (1024, 16, 1, "bf16"), (1024, 16, 1, "fp16"),
                                              (128, 4, 1, "fp32")])
        prefill = rng.random() < 0.4
        hi = _logint(rng, 32, 512 if dtype == "fp32" else 2048)
        return dict(kind="block", decodes=0 if prefill else _logint(rng, 1, 256),
                    prompts=rng.randint(1, 8) if prefill else 0, plo=max(2, hi // 8) if prefill
                    else 0, phi=min(hi, 512) if prefill else 0, d_model=d_model, hq=hq, hkv=hkv,
                    bs=bs, dtype=dtype, lo=max(1, hi // 8), hi=hi, shape=shape)
    if kind == "head":
        return dict(kind="head", rows=_logint(rng, 1, 256), d_model=rng.choice([128, 512, 1024]),
                    vocab=rng.choice([50257, 50257, _logint(rng, 1000, 50000)]),
                    dtype=rng.choice(["fp32", "bf16", "fp16"]),
                    pick=rng.choice(["sample", "greedy"]), top_k=rng.choice([1, 8, 32, 50]),
                    top_p=rng.choice([0.7, 0.9, 1.0]), temperature=rng.choice([0.7, 1.0, 1.3]))
    if kind == "append":
        return dict(kind="append", rows=_logint(rng, 1, 16384), hkv=rng.choice([1, 1, 2]),
                    d=rng.choice([32, 64, 128]), bs=bs, dtype=rng.choice(["fp32", "bf16", "fp16"]))
    mode = rng.choice(["graph", "batch"])
    layers, d_model, hq, dtype, cap = rng.choice([(4, 128, 4, "fp32", 256), (8, 512, 8, "fp32", 512),
                                                  (8, 512, 8, "bf16", 512),
                                                  (6, 1024, 16, "bf16", 1024)])
    prefill = mode == "batch" and rng.random() < 0.5
    hi = _logint(rng, 32, cap - 8)
    return dict(kind="model", mode=mode, layers=layers, d_model=d_model, hq=hq, hkv=1,
                vocab=50257, max_seq=cap, bs=bs, dtype=dtype,
                decodes=0 if prefill else _logint(rng, 1, 128), lo=max(1, hi // 8), hi=hi,
                prompts=rng.randint(1, 8) if prefill else 0, plo=max(2, hi // 8) if prefill else 0,
                phi=hi if prefill else 0, shape=shape)


# ---------------------------------------------------------------- geometry
def _contexts(case, n):
    """Tokens already cached of n decoding sequences."""
    if n == 0:
        return []
    rng = np.random.default_rng(case["shape"])
    lo, hi = case["lo"], case["hi"]
    if case.get("dist", "uniform") == "uniform":
        return [int(x) for x in rng.integers(lo, hi + 1, size=n)]
    x = rng.lognormal(math.log(lo) - 0.5, 1.0, size=n)  # mean lo, sigma 1
    return [int(v) for v in np.clip(np.rint(x), 1, hi)]


def _runs(case):
    """(start, new tokens) of every sequence of a step: decodes, then prompts."""
    runs = [(c, 1) for c in _contexts(case, case["decodes"])]
    rng = np.random.default_rng(case["shape"] + 1)
    for i in range(case["prompts"]):
        new = int(rng.integers(case["plo"], case["phi"] + 1))
        past = case.get("past", 0)
        runs.append((int(rng.integers(1, past + 1)) if past and i % 2 else 0, new))
    return runs


def _blocks(ends, bs):
    return sum(-(-e // bs) for e in ends) * 5 // 4 + 2


def _tables(ends, bs, seed):
    """Scattered, disjoint block lists covering each sequence's tokens."""
    perm = np.random.default_rng(seed).permutation(np.arange(1, _blocks(ends, bs)))
    tables, at = [], 0
    for e in ends:
        n = -(-e // bs)
        tables.append([int(b) for b in perm[at:at + n]])
        at += n
    return tables


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * std).to(dtype)


def _positions(runs):
    return [p for s, n in runs for p in range(s, s + n)]


def _starts(runs):
    return np.concatenate([[0], np.cumsum([n for _, n in runs])]).tolist()


# ---------------------------------------------------------------- inputs
def _decode_inputs(case, seed):
    lens = _contexts(case, case["batch"])
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    nb = _blocks(lens, case["bs"])
    shape = (nb, case["bs"], case["hkv"], case["d"])
    pdt = torch.float8_e4m3fn if case["kv"] == "fp8" else dt
    return dict(lens=lens, tables=_tables(lens, case["bs"], seed),
                q=_normal(g, len(lens), case["hq"], case["d"], dtype=dt),
                k=_normal(g, *shape, dtype=pdt), v=_normal(g, *shape, dtype=pdt))


def _step_inputs(case, seed, layers, d):
    runs = _runs(case)
    ends = [s + n for s, n in runs]
    T = sum(n for _, n in runs)
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    kv = _normal(g, layers, 2, _blocks(ends, case["bs"]), case["bs"], case["hkv"], d, dtype=dt)
    return dict(runs=runs, ends=ends, T=T, g=g, dt=dt, kv=kv,
                tables=_tables(ends, case["bs"], seed))


def _pool(i, case, layers, d):
    pool = KVPool(layers, case["bs"], i["kv"].shape[2], case["hkv"], d, i["dt"], DEV)
    pool.kv.copy_(i["kv"])
    return pool


def _block_weights(g, dm, hkv_d, dt):
    std = 1 / math.sqrt(3 * dm)  # the variance of nn.Linear's default
    lin = lambda n: _normal(g, n, dm, dtype=dt, std=std)  # noqa: E731
    norm = lambda: (1 + 0.1 * torch.randn(dm, generator=g, device=DEV)).to(dt)  # noqa: E731
    return {"attn_norm.weight": norm(), "attn.q_proj.weight": lin(dm),
            "attn.k_proj.weight": lin(hkv_d), "attn.v_proj.weight": lin(hkv_d),
            "attn.out.weight": lin(dm), "mlp_norm.weight": norm(),
            "mlp.gate_proj.weight": lin(dm), "mlp.up_proj.weight": lin(dm),
            "mlp.down_proj.weight": lin(dm)}


def _config(case, layers=1, vocab=8, max_seq=4096):
    return ModelConfig(vocab_size=vocab, d_model=case["d_model"], num_layers=layers,
                       num_heads=case["hq"], num_kv_heads=case["hkv"], max_seq_len=max_seq,
                       dtype=DTYPES[case["dtype"]])


def _head_inputs(case, seed):
    g, dt, dm = _gen(seed), DTYPES[case["dtype"]], case["d_model"]
    return dict(x=_normal(g, case["rows"], dm, dtype=dt, std=3.0),
                norm=(1 + 0.1 * torch.randn(dm, generator=g, device=DEV)).to(dt),
                w=_normal(g, case["vocab"], dm, dtype=dt, std=2 / math.sqrt(dm)),
                u=torch.rand(case["rows"], generator=g, device=DEV))


def _model_inputs(case, seed):
    i = _step_inputs(case, seed, case["layers"], case["d_model"] // case["hq"])
    g, dm, dt = i["g"], case["d_model"], i["dt"]
    hkv_d = case["hkv"] * dm // case["hq"]
    w = {"embedding.embedding.weight": _normal(g, case["vocab"], dm, dtype=dt)}
    for n in range(case["layers"]):
        w.update({f"layers.{n}.{k}": t for k, t in _block_weights(g, dm, hkv_d, dt).items()})
    w["final_norm.weight"] = (1 + 0.1 * torch.randn(dm, generator=g, device=DEV)).to(dt)
    w["lm_head.weight"] = _normal(g, case["vocab"], dm, dtype=dt, std=2 / math.sqrt(dm))
    i["w"] = w
    i["ids"] = torch.randint(0, case["vocab"], (i["T"],), generator=g, device=DEV)
    return i


def _append_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    nb = case["rows"] // case["bs"] * 5 // 4 + 3
    slots = np.random.default_rng(seed).permutation(np.arange(1, nb))
    pos = np.arange(case["rows"])
    slots = slots[pos // case["bs"]] * case["bs"] + pos % case["bs"]
    shape = (case["rows"], case["hkv"], case["d"])
    return dict(nb=nb, slots=torch.from_numpy(slots.astype(np.int64)).to(DEV),
                k=_normal(g, *shape, dtype=dt), v=_normal(g, *shape, dtype=dt))


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        i = _decode_inputs(case, seed)
        width = max(len(t) for t in i["tables"])
        tab = torch.zeros((len(i["tables"]), width), dtype=torch.int32)
        for n, t in enumerate(i["tables"]):
            tab[n, :len(t)] = torch.tensor(t, dtype=torch.int32)
        return dict(kind=kind, q=i["q"], k=i["k"], v=i["v"], tables=tab.to(DEV),
                    lens=torch.tensor(i["lens"], dtype=torch.int32).to(DEV),
                    max_kv=max(i["lens"]))
    if kind == "step":
        i = _step_inputs(case, seed, case["layers"], case["d"])
        rows = [[_normal(i["g"], i["T"], h, case["d"], dtype=i["dt"])
                 for h in (case["hq"], case["hkv"], case["hkv"])] for _ in range(case["layers"])]
        meta = pack_batch_meta(i["tables"], _starts(i["runs"]), _positions(i["runs"]), i["T"],
                               DEV, case["bs"])
        return dict(kind=kind, pool=_pool(i, case, case["layers"], case["d"]), rows=rows,
                    meta=meta)
    if kind == "block":
        d = case["d_model"] // case["hq"]
        i = _step_inputs(case, seed, 1, d)
        with torch.device(DEV):
            block = PagedBlock(_config(case), 0).to(i["dt"]).eval()
        block.load_state_dict(_block_weights(i["g"], case["d_model"], case["hkv"] * d, i["dt"]))
        x = _normal(i["g"], i["T"], case["d_model"], dtype=i["dt"])
        meta = pack_batch_meta(i["tables"], _starts(i["runs"]), _positions(i["runs"]), i["T"],
                               DEV, case["bs"])
        return dict(kind=kind, pool=_pool(i, case, 1, d), block=block, x=x, meta=meta)
    if kind == "head":
        i = _head_inputs(case, seed)
        with torch.device(DEV):
            norm = RMSNorm(case["d_model"], EPS).to(i["w"].dtype)
            head = torch.nn.Linear(case["d_model"], case["vocab"], bias=False).to(i["w"].dtype)
        norm.load_state_dict({"weight": i["norm"]})
        head.load_state_dict({"weight": i["w"]})
        return dict(kind=kind, x=i["x"], u=i["u"], norm=norm, head=head, pick=case["pick"],
                    args=(case["temperature"], case["top_k"], case["top_p"]))
    if kind == "append":
        i = _append_inputs(case, seed)
        return dict(kind=kind, slots=i["slots"], k=i["k"], v=i["v"],
                    pool=KVPool(1, case["bs"], i["nb"], case["hkv"], case["d"],
                                DTYPES[case["dtype"]], DEV))
    i = _model_inputs(case, seed)
    with torch.device(DEV):
        model = PagedTransformer(_config(case, case["layers"], case["vocab"],
                                         case["max_seq"])).to(i["dt"]).eval()
    model.load_state_dict(i["w"])
    pool = _pool(i, case, case["layers"], case["d_model"] // case["hq"])
    if case["mode"] == "batch":
        step = BatchStep(input_ids=i["ids"], positions=_positions(i["runs"]),
                         query_start_loc=_starts(i["runs"]), block_tables=i["tables"],
                         seq_lens=i["ends"])
        return dict(kind="batch", model=model, pool=pool, step=step)
    meta = pack_batch_meta(i["tables"], _starts(i["runs"]), _positions(i["runs"]), i["T"], DEV,
                           case["bs"])
    state = dict(kind="graph", pool=pool, ids=i["ids"], at=meta.step_view.clone())
    state["graph"] = DecodeStepGraph(model, pool, meta, i["ids"])
    return state


# ---------------------------------------------------------------- run
@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "decode":
        return paged_mqa_decode(state["q"], state["k"], state["v"], state["tables"],
                                state["lens"], max_kv_len=state["max_kv"])
    if kind == "step":
        outs = [paged_attention_append_meta(q, k, v, state["pool"], n, state["meta"])
                for n, (q, k, v) in enumerate(state["rows"])]
        return outs + [state["pool"].kv]
    if kind == "block":
        x, b = state["x"].clone(), state["block"]
        b.attn.forward_meta_residual_(x, b.attn_norm, state["pool"], 0, state["meta"])
        b.mlp.forward_residual_(x, b.mlp_norm)
        return [x, state["pool"].kv]
    if kind == "head":
        logits = state["head"](state["norm"](state["x"]))
        if state["pick"] == "greedy":
            return [logits, fused_ops.argmax_rows(logits)]
        return [logits, fused_ops.sample_rows(logits, *state["args"], state["u"])[0]]
    if kind == "append":
        state["pool"].write(0, state["slots"], state["k"], state["v"])
        return state["pool"].kv
    if kind == "batch":
        return [state["model"].forward_batch(state["step"], state["pool"]), state["pool"].kv]
    # the server writes the step's tokens and positions, then replays
    graph = state["graph"]
    graph.ids.copy_(state["ids"])
    graph.meta.step_view.copy_(state["at"])
    ids = graph.replay()
    return [graph.logits, ids, state["pool"].kv]


# ---------------------------------------------------------------- work
def _attn_work(runs, hq, hkv, d, bs, es, kes):
    T = sum(n for _, n in runs)
    kv = sum(s + n for s, n in runs)
    seen = sum(n * s + n * (n + 1) // 2 for s, n in runs)
    bytes_ = (2 * kv * hkv * d * kes + 2 * T * hq * d * es
              + 4 * sum(-(-(s + n) // bs) for s, n in runs) + 8 * len(runs))
    return bytes_, 4 * hq * d * seen


def work(case):
    kind, es = case["kind"], ESIZE[case["dtype"]]
    if kind == "decode":
        runs = [(c - 1, 1) for c in _contexts(case, case["batch"])]
        b, f = _attn_work(runs, case["hq"], case["hkv"], case["d"], case["bs"], es,
                          1 if case["kv"] == "fp8" else es)
        return {"bytes": b, "flops": f}
    if kind == "append":
        n = 4 * case["rows"] * case["hkv"] * case["d"] * es + 8 * case["rows"]
        return {"bytes": n, "flops": 0}
    if kind == "head":
        m, n, k = case["rows"], case["vocab"], case["d_model"]
        return {"bytes": (n * k + m * k + m * n) * es + 12 * m, "flops": 2 * m * n * k}
    runs = _runs(case)
    T = sum(n for _, n in runs)
    d = case["d"] if kind == "step" else case["d_model"] // case["hq"]
    b, f = _attn_work(runs, case["hq"], case["hkv"], d, case["bs"], es, es)
    row = case["hkv"] * d * es
    if kind == "step":  # the new rows come from memory and go to the pool
        return {"bytes": case["layers"] * (b + 2 * T * row), "flops": case["layers"] * f}
    # weights once; activations between a layer's kernels need not reach memory
    dm = case["d_model"]
    wn = 2 * dm * dm + 2 * case["hkv"] * d * dm + 3 * dm * dm
    b = b - 2 * T * case["hq"] * d * es + wn * es
    f = f + 2 * T * wn
    if kind == "block":
        return {"bytes": b + 2 * T * dm * es, "flops": f}
    n = len(runs)
    head = case["vocab"] * dm * es + n * case["vocab"] * es + T * dm * es + 8 * T
    return {"bytes": case["layers"] * b + head,
            "flops": case["layers"] * f + 2 * n * case["vocab"] * dm}


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times the distance to exact() measured on one MI355X: fp32
    attention 2.4e-7, block 1.2e-7, head 5.8e-7, 34-layer model 7e-7; bf16
    attention 0.0028, block 0.0024, head 0.0023, 12-layer model 0.009; fp16
    an eighth of bf16 (three more mantissa bits). Token choices move where two
    candidates lie within that distance."""
    kind, dt = case["kind"], case["dtype"]
    if kind == "append":
        return "exact"
    half = {"bf16": 1.0, "fp16": 0.125}.get(dt)
    if kind == "model":
        return {"rel": 4e-6 if half is None else 4e-2 * half, "differ": 0.2}
    if kind == "head":
        return {"rel": 2.5e-6 if half is None else 1e-2 * half, "differ": 0.05}
    return {"rel": 2e-6 if half is None else 1.1e-2 * half}


# ---------------------------------------------------------------- exact
def _rows_of(table, n, bs):
    p = torch.arange(n, device=DEV)
    return torch.tensor(table, device=DEV)[p // bs] * bs + p % bs


def _attend(q, k, v, start):
    """q [n, hq, d], k / v [kv, hkv, d] in 64 bits; query i sees key j <= start + i."""
    n, hq, d = q.shape
    kv, hkv, _ = k.shape
    out = torch.empty_like(q)
    grp = hq // hkv
    for h in range(hkv):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for a in range(0, n, 256):
            m = min(256, n - a)
            s = (q[a:a + m, h * grp:(h + 1) * grp].reshape(m * grp, d) @ kt) / math.sqrt(d)
            s = s.view(m, grp, kv)
            if n > 1:
                last = start + a + torch.arange(m, device=DEV)
                hide = torch.arange(kv, device=DEV)[None, :] > last[:, None]
                s = s.masked_fill(hide[:, None, :], -math.inf)
            p = torch.softmax(s, -1).view(m * grp, kv)
            out[a:a + m, h * grp:(h + 1) * grp] = (p @ vh).view(m, grp, d)
    return out


def _step_exact(i, case, kv, q, k, v):
    """One layer: rows into kv [2, blocks, bs, hkv, d], then attention."""
    flat = kv.view(2, -1, *kv.shape[3:])
    outs, at = [], 0
    for (start, n), table in zip(i["runs"], i["tables"]):
        rows = _rows_of(table, start + n, case["bs"])
        flat[0, rows[start:]] = k[at:at + n]
        flat[1, rows[start:]] = v[at:at + n]
        outs.append(_attend(q[at:at + n], flat[0, rows], flat[1, rows], start))
        at += n
    return torch.cat(outs)


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, positions, theta=10000.0):
    d = x.shape[-1]
    inv = 1.0 / (theta ** (torch.arange(0, d, 2, device=DEV).float() / d))
    # the rotation tables are the model's fp32 buffers
    ang = torch.outer(positions.float(), inv)
    c, s = ang.cos().double()[:, None], ang.sin().double()[:, None]
    y = torch.empty_like(x)
    y[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * s
    y[..., 1::2] = x[..., 0::2] * s + x[..., 1::2] * c
    return y


def _block64(x, w, i, case, kv, positions):
    T, hq, hkv = x.shape[0], case["hq"], case["hkv"]
    d = case["d_model"] // hq
    lin = lambda a, name: a @ w[name].double().t()  # noqa: E731
    h = _norm64(x, w["attn_norm.weight"])
    q = _rope64(lin(h, "attn.q_proj.weight").view(T, hq, d), positions)
    k = _rope64(lin(h, "attn.k_proj.weight").view(T, hkv, d), positions)
    v = lin(h, "attn.v_proj.weight").view(T, hkv, d)
    x = x + lin(_step_exact(i, case, kv, q, k, v).view(T, -1), "attn.out.weight")
    h = _norm64(x, w["mlp_norm.weight"])
    gate = torch.nn.functional.silu(lin(h, "mlp.gate_proj.weight"))
    return x + lin(gate * lin(h, "mlp.up_proj.weight"), "mlp.down_proj.weight")


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "append":
        return None  # a copy: compared byte for byte
    if kind == "decode":
        i = _decode_inputs(case, seed)
        k, v = (i[n].double().view(-1, case["hkv"], case["d"]) for n in ("k", "v"))
        outs = []
        for n, (table, kv) in enumerate(zip(i["tables"], i["lens"])):
            rows = _rows_of(table, kv, case["bs"])
            outs.append(_attend(i["q"][n:n + 1].double(), k[rows], v[rows], kv - 1))
        return torch.cat(outs)
    if kind == "head":
        i = _head_inputs(case, seed)
        return [_norm64(i["x"].double(), i["norm"]) @ i["w"].double().t(), None]
    if kind == "step":
        i = _step_inputs(case, seed, case["layers"], case["d"])
        kv, outs = i["kv"].double(), []
        for n in range(case["layers"]):
            q, k, v = (_normal(i["g"], i["T"], h, case["d"], dtype=i["dt"]).double()
                       for h in (case["hq"], case["hkv"], case["hkv"]))
            outs.append(_step_exact(i, case, kv[n], q, k, v))
        return outs + [kv]
    if kind == "block":
        d = case["d_model"] // case["hq"]
        i = _step_inputs(case, seed, 1, d)
        w = _block_weights(i["g"], case["d_model"], case["hkv"] * d, i["dt"])
        x = _normal(i["g"], i["T"], case["d_model"], dtype=i["dt"]).double()
        kv = i["kv"].double()
        pos = torch.tensor(_positions(i["runs"]), device=DEV)
        return [_block64(x, w, i, case, kv[0], pos), kv]
    i = _model_inputs(case, seed)
    w, kv = i["w"], i["kv"].double()
    pos = torch.tensor(_positions(i["runs"]), device=DEV)
    x = w["embedding.embedding.weight"][i["ids"]].double()
    for n in range(case["layers"]):
        part = {k[len(f"layers.{n}."):]: t for k, t in w.items() if k.startswith(f"layers.{n}.")}
        x = _block64(x, part, i, case, kv[n], pos)
    last = torch.tensor(_starts(i["runs"])[1:], device=DEV) - 1
    logits = _norm64(x[last], w["final_norm.weight"]) @ w["lm_head.weight"].double().t()
    return [logits, kv] if case["mode"] == "batch" else [logits, None, kv]
