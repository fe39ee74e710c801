"""The work this package is used for, as measurable cases: steps of a serving engine through ``Attention.forward`` and
the attention operators, over the real range of batch sizes, prompt and context lengths.

A case is one engine step's attention over a stack of layers that share the step's lengths and block tables, each layer
with its own rows and cache planes, as the model's layers have them: 16 query heads over 2 kv heads, head_dim 128, bf16,
256-token cache blocks from a shuffled pool. Steps that an engine captures (decode, prefill over a cached prefix, mixed
steps, the diffusion transformer's rows) are HIP graphs over static buffers, captured once and replayed; the others run
eagerly. A pass returns every layer's output and, where the step writes it, the whole KV cache.

Kinds: ``decode`` (one query per sequence), ``prefill`` (new tokens, with or without cached prefixes and the int8
output of the W8A8 layers), ``mixed`` (prefills and decode rows in one step), ``local`` (non-causal rows of a fixed
short length)."""

from __future__ import annotations

import random

import torch

from voxcpm2_arabic_dialects_turbo_amd import runner
from voxcpm2_arabic_dialects_turbo_amd.context import reset_context
from voxcpm2_arabic_dialects_turbo_amd.layers import Attention
from voxcpm2_arabic_dialects_turbo_amd.ops import prefill_attention_store

H, HK, D, BS = 16, 2, 128, 256
SCALE = D ** -0.5
DEV = "cuda"


def listed():
    return [
        # one speaker being served alone: the latency of every generated frame
        {"name": "decode_1", "kind": "decode", "batch": 1, "lo": 420, "hi": 420, "max_len": 1024, "layers": 28},
        # a handful of streams at the production length limit of 1024
        {"name": "decode_6", "kind": "decode", "batch": 6, "lo": 100, "hi": 1000, "max_len": 1024, "layers": 28},
        # an ordinary load: 40 streams
        {"name": "decode_40", "kind": "decode", "batch": 40, "lo": 200, "hi": 1500, "max_len": 2048, "layers": 28},
        # peak concurrency, the headline decode step
        {"name": "decode_150", "kind": "decode", "batch": 150, "lo": 256, "hi": 2048, "max_len": 2048, "layers": 28},
        # long-form reading: few streams near the engine's default length limit of 4096
        {"name": "decode_long", "kind": "decode", "batch": 13, "lo": 2500, "hi": 4096, "max_len": 4096, "layers": 28},
        # one request's prompt: the attention part of the time to its first frame (keys through the block tables, as
        # in a captured prefill)
        {"name": "prefill_1", "kind": "prefill", "batch": 1, "lo": 237, "hi": 237, "prefix_lo": 0, "prefix_hi": 0,
         "tables": True, "int8": False, "graph": True, "layers": 28},
        # eight prompts admitted together
        {"name": "prefill_8", "kind": "prefill", "batch": 8, "lo": 64, "hi": 512, "prefix_lo": 0, "prefix_hi": 0,
         "tables": False, "int8": False, "graph": True, "layers": 8},
        # a burst of short texts after a cached voice prompt, keys through the block tables
        {"name": "prefill_prefix", "kind": "prefill", "batch": 44, "lo": 33, "hi": 59, "prefix_lo": 50,
         "prefix_hi": 50, "tables": True, "int8": False, "graph": True, "layers": 8},
        # long texts: compute-bound
        {"name": "prefill_long", "kind": "prefill", "batch": 9, "lo": 1500, "hi": 4096, "prefix_lo": 0, "prefix_hi": 0,
         "tables": False, "int8": False, "graph": False, "layers": 2},
        # prompts admitted while other streams decode, in one step
        {"name": "mixed", "kind": "mixed", "batch": 6, "lo": 300, "hi": 600, "decodes": 120, "ctx_lo": 128,
         "ctx_hi": 1800, "layers": 8},
        # the head-start step of a burst, W8A8 layers (int8 output), run eagerly as the W8A8 prefill is
        {"name": "headstart_int8", "kind": "prefill", "batch": 200, "lo": 5, "hi": 9, "prefix_lo": 0, "prefix_hi": 0,
         "tables": False, "int8": True, "graph": False, "layers": 8},
        # the diffusion transformer's non-causal rows of 150 streams, its 12 layers
        {"name": "local_150", "kind": "local", "batch": 150, "length": 11, "layers": 12},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["decode", "decode", "prefill", "prefill", "int8", "mixed", "local"])
    if kind == "decode":
        batch = log(1, 256)
        max_len = rng.choice([1024, 2048, 4096])
        hi = min(max_len, 150 * 1100 // batch)  # at most the tokens of the peak step
        lo = rng.randint(max(1, hi // 20), hi)
        return {"kind": "decode", "batch": batch, "lo": lo, "hi": hi, "max_len": max_len, "layers": 28}
    if kind == "local":
        return {"kind": "local", "batch": log(1, 256), "length": rng.choice([5, 7, 11, 16]), "layers": 12}
    if kind == "mixed":
        hi = log(40, 1000)
        return {"kind": "mixed", "batch": rng.randint(1, 8), "lo": max(2, hi // 2), "hi": hi,
                "decodes": log(12, 200), "ctx_lo": 60, "ctx_hi": log(200, 2048), "layers": 8}
    if kind == "int8":  # short texts, alone or after a voice prompt
        prefix = rng.choice([0, rng.randint(20, 120)])
        hi = rng.randint(6, 60)
        return {"kind": "prefill", "batch": log(1, 200), "lo": max(2, hi // 2), "hi": hi, "prefix_lo": prefix // 2,
                "prefix_hi": prefix, "tables": prefix > 0, "int8": True, "graph": False, "layers": 8}
    hi = log(8, 4096)
    batch = log(1, max(1, min(64, 20000 // hi)))
    prefix = rng.choice([0, rng.randint(20, 300)])
    return {"kind": "prefill", "batch": batch, "lo": max(2, rng.randint(hi // 8, hi)), "hi": hi,
            "prefix_lo": prefix // 2, "prefix_hi": prefix, "tables": prefix > 0 or rng.random() < 0.5, "int8": False,
            "graph": hi <= 1024, "layers": 8 if hi <= 1024 else 2}


def _lens(case, what, n, lo, hi):
    """n lengths uniform in [lo, hi], the same for every seed of a case (the work depends on them)."""
    rng = random.Random("%s %d %d %d" % (what, n, lo, hi))
    return [rng.randint(lo, hi) for _ in range(n)]


def _sequences(case):
    """(new tokens, all tokens) of each sequence of the step."""
    if case["kind"] == "decode":
        return [(1, n) for n in _lens(case, "ctx", case["batch"], case["lo"], case["hi"])]
    new = _lens(case, "new", case["batch"], case["lo"], case["hi"])
    if case["kind"] == "mixed":
        return [(n, n) for n in new] + [(1, n) for n in _lens(case, "ctx", case["decodes"], case["ctx_lo"],
                                                              case["ctx_hi"])]
    return [(n, n + p) for n, p in zip(new, _lens(case, "prefix", case["batch"], case["prefix_lo"],
                                                  case["prefix_hi"]))]


def _tables(seqs, seed):
    """Block tables from a shuffled pool a little larger than the step needs, and the pool's size."""
    need = [-(-n // BS) for _, n in seqs]
    pool = sum(need) + max(4, sum(need) // 16)
    perm = list(range(pool))
    random.Random(seed).shuffle(perm)
    tables, at = [], 0
    for nb in need:
        tables.append(perm[at:at + nb])
        at += nb
    return tables, pool


def _normal(shape, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)


def _rows(case, layers, n, seed):
    """Per layer: a qkv projection's output rows [n, (H + 2 HK) D], and q / k / v as views of them."""
    qkv = _normal((layers, n, (H + 2 * HK) * D), seed)
    return [(x[:, :H * D].view(n, H, D), x[:, H * D:(H + HK) * D].view(n, HK, D),
             x[:, (H + HK) * D:].view(n, HK, D)) for x in qkv]


def _inputs(case, seed):
    layers = case["layers"]
    if case["kind"] == "local":
        b, n = case["batch"], case["length"]
        rows = _rows(case, layers, b * n, 2 * seed)
        return {"rows": [(q.view(b, n, H, D), k.view(b, n, HK, D), v.view(b, n, HK, D)) for q, k, v in rows]}
    seqs = _sequences(case)
    tables, pool = _tables(seqs, seed)
    kv = _normal((layers, 2, pool, BS, HK, D), 2 * seed + 1)
    rows = _rows(case, layers, _step_rows(case, seqs), 2 * seed)
    smooth = None
    if case.get("int8"):
        gen = torch.Generator(device=DEV).manual_seed(2 * seed + 5)
        smooth = 0.5 + torch.rand(layers, H * D, generator=gen, device=DEV)
    return {"seqs": seqs, "tables": tables, "kv": kv, "rows": rows, "smooth": smooth}


def _step_rows(case, seqs):
    """Rows of the step: every new token, and in a decode step the padding up to the captured batch size."""
    if case["kind"] != "decode":
        return sum(n for n, _ in seqs)
    return min(b for b in runner.graph_batch_sizes(256) if b >= case["batch"])


def _capture(forward):
    """Captures forward() after warm-up runs on a side stream; returns the graph and the captured outputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        forward()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = forward()
    return graph, out


def prepare(case, seed):
    reset_context()
    x = _inputs(case, seed)
    layers = case["layers"]
    if case["kind"] == "local":
        model = [Attention(H, D, SCALE, HK, is_causal=False) for _ in range(layers)]
        graph, out = _capture(lambda: [m(*r) for m, r in zip(model, x["rows"])])
        return {"graph": graph, "out": out, "inputs": x}
    model = [Attention(H, D, SCALE, HK) for _ in range(layers)]
    kv = runner.allocate_kv_cache(model, x["kv"].shape[2], BS, device=DEV)
    kv.copy_(x.pop("kv"))
    tasks = [runner.RunnerTask(t, n, n - new, BS) for t, (new, n) in zip(x["tables"], x["seqs"])]
    s = {"inputs": x, "model": model, "kv": kv}
    if case["kind"] == "decode":
        bs = x["rows"][0][0].shape[0]
        bufs = runner.DecodeGraphBuffers(bs, runner.num_blocks_for(case["max_len"], BS), device=DEV)
        runner.prepare_decode_context(tasks, BS, device=DEV)
        bufs.load()
        bufs.bind(bs)
        graph, out = _capture(lambda: [m(*r) for m, r in zip(model, x["rows"])])
        reset_context()
        s.update(graph=graph, out={"o": out, "kv": kv}, bufs=bufs)
        return s
    if case["kind"] == "mixed" or case["graph"]:
        staging = runner.StepStaging(DEV)
        runner.prepare_prefill_context(tasks, BS, device=DEV, graphs=case.get("tables", True), staging=staging)
        context = runner.get_context()
        graph, out = _capture(lambda: [m(*r) for m, r in zip(model, x["rows"])])
        reset_context()
        s.update(graph=graph, out={"o": out, "kv": kv}, context=context)
        return s
    s.update(tasks=tasks, staging=runner.StepStaging(DEV), int8=case["int8"], tables=case["tables"])
    return s


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    # an eager prefill step: its context from the host, then every layer
    x, staging = state["inputs"], state["staging"]
    runner.prepare_prefill_context(state["tasks"], BS, device=DEV, graphs=state["tables"], staging=staging)
    c = runner.get_context()
    out = []
    for i, (m, (q, k, v)) in enumerate(zip(state["model"], x["rows"])):
        if state["int8"]:
            out.append(prefill_attention_store(q, k, v, m.k_cache, m.v_cache, c.slot_mapping,
                                               cu_seqlens_q=c.cu_seqlens_q, cu_seqlens_k=c.cu_seqlens_k,
                                               max_seqlen_q=c.max_seqlen_q, softmax_scale=SCALE,
                                               block_table=c.block_tables, quant=True, inv_smooth=x["smooth"][i]))
        else:
            out.append(m(q, k, v))
    reset_context()
    return {"o": out, "kv": state["kv"]}


def work(case):
    layers = case["layers"]
    if case["kind"] == "local":
        b, n = case["batch"], case["length"]
        return {"bytes": layers * b * n * (2 * H + 2 * HK) * D * 2, "flops": layers * 4 * D * H * b * n * n}
    seqs = _sequences(case)
    rows = sum(n for n, _ in seqs)
    keys = sum(n for _, n in seqs)
    pairs = sum(new * (n - new) + new * (new + 1) // 2 for new, n in seqs)
    out = H * D + 4 if case.get("int8") else H * D * 2
    # q read, output written, every key and value read once, the new rows written to the cache
    per_layer = rows * (H * D * 2 + out) + (keys + rows) * 2 * HK * D * 2
    return {"bytes": layers * per_layer, "flops": layers * 4 * D * H * pairs}


def tolerance(case):
    # bf16 outputs of fp32 sums: the probabilities' and the output's roundings, 2^-9 each, beside another order of sums
    if case.get("int8"):
        return {"rel": 1e-2, "max": 0.4, "differ": 0.01}
    return {"rel": 1e-2, "max": 0.4}


def _attend(q, k, v, causal):
    """q [n, H, D] over k / v [m, HK, D] in 64 bits, query i at position m - n + i."""
    n, m = q.shape[0], k.shape[0]
    q = q.double().view(n, HK, H // HK, D).permute(1, 2, 0, 3).reshape(HK, -1, D)
    s = torch.matmul(q, k.double().permute(1, 2, 0).contiguous()).view(HK, H // HK, n, m) * SCALE
    if causal:
        i = torch.arange(n, device=DEV)[:, None] + (m - n)
        s.masked_fill_(torch.arange(m, device=DEV)[None, :] > i, float("-inf"))
    p = torch.softmax(s, -1).view(HK, -1, m)
    del s
    o = torch.matmul(p, v.double().permute(1, 0, 2).contiguous())
    return o.view(HK, H // HK, n, D).permute(2, 0, 1, 3).reshape(n, H, D)


def exact(case, seed):
    x = _inputs(case, seed)
    if case["kind"] == "local":
        return [torch.stack([_attend(q[b], k[b], v[b], False) for b in range(case["batch"])]) for q, k, v in x["rows"]]
    kv, out = x["kv"], []
    for i, (q, k, v) in enumerate(x["rows"]):
        o, at = torch.zeros(q.shape[0], H, D, dtype=torch.float64, device=DEV), 0
        for (new, n), table in zip(x["seqs"], x["tables"]):
            pos = torch.arange(n - new, n, device=DEV)
            t = torch.tensor(table, device=DEV)
            kv[i, 0, t[pos // BS], pos % BS] = k[at:at + new]
            kv[i, 1, t[pos // BS], pos % BS] = v[at:at + new]
            keys, values = (kv[i, j, t].reshape(-1, HK, D)[:n] for j in (0, 1))
            for a in range(0, new, 512):  # queries in slices, for their scores' memory
                e = min(new, a + 512)
                m = n - new + e
                o[at + a:at + e] = _attend(q[at + a:at + e], keys[:m], values[:m], True)
            at += new
        if case.get("int8"):
            y = o.view(-1, H * D) * x["smooth"][i].double()
            out.append((None, y.abs().amax(1).clamp_min(1e-6) / 127))
        else:
            out.append(o.unsqueeze(1) if case["kind"] == "decode" else o)
    return {"o": out, "kv": kv}
