"""The workloads whose time is followed here: the calls a serving engine makes
of this framework, from one user's decode step to a full mixed batch.

  listed()              the fixed cases
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   inputs, pools, layers and captured graphs on the GPU
  run(state)            one pass through the public entry points; its outputs
  work(case)            bytes and operations a pass cannot do without
  tolerance(case)       how far another correct implementation may be
  exact(case, seed)     the outputs in 64-bit torch, without this package

Three kinds of case:

  attention  AttentionLayer.forward (qk-norm, RoPE, KV store, paged attention)
             on decode, prefill and mixed batches; eagerly for one layer, or a
             whole step of layers through a captured graph with the step's
             prepare_metadata and prepare_for_replay.
  block      the rest of a transformer block between the GEMMs: fused add +
             RMSNorm and the gated activation; eagerly, or as a captured step.
  sampler    the Sampler step: a token per row of logits, either with
             sample_from_logits or as probabilities and then a draw.

Sizes are those of the Qwen3 models the benchmark uses (0.6B 16q/8kv, 8B
32q/8kv, 30B-A3B 32q/4kv, head dim 128, vocabulary 151,936). Request lengths
are drawn from the case's own `lengths` number, so a case's work is the same
for every seed; the seed makes the data.
"""
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
D = 128
VOCAB = 151_936
ROUNDS = 32       # uniforms per row the Sampler hands to the rejection draws
MAX_POS = 40_960  # Qwen3's position range
EPS = 1e-6
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _backend():
    """The C++ backend module (the package's directory name is not a Python
    identifier, so it is loaded by path)."""
    name = "sglang_cpp_amd"
    if name not in sys.modules:
        pkg = ROOT / "sglang.cpp_amd"
        spec = importlib.util.spec_from_file_location(
            name, pkg / "__init__.py", submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name].backend.load()


# ------------------------------------------------------------------ cases

def _attention(hq, hkv, page, lengths, dec=0, dec_lo=1, dec_hi=1, pre=0, new_lo=1, new_hi=1,
               cached_lo=0, cached_hi=0, layers=1, graph=False):
    return dict(kind="attention", hq=hq, hkv=hkv, page=page, lengths=lengths, dec=dec,
                dec_lo=dec_lo, dec_hi=dec_hi, pre=pre, new_lo=new_lo, new_hi=new_hi,
                cached_lo=cached_lo, cached_hi=cached_hi, layers=layers, graph=graph)


def _block(tokens, hidden, inter, dtype="bf16", act="silu", layers=1, graph=False):
    return dict(kind="block", tokens=tokens, hidden=hidden, inter=inter, dtype=dtype, act=act,
                layers=layers, graph=graph)


def _sampler(rows, dtype="bf16", mode="top_k_top_p", route="logits"):
    return dict(kind="sampler", rows=rows, dtype=dtype, mode=mode, route=route)


def listed():
    return [
        # A few chat users on the smallest model: every layer of one captured
        # decode step, where launches and latency are all there is.
        dict(name="decode_step_b4", **_attention(16, 8, 1, 1, dec=4, dec_lo=380, dec_hi=640,
                                                 layers=28, graph=True)),
        # One user far into a long chat, one layer.
        dict(name="decode_b1_long", **_attention(32, 8, 16, 2, dec=1, dec_lo=12_001,
                                                 dec_hi=12_001)),
        # A usual batch of a busy server, ragged lengths.
        dict(name="decode_b32", **_attention(32, 8, 16, 3, dec=32, dec_lo=128, dec_hi=4096)),
        # A full batch: the benchmark's large decode.
        dict(name="decode_b256", **_attention(32, 8, 16, 4, dec=256, dec_lo=128, dec_hi=4096)),
        # Next turns of running chats: short new messages behind long cached
        # prefixes, odd lengths.
        dict(name="extend_turns", **_attention(32, 8, 16, 5, pre=4, new_lo=17, new_hi=90,
                                               cached_lo=2000, cached_hi=12_000)),
        # New prompts arriving together, no cache hit, ragged.
        dict(name="prefill_prompts", **_attention(32, 8, 16, 6, pre=12, new_lo=31,
                                                  new_hi=1500)),
        # One chunk of a long prompt: 2,048 tokens behind 4,096 cached.
        dict(name="prefill_chunk", **_attention(32, 4, 16, 7, pre=1, new_lo=2048, new_hi=2048,
                                                cached_lo=4096, cached_hi=4096)),
        # A chunked-prefill step with decode rows beside the chunk.
        dict(name="mixed_step", **_attention(32, 4, 16, 8, dec=64, dec_lo=1024, dec_hi=32_768,
                                             pre=1, new_lo=2048, new_hi=2048, cached_lo=4096,
                                             cached_hi=4096)),
        # Norms and activations of a decode step of 64 requests, all layers.
        dict(name="block_step_b64", **_block(64, 4096, 12_288, layers=36, graph=True)),
        # The same for one layer of a prefill batch, an odd token count.
        dict(name="block_prefill", **_block(8191, 4096, 12_288)),
        # The Sampler for a small batch, as the reference's two calls.
        dict(name="sampler_b16", **_sampler(16, route="probs")),
        # The Sampler for a full batch, straight from the logits.
        dict(name="sampler_b256", **_sampler(256)),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "extend", "prompts", "mixed", "block", "sampler",
                       "sampler"))
    seed = rng.randrange(1 << 20)
    hq, hkv = rng.choice(((16, 8), (32, 8), (32, 4)))
    page = rng.choice((1, 16))
    if kind == "decode":
        rows = _log_int(rng, 1, 256)
        hi = _log_int(rng, 200, min(32_768, 1_000_000 // rows))
        lo = max(1, int(hi * rng.uniform(0.05, 1.0)))
        graph = rows * hi <= 40_000 and rng.random() < 0.4
        return _attention(hq, hkv, page, seed, dec=rows, dec_lo=lo, dec_hi=hi,
                          layers=rng.randint(4, 28) if graph else 1, graph=graph)
    if kind == "extend":
        n = rng.randint(1, 8)
        new = _log_int(rng, 2, 300)
        cached = _log_int(rng, 64, 16_384)
        return _attention(hq, hkv, page, seed, pre=n, new_lo=max(2, new // 3), new_hi=new,
                          cached_lo=max(1, cached // 4), cached_hi=cached)
    if kind == "prompts":
        n = _log_int(rng, 1, 16)
        new = _log_int(rng, 100, min(6000, 16_000 // n))
        cached = rng.choice((0, 0, _log_int(rng, 64, 4096)))
        return _attention(hq, hkv, page, seed, pre=n, new_lo=max(2, new // 8), new_hi=new,
                          cached_lo=cached // 2, cached_hi=cached)
    if kind == "mixed":
        rows = _log_int(rng, 2, 64)
        hi = _log_int(rng, 500, 24_000)
        new = _log_int(rng, 128, 2048)
        return _attention(hq, hkv, page, seed, dec=rows, dec_lo=max(1, hi // 6), dec_hi=hi,
                          pre=rng.randint(1, 2), new_lo=max(2, new // 2), new_hi=new,
                          cached_lo=64, cached_hi=_log_int(rng, 128, 4096))
    if kind == "block":
        hidden, inter = rng.choice(((1024, 3072), (4096, 12_288), (2048, 6144)))
        tokens = _log_int(rng, 1, 8192)
        graph = tokens <= 256 and rng.random() < 0.6
        return _block(tokens, hidden, inter, dtype=rng.choice(("bf16", "bf16", "fp16")),
                      act=rng.choice(("silu", "silu", "gelu")),
                      layers=rng.randint(8, 36) if graph else 1, graph=graph)
    return _sampler(_log_int(rng, 1, 256), dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")),
                    mode=rng.choice(("top_k_top_p", "top_k_top_p", "top_k", "top_p", "plain")),
                    route=rng.choice(("logits", "probs")))


# ------------------------------------------------------------------ attention

def _lengths(case):
    """(cached, new) of each request, decode rows first."""
    rng = np.random.default_rng(case["lengths"])
    kv = rng.integers(case["dec_lo"], case["dec_hi"] + 1, size=case["dec"])
    new = rng.integers(case["new_lo"], case["new_hi"] + 1, size=case["pre"])
    cached = rng.integers(case["cached_lo"], case["cached_hi"] + 1, size=case["pre"])
    return (np.concatenate([kv - 1, cached]).astype(np.int64),
            np.concatenate([np.ones(case["dec"], np.int64), new]).astype(np.int64))


def _layout(case, seed):
    """Page table (token granular, pages handed out in random order, a spare
    page last), positions and slots of the new tokens: host arrays."""
    cached, new = _lengths(case)
    page, total = case["page"], cached + new
    pages = -(-total // page)
    order = np.random.default_rng([seed, case["lengths"]]).permutation(int(pages.sum()))
    # Captured graphs are sized for longer rows than this step's.
    width = -(-int(total.max()) // 32) * 32
    if case["graph"]:
        width = max(4096, 1 << int(width - 1).bit_length())
    spare = int(pages.sum()) * page
    table = np.full((len(total) + 1, width), spare, dtype=np.int32)
    at, positions, slots = 0, [], []
    for r, n in enumerate(pages):
        row = (order[at:at + n, None] * page + np.arange(page)[None, :]).reshape(-1)
        at += int(n)
        table[r, :total[r]] = row[:total[r]]
        pos = np.arange(cached[r], total[r])
        positions.append(pos)
        slots.append(row[pos])
    return dict(cached=cached, new=new, total=total, pages=int(pages.sum()) + 1, table=table,
                positions=np.concatenate(positions).astype(np.int32),
                slots=np.concatenate(slots).astype(np.int32))


def _randn(shape, g, dtype=torch.bfloat16):
    out = torch.empty(shape, device=DEV, dtype=dtype)
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        flat[i:i + (1 << 28)].normal_(generator=g)
    return out


def _attention_data(case, seed, lay, pool):
    """Fills the pool and makes the qkv rows and norm weights of each layer:
    cached keys and values of unit scale, as qk-normalised rows have."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    flat = pool.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        flat[i:i + (1 << 28)].normal_(generator=g)
    tokens = int(lay["new"].sum())
    qkv = _randn((case["layers"], tokens, (case["hq"] + 2 * case["hkv"]) * D), g)
    weights = (torch.rand((case["layers"], 2, D), device=DEV, generator=g) + 0.5).to(torch.bfloat16)
    return qkv, weights


def _prepare_attention(case, seed):
    sb = _backend()
    lay = _layout(case, seed)
    hq, hkv, layers = case["hq"], case["hkv"], case["layers"]
    pool = sb.MHAKVCache(hkv, layers, D, lay["pages"], case["page"])
    qkv, weights = _attention_data(case, seed, lay, pool.buffer())
    backend = sb.HipAttnBackend(pool, hq, hkv, D)
    backend.set_page_table(torch.from_numpy(lay["table"]).to(DEV))
    rotary = sb.RotaryEmbedding(D, D, MAX_POS, 1e6)
    stack = []
    for l in range(layers):
        norms = [sb.RMSNorm(D, EPS), sb.RMSNorm(D, EPS)]
        for norm, w in zip(norms, weights[l]):
            norm.weight = w.contiguous()
        stack.append(sb.AttentionLayer(l, hq, hkv, D, backend, rotary, *norms))
    positions = torch.from_numpy(lay["positions"]).to(DEV)
    slots = torch.from_numpy(lay["slots"]).to(DEV)
    reqs = [sb.Req(r, int(c), int(t)) for r, (c, t) in enumerate(zip(lay["cached"], lay["total"]))]
    batch = sb.Batch(case["pre"] > 0, reqs, positions, slots)
    state = dict(case=case, backend=backend, pool=pool, stack=stack, qkv=qkv, batch=batch,
                 positions=positions)
    if not case["graph"]:
        backend.prepare_metadata(batch)
        return state
    rows, longest = len(reqs), lay["table"].shape[1]
    backend.init_capture_graph(longest, [rows])
    capture = sb.Batch(False, [sb.Req(r, longest - 1, longest) for r in range(rows)], positions,
                       slots)
    backend.prepare_for_capture(capture)
    spare = qkv[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        keep = pool.buffer()[:, 0].index_select(1, slots.long())
        stack[0].forward(spare, positions, capture)  # warm-up, its stores undone
        pool.buffer()[:, 0].index_copy_(1, slots.long(), keep)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [layer.forward(qkv[l], positions, capture) for l, layer in enumerate(stack)]
    state.update(graph=graph, outs=outs, capture=capture)
    return state


def _run_attention(s):
    if s["case"]["graph"]:
        s["backend"].prepare_metadata(s["batch"])
        s["backend"].prepare_for_replay(s["batch"])
        s["graph"].replay()
        outs = s["outs"]
    else:
        outs = [layer.forward(s["qkv"][l], s["positions"], s["batch"])
                for l, layer in enumerate(s["stack"])]
    # The layers' outputs, the rotated q beside k and v, and the pool with the
    # step's keys and values stored.
    return {"out": outs, "qkv": s["qkv"], "pool": s["pool"].buffer()}


def _exact_attention(case, seed):
    lay = _layout(case, seed)
    hq, hkv, layers, group = case["hq"], case["hkv"], case["layers"], case["hq"] // case["hkv"]
    pool = torch.empty((2, layers, lay["pages"] * case["page"], hkv, D), device=DEV,
                       dtype=torch.bfloat16)
    qkv, weights = _attention_data(case, seed, lay, pool)
    pool, qkv, weights = pool.double(), qkv.double(), weights.double()
    pos = torch.from_numpy(lay["positions"]).to(DEV).double()
    slots = torch.from_numpy(lay["slots"]).to(DEV).long()
    table = torch.from_numpy(lay["table"]).to(DEV).long()
    freq = 1e6 ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
    cos = torch.cos(pos[:, None] * freq)[:, None]
    sin = torch.sin(pos[:, None] * freq)[:, None]
    outs = []
    for l in range(layers):
        rows = qkv[l].view(len(pos), hq + 2 * hkv, D)
        x = rows[:, :hq + hkv]
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
        x = torch.cat([x[:, :hq] * weights[l, 0], x[:, hq:] * weights[l, 1]], 1)
        a, b = x[..., :D // 2], x[..., D // 2:]
        x = torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
        rows[:, :hq] = x[:, :hq]  # k is left as it came; the pool holds its rotation
        pool[0, l, slots] = x[:, hq:]
        pool[1, l, slots] = rows[:, hq + hkv:]
        out = torch.empty((len(pos), hq, D), device=DEV, dtype=torch.float64)
        at = 0
        for r in range(len(lay["new"])):
            n, total = int(lay["new"][r]), int(lay["total"][r])
            k = pool[0, l, table[r, :total]].permute(1, 2, 0).contiguous()  # [hkv, D, total]
            v = pool[1, l, table[r, :total]].permute(1, 0, 2).contiguous()  # [hkv, total, D]
            q = x[at:at + n, :hq].view(n, hkv, group, D).permute(1, 2, 0, 3)
            seen = torch.arange(total, device=DEV)[None] <= \
                torch.arange(total - n, total, device=DEV)[:, None]
            for h in range(hkv):
                s = q[h].reshape(group * n, D) @ k[h] / math.sqrt(D)
                s = s.view(group, n, total).masked_fill(~seen, -math.inf)
                o = torch.softmax(s, -1).view(group * n, total) @ v[h]
                out[at:at + n, h * group:(h + 1) * group] = o.view(group, n, D).transpose(0, 1)
            at += n
        outs.append(out.view(len(pos), hq * D))
    return {"out": outs, "qkv": qkv, "pool": pool}


def _work_attention(case):
    cached, new = _lengths(case)
    total, hq, hkv = cached + new, case["hq"], case["hkv"]
    tokens = int(new.sum())
    pairs = int((new * total - new * (new - 1) // 2).sum())
    per_layer = (2 * 2 * hkv * D * int(cached.sum())      # cached keys and values read
                 + 2 * (hq + 2 * hkv) * D * tokens        # qkv rows read
                 + 2 * (2 * hq + 2 * hkv) * D * tokens    # rotated q, k and v rows, o written
                 + 4 * int(total.sum()))                  # slots
    return {"bytes": per_layer * case["layers"], "flops": 4 * D * hq * pairs * case["layers"]}


# ------------------------------------------------------------------ block

def _block_data(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt, L, T, H, I = (DTYPES[case["dtype"]], case["layers"], case["tokens"], case["hidden"],
                      case["inter"])
    x = _randn((L, T, H), g, dt)
    residual = _randn((L, T, H), g, dt) * 4  # the residual stream outgrows a block's output
    gate_up = _randn((L, T, 2 * I), g, dt)
    weights = (torch.rand((L, H), device=DEV, generator=g) + 0.5).to(dt)
    return x, residual, gate_up, weights


def _prepare_block(case, seed):
    sb = _backend()
    x, residual, gate_up, weights = _block_data(case, seed)
    norms = []
    for l in range(case["layers"]):
        norms.append(sb.RMSNorm(case["hidden"], EPS))
        norms[-1].weight = weights[l]
    out = torch.empty((case["layers"], case["tokens"], case["inter"]), device=DEV, dtype=x.dtype)
    act = sb.silu_and_mul if case["act"] == "silu" else sb.gelu_and_mul
    state = dict(x=x, residual=residual, gate_up=gate_up, out=out)

    def step():
        for l, norm in enumerate(norms):
            norm.fused_add_forward_inplace(x[l], residual[l])
            act(out[l], gate_up[l])

    state["step"] = step
    if case["graph"]:
        warm = torch.cuda.Stream()
        warm.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(warm):
            norms[0].fused_add_forward_inplace(x[0].clone(), residual[0].clone())
            act(out[0], gate_up[0])
        torch.cuda.current_stream().wait_stream(warm)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        state["step"], state["graph"] = graph.replay, graph
    return state


def _run_block(s):
    s["step"]()
    return {"x": s["x"], "residual": s["residual"], "act": s["out"]}


def _exact_block(case, seed):
    x, residual, gate_up, weights = (t.double() for t in _block_data(case, seed))
    s = x + residual
    gate, up = gate_up[..., :case["inter"]], gate_up[..., case["inter"]:]
    gate = torch.nn.functional.silu(gate) if case["act"] == "silu" else \
        torch.nn.functional.gelu(gate, approximate="tanh")
    normed = s * torch.rsqrt(s.square().mean(-1, keepdim=True) + EPS) * weights[:, None]
    return {"x": normed, "residual": s, "act": gate * up}


def _work_block(case):
    T, H, I, L = case["tokens"], case["hidden"], case["inter"], case["layers"]
    return {"bytes": 2 * L * (T * (4 * H + 3 * I) + H), "flops": L * T * (5 * H + 6 * I)}


# ------------------------------------------------------------------ sampler

def _sampler_data(case, seed):
    """Logits as a language model's head gives them: a broad bulk, and in
    every row a few dozen favoured tokens, from rows that are almost certain
    of the next token to rows that are not."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    B = case["rows"]
    logits = torch.randn((B, VOCAB), device=DEV, generator=g) * 2.5
    ranks = torch.arange(64, device=DEV, dtype=torch.float32)
    top = 8 + 12 * torch.rand((B, 1), device=DEV, generator=g)
    where = torch.randint(0, VOCAB, (B, 64), device=DEV, generator=g)
    logits.scatter_(1, where, top - 1.5 * torch.log2(ranks + 1))
    temps = 0.6 + 0.6 * torch.rand(B, device=DEV, generator=g)
    top_k = torch.randint(20, 101, (B,), device=DEV, generator=g)
    top_p = 0.8 + 0.15 * torch.rand(B, device=DEV, generator=g)
    rounds = (B,) if case["mode"] == "plain" else (ROUNDS, B)
    uniform = torch.rand(rounds, device=DEV, generator=g)
    return logits.to(DTYPES[case["dtype"]]), temps, top_k, top_p, uniform


def _prepare_sampler(case, seed):
    logits, temps, top_k, top_p, uniform = _sampler_data(case, seed)
    top_k = top_k.to(torch.int32 if case["mode"] == "top_k_top_p" else torch.float32)
    return dict(case=case, sb=_backend(), logits=logits, temps=temps, top_k=top_k, top_p=top_p,
                uniform=uniform)


def _run_sampler(s):
    sb, case, u = s["sb"], s["case"], s["uniform"]
    mode = case["mode"]
    top_k = s["top_k"] if mode in ("top_k", "top_k_top_p") else None
    top_p = s["top_p"] if mode in ("top_p", "top_k_top_p") else None
    if case["route"] == "logits":
        samples, success = sb.sample_from_logits(s["logits"], s["temps"], u, top_k, top_p)
        return {"samples": samples, "success": success}
    probs = sb.sampling_probs(s["logits"], s["temps"])
    success = None
    if mode == "plain":
        samples = sb.flashinfer_sample_from_probs(probs, u)
    elif mode == "top_k":
        samples, success = sb.flashinfer_top_k_sample_from_probs(probs, u, top_k)
    elif mode == "top_p":
        samples, success = sb.flashinfer_top_p_sample_from_probs(probs, u, top_p)
    else:
        samples, success = sb.flashinfer_top_k_top_p_sample_from_probs(probs, u, top_k, 0, top_p,
                                                                      0.0)
    return {"probs": probs, "samples": samples, "success": success}


def _exact_sampler(case, seed):
    if case["route"] == "logits":
        return None  # whole numbers only
    logits, temps, _, _, _ = _sampler_data(case, seed)
    return {"probs": torch.softmax(logits.double() / temps.double()[:, None], -1),
            "samples": None, "success": None}


def _work_sampler(case):
    n = case["rows"] * VOCAB
    esize = 4 if case["dtype"] == "fp32" else 2
    small = case["rows"] * (4 * ROUNDS + 20)
    # Probabilities that are handed out are written, and read by the draw.
    return {"bytes": n * (esize + (8 if case["route"] == "probs" else 0)) + small, "flops": 8 * n}


# ------------------------------------------------------------------ entry points

def prepare(case, seed):
    return {"attention": _prepare_attention, "block": _prepare_block,
            "sampler": _prepare_sampler}[case["kind"]](case, seed) | {"kind": case["kind"]}


def run(state):
    return {"attention": _run_attention, "block": _run_block,
            "sampler": _run_sampler}[state["kind"]](state)


def work(case):
    return {"attention": _work_attention, "block": _work_block,
            "sampler": _work_sampler}[case["kind"]](case)


def tolerance(case):
    if case["kind"] == "attention":
        # bf16 q, k, weights and outputs.
        return {"rel": 1.2e-2, "max": 0.1}
    if case["kind"] == "block":
        # One rounding of each output to 16 bits.
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 1e-3,
                "max": 2e-2 if case["dtype"] == "bf16" else 3e-3}
    # fp32 probabilities; tokens and flags are whole and stay the same.
    return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}


def exact(case, seed):
    return {"attention": _exact_attention, "block": _exact_block,
            "sampler": _exact_sampler}[case["kind"]](case, seed)
