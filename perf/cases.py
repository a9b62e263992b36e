"""Performance cases: the work that a serving program gives this framework.

Six kinds, each through the entry points such a program calls:

  decode   one decode step of the paged-KV decoder, captured in a hipGraph as
           the serving engine keeps it (a row per sequence, logits out)
  prefill  one packed step of prompt rows through the same model: whole
           prompts, a prompt portion behind cached history, or the few rows
           per sequence with which speculation verifies a draft
  moe      the routed feed-forward of the mixture model on prompt rows
  sample   temperature / top-k / top-p sampling of a batch's logits
  session  caller-paced requests of the hybrid family through the engine:
           prompts in one packed step, then single tokens, logits of each

Sizes are those of the repository's model configurations (the deep ones cut to
half their layers, which are all alike: the bf16 rounding of random weights
grows with depth, to 1.5% of the logits at 16 layers); batches and lengths
are those of its serving benchmark (128 calls of 512 prompt and 64 generated
tokens, 64-token pages) and of shorter, longer and ragged traffic around it.
Weights are random at the scales the models are initialised with.
"""
from __future__ import annotations

import math
from dataclasses import replace

import torch

from agentfield_amd import ops
from agentfield_amd.engine import LLMEngine
from agentfield_amd.engine.engine import choose_nsplit
from agentfield_amd.models import CONFIGS
from agentfield_amd.models.hybrid import ReperaxForCausalLM
from agentfield_amd.models.llama import (AttnMetadata, KVCache,
                                         LlamaForCausalLM, MoEMLP)

DEV = "cuda"
PAGE = 64
F64 = torch.float64


# ------------------------------------------------------------------- the list
def listed():
    return [
        # one interactive caller: every launch and every byte of weights counts
        dict(name="decode-one", kind="decode", model="llama-3-8b", layers=16,
             batch=1, lo=387, hi=387),
        # half a node's share of the serving benchmark
        dict(name="decode-64", kind="decode", model="llama-3-8b", layers=16,
             batch=64, lo=513, hi=576),
        # the serving benchmark's decode step
        dict(name="decode-128", kind="decode", model="llama-3-8b", layers=16,
             batch=128, lo=513, hi=576),
        # long, ragged conversations: the K/V stream dominates
        dict(name="decode-long", kind="decode", model="llama-3-8b", layers=16,
             batch=24, lo=1800, hi=8100),
        # sliding-window attention past its window
        dict(name="decode-window", kind="decode", model="mistral-7b",
             layers=16, batch=12, lo=4500, hi=8000),
        # one short prompt: time to first token of a small call
        dict(name="prefill-short", kind="prefill", model="llama-3-8b",
             layers=16, batch=1, lo=45, hi=45, hist=0, every=False),
        # a ragged batch of benchmark-sized prompts
        dict(name="prefill-batch", kind="prefill", model="llama-3-8b",
             layers=16, batch=20, lo=300, hi=700, hist=0, every=False),
        # one long document
        dict(name="prefill-long", kind="prefill", model="llama-3-8b",
             layers=16, batch=1, lo=8000, hi=8000, hist=0, every=False),
        # four drafted tokens and the last one, verified behind a history
        dict(name="verify", kind="prefill", model="llama-3-8b", layers=16,
             batch=16, lo=5, hi=5, hist=3000, every=True),
        # a mixture layer's feed-forward over a few prompts
        dict(name="moe-prompt", kind="moe", model="mixtral-8x7b", rows=1100),
        # sampled (not greedy) traffic
        dict(name="sample-top", kind="sample", batch=64, vocab=128256),
        # the hybrid family, caller-paced
        dict(name="session", kind="session", model="reperax-1b", batch=6,
             lo=500, hi=1900, steps=6),
    ]


#: K/V positions and prompt rows that a drawn case may have at most, per model
#: (those of the largest listed cases, or what their K/V bytes allow).
DENSE = {
    "llama-3-8b": dict(layers=16, ctx=8100, keys=120_000, rows=9_000),
    "mistral-7b": dict(layers=16, ctx=8000, keys=120_000, rows=9_000),
    "llama-2-7b": dict(layers=16, ctx=4000, keys=30_000, rows=9_000),
    "debug-1b": dict(layers=16, ctx=8000, keys=200_000, rows=9_000),
    # one pipeline's worth of the large model's layers
    "llama-3-70b": dict(layers=8, ctx=8000, keys=200_000, rows=6_000),
}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "prefill", "moe", "sample", "session"],
                       [4, 4, 1, 1, 1])[0]
    if kind == "decode":
        model = rng.choice(sorted(DENSE))
        top = DENSE[model]
        batch = _log(rng, 1, 128)
        hi = _log(rng, 40, max(41, min(top["ctx"], top["keys"] // batch)))
        return dict(kind=kind, model=model, layers=top["layers"], batch=batch,
                    lo=max(2, int(hi * rng.uniform(0.2, 1.0))), hi=hi)
    if kind == "prefill":
        model = rng.choice(sorted(DENSE))
        top = DENSE[model]
        if rng.random() < 0.3:   # a few rows per sequence behind a history
            batch = _log(rng, 1, 32)
            hi = rng.randint(2, 9)
            hist = _log(rng, 60, min(top["ctx"] - 16, top["keys"] // batch))
            return dict(kind=kind, model=model, layers=top["layers"],
                        batch=batch, lo=2, hi=hi, hist=hist, every=True)
        rows = _log(rng, 20, top["rows"])
        batch = _log(rng, 1, max(1, min(32, rows // 20)))
        hi = min(rows // batch, top["ctx"] - 8)
        hist = 0
        if rng.random() < 0.3 and hi < top["ctx"] // 2:
            hist = _log(rng, 10, min(top["ctx"] - hi, top["keys"] // batch))
        return dict(kind=kind, model=model, layers=top["layers"], batch=batch,
                    lo=max(1, int(hi * rng.uniform(0.3, 1.0))), hi=hi,
                    hist=hist, every=False)
    if kind == "moe":
        return dict(kind=kind, model="mixtral-8x7b", rows=_log(rng, 20, 4096))
    if kind == "sample":
        return dict(kind=kind, batch=_log(rng, 1, 128),
                    vocab=rng.choice([32000, 32003, 128256]))
    batch = rng.randint(1, 6)
    hi = _log(rng, 30, 1900)
    return dict(kind=kind, model="reperax-1b", batch=batch,
                lo=max(2, int(hi * rng.uniform(0.3, 1.0))), hi=hi,
                steps=rng.randint(1, 6))


# ----------------------------------------------------------------- inputs
def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(int(seed))


def _lengths(case, seed):
    """Ragged lengths lo..hi, the longest among them."""
    g = _gen(seed * 7919 + 13, "cpu")
    n = torch.randint(case["lo"], case["hi"] + 1, (case["batch"],),
                      generator=g).tolist()
    n[-1] = case["hi"]
    if case.get("every"):      # all rows' logits come back: a fixed number
        n = sorted(n)
        n = [min(case["hi"], max(case["lo"], round(
            case["lo"] + (case["hi"] - case["lo"]) * (i + 1) / len(n))))
            for i in range(len(n))]
    return n


def _dense_cfg(case):
    return replace(CONFIGS[case["model"]], num_layers=case["layers"])


def _dense_shapes(cfg):
    H, I = cfg.hidden_size, cfg.intermediate_size
    yield "embed", (cfg.vocab_size, H)
    for i in range(cfg.num_layers):
        p = f"layers.{i}."
        yield p + "input_norm", (H,)
        yield p + "attn.qkv", (cfg.q_size + 2 * cfg.kv_size, H)
        yield p + "attn.o", (H, cfg.q_size)
        yield p + "post_norm", (H,)
        yield p + "mlp.gate_up", (2 * I, H)
        yield p + "mlp.down", (H, I)
    yield "final_norm", (H,)
    yield "lm_head", (cfg.vocab_size, H)


def _fill(t, name, g, layers=1):
    """Unit-scale embeddings, projections at the usual 0.02, those that write
    the residual smaller with depth, so that its rows stay of one scale."""
    if "norm" in name:
        t.normal_(1.0, 0.1, generator=g)
    elif name == "embed":
        t.normal_(0.0, 1.0, generator=g)
    elif name.endswith(("attn.o", "mlp.down")):
        t.normal_(0.0, 0.02 / math.sqrt(2 * layers), generator=g)
    else:
        t.normal_(0.0, 0.02, generator=g)


def _dense_batch(case, seed):
    """Rows, pages and cached history of one step, on the device."""
    cfg = _dense_cfg(case)
    n = _lengths(case, seed)
    if case["kind"] == "decode":       # n counts the token being decoded
        hist, rows = [x - 1 for x in n], [1] * len(n)
    else:
        g = _gen(seed * 31 + 5, "cpu")
        hist = [int(case["hist"] * (0.6 + 0.4 * f)) for f in
                torch.rand(len(n), generator=g).tolist()]
        rows = n
    need = [(h + r + PAGE - 1) // PAGE for h, r in zip(hist, rows)]
    top = case["hi"] + case.get("hist", 0)
    pages = len(n) * ((top + PAGE - 1) // PAGE) + 1
    maxp = (cfg.max_position + PAGE - 1) // PAGE
    # page 0 is the null page; pages change hands, so order is arbitrary
    perm = (torch.randperm(pages - 1, generator=_gen(seed + 1, "cpu")) + 1
            ).to(torch.int32)
    bt = torch.zeros(len(n), maxp, dtype=torch.int32)
    at = 0
    for i, k in enumerate(need):
        bt[i, :k] = perm[at:at + k]
        at += k
    pos = torch.cat([torch.arange(h, h + r) for h, r in zip(hist, rows)])
    seq = torch.cat([torch.full((r,), i) for i, r in enumerate(rows)])
    slots = bt[seq, pos // PAGE].long() * PAGE + pos % PAGE
    cu = [0]
    for r in rows:
        cu.append(cu[-1] + r)
    ids = torch.randint(0, cfg.vocab_size, (len(pos),),
                        generator=_gen(seed + 2, "cpu"))
    return dict(cfg=cfg, hist=hist, rows=rows, pages=pages, cu=cu,
                bt=bt.to(DEV), pos=pos.to(torch.int32).to(DEV),
                slots=slots.to(DEV), ids=ids.to(torch.int32).to(DEV))


def _cache_fill(k, v, g):
    """Cached keys and values of earlier tokens (unit-scale rows)."""
    k.normal_(0.0, 1.3, generator=g)
    v.normal_(0.0, 1.3, generator=g)


def _prepare_dense(case, seed):
    b = _dense_batch(case, seed)
    cfg = b["cfg"]
    model = LlamaForCausalLM(cfg, device=DEV).eval()
    g = _gen(seed)
    own = dict(model.named_parameters())
    with torch.no_grad():
        for name, shape in _dense_shapes(cfg):
            assert own[name].shape == shape
            _fill(own[name], name, g, cfg.num_layers)
    model.fold_norm_weights()          # as the engine does on load
    kv = KVCache(cfg, b["pages"], PAGE, DEV)
    if max(b["hist"]) > 0:
        g = _gen(seed + 3)
        for k, v in zip(kv.k, kv.v):
            _cache_fill(k, v, g)
    st = dict(case=case, model=model, kv=kv, ids=b["ids"], pos=b["pos"])
    if case["kind"] == "decode":
        lens = torch.tensor([h + 1 for h in b["hist"]], dtype=torch.int32,
                            device=DEV)
        st["md"] = AttnMetadata(
            is_prefill=False, slots=b["slots"], block_table=b["bt"],
            seq_lens_t=lens, nsplit=choose_nsplit(len(lens), cfg.num_kv_heads))
        st["rows"] = None
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                _dense_forward(st)
        torch.cuda.current_stream().wait_stream(side)
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            st["logits"] = _dense_forward(st)
    else:
        st["md"] = AttnMetadata(
            is_prefill=True, slots=b["slots"],
            cu_seqlens=torch.tensor(b["cu"], dtype=torch.int32, device=DEV),
            seq_lens=b["rows"],
            q_start=torch.tensor(b["hist"], dtype=torch.int32, device=DEV),
            block_table=b["bt"])
        st["rows"] = None if case["every"] else torch.tensor(
            [c - 1 for c in b["cu"][1:]], dtype=torch.int32, device=DEV)
    return st


@torch.inference_mode()
def _dense_forward(st):
    return st["model"](st["ids"], st["pos"], st["kv"], st["md"],
                       logit_rows=st["rows"])


def _moe_tensors(case, seed):
    cfg = CONFIGS[case["model"]]
    E, H, I = cfg.num_experts, cfg.hidden_size, cfg.intermediate_size
    g = _gen(seed)
    t = {"x": torch.empty(case["rows"], H, device=DEV, dtype=torch.bfloat16)}
    t["x"].normal_(0.0, 1.0, generator=g)       # rows behind a norm
    for name, shape in (("router", (E, H)), ("gate_up", (E, 2 * I, H)),
                        ("down", (E, H, I))):
        t[name] = torch.empty(shape, device=DEV, dtype=torch.bfloat16)
        _fill(t[name], name, g)
    return cfg, t


def _sample_tensors(case, seed):
    B, V = case["batch"], case["vocab"]
    g = _gen(seed)
    logits = torch.empty(B, V, device=DEV)
    logits.normal_(0.0, 2.5, generator=g)
    c = _gen(seed + 1, "cpu")
    temps = 0.3 + torch.rand(B, generator=c)
    temps[torch.rand(B, generator=c) < 0.2] = 0.0      # greedy rows among them
    topk = torch.randint(5, 100, (B,), generator=c).to(torch.int32)
    topk[torch.rand(B, generator=c) < 0.4] = 0          # off
    topp = 0.7 + 0.3 * torch.rand(B, generator=c)
    topp[torch.rand(B, generator=c) < 0.3] = 1.0        # off
    return logits.bfloat16(), temps.to(DEV), topk.to(DEV), topp.to(DEV)


def _hybrid_weights(cfg, seed):
    """Checkpoint-named bf16 tensors at scales that keep rows O(1)."""
    g = _gen(seed)
    W, w = cfg.width, {}

    def mat(name, o, i, gain=1.0):
        w[name] = torch.empty(o, i, device=DEV).normal_(
            0.0, gain / math.sqrt(i), generator=g).bfloat16()

    def vec(name, n, mean=0.0, std=0.1):
        w[name] = torch.empty(n, device=DEV).normal_(
            mean, std, generator=g).bfloat16()

    w["embed"] = torch.empty(cfg.vocab_size, W, device=DEV).normal_(
        0.0, 1.0, generator=g).bfloat16()
    vec("final.norm", W)
    for i, L in enumerate(cfg.layers):
        p = f"l{i}."
        vec(p + "norm1", W)
        w[p + "shift"] = torch.rand(W, device=DEV, generator=g).bfloat16()
        mat(p + "rg1", W, W)
        vec(p + "rg1.b", W, 0.0, 0.5)
        if L.kind == "parallel":
            a, r = L.attn, L.gla
            q = p + "mix.left."
            mat(q + "q", a.heads * a.dim, W)
            mat(q + "k", a.kv_heads * a.dim, W)
            mat(q + "v", a.kv_heads * a.vdim, W)
            mat(q + "o", W, a.heads * a.vdim)
            vec(q + "q.norm", a.heads * a.dim, 1.0)
            vec(q + "k.norm", a.kv_heads * a.dim, 1.0)
            q = p + "mix.right."
            for n, o in (("q", r.heads * r.dim), ("k", r.heads * r.dim),
                         ("v", r.heads * r.vdim), ("g", r.heads * r.vdim),
                         ("a1", r.rank)):
                mat(q + n, o, W)
            mat(q + "a2", r.heads * r.dim, r.rank, 2.0)
            vec(q + "a2.b", r.heads * r.dim, 2.0, 1.0)
            vec(q + "norm", r.vdim, 1.0)
            mat(q + "o", W, r.heads * r.vdim)
        else:
            r = L.ret
            q = p + "mix."
            for n, o in (("q", r.heads * r.dim), ("k", r.heads * r.dim),
                         ("v", r.heads * r.vdim), ("g", r.heads * r.vdim)):
                mat(q + n, o, W)
            mat(q + "o", W, r.heads * r.vdim)
        vec(p + "norm2", W)
        mat(p + "mlp.up", L.ff, W)
        mat(p + "mlp.down", W, L.ff)
        w[p + "mlp.act"] = torch.tensor([0.6, 0.3, 0.1, 0.0], device=DEV)
        mat(p + "rg2", W, W)
        vec(p + "rg2.b", W, 0.0, 0.5)
    return w


def _session_tokens(case, seed):
    cfg = CONFIGS[case["model"]]
    g = _gen(seed + 9, "cpu")
    return [torch.randint(0, cfg.vocab_size, (n + case["steps"],),
                          generator=g).tolist()
            for n in _lengths(case, seed)]


def _prepare_session(case, seed):
    cfg = CONFIGS[case["model"]]
    w = _hybrid_weights(cfg, seed)
    model = ReperaxForCausalLM(cfg, device=DEV).load_tensors(w.__getitem__)
    tokens = _session_tokens(case, seed)
    pages = sum((len(t) + PAGE - 1) // PAGE for t in tokens) + 1
    eng = LLMEngine(cfg, device=DEV, page_size=PAGE, num_pages=pages,
                    max_num_seqs=case["batch"], model=model,
                    max_prefill_tokens=sum(map(len, tokens)),
                    enable_graphs=False, caller_paced=True)
    return dict(case=case, engine=eng, tokens=tokens)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _prepare_dense(case, seed)
    if kind == "moe":
        cfg, t = _moe_tensors(case, seed)
        with torch.device(DEV):
            mlp = MoEMLP(cfg)
        mlp = mlp.to(torch.bfloat16).eval()
        with torch.no_grad():
            for name in ("router", "gate_up", "down"):
                getattr(mlp, name).copy_(t[name])
        return dict(case=case, mlp=mlp, x=t["x"])
    if kind == "sample":
        logits, temps, topk, topp = _sample_tensors(case, seed)
        return dict(case=case, logits=logits, temps=temps, topk=topk,
                    topp=topp,
                    sampler=ops.SamplerState(case["batch"], DEV, seed=1234))
    return _prepare_session(case, seed)


# ------------------------------------------------------------------- one pass
@torch.inference_mode()
def run(st):
    kind = st["case"]["kind"]
    if kind == "decode":
        st["graph"].replay()
        return {"logits": st["logits"], "k": st["kv"].k[-1],
                "v": st["kv"].v[-1]}
    if kind == "prefill":
        logits = _dense_forward(st)
        return {"logits": logits, "k": st["kv"].k[-1], "v": st["kv"].v[-1]}
    if kind == "moe":
        return {"y": st["mlp"](st["x"])}
    if kind == "sample":
        return {"tokens": ops.sample(st["logits"], st["temps"], st["sampler"],
                                     topk=st["topk"], topp=st["topp"])}
    eng, steps = st["engine"], st["case"]["steps"]
    reqs = [eng.open_request() for _ in st["tokens"]]
    out = [eng.feed_step([(r, t[:-steps], [len(t) - steps - 1])
                          for r, t in zip(reqs, st["tokens"])])]
    for j in range(-steps, 0):
        out.append(eng.feed_step([(r, [t[j]], [0])
                                  for r, t in zip(reqs, st["tokens"])]))
    for r in reqs:
        eng.close_request(r)
    return {"logits": out}


# ------------------------------------------------------------- necessary work
def _seen(hist, rows, window):
    """Keys that a sequence's rows attend to, in all."""
    if window <= 0:
        return rows * hist + rows * (rows + 1) // 2
    return sum(min(window, hist + r + 1) for r in range(rows))


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        cfg = _dense_cfg(case)
        mean = (case["lo"] + case["hi"]) / 2
        B = case["batch"]
        if kind == "decode":
            hist, rows, heads = int(mean) - 1, 1, B
        else:
            hist, rows = int(case["hist"] * 0.8), int(mean)
            heads = B * rows if case["every"] else B
        per_layer = (cfg.hidden_size * (2 * cfg.q_size + 2 * cfg.kv_size)
                     + 3 * cfg.hidden_size * cfg.intermediate_size)
        head = cfg.hidden_size * cfg.vocab_size
        win = cfg.sliding_window
        flops = (2.0 * B * rows * per_layer * cfg.num_layers
                 + 4.0 * cfg.q_size * cfg.num_layers * B
                 * _seen(hist, rows, win) + 2.0 * heads * head)
        first = min(hist, win + rows) if win else hist
        kv = 4.0 * cfg.kv_size * cfg.num_layers * B * (first + rows)
        return {"bytes": 2.0 * (per_layer * cfg.num_layers + head) + kv
                + 2.0 * heads * cfg.vocab_size, "flops": flops}
    if kind == "moe":
        cfg = CONFIGS[case["model"]]
        unit = 3 * cfg.hidden_size * cfg.intermediate_size
        used = min(cfg.num_experts, case["rows"] * cfg.num_experts_per_tok)
        return {"bytes": 2.0 * unit * used
                + 4.0 * case["rows"] * cfg.hidden_size,
                "flops": 2.0 * unit * case["rows"] * cfg.num_experts_per_tok}
    if kind == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 2.0 * n, "flops": 4.0 * n}
    cfg = CONFIGS[case["model"]]
    W, mean = cfg.width, (case["lo"] + case["hi"]) / 2
    per = state = 0
    for L in cfg.layers:
        per += W * (2 * W + 2 * L.ff)
        if L.kind == "parallel":
            a, r = L.attn, L.gla
            per += W * (2 * a.heads * a.dim + 2 * a.kv_heads * a.dim
                        + r.heads * (2 * r.dim + 3 * r.vdim))
        else:
            r = L.ret
            per += W * r.heads * (2 * r.dim + 3 * r.vdim)
        state += r.heads * r.dim * r.vdim
    head = W * cfg.vocab_size
    B, steps = case["batch"], case["steps"]
    return {"bytes": (1 + steps) * (2.0 * (per + head) + 8.0 * B * state),
            "flops": 2.0 * B * (mean + steps) * per
            + 4.0 * B * (mean + steps) * state + 2.0 * B * (1 + steps) * head}


# ----------------------------------------------------------------- tolerances
def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return {"rel": 0.0, "differ": 0.01}
    if kind == "moe":
        return {"rel": 1e-2}
    if kind == "session":
        return {"rel": 2e-2}
    # bf16 activations through 16 layers: 1.5% off 64 bits, so two correct
    # implementations are up to 2% apart
    return {"rel": 3e-2}


# ------------------------------------------------- the same results in 64 bits
def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rotate(x, pos, theta):
    """Rotate-half positions on [rows, heads, dim]."""
    half = x.shape[-1] // 2
    inv = theta ** (-torch.arange(half, dtype=F64, device=x.device) / half)
    ang = pos.to(F64)[:, None, None] * inv
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(),
                      b * ang.cos() + a * ang.sin()], -1)


def _attend(q, k, v, hist, window):
    """q [r, Hq, D] against k / v [hist + r, Hk, D], causal."""
    r, Hq, D = q.shape
    G = Hq // k.shape[1]
    out = torch.empty_like(q)
    for r0 in range(0, r, 2048):
        r1 = min(r, r0 + 2048)
        row = torch.arange(hist + r0, hist + r1, device=q.device)[:, None]
        col = torch.arange(hist + r1, device=q.device)[None, :]
        hide = col > row
        if window > 0:
            hide |= col <= row - window
        for h in range(k.shape[1]):
            s = torch.einsum("rgd,kd->grk", q[r0:r1, h * G:(h + 1) * G],
                             k[:hist + r1, h]) / math.sqrt(D)
            s.masked_fill_(hide, -math.inf)
            out[r0:r1, h * G:(h + 1) * G] = torch.einsum(
                "grk,kd->rgd", torch.softmax(s, -1), v[:hist + r1, h])
    return out


@torch.no_grad()
def _exact_dense(case, seed):
    b = _dense_batch(case, seed)
    cfg = b["cfg"]
    g = _gen(seed)
    w = {}
    for name, shape in _dense_shapes(cfg):
        w[name] = torch.empty(shape, device=DEV, dtype=torch.bfloat16)
        _fill(w[name], name, g, cfg.num_layers)
    shape = (b["pages"], cfg.num_kv_heads, PAGE, cfg.head_dim)
    cg = _gen(seed + 3)
    pos, bt = b["pos"].long(), b["bt"].long()
    x = w["embed"].double()[b["ids"].long()]
    kc = vc = None
    for i in range(cfg.num_layers):
        p = f"layers.{i}."
        kc = torch.zeros(shape, dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros_like(kc)
        if max(b["hist"]) > 0:
            _cache_fill(kc, vc, cg)
        h = _rms(x, w[p + "input_norm"].double(), cfg.rms_eps)
        qkv = h @ w[p + "attn.qkv"].double().T
        q, k, v = qkv.split([cfg.q_size, cfg.kv_size, cfg.kv_size], -1)
        q = _rotate(q.unflatten(-1, (-1, cfg.head_dim)), pos, cfg.rope_theta)
        k = _rotate(k.unflatten(-1, (-1, cfg.head_dim)), pos, cfg.rope_theta)
        v = v.unflatten(-1, (-1, cfg.head_dim))
        o = torch.empty_like(q)
        for s, (hist, r) in enumerate(zip(b["hist"], b["rows"])):
            c = slice(b["cu"][s], b["cu"][s] + r)
            ks, vs = k[c], v[c]
            if hist:
                at = torch.arange(hist, device=DEV)
                pg = bt[s, at // PAGE]
                ks = torch.cat([kc[pg, :, at % PAGE].double(), ks])
                vs = torch.cat([vc[pg, :, at % PAGE].double(), vs])
            o[c] = _attend(q[c], ks, vs, hist, cfg.sliding_window)
        x = x + o.flatten(1) @ w[p + "attn.o"].double().T
        h = _rms(x, w[p + "post_norm"].double(), cfg.rms_eps)
        gu = h @ w[p + "mlp.gate_up"].double().T
        a, u = gu.chunk(2, -1)
        x = x + (torch.nn.functional.silu(a) * u) @ \
            w[p + "mlp.down"].double().T
    x = _rms(x, w["final_norm"].double(), cfg.rms_eps)
    if case["kind"] == "prefill" and not case["every"]:
        x = x[torch.tensor([c - 1 for c in b["cu"][1:]], device=DEV)]
    out = {"logits": x @ w["lm_head"].double().T}
    del w
    for name, cache, new in (("k", kc, k), ("v", vc, v)):
        full = cache.double()
        full[b["slots"] // PAGE, :, b["slots"] % PAGE] = new
        out[name] = full
    return out


@torch.no_grad()
def _exact_moe(case, seed):
    cfg, t = _moe_tensors(case, seed)
    x = t["x"].double()
    probs = torch.softmax(x @ t["router"].double().T, -1)
    val, idx = probs.topk(cfg.num_experts_per_tok, -1)
    val = val / val.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for e in range(cfg.num_experts):
        row, slot = (idx == e).nonzero(as_tuple=True)
        a, u = (x[row] @ t["gate_up"][e].double().T).chunk(2, -1)
        y[row] += val[row, slot, None] * (
            (torch.nn.functional.silu(a) * u) @ t["down"][e].double().T)
    return {"y": y}


def _shift(x):
    return torch.cat([torch.zeros_like(x[:, :1]), x[:, :-1]], 1)


def _heads(x, n):
    return x.unflatten(-1, (n, -1)).transpose(1, 2)    # [B, n, T, d]


@torch.no_grad()
def _exact_session(case, seed):
    cfg = CONFIGS[case["model"]]
    w = {k: v.double() for k, v in _hybrid_weights(cfg, seed).items()}
    tokens = _session_tokens(case, seed)
    B, T, steps = len(tokens), max(map(len, tokens)), case["steps"]
    ids = torch.zeros(B, T, dtype=torch.long)
    for i, t in enumerate(tokens):
        ids[i, :len(t)] = torch.tensor(t)
    x = w["embed"][ids.to(DEV)]
    eps = cfg.eps
    at = torch.arange(T, device=DEV)
    past = at[:, None] - at[None, :]

    def silu(z):
        return z * torch.sigmoid(z)

    for i, L in enumerate(cfg.layers):
        p = f"l{i}."
        n1 = _rms(x, 1.0 + w[p + "norm1"], eps)
        hs = n1 + (_shift(n1) - n1) * w[p + "shift"]
        if L.kind == "parallel":
            a, r, q_ = L.attn, L.gla, p + "mix.left."
            q = _heads(_rms(hs @ w[q_ + "q"].T, w[q_ + "q.norm"], eps),
                       a.heads)
            k = _heads(_rms(hs @ w[q_ + "k"].T, w[q_ + "k.norm"], eps),
                       a.kv_heads)
            v = _heads(hs @ w[q_ + "v"].T, a.kv_heads)
            k, v = (t.repeat_interleave(a.heads // a.kv_heads, 1)
                    for t in (k, v))
            hide = past < 0
            if a.chunk > 0:
                hide = hide | (at[:, None] // a.chunk != at[None] // a.chunk)
            o = torch.empty(B, a.heads, T, a.vdim, dtype=F64, device=DEV)
            for h in range(a.heads):
                s = (q[:, h] @ k[:, h].transpose(1, 2).contiguous()) * a.scale
                o[:, h] = torch.softmax(s.masked_fill(hide, -math.inf),
                                        -1) @ v[:, h]
            mixed = L.left_scale * (
                o.transpose(1, 2).flatten(2) @ w[q_ + "o"].T)
            q_ = p + "mix.right."
            q = _heads(hs @ w[q_ + "q"].T, r.heads) / math.sqrt(r.dim)
            k = _heads(hs @ w[q_ + "k"].T, r.heads)
            v = _heads(hs @ w[q_ + "v"].T, r.heads)
            z = (hs @ w[q_ + "a1"].T) @ w[q_ + "a2"].T + w[q_ + "a2.b"]
            keep = _heads(torch.sigmoid(z) ** (1.0 / r.tau), r.heads)
            S = torch.zeros(B, r.heads, r.dim, r.vdim, dtype=F64, device=DEV)
            o = torch.empty(B, r.heads, T, r.vdim, dtype=F64, device=DEV)
            for t in range(T):
                S = S * keep[:, :, t, :, None] + \
                    k[:, :, t, :, None] * v[:, :, t, None, :]
                o[:, :, t] = (S * q[:, :, t, :, None]).sum(2)
            o = _rms(o, w[q_ + "norm"], eps).transpose(1, 2).flatten(2)
            mixed = mixed + L.right_scale * (
                (o * silu(hs @ w[q_ + "g"].T)) @ w[q_ + "o"].T)
        else:
            r, q_ = L.ret, p + "mix."
            q, k, v = (_heads(hs @ w[q_ + n].T, r.heads) for n in "qkv")
            d = r.rot_dims
            ang = at.to(F64)[:, None] * r.rot_base ** (
                -2.0 * torch.arange(d // 2, dtype=F64, device=DEV) / d)

            def rot(u):
                a, b = u[..., :d // 2], u[..., d // 2:d]
                return torch.cat([a * ang.cos() - b * ang.sin(),
                                  b * ang.cos() + a * ang.sin(),
                                  u[..., d:]], -1)
            q, k = rot(q), rot(k) / math.sqrt(r.dim)
            o = torch.empty(B, r.heads, T, r.vdim, dtype=F64, device=DEV)
            for h in range(r.heads):
                fade = torch.where(past >= 0,
                                   r.decay[h] ** past.clamp(min=0).to(F64),
                                   torch.zeros((), dtype=F64, device=DEV))
                s = q[:, h] @ k[:, h].transpose(1, 2).contiguous()
                o[:, h] = (s * fade) @ v[:, h]
            o = _rms(o, 1.0, eps).transpose(1, 2).flatten(2)
            mixed = (o * silu(hs @ w[q_ + "g"].T)) @ w[q_ + "o"].T
        n2 = _rms(x, 1.0 + w[p + "norm2"], eps)
        z, c = n2 @ w[p + "mlp.up"].T, w[p + "mlp.act"]
        act = (c[0] * _rms(z, 1.0, eps) + c[1] * _rms(z ** 2, 1.0, eps)
               + c[2] * _rms(z ** 3, 1.0, eps) + c[3])
        x = x + mixed * torch.sigmoid(n1 @ w[p + "rg1"].T + w[p + "rg1.b"]) \
            + (act @ w[p + "mlp.down"].T) * torch.sigmoid(
                n2 @ w[p + "rg2"].T + w[p + "rg2.b"])
    rows = torch.tensor([[len(t) - steps - 1 + j for t in tokens]
                         for j in range(steps + 1)], device=DEV)
    x = x[torch.arange(B, device=DEV)[None, :], rows]      # [steps + 1, B, W]
    logits = _rms(x, 1.0 + w["final.norm"], eps) @ w["embed"].T
    if cfg.logit_softcap > 0:
        logits = cfg.logit_softcap * torch.tanh(logits / cfg.logit_softcap)
    return {"logits": list(logits)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_dense(case, seed)
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "sample":
        return None        # draws come from the framework's own generator
    return _exact_session(case, seed)
