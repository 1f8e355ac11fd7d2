"""Timed cases of the self-speculative decoder: what a program that serves the hybrid model has the
framework do, each through a public entry point.

Seven families, all at the head geometry of the 4B-shape model (hidden 2560; gated-delta layers of 16 heads
of 128; attention of 16 query / 4 KV heads of 256; FFN 9728; vocabulary 248320):

  greedy     greedy acceptance of a verify pass's logits
  accept     rejection-sampling acceptance of a verify pass
  draft      the sampled draft pass behind the LM head: truncation statistics, draws, q rows
  attention  canvas attention of a block (or of a prefill chunk) against the KV cache
  gdn        a gated-delta layer between its projections: conv, gates, delta rule
  forward    a decoder forward over a block of canvas rows, replayed from a HIP graph as the decode loops do
  prefill    the causal prefill of new prompts into a fresh cache

listed() are the cases that are followed, draw() gives more of the same ranges, exact() computes a case's
outputs in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from trida_stack_amd import kernels as K
from trida_stack_amd.model import HybridConfig, TridaRuntime
from trida_stack_amd.sampling import prefill_batch

DEV = "cuda:0"
VOCAB = 248320
HQ, HKV, HEAD = 16, 4, 256      # attention heads
DK = 128                        # gated-delta key / value width
MODES = {"verify": K.MASK_VERIFY, "draft": K.MASK_DRAFT, "canvas": K.MASK_CANVAS}
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64


# ------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one sequence's greedy verify, the smallest call: 33 rows of a 151936-token vocabulary
        dict(name="greedy_b1", kind="greedy", batch=1, drafts=32, vocab=151936, dtype="fp32"),
        # a batched sampled step's acceptance: 64 sequences of 33 verify rows
        dict(name="accept_b64", kind="accept", batch=64, drafts=32, vocab=VOCAB, temperature=0.7, top_p=0.95, top_k=0),
        # one of the four draft passes of that step: 8 slots of each sequence drawn, their q rows kept
        dict(name="draft_b64", kind="draft", batch=64, slots=8, vocab=VOCAB, temperature=0.7, top_p=0.95, top_k=0),
        # a verify block over a long context of one sequence
        dict(name="attn_verify_8k", kind="attention", batch=1, rows=33, ctx_lo=8192, ctx_hi=8192, mode="verify", gate=True),
        # a denoise block over a batch of ragged contexts
        dict(name="attn_draft_b64", kind="attention", batch=64, rows=33, ctx_lo=512, ctx_hi=4096, mode="draft", gate=True),
        # a prefill chunk in the middle of a prompt
        dict(name="attn_chunk_512", kind="attention", batch=1, rows=512, ctx_lo=3584, ctx_hi=3584, mode="verify", gate=True),
        # a gated-delta layer over a whole prompt
        dict(name="gdn_prefill_4k", kind="gdn", batch=1, rows=4096, heads=16, mode="prefill"),
        # a gated-delta layer over a denoise block of a batch
        dict(name="gdn_block_b64", kind="gdn", batch=64, rows=33, heads=16, mode="draft"),
        # the forward that bounds one user's latency: every layer, one verify block
        dict(name="forward_b1", kind="forward", layers=32, batch=1, rows=33, ctx=2048, mode="verify", head_rows=33),
        # a small batch's verify forward (a quarter of the layers)
        dict(name="forward_b8", kind="forward", layers=8, batch=8, rows=33, ctx=2048, mode="verify", head_rows=33),
        # the largest batch's denoise forward, the LM head over the 8 slots that the pass draws
        dict(name="forward_b64", kind="forward", layers=8, batch=64, rows=33, ctx=2048, mode="draft", head_rows=8),
        # a new request's prompt (a quarter of the layers)
        dict(name="prefill_2k", kind="prefill", layers=8, prompts=1, tokens=2048),
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["greedy", "accept", "draft", "attention", "attention", "gdn", "gdn", "forward", "forward", "prefill"])
    block = rng.choice([1, 7, 15, 32, 33])   # an AR step, the canvases of n = 4 and 8, the denoise blocks
    if kind == "greedy":
        return dict(kind=kind, batch=log(1, 64), drafts=rng.choice([3, 7, 15, 32]), vocab=log(30001, 262144),
                    dtype=rng.choice(["fp32", "bf16"]))
    if kind in ("accept", "draft"):
        c = dict(kind=kind, batch=log(1, 64), vocab=log(30001, VOCAB), temperature=round(rng.uniform(0.5, 1.2), 2),
                 top_p=round(rng.uniform(0.8, 0.98), 3), top_k=rng.choice([0, 0, 50]))
        if kind == "accept":
            c["drafts"] = rng.choice([3, 7, 15, 32])
        else:
            c["slots"] = rng.choice([1, 2, 4, 8])
        return c
    if kind == "attention":
        if rng.random() < 0.4:
            return dict(kind=kind, batch=1, rows=log(65, 512), ctx_lo=(p := rng.choice([0, log(64, 3584)])), ctx_hi=p,
                        mode="verify", gate=True)
        batch = log(1, 64)
        hi = log(128, 8192 if batch <= 32 else 4096)
        return dict(kind=kind, batch=batch, rows=block, ctx_lo=max(1, hi // rng.choice([1, 3, 8])), ctx_hi=hi,
                    mode=rng.choice(["verify", "draft", "canvas"]), gate=rng.random() < 0.8)
    if kind == "gdn":
        heads = rng.choice([16, 16, 32])
        if rng.random() < 0.5:
            rows = log(65, 4096)
            return dict(kind=kind, batch=rng.randint(1, max(1, min(8, 8192 // rows))), rows=rows, heads=heads, mode="prefill")
        return dict(kind=kind, batch=log(1, 64), rows=block, heads=heads, mode=rng.choice(["verify", "draft"]))
    if kind == "forward":
        batch = log(1, 64)
        mode = rng.choice(["verify", "draft"]) if batch * block <= 512 else "draft"
        return dict(kind=kind, layers=4, batch=batch, rows=block, ctx=log(64, 4096), mode=mode,
                    head_rows=block if batch * block <= 512 else min(8, block))
    return dict(kind=kind, layers=4, prompts=rng.choice([1, 1, 2, 3]), tokens=log(5, 2048))


# ------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _logits(g, *shape):
    """Logit rows as a language model has them: a broad bulk, and in every other row a few likely tokens."""
    x = torch.randn(*shape, generator=g, device=DEV) * 2
    flat = x.view(-1, shape[-1])
    rows = flat[::2]
    at = torch.randint(0, shape[-1], (rows.shape[0], 20), generator=g, device=DEV)
    rows.scatter_add_(1, at, torch.rand(rows.shape[0], 20, generator=g, device=DEV) * 8 + 8)
    return x


def _greedy_inputs(c, seed):
    g = _gen(seed)
    B, Kd, V = c["batch"], c["drafts"], c["vocab"]
    logits = _logits(g, B, Kd + 1, V).to(F32 if c["dtype"] == "fp32" else BF)
    drafts = torch.randint(0, V, (B, Kd), generator=g, device=DEV)
    # geometric accepted prefixes: each draft is the row's argmax with probability 0.7
    hit = torch.rand(B, Kd, generator=g, device=DEV) < 0.7
    drafts = torch.where(hit, logits[:, :Kd].float().argmax(-1), drafts)
    ctx = torch.randint(512, 4097, (B,), generator=g, device=DEV)
    return dict(logits=logits, drafts=drafts, ctx=ctx)


def _accept_inputs(c, seed):
    g = _gen(seed)
    B, Kd, V, T = c["batch"], c["drafts"], c["vocab"], c["temperature"]
    p = _logits(g, B, Kd + 1, V)
    q = torch.empty(B, Kd, V, device=DEV)
    drafts = torch.empty(B, Kd, dtype=torch.int64, device=DEV)
    for b in range(B):  # the draft's distribution: near the verify pass's, its tail cut
        y = (p[b, :Kd] + torch.randn(Kd, V, generator=g, device=DEV) * 0.3) / T
        e = torch.exp(y - y.amax(-1, keepdim=True))
        e = torch.where(e > 1e-3, e, torch.zeros_like(e))
        q[b] = e / e.sum(-1, keepdim=True)
        drafts[b] = torch.multinomial(q[b], 1, generator=g)[:, 0]
    return dict(p=p, q=q, drafts=drafts, ua=torch.rand(B, Kd, generator=g, device=DEV),
                us=torch.rand(B, generator=g, device=DEV), ctx=torch.randint(512, 4097, (B,), generator=g, device=DEV))


def _draft_inputs(c, seed):
    g = _gen(seed)
    B, k, V = c["batch"], c["slots"], c["vocab"]
    sel = torch.arange(k, device=DEV).repeat(B, 1).contiguous()
    return dict(logits=_logits(g, B, k, V).to(BF), sel=sel, u=torch.rand(B * k, generator=g, device=DEV))


def _lengths(c, g):
    return torch.randint(c["ctx_lo"], c["ctx_hi"] + 1, (c["batch"],), generator=g, device=DEV, dtype=torch.int32)


def _attention_inputs(c, seed):
    g = _gen(seed)
    B, T = c["batch"], c["rows"]
    cap = c["ctx_hi"] + T
    rn = lambda *sh: torch.randn(*sh, generator=g, device=DEV, dtype=F32).to(BF)  # noqa: E731
    length = _lengths(c, g)
    # the q projection holds [q | gate] per head
    gate = rn(B, T, HQ, 2 * HEAD)[..., HEAD:] if c["gate"] else None
    return dict(q=rn(B, T, HQ, HEAD), k=rn(B, HKV, cap, HEAD), v=rn(B, HKV, cap, HEAD), length=length, gate=gate, cap=cap)


def _gates(g, heads):
    """A_log and dt_bias of a gated-delta layer: decay rates in 1..16, time steps in 1e-3..1e-1."""
    A_log = torch.log(torch.rand(heads, generator=g, device=DEV) * 15 + 1)
    dt = torch.exp(torch.rand(heads, generator=g, device=DEV) * math.log(100.0) + math.log(1e-3))
    return A_log, dt + torch.log(-torch.expm1(-dt))


def _gdn_inputs(c, seed):
    g = _gen(seed)
    B, T, Hv = c["batch"], c["rows"], c["heads"]
    C = (2 * 16 + Hv) * DK
    rn = lambda *sh: torch.randn(*sh, generator=g, device=DEV, dtype=F32)  # noqa: E731
    A_log, dt_bias = _gates(g, Hv)
    return dict(proj=rn(B, T, C + Hv * DK + 2 * Hv).to(BF), window=rn(B, 3, C).to(BF), conv=((torch.rand(C, 4, generator=g, device=DEV) - 0.5)).to(BF),
                A_log=A_log, dt_bias=dt_bias, state=rn(B, Hv, DK, DK) * 0.05, C=C)


def _config(layers):
    return HybridConfig(n_layers=layers)


def _weights(layers, g):
    """Random weights of the hybrid decoder in the [out, in] layout of checkpoints: projections normal(0, 0.02),
    the ones that write the residual stream scaled down with the depth, a unit-scale embedding."""
    c = _config(layers)
    h, out = c.hidden, 0.02 / math.sqrt(2 * layers)

    def nrm(n, k, std=0.02):
        return (torch.randn(n, k, generator=g, device=DEV, dtype=BF) * std)

    w = {"embed": nrm(c.vocab, h, 1.0), "final_norm": torch.randn(h, generator=g, device=DEV).mul(0.05).to(BF)}
    w["lm_head"] = nrm(c.vocab, h)
    for i in range(layers):
        p = f"l{i}."
        for n in ("in_norm", "post_norm"):
            w[p + n] = torch.randn(h, generator=g, device=DEV).mul(0.05).to(BF)
        w[p + "w_gu"] = nrm(2 * c.intermediate, h)
        w[p + "w_down"] = nrm(h, c.intermediate, out)
        if c.is_attention(i):
            w[p + "w_qkv"] = nrm((2 * HQ + 2 * HKV) * HEAD, h)
            w[p + "q_norm"] = torch.randn(HEAD, generator=g, device=DEV).mul(0.05).to(BF)
            w[p + "k_norm"] = torch.randn(HEAD, generator=g, device=DEV).mul(0.05).to(BF)
            w[p + "w_o"] = nrm(h, HQ * HEAD, out)
        else:
            w[p + "w_in"] = nrm(c.conv_dim + c.value_dim + 2 * c.lin_v_heads, h)
            w[p + "conv_w"] = (torch.rand(c.conv_dim, c.conv_kernel, generator=g, device=DEV) - 0.5).to(BF)
            w[p + "A_log"], w[p + "dt_bias"] = _gates(g, c.lin_v_heads)
            w[p + "gnorm"] = (torch.randn(c.lin_v_dim, generator=g, device=DEV) * 0.05 + 1).to(BF)
            w[p + "w_out"] = nrm(h, c.value_dim, out)
    return w


def _forward_inputs(c, seed):
    """Weights, block token ids and the decode state of every sequence (its KV entries, gated-delta states and
    conv windows), contexts between half of ctx and ctx."""
    g = _gen(seed)
    cfg = _config(c["layers"])
    w = _weights(c["layers"], g)
    B, T = c["batch"], c["rows"]
    n_attn = sum(cfg.is_attention(i) for i in range(cfg.n_layers))
    n_gdn = cfg.n_layers - n_attn
    cap = c["ctx"] + T
    ids = torch.randint(0, cfg.vocab, (B, T), generator=g, device=DEV)
    if c["mode"] == "draft" and T > 1:
        ids[:, 1 + T // 2:] = cfg.mask_id
    length = torch.randint(max(1, c["ctx"] // 2), c["ctx"] + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    if B == 1:
        length.fill_(c["ctx"])
    rn = lambda *sh: torch.randn(*sh, generator=g, device=DEV, dtype=F32)  # noqa: E731
    kv = torch.randn(2, n_attn, B, HKV, cap, HEAD, generator=g, device=DEV, dtype=BF)
    state = rn(n_gdn, B, 16, DK, DK) * 0.05
    window = rn(n_gdn, B, 3, cfg.conv_dim).to(BF)
    return dict(cfg=cfg, w=w, ids=ids, length=length, kv=kv, state=state, window=window, cap=cap)


def _prefill_inputs(c, seed):
    g = _gen(seed)
    w = _weights(c["layers"], g)
    cfg = _config(c["layers"])
    # ragged prompts, the first one the longest
    lens = [max(1, c["tokens"] * (4 - i) // 4) for i in range(c["prompts"])]
    prompts = [torch.randint(0, cfg.vocab, (n,), generator=g, device=DEV).tolist() for n in lens]
    return dict(cfg=cfg, w=w, prompts=prompts)


INPUTS = dict(greedy=_greedy_inputs, accept=_accept_inputs, draft=_draft_inputs, attention=_attention_inputs,
              gdn=_gdn_inputs, forward=_forward_inputs, prefill=_prefill_inputs)


def prepare(case, seed):
    s = INPUTS[case["kind"]](case, seed)
    s["case"] = case
    if case["kind"] == "draft":  # the q rows that the step keeps, and its fp32 rows
        B, k, V = case["batch"], case["slots"], case["vocab"]
        s["lf"], s["q"] = torch.empty(B, k, V, device=DEV), torch.zeros(B, k, V, device=DEV)
    elif case["kind"] == "prefill":
        s["rt"] = TridaRuntime(s["cfg"], s.pop("w"), device=DEV)
    elif case["kind"] == "forward":
        rt = s["rt"] = TridaRuntime(s["cfg"], s.pop("w"), device=DEV)
        cache = rt.make_cache(case["batch"], s["cap"])
        kv = s.pop("kv")
        cache.kv_k.copy_(kv[0])
        cache.kv_v.copy_(kv[1])
        cache.state.copy_(s.pop("state"))
        cache.window.copy_(s.pop("window"))
        cache.length.copy_(s["length"])
        cache.pos.copy_(s["length"])
        cache.ctx_hint = case["ctx"]
        # the decode loops replay their forwards from a HIP graph
        s["cache"] = cache
        side = torch.cuda.Stream(DEV)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _forward(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["logits"] = _forward(s)
    return s


def _forward(s):
    c = s["case"]
    return s["rt"].forward(s["ids"], s["cache"], c["mode"], rows=c["head_rows"])


# ------------------------------------------------------------------------------------------- one pass
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "greedy":
        am, n_acc, bonus, crop = K.greedy_accept(s["logits"], s["drafts"], ctx_len=s["ctx"])
        return dict(argmax=am, n_acc=n_acc, bonus=bonus, crop=crop)
    if kind == "accept":
        n_acc, token, crop, _, status = K.sample_accept(
            s["p"], s["q"], s["drafts"], s["ua"], s["us"], temperature=c["temperature"], top_k=c["top_k"],
            top_p=c["top_p"], ctx_len=s["ctx"])
        return dict(n_acc=n_acc, token=token, crop=crop, status=status)
    if kind == "draft":
        lf = K.gather_rows(s["logits"], s["sel"], out=s["lf"])
        m, thr, zk, status = K.truncate_stats(lf, temperature=c["temperature"], top_k=c["top_k"], top_p=c["top_p"])
        token = K.sample_rows(lf, (m, thr, zk), s["u"], temperature=c["temperature"])
        q = K.truncated_probs_rows(lf, (m, thr, zk), s["sel"], s["sel"], s["q"], temperature=c["temperature"])
        return dict(m=m, thr=thr, zk=zk, status=status, token=token, q=q)
    if kind == "attention":
        return K.attn_canvas(s["q"], s["k"], s["v"], s["length"], mask_mode=MODES[c["mode"]], n_clean=(c["rows"] + 1) // 2,
                             gate=s["gate"], max_keys=s["cap"])
    if kind == "gdn":
        return _run_gdn(s, c)
    if kind == "forward":
        s["graph"].replay()
        return s["logits"]
    rt, prompts = s["rt"], s["prompts"]
    cache = rt.make_cache(len(prompts), max(len(p) for p in prompts) + 64)
    logits = prefill_batch(rt, cache, prompts)
    return dict(logits=logits, k=cache.kv_k, v=cache.kv_v, state=cache.state, window=cache.window)


def _run_gdn(s, c):
    proj, C, Hv, prefill = s["proj"], s["C"], c["heads"], c["mode"] == "prefill"
    B, T = proj.shape[:2]
    at = C + Hv * DK
    win = torch.empty_like(s["window"]) if prefill else None
    pre = None if prefill else torch.empty(B, T, C, dtype=BF, device=DEV)
    q, k, v, g, beta = K.gdn_prep(proj[..., :C], s["window"], s["conv"], proj[..., at + Hv: at + 2 * Hv], proj[..., at: at + Hv],
                                  s["A_log"], s["dt_bias"], Hk=16, Hv=Hv, Dk=DK, Dv=DK, window_out=win, pre_out=pre)
    if prefill:
        state = torch.empty_like(s["state"])
        out = K.gdr_chunk(q, k, v, g, beta, s["state"], state_out=state)
        return dict(out=out, state=state, window=win)
    mode = dict(causal_mode=2, num_clean=1) if c["mode"] == "draft" else dict(causal_mode=1)
    # the block readout on matrix cores for batches, the token recurrence for a few sequences
    if B * Hv >= TridaRuntime.GDR_BLOCK_MIN_HEADS and T <= 64:
        out = K.gdr_chunk(q, k, v, g, beta, s["state"], **mode)
    else:
        out, _ = K.gdr_recurrent(q, k, v, g, beta, s["state"], **mode)
    return dict(out=out, k=k, v=v, g=g, beta=beta, rows=pre)


# ------------------------------------------------------------------------------------------- work
def work(case):
    c, kind = case, case["kind"]
    if kind == "greedy":
        return {"bytes": c["batch"] * (c["drafts"] + 1) * c["vocab"] * (4 if c["dtype"] == "fp32" else 2), "flops": 0}
    if kind == "accept":
        # each sequence's first verify row, and the correction's rows of p and q (how many more rows are read
        # depends on what is accepted)
        return {"bytes": c["batch"] * 3 * c["vocab"] * 4, "flops": 0}
    if kind == "draft":
        return {"bytes": c["batch"] * c["slots"] * c["vocab"] * (2 + 4), "flops": 0}
    if kind == "attention":
        B, T = c["batch"], c["rows"]
        keys = B * ((c["ctx_lo"] + c["ctx_hi"]) / 2 + T)
        return {"bytes": keys * HKV * HEAD * 2 * 2 + B * T * HQ * HEAD * 2 * (3 if c["gate"] else 2),
                "flops": 4.0 * HQ * HEAD * T * (keys - (B * (T - 1) / 2 if c["mode"] == "verify" else 0))}
    if kind == "gdn":
        B, T, Hv = c["batch"], c["rows"], c["heads"]
        C = (32 + Hv) * DK
        rows = B * T
        state = B * Hv * DK * DK * 4 * (2 if c["mode"] == "prefill" else 1)
        kept = 0 if c["mode"] == "prefill" else rows * (2 * C + (16 + Hv) * DK * 2)
        return {"bytes": rows * (C * 2 + 4 * Hv + Hv * DK * 2) + state + kept, "flops": 8.0 * rows * Hv * DK * DK}
    cfg = _config(c["layers"])
    h = cfg.hidden
    body = cfg.n_params() - cfg.vocab * h
    n_attn = sum(cfg.is_attention(i) for i in range(cfg.n_layers))
    n_gdn = cfg.n_layers - n_attn
    if kind == "forward":
        B, T, R = c["batch"], c["rows"], c["head_rows"]
        keys = B * ((c["ctx"] if B == 1 else 0.75 * c["ctx"]) + T)
        return {"bytes": 2.0 * (body + cfg.vocab * h) + n_attn * keys * HKV * HEAD * 4 + n_gdn * B * 16 * DK * DK * 4
                + 2.0 * B * R * cfg.vocab,
                "flops": 2.0 * body * B * T + 2.0 * cfg.vocab * h * B * R + n_attn * 4.0 * HQ * HEAD * T * keys
                + n_gdn * B * T * 8.0 * 16 * DK * DK}
    lens = [max(1, c["tokens"] * (4 - i) // 4) for i in range(c["prompts"])]
    n, sq = sum(lens), sum(t * t for t in lens)
    return {"bytes": 2.0 * (body + cfg.vocab * h) + n_attn * n * HKV * HEAD * 4 + n_gdn * len(lens) * 16 * DK * DK * 4,
            "flops": 2.0 * body * n + 2.0 * cfg.vocab * h * len(lens) + n_attn * 2.0 * HQ * HEAD * sq
            + n_gdn * n * 8.0 * 16 * DK * DK}


def tolerance(case):
    kind = case["kind"]
    if kind == "greedy":
        return "exact"
    if kind == "accept":   # decisions on given uniforms: a tie may fall either way
        return {"rel": 0.0, "differ": 0.01}
    if kind == "draft":    # 32-bit exponentials; a token at the nucleus boundary may fall either way
        return {"rel": 2e-5, "max": 0.1, "differ": 0.01}
    if kind == "attention":
        return {"rel": 1e-2}
    if kind == "gdn":
        return {"rel": 1e-2}
    return {"rel": 0.03}


# ------------------------------------------------------------------------------------------- 64 bits
def exact(case, seed):
    s = INPUTS[case["kind"]](case, seed)
    kind = case["kind"]
    if kind in ("greedy", "accept"):
        return None  # whole numbers
    if kind == "draft":
        return _exact_draft(case, s)
    if kind == "attention":
        return _exact_attention(s["q"].double(), s["k"], s["v"], s["length"].tolist(), case["mode"], (case["rows"] + 1) // 2,
                                None if s["gate"] is None else s["gate"].double())
    if kind == "gdn":
        return _exact_gdn(case, s)
    if kind == "forward":
        return _exact_forward(case, s)
    return _exact_prefill(case, s)


def _exact_draft(c, s):
    y = (s["logits"].float() / torch.tensor(c["temperature"], dtype=F32, device=DEV)).view(-1, c["vocab"])
    q, stats = torch.empty(y.shape, dtype=F32, device=DEV), []
    for r0 in range(0, y.shape[0], 64):
        row = y[r0: r0 + 64].double()
        top = row.sort(-1, descending=True).values
        n = min(c["top_k"], c["vocab"]) if c["top_k"] else c["vocab"]
        cand = top[:, :n]
        e = torch.exp(cand - cand[:, :1])
        p = e / e.sum(-1, keepdim=True)
        kept = ((p.cumsum(-1) - p) < c["top_p"]).sum(-1, keepdim=True).clamp_min(1)
        thr = cand.gather(1, kept - 1)
        e = torch.where(row >= thr, torch.exp(row - cand[:, :1]), torch.zeros_like(row))
        zk = e.sum(-1, keepdim=True)
        q[r0: r0 + 64] = (e / zk).float()
        stats.append(torch.cat([cand[:, :1], thr, zk], 1))
    st = torch.cat(stats)
    shape = s["logits"].shape[:2]
    m, thr, zk = (st[:, i].reshape(shape) for i in range(3))
    return dict(m=m, thr=thr, zk=zk, status=None, token=None, q=q.view(*shape, -1))


def _exact_attention(q, k_cache, v_cache, lengths, mode, n_clean, gate):
    B, T = q.shape[:2]
    out = torch.empty_like(q)
    r, col = torch.arange(T, device=DEV)[:, None], torch.arange(T, device=DEV)[None]
    inner = col <= r
    if mode == "draft":
        inner = torch.ones_like(inner)
    elif mode == "canvas":
        inner = inner | (r >= n_clean)
    for b in range(B):
        n = lengths[b] + T
        seen = torch.cat([torch.ones(T, lengths[b], dtype=torch.bool, device=DEV), inner], 1)
        for j in range(HKV):
            heads = slice(j * (HQ // HKV), (j + 1) * (HQ // HKV))
            k, v = k_cache[b, j, :n].double(), v_cache[b, j, :n].double()
            qq = q[b, :, heads].transpose(0, 1).contiguous()
            sc = torch.matmul(qq, k.t().contiguous()) * HEAD ** -0.5
            sc = sc.masked_fill(~seen, float("-inf"))
            out[b, :, heads] = torch.matmul(torch.softmax(sc, -1), v).transpose(0, 1)
    return out if gate is None else out * torch.sigmoid(gate)


def _exact_delta(x, window, conv, a, b, A_log, dt_bias, state, Hv, num_clean):
    """Conv, gates and the delta rule of rows x [B, T, C]: (readout, the rows k, v, g, beta, the final state
    [B, Hv, Dv, Dk], the new window). num_clean: rows from there on read the final state."""
    B, T, C = x.shape
    full = torch.cat([window.double(), x.double()], 1)
    y = F.silu(sum(full[:, j: j + T] * conv[:, j].double() for j in range(4)))
    q, k, v = (t.reshape(B, T, -1, DK) for t in torch.split(y, [16 * DK, 16 * DK, Hv * DK], -1))
    q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    g = -torch.exp(A_log.double()) * F.softplus(a.double() + dt_bias.double())
    beta = torch.sigmoid(b.double())
    kk = k.repeat_interleave(Hv // 16, 2)
    qq = q.repeat_interleave(Hv // 16, 2) * DK ** -0.5
    S = state.double()
    out = torch.empty(B, T, Hv, DK, dtype=F64, device=DEV)
    decay = torch.exp(g)
    for t in range(T):
        S = S * decay[:, t, :, None, None]
        kt = kk[:, t, :, None, :]
        delta = (v[:, t] - (S * kt).sum(-1)) * beta[:, t, :, None]
        S = S + delta[..., None] * kt
        if t < num_clean:
            out[:, t] = (S * qq[:, t, :, None, :]).sum(-1)
    for t in range(num_clean, T):
        out[:, t] = (S * qq[:, t, :, None, :]).sum(-1)
    return out, k, v, g, beta, S, full[:, -3:]


def _exact_gdn(c, s):
    proj, C, Hv = s["proj"], s["C"], c["heads"]
    at = C + Hv * DK
    T = c["rows"]
    out, k, v, g, beta, S, win = _exact_delta(
        proj[..., :C], s["window"], s["conv"], proj[..., at + Hv: at + 2 * Hv], proj[..., at: at + Hv], s["A_log"],
        s["dt_bias"], s["state"], Hv, 1 if c["mode"] == "draft" else T)
    if c["mode"] == "prefill":
        return dict(out=out, state=S, window=win)
    return dict(out=out, k=k, v=v, g=g, beta=beta, rows=proj[..., :C].double())


def _norm(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * (1 + w.double())


def _rope(x, pos, cfg):
    half = cfg.rot_dim // 2
    inv = cfg.rope_theta ** (-2.0 * torch.arange(half, dtype=F64, device=DEV) / cfg.rot_dim)
    ang = pos.double()[..., None, None] * inv
    x1, x2 = x[..., :half], x[..., half: 2 * half]
    return torch.cat([x1 * ang.cos() - x2 * ang.sin(), x2 * ang.cos() + x1 * ang.sin(), x[..., 2 * half:]], -1)


def _exact_model(cfg, w, ids, length, kv_k, kv_v, state, window, mode):
    """The decoder on a block of ids [B, T] over fp64 caches kv_k / kv_v [A, B, Hkv, cap, D], states and windows (all
    updated in place with the block): the last hidden rows after the final norm."""
    B, T = ids.shape
    lin = lambda x, name: torch.matmul(x.reshape(B * T, -1), w[name].double().t()).view(B, T, -1)  # noqa: E731
    x = w["embed"][ids].double()
    pos = length[:, None].long() + torch.arange(T, device=DEV)[None]
    na = ng = 0
    for i in range(cfg.n_layers):
        p = f"l{i}."
        n = _norm(x, w[p + "in_norm"], cfg.rms_eps)
        if cfg.is_attention(i):
            qkv = lin(n, p + "w_qkv")
            q, gate = qkv[..., : 2 * HQ * HEAD].reshape(B, T, HQ, 2 * HEAD).split(HEAD, -1)
            k, v = qkv[..., 2 * HQ * HEAD:].reshape(B, T, 2, HKV, HEAD).unbind(2)
            q = _rope(_norm(q, w[p + "q_norm"], cfg.rms_eps), pos, cfg)
            k = _rope(_norm(k, w[p + "k_norm"], cfg.rms_eps), pos, cfg)
            for b in range(B):
                n0 = int(length[b])
                kv_k[na, b, :, n0: n0 + T] = k[b].transpose(0, 1)
                kv_v[na, b, :, n0: n0 + T] = v[b].transpose(0, 1)
            o = _exact_attention(q, kv_k[na], kv_v[na], length.tolist(), mode, T, gate)
            x = x + lin(o, p + "w_o")
            na += 1
        else:
            proj = lin(n, p + "w_in")
            C, VD, H = cfg.conv_dim, cfg.value_dim, cfg.lin_v_heads
            out, _, _, _, _, S, win = _exact_delta(
                proj[..., :C], window[ng], w[p + "conv_w"], proj[..., C + VD + H:], proj[..., C + VD: C + VD + H],
                w[p + "A_log"], w[p + "dt_bias"], state[ng], H, 1 if mode == "draft" else T)
            state[ng], window[ng] = S, win
            z = proj[..., C: C + VD].reshape(B, T, H, -1)
            y = out * torch.rsqrt((out * out).mean(-1, keepdim=True) + cfg.rms_eps) * w[p + "gnorm"].double() * F.silu(z)
            x = x + lin(y, p + "w_out")
            ng += 1
        gu = lin(_norm(x, w[p + "post_norm"], cfg.rms_eps), p + "w_gu")
        x = x + lin(F.silu(gu[..., : cfg.intermediate]) * gu[..., cfg.intermediate:], p + "w_down")
    return _norm(x, w["final_norm"], cfg.rms_eps)


def _exact_forward(c, s):
    x = _exact_model(s["cfg"], s["w"], s["ids"], s["length"], s["kv"][0].double(), s["kv"][1].double(), s["state"].double(),
                     s["window"].double(), c["mode"])[:, : c["head_rows"]]
    head = s["w"]["lm_head"].double().t()
    return torch.stack([torch.matmul(row, head).float() for row in x])


def _exact_prefill(c, s):
    cfg, w, prompts = s["cfg"], s["w"], s["prompts"]
    B, cap = len(prompts), max(len(p) for p in prompts) + 64
    n_attn = sum(cfg.is_attention(i) for i in range(cfg.n_layers))
    new = lambda *sh: torch.zeros(*sh, dtype=F64, device=DEV)  # noqa: E731
    kv_k, kv_v = new(n_attn, B, HKV, cap, HEAD), new(n_attn, B, HKV, cap, HEAD)
    state, window = new(cfg.n_layers - n_attn, B, 16, DK, DK), new(cfg.n_layers - n_attn, B, 3, cfg.conv_dim)
    zero = torch.zeros(1, dtype=torch.int32, device=DEV)
    logits = []
    for b, prompt in enumerate(prompts):
        one = slice(b, b + 1)
        x = _exact_model(cfg, w, torch.tensor([prompt], device=DEV), zero, kv_k[:, one], kv_v[:, one], state[:, one],
                         window[:, one], "verify")
        logits.append(torch.matmul(x[0, -1], w["lm_head"].double().t()))
    return dict(logits=torch.stack(logits), k=kv_k, v=kv_v, state=state, window=window)
