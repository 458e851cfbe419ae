"""The work that users of this framework have it do, as cases that can be timed and compared.

Kinds of case (the `kind` of each dict):

  forward  flash_attn_key_bias without gradients: an attention layer of a prefill or an evaluation.
  train    flash_attn_key_bias with gradients: out, dq, dk, dv and the key bias's gradient of a
           training step of the gate.
  varlen   flash_attn_key_bias_varlen with gradients over packed sequences (packed training).
  score    ScoringHead.scores: the gate's score of every prompt row.
  select   gate.select_pack: the keep lists of a batch, its kept hidden rows and the K/V rows of the
           layers at or below the gate, the kept positions and their gate bias.
  decode   DecodeState.step: one token for every sequence of a batch, all 28 layers, as the step of a
           generation under way (the step's HIP graph is captured by then).  The input tokens are
           given (a forced continuation), so that a near tie of two logits does not change the work.
  prefill  prefill_batch: the whole gated prefill of a Qwen3-1.7B-shaped model up to the first token's
           logits.  It returns the logits and the caches of the layers at or below the gate.  The kept
           rows' caches are left out: their order depends on which of two nearly equal scores is
           larger, so that one rounding anywhere below moves every row behind it.

Every number is drawn on the GPU from the seed.  Queries and keys have unit variance, as the q/k norms
of the model leave them.
"""
import math

import torch

D = 128                      # head dim
SCALE = D ** -0.5
D_MODEL = 2048
DEVICE = "cuda"


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # two short odd-length prompts: launches and host work count
        dict(name="forward_b2_517", kind="forward", batch=2, seq=517, heads=16, kv_heads=8, causal=True),
        # a 4k prompt's attention layer
        dict(name="forward_4k", kind="forward", batch=1, seq=4096, heads=16, kv_heads=8, causal=True),
        # the long-context layer, the benchmark's headline shape
        dict(name="forward_32k", kind="forward", batch=1, seq=32768, heads=16, kv_heads=8, causal=True),
        # a small training step (one 2k sequence)
        dict(name="train_2k", kind="train", batch=1, seq=2048, heads=16, kv_heads=8, causal=True),
        # the large training step of the benchmark
        dict(name="train_b4_8k", kind="train", batch=4, seq=8192, heads=16, kv_heads=8, causal=True),
        # packed training over ragged sequences
        dict(name="varlen_packed6", kind="varlen", lens="4021,1733,897,3210,260,2048", heads=16, kv_heads=8),
        # the scores of a 32k prompt
        dict(name="score_32k", kind="score", rows=32768),
        # keep 2000 of a 32k prompt: hidden rows and two layers of K/V
        dict(name="select_32k_k2000", kind="select", lens="32768", keep="2000", layers=2, bf16_scores=False),
        # eight ragged prompts of 42k to 124k, each with its own K; bf16-valued scores (ties)
        dict(name="select_ragged8", kind="select", lens="114517,57946,113394,80391,42386,123699,106754,74151",
             keep="2000,4000,100,4000,100,100,4000,500", layers=2, bf16_scores=True),
        # one user's generation after a pruned 32k prompt
        dict(name="decode_b1_32k", kind="decode", lens="32768", keep="2000", prune_below=False),
        # a batch of eight generations after ragged prompts
        dict(name="decode_b8", kind="decode", lens="4096,2711,6002,3517,5120,1999,4444,7001",
             keep="500,500,1000,100,2000,500,100,1000", prune_below=False),
        # time to first token of a 32k prompt pruned to 2000
        dict(name="prefill_32k_k2000", kind="prefill", lens="32768", keep="2000", branch=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "train", "train", "varlen", "score", "select", "decode", "prefill"])
    heads, kv_heads = rng.choice([(16, 8), (16, 8), (16, 8), (8, 8), (12, 4), (8, 2)])
    if kind in ("forward", "train"):
        seq = _log_int(rng, 128, 24000 if kind == "forward" else 8000)
        batch = rng.randint(1, max(1, min(4, 32768 // seq)))
        causal = rng.random() < 0.85 or seq * batch > 8192
        return dict(kind=kind, batch=batch, seq=seq, heads=heads, kv_heads=kv_heads, causal=causal)
    if kind == "varlen":
        lens = [_log_int(rng, 100, 5000) for _ in range(rng.randint(2, 8))]
        return dict(kind=kind, lens=",".join(map(str, lens)), heads=heads, kv_heads=kv_heads)
    if kind == "score":
        return dict(kind=kind, rows=_log_int(rng, 512, 400000))
    if kind == "select":
        n = rng.randint(1, 8)
        lens = [_log_int(rng, 600, 120000) for _ in range(n)]
        return dict(kind=kind, lens=",".join(map(str, lens)),
                    keep=",".join(str(rng.choice([100, 500, 2000, 4000])) for _ in lens), layers=rng.choice([0, 1, 2]),
                    bf16_scores=rng.random() < 0.5)
    if kind == "decode":
        lens = [_log_int(rng, 600, 8000) for _ in range(rng.randint(1, 8))]
        return dict(kind=kind, lens=",".join(map(str, lens)),
                    keep=",".join(str(rng.choice([100, 500, 2000])) for _ in lens), prune_below=rng.random() < 0.3)
    n = rng.randint(1, 3)
    lens = [_log_int(rng, 700, 24000 // n) for _ in range(n)]
    return dict(kind="prefill", lens=",".join(map(str, lens)), keep=",".join(str(rng.choice([100, 500])) for _ in lens),
                branch=rng.random() < 0.3)


# ---- inputs --------------------------------------------------------------------------------------

def _ints(text):
    return [int(x) for x in text.split(",")]


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEVICE).to(torch.bfloat16)


def _spans(lens):
    """State spans: all of a prompt but a 64-token prefix and a 256-token suffix."""
    return [64] * len(lens), [n - 256 for n in lens]


def _key_bias(g, rows, heads, seq):
    """log(sigmoid(z)) per key, times a factor per head: what the gate adds to the logits."""
    kb = torch.nn.functional.logsigmoid(torch.randn(rows, 1, seq, generator=g, device=DEVICE) * 2.0)
    return kb * (0.75 + 0.5 * torch.rand(1, heads, 1, generator=g, device=DEVICE))


def _attention_inputs(case, g):
    H, Hkv = case["heads"], case["kv_heads"]
    if case["kind"] == "varlen":
        lens = _ints(case["lens"])
        lead, rows, seq = (sum(lens),), len(lens), max(lens)
    else:
        lead, rows, seq = (case["batch"], case["seq"]), case["batch"], case["seq"]
    q, k, v = _normal(g, *lead, H, D), _normal(g, *lead, Hkv, D), _normal(g, *lead, Hkv, D)
    dout = _normal(g, *lead, H, D)
    kb = _key_bias(g, rows, H, seq)
    if case["kind"] == "varlen":
        for b, n in enumerate(lens):
            kb[b, :, n:] = 0.0
    return q, k, v, kb, dout


def _gate_inputs(case, g):
    lens = _ints(case["lens"])
    scores = torch.randn(sum(lens), generator=g, device=DEVICE)
    if case["bf16_scores"]:
        scores = scores.to(torch.bfloat16).float()
    hidden = _normal(g, sum(lens), D_MODEL)
    kv = [_normal(g, sum(lens), 8, D) for _ in range(2 * case["layers"])]
    return lens, scores, [hidden] + kv


def _score_inputs(case, g):
    from tokengate_amd import gate
    head = gate.random_head(26, 16, seed=5, device=DEVICE)
    head.b1 = 0.1 * torch.randn(256, generator=g, device=DEVICE)
    return head, _normal(g, case["rows"], D_MODEL)


def _model(case, seed):
    from tokengate_amd import decoder, gate
    wts = decoder.random_decoder(decoder.QWEN3_1P7B, seed=int(seed) % (1 << 31), device=DEVICE)
    if case.get("branch"):
        head = gate.random_branch_head(wts, 1, seed=5)
    else:
        head = gate.random_head(wts.shape.n_layers - 2, wts.shape.n_heads, seed=5, device=DEVICE)
    g = _gen(seed + 1)
    ids = [torch.randint(0, wts.shape.vocab, (n,), generator=g, device=DEVICE) for n in _ints(case["lens"])]
    return wts, head, ids, g


MAX_NEW_TOKENS = 1024


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train", "varlen"):
        q, k, v, kb, dout = _attention_inputs(case, _gen(seed))
        state = dict(case=case, q=q, k=k, v=v, kb=kb)
        if kind != "forward":
            for t in (q, k, v, kb):
                t.requires_grad_(True)
            state["dout"] = dout
        if kind == "varlen":
            cu = [0]
            for n in _ints(case["lens"]):
                cu.append(cu[-1] + n)
            state["cu"] = torch.tensor(cu, dtype=torch.int32, device=DEVICE)
            state["max"] = max(_ints(case["lens"]))
        return state
    if kind == "score":
        head, x = _score_inputs(case, _gen(seed))
        return dict(case=case, head=head, x=x)
    if kind == "select":
        from tokengate_amd import gate
        lens, scores, rows = _gate_inputs(case, _gen(seed))
        starts, ends = _spans(lens)
        first = [sum(lens[:b]) for b in range(len(lens))]
        plan = gate.plan(first, lens, starts, ends, _ints(case["keep"]), torch.device(DEVICE, torch.cuda.current_device()))
        return dict(case=case, scores=scores, rows=rows, plan=plan)
    wts, head, ids, g = _model(case, seed)
    starts, ends = _spans(_ints(case["lens"]))
    if kind == "prefill":
        return dict(case=case, wts=wts, head=head, ids=ids, starts=starts, ends=ends, keep=_ints(case["keep"]))
    from tokengate_amd.prefill import prefill_batch
    result = prefill_batch(wts, head, ids, starts, ends, 1, _ints(case["keep"]), prune_below_gate=case["prune_below"],
                           decode_headroom=MAX_NEW_TOKENS)
    tokens = torch.randint(0, wts.shape.vocab, (len(ids),), generator=g, device=DEVICE)
    state = dict(case=case, wts=wts, head=head, result=result, tokens=tokens)
    _start_generation(state)
    return state


def _start_generation(state):
    """A generation under way: its first step has run and the graph of the others is captured."""
    from tokengate_amd.decode import DecodeState
    state["decode"] = DecodeState(state["wts"], state["head"], 1, state["result"], MAX_NEW_TOKENS,
                                  prune_below_gate=state["case"]["prune_below"], graph=True)
    for _ in range(2):
        state["decode"].step(state["tokens"])


# ---- one pass ------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("forward", "train"):
        from tokengate_amd.fa2bias.keybias import flash_attn_key_bias
        if kind == "forward":
            with torch.no_grad():
                return flash_attn_key_bias(state["q"], state["k"], state["v"], state["kb"], SCALE, case["causal"])
        out = flash_attn_key_bias(state["q"], state["k"], state["v"], state["kb"], SCALE, case["causal"])
        return [out.detach()] + list(torch.autograd.grad(out, [state[n] for n in ("q", "k", "v", "kb")], state["dout"]))
    if kind == "varlen":
        from tokengate_amd.fa2bias.keybias import flash_attn_key_bias_varlen
        out = flash_attn_key_bias_varlen(state["q"], state["k"], state["v"], state["kb"], state["cu"], state["max"],
                                         SCALE)
        return [out.detach()] + list(torch.autograd.grad(out, [state[n] for n in ("q", "k", "v", "kb")], state["dout"]))
    if kind == "score":
        return state["head"].scores(state["x"])
    if kind == "select":
        from tokengate_amd import gate
        plan = state["plan"]
        n = plan.total_kept
        packed = [torch.empty(n, *t.shape[1:], dtype=t.dtype, device=t.device) for t in state["rows"]]
        positions = torch.empty(n, dtype=torch.int64, device=DEVICE)
        bias = torch.empty(n, dtype=torch.float32, device=DEVICE)
        keep = gate.select_pack(state["scores"], plan, list(zip(state["rows"], packed)), positions=positions,
                                bias_out=bias)
        return [keep, positions, bias] + packed
    if kind == "decode":
        if state["decode"].steps >= MAX_NEW_TOKENS:      # the generation is at its end: the next one begins
            _start_generation(state)
        state["decode"].step(state["tokens"])
        return state["decode"].last_logits
    from tokengate_amd.prefill import prefill_batch
    r = prefill_batch(state["wts"], state["head"], state["ids"], state["starts"], state["ends"], 1, state["keep"])
    return [r.logits] + [t for layer in r.kv[:2] for t in (layer.k, layer.v)]


# ---- what a pass cannot do without ---------------------------------------------------------------

LAYER_WEIGHTS = 2048 * 4096 + 2048 * 2048 + 3 * 2048 * 6144      # q|k|v, o, gate|up, down
VOCAB = 151936


def _pairs(lens, causal=True):
    return sum(n * (n + 1) // 2 if causal else n * n for n in lens)


def work(case):
    kind = case["kind"]
    if kind in ("forward", "train", "varlen"):
        H, Hkv = case["heads"], case["kv_heads"]
        lens = _ints(case["lens"]) if kind == "varlen" else [case["seq"]] * case["batch"]
        rows, pairs = sum(lens), _pairs(lens, case.get("causal", True))
        bias = 4 * H * (rows if kind != "varlen" else len(lens) * max(lens))
        fwd_bytes = 2 * D * rows * (2 * H + 2 * Hkv) + bias
        if kind == "forward":
            return dict(bytes=fwd_bytes, flops=4 * D * H * pairs)
        # read q, k, v, bias, dout; write out, dq, dk, dv, dbias
        return dict(bytes=2 * D * rows * (4 * H + 4 * Hkv) + 2 * bias, flops=14 * D * H * pairs)
    if kind == "score":
        return dict(bytes=2 * D_MODEL * (case["rows"] + 256) + 4 * case["rows"], flops=2 * 256 * D_MODEL * case["rows"])
    lens, keep = _ints(case["lens"]), _ints(case["keep"])
    n_state = [n - 320 for n in lens]
    kept = [320 + max(1, min(k, n)) for k, n in zip(keep, n_state)]
    if kind == "select":
        row = 2 * D_MODEL + case["layers"] * 2 * 2 * 8 * D
        return dict(bytes=4 * sum(n_state) + sum(kept) * (2 * row + 8 + 8 + 4), flops=0)
    if kind == "decode":
        below = kept if case["prune_below"] else lens
        weights = 28 * LAYER_WEIGHTS + VOCAB * D_MODEL
        cache = 2 * sum(below) + 26 * sum(kept)
        return dict(bytes=2 * weights + 2 * 2 * 8 * D * cache + 26 * 16 * 4 * sum(kept) + 4 * VOCAB * len(lens),
                    flops=2 * weights * len(lens) + 4 * D * 16 * cache)
    mlp = 3 * 2048 * 6144
    below_weights = 2 * LAYER_WEIGHTS * sum(lens) + (mlp * sum(kept) - (mlp / 3) * sum(lens) if case["branch"]
                                                     else 256 * D_MODEL * sum(lens))
    flops = 2 * (below_weights + 26 * LAYER_WEIGHTS * sum(kept)) + 4 * D * 16 * (2 * _pairs(lens) + 26 * _pairs(kept))
    flops += 2 * VOCAB * D_MODEL * len(lens)
    return dict(bytes=2 * (28 * LAYER_WEIGHTS + VOCAB * D_MODEL) + 2 * D_MODEL * sum(lens) + 2 * 2 * 2 * 8 * D * sum(lens),
                flops=flops)


# ---- how far another correct implementation may be off -------------------------------------------

def tolerance(case):
    """Measured, then about four times that: another implementation of the same precision against this one."""
    kind = case["kind"]
    if kind in ("forward", "train", "varlen"):
        return {"rel": 1e-2}      # bf16 results with fp32 sums: 2.9e-3 from a torch fp32 softmax with bf16 weights
    if kind == "score":
        return {"rel": 2e-6}      # fp32 sums over 2048 inputs: 3.4e-7 from float64
    if kind == "select":
        return {"rel": 5e-7}      # copies; the bias alone is computed: 0.9e-7 from float64
    # 28 bf16 layers: 3.0e-2 to 4.0e-2 with the norms, the SwiGLU product and the decode projections in torch
    return {"rel": 0.15}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _exact_attention(q, k, v, kb, dout, causal):
    """One sequence in float64: q, dout (S, H, D), k, v (S, Hkv, D), kb (H, S).  Returns out and, with
    dout, dq, dk, dv and dkb."""
    S, H, _ = q.shape
    group = H // k.shape[1]
    q, k, v, kb = (t.detach().double() for t in (q, k, v, kb))
    out = torch.empty_like(q)
    grads = None
    if dout is not None:
        dout = dout.double()
        grads = [torch.zeros_like(t) for t in (q, k, v, kb)]
    step = max(64, min(S, (1 << 27) // S))
    cols = torch.arange(S, device=q.device)
    for h in range(H):
        kh, vh = k[:, h // group], v[:, h // group]
        for r0 in range(0, S, step):
            r1 = min(S, r0 + step)
            n = r1 if causal else S
            z = SCALE * (q[r0:r1, h] @ kh[:n].t()) + kb[h, :n]
            if causal:
                z.masked_fill_(cols[None, :n] > cols[r0:r1, None], float("-inf"))
            p = torch.softmax(z, -1)
            out[r0:r1, h] = p @ vh[:n]
            if dout is None:
                continue
            do = dout[r0:r1, h]
            ds = p * (do @ vh[:n].t() - (do * out[r0:r1, h]).sum(-1, keepdim=True))
            grads[0][r0:r1, h] = SCALE * (ds @ kh[:n])
            grads[1][:n, h // group] += SCALE * (ds.t() @ q[r0:r1, h])
            grads[2][:n, h // group] += p.t() @ do
            grads[3][h, :n] += ds.sum(0)
    return [out] + (grads or [])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train"):
        q, k, v, kb, dout = _attention_inputs(case, _gen(seed))
        parts = [_exact_attention(q[b], k[b], v[b], kb[b], dout[b] if kind == "train" else None, case["causal"])
                 for b in range(case["batch"])]
        whole = [torch.stack(t) for t in zip(*parts)]
        return whole if kind == "train" else whole[0]
    if kind == "varlen":
        q, k, v, kb, dout = _attention_inputs(case, _gen(seed))
        parts, r0 = [], 0
        dkb = torch.zeros(kb.shape, dtype=torch.float64, device=DEVICE)
        for b, n in enumerate(_ints(case["lens"])):
            s = slice(r0, r0 + n)
            parts.append(_exact_attention(q[s], k[s], v[s], kb[b, :, :n], dout[s], True))
            dkb[b, :, :n] = parts[-1].pop()
            r0 += n
        return [torch.cat(t) for t in zip(*parts)] + [dkb]
    if kind == "score":
        head, x = _score_inputs(case, _gen(seed))
        w1, b1, w2 = head.w1.double(), head.b1.double(), head.w2.double()
        return torch.cat([torch.nn.functional.silu(c.double() @ w1.t() + b1) @ w2 + head.b2 for c in x.split(65536)])
    if kind == "select":
        lens, scores, rows = _gate_inputs(case, _gen(seed))
        keep, bias, first, r0 = [], [], [], 0
        for n, k, s, e in zip(lens, _ints(case["keep"]), *_spans(lens)):
            span = scores[r0 + s:r0 + e].double()
            best = torch.argsort(span, descending=True, stable=True)[:max(1, min(k, e - s))].sort().values + s
            at = torch.arange(n, device=DEVICE)
            keep.append(torch.cat([at[:s], best, at[e:]]))
            b = torch.zeros(keep[-1].numel(), dtype=torch.float64, device=DEVICE)
            b[s:s + best.numel()] = span[best - s] / torch.sqrt((span * span).mean() + 1e-6)
            bias.append(b)
            first.append(keep[-1] + r0)
            r0 += n
        keep, first = torch.cat(keep), torch.cat(first)
        return [keep, keep, torch.cat(bias)] + [t.index_select(0, first) for t in rows]
    return None      # a whole model in 64 bits takes too long
