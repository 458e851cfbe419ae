"""tg_decode_attention (q/k norm, RoPE, cache append and attention of a decode step in one launch): the
appended rows equal tg_qk_norm_rope's bit for bit, and the output is bit for bit that of tg_qk_norm_rope
followed by tg_keybias_varlen_kv_fwd, whose tile arithmetic and merge order it keeps.  Against the float64
attention over the cache: the weights and the chunks' partial results are rounded to bf16 (2^-9 of
sum p |v| each), then the output (2^-9 of it); 2e-5 for the fp32 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(dev, used, gap, H, Hkv, seed, bias, scaled):
    from tokengate_amd import decoder as dec
    g = torch.Generator(device=dev).manual_seed(seed)
    B, D = len(used), 128
    shape = dec.DecoderShape(n_layers=1, n_heads=H, n_kv_heads=Hkv, d_model=H * D)
    bf = lambda *s, std=1.0, mean=0.0: (mean + std * torch.randn(*s, generator=g, device=dev)).to(torch.bfloat16)
    lw = dec.LayerWeights(None, None, bf(D, std=0.3, mean=1.0), bf(D, std=0.3, mean=1.0), None, None, None, None)
    start, r = [], 3
    for n in used:
        start.append(r)
        r += n + gap
    k, v = bf(r, Hkv, D), bf(r, Hkv, D)
    qkv = bf(B, (H + 2 * Hkv) * D)
    pos = torch.tensor([n + 7 for n in used], device=dev)
    max_k = max(used) + gap
    bias = 3 * torch.randn(B, H, max_k + 5, generator=g, device=dev) if bias else None
    qs = 0.5 + torch.rand(H, generator=g, device=dev) if scaled else None
    rs = torch.rand(B, generator=g, device=dev) if scaled else None
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    return shape, lw, qkv, pos, dec.rope_inv_freq(shape, dev), k, v, i32(start), i32(used), max_k, bias, qs, rs


def _check(c, out, k, v):
    from tokengate_amd import decoder as dec
    shape, lw, qkv, pos, inv, k0, v0, start, used, max_k, bias, qs, rs = c
    k1, v1 = k0.clone(), v0.clone()
    q = dec.qk_norm_rope(qkv.clone(), pos, lw, shape, inv, k1, v1, qs, rs, kv_rows=start + used - 1)
    assert torch.equal(k, k1) and torch.equal(v, v1), "appended cache rows"
    group = shape.n_heads // shape.n_kv_heads
    for b in range(q.shape[0]):
        s, n = int(start[b]), int(used[b])
        kk, vv = (t[s:s + n].double().repeat_interleave(group, 1) for t in (k1, v1))
        z = (q[b].double()[:, None] * kk.transpose(0, 1)).sum(-1)
        if bias is not None:
            z = z + bias[b, :, :n].double()
        p = torch.softmax(z * 128 ** -0.5, -1)[..., None]
        ref, mass = (p * vv.transpose(0, 1)).sum(1), (p * vv.abs().transpose(0, 1)).sum(1)
        err = (out[b].double() - ref).abs()
        assert bool((err <= 2.0 ** -8 * mass + 2.0 ** -9 * ref.abs() + 2e-5).all()), (b, float(err.max()))
    cu = torch.arange(q.shape[0] + 1, dtype=torch.int32, device=q.device)
    two = dec.varlen_kv_attention(q, k1, v1, cu, start, used, 1, max_k, 128 ** -0.5, bias)
    assert torch.equal(out, two), "the two launches' output"


@pytest.mark.parametrize("used,gap,H,Hkv,bias,scaled", [
    ([1], 0, 16, 8, True, False),                       # the new key alone
    ([2, 1, 3], 900, 16, 8, True, True),                # more chunks than keys: empty chunks
    ([65], 0, 16, 8, False, False), ([129, 128, 127], 1, 16, 8, True, False),
    ([2321], 1023, 16, 8, True, True), ([32769], 7, 16, 8, False, False),
    ([700, 5000, 33, 1600, 64, 63, 2, 9000], 5, 16, 8, True, True),
    ([1300, 40], 3, 5, 5, True, False), ([900], 0, 16, 2, True, True), ([450] * 40, 2, 12, 4, True, False)])
def test_decode_attention(cuda, used, gap, H, Hkv, bias, scaled):
    from tokengate_amd import decoder as dec
    c = _case(cuda, used, gap, H, Hkv, 11 + sum(used), bias, scaled)
    shape, lw, qkv, pos, inv, k0, v0, start, n, max_k, kb, qs, rs = c
    rope, _ = dec.decode_begin(pos.clone(), inv)
    ws = dec.decode_attention_workspace(len(used), shape, max_k, cuda)
    outs = []
    for _ in range(3):                                  # the workspace's counters are zero again after each
        k, v = k0.clone(), v0.clone()
        outs.append(dec.decode_attention(qkv, rope, lw, shape, k, v, start, n, max_k, 128 ** -0.5, ws, kb, qs, rs))
    torch.cuda.synchronize()
    _check(c, outs[0], k, v)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_decode_attention_shared_workspace(cuda):
    """Launches of different batch sizes, head counts and key counts share one workspace: the counters stay
    apart from every launch's partials and are zero again after each."""
    from tokengate_amd import decoder as dec
    sizes = [([3000] * 4, 16, 8), ([2500] * 12, 16, 8), ([900] * 40, 12, 4), ([20000], 16, 8), ([700] * 30, 16, 8)]
    cases = [_case(cuda, used, 3, H, Hkv, 40 + len(used), True, False) for used, H, Hkv in sizes]
    ws = max((dec.decode_attention_workspace(len(c[7]), c[0], c[9], cuda) for c in cases), key=lambda t: t.numel())
    for i in (0, 1, 2, 0, 4, 3, 1, 2, 4):
        shape, lw, qkv, pos, inv, k0, v0, start, n, max_k, kb, qs, rs = cases[i]
        rope, _ = dec.decode_begin(pos.clone(), inv)
        k, v = k0.clone(), v0.clone()
        out = torch.full((len(n), shape.n_heads, 128), float("nan"), dtype=torch.bfloat16, device=cuda)
        dec.decode_attention(qkv, rope, lw, shape, k, v, start, n, max_k, 128 ** -0.5, ws, kb, out=out)
        torch.cuda.synchronize()
        _check(cases[i], out, k, v)


def test_decode_attention_masked_keys(cuda):
    """Bias of -inf hides a key; a head that sees no key at all gets zeros."""
    from tokengate_amd import decoder as dec
    c = _case(cuda, [300, 40], 2000, 16, 8, 5, True, False)
    shape, lw, qkv, pos, inv, k0, v0, start, n, max_k, kb, qs, rs = c
    rope, _ = dec.decode_begin(pos.clone(), inv)
    kb[:, 3] = -float("inf")
    kb[:, 3, 17] = 0.5
    kb[1, 6] = -float("inf")
    k, v = k0.clone(), v0.clone()
    ws = dec.decode_attention_workspace(2, shape, max_k, cuda)
    out = dec.decode_attention(qkv, rope, lw, shape, k, v, start, n, max_k, 128 ** -0.5, ws, kb)
    torch.cuda.synchronize()
    for b in range(2):
        assert torch.equal(out[b, 3], v0[int(start[b]) + 17, 1])
    assert bool((out[1, 6] == 0).all())
    kb[1, 6] = 0.0
    out[1, 6] = dec.decode_attention(qkv, rope, lw, shape, k, v, start, n, max_k, 128 ** -0.5, ws, kb)[1, 6]
    _check(c, out, k, v)


def test_decode_attention_rejects(cuda):
    from tokengate_amd import decoder as dec
    shape, lw, qkv, pos, inv, k, v, start, n, max_k, kb, qs, rs = _case(cuda, [500], 0, 16, 8, 1, True, False)
    rope, _ = dec.decode_begin(pos.clone(), inv)
    ws = dec.decode_attention_workspace(1, shape, max_k, cuda)
    with pytest.raises(RuntimeError, match="workspace"):
        dec.decode_attention(qkv, rope, lw, shape, k, v, start, n, max_k, 0.1, ws[:16], kb)
    with pytest.raises(RuntimeError, match="key axis"):
        dec.decode_attention(qkv, rope, lw, shape, k, v, start, n, max_k, 0.1, ws, kb[..., :max_k - 1])
    with pytest.raises(RuntimeError, match="int32"):
        dec.decode_attention(qkv, rope, lw, shape, k, v, start.long(), n, max_k, 0.1, ws, kb)


def test_decode_begin(cuda):
    """The step's rotary table, counters and scaled-softmax ratio against float64."""
    from tokengate_amd import decoder as dec
    pos = torch.tensor([0, 1, 131071, 5000, 2], device=cuda)
    p0 = pos.clone()
    inv = dec.rope_inv_freq(dec.DecoderShape(), cuda)
    used = torch.arange(10, dtype=torch.int32, device=cuda).view(2, 5).contiguous()
    slots = torch.tensor([0.0, 5.0, 2000.0, 4999.0, 1.0], device=cuda)
    rope, ratio = dec.decode_begin(pos, inv, used, slots)
    torch.cuda.synchronize()
    ang = (p0.float()[:, None] * inv).double()             # the table's angles are fp32 products
    ref = torch.stack([ang.cos(), ang.sin()], -1)
    assert float((rope.double() - ref).abs().max()) <= 2.0 ** -22
    assert torch.equal(pos, p0 + 1) and torch.equal(used.flatten().cpu(), torch.arange(10, dtype=torch.int32) + 1)
    assert slots.tolist() == [1.0, 6.0, 2001.0, 5000.0, 2.0]
    r = (slots.double().clamp(min=2).log() / (p0.double() + 1).clamp(min=2).log()).clamp(max=1)
    assert float((ratio.double() - r).abs().max()) <= 1e-6
    assert dec.decode_begin(pos, inv)[1] is None
