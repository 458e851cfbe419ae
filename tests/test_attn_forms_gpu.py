"""GPU parity of the dense attention at the sizes where its launch forms can go wrong: the forward's
key groups (two or four groups of waves that share a workgroup's keys and merge through LDS) at
the edges of their 128-key steps and 32 / 64-row tiles, odd GQA groups, rows that see no key, key
groups that see no key, and masked keys at the lowest float, against a float64 evaluation on the
device.  Tolerance: max-abs 2e-2 and rel-L2 1e-2 (tests/attn_util), bf16 outputs of unit-variance V.
"""
import pytest
import torch

from tests.attn_util import assert_close, to_np

pytestmark = pytest.mark.gpu


def _reference(q, k, v, bias_raw, scale, causal):
    """out, lse of every row in float64 (a row without a key: out 0, lse +inf)."""
    B, Sq, H, D = q.shape
    Sk, g = k.shape[1], H // k.shape[2]
    out = torch.empty(B, Sq, H, D, dtype=torch.float64, device=q.device)
    lse = torch.empty(B, H, Sq, dtype=torch.float64, device=q.device)
    hidden = torch.arange(Sk, device=q.device)[None, :] > torch.arange(Sq, device=q.device)[:, None] + Sk - Sq
    for b in range(B):
        for h in range(H):
            z = q[b, :, h].double() @ k[b, :, h // g].double().t()
            if bias_raw is not None:
                z = z + bias_raw[b, h].double()
            z = z * scale
            if causal:
                z = z.masked_fill(hidden, float("-inf"))
            m = z.amax(-1, keepdim=True).clamp(min=-1e300)
            p = torch.exp(z - m)
            s = p.sum(-1, keepdim=True)
            out[b, :, h] = torch.where(s > 0, p / s, 0.0) @ v[b, :, h // g].double()
            lse[b, h] = torch.where(s > 0, m + torch.log(s), float("inf"))[:, 0]
    return out, lse


SHAPES = [
    # B, Sq, Sk, H, Hkv, causal, bias
    (1, 1, 1, 16, 8, True, True), (1, 31, 31, 16, 8, True, True), (1, 33, 33, 16, 8, True, False),
    (1, 127, 127, 16, 8, True, True), (1, 129, 129, 16, 8, True, True), (2, 517, 517, 16, 8, True, True),
    (1, 161, 417, 16, 8, True, True), (1, 300, 140, 16, 8, True, True), (1, 257, 129, 16, 8, False, True),
    (1, 777, 777, 16, 8, False, True), (1, 1025, 1025, 16, 8, True, True), (1, 1000, 1000, 3, 1, True, True),
    (3, 999, 999, 4, 4, True, False), (1, 2049, 2049, 16, 8, True, True), (1, 2320, 2320, 12, 4, True, True),
    (1, 2320, 2320, 16, 8, True, True), (2, 1500, 1500, 6, 2, True, True), (1, 2048, 2048, 16, 8, False, True),
    (1, 3071, 3071, 16, 8, True, True), (1, 4097, 4097, 16, 8, True, False), (1, 4096, 4096, 8, 8, True, True),
]


@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,causal,has_bias", SHAPES, ids=[f"{s[1]}x{s[2]}h{s[3]}b{s[0]}" for s in SHAPES])
def test_forward_forms(cuda, B, Sq, Sk, H, Hkv, causal, has_bias):
    from tokengate_amd.fa2bias.keybias import ext
    g = torch.Generator(device=cuda).manual_seed(Sq + 3 * Sk + H)
    q, k, v = (torch.randn(B, s, h, 128, generator=g, device=cuda).to(torch.bfloat16)
               for s, h in ((Sq, H), (Sk, Hkv), (Sk, Hkv)))
    scale = 128 ** -0.5
    bias_raw = None
    if has_bias:
        bias_raw = torch.randn(B, H, Sk, generator=g, device=cuda) * 2.0 / scale
        bias_raw[:, :, 5:Sk:7] = torch.finfo(torch.float32).min      # masked keys; key 0 stays visible
        if Sk > 200:
            bias_raw[:, ::2, 128:192] = float("-inf")                # whole keys of one group and step
    out, lse, _, _ = ext().fwd(q, k, v, None, bias_raw, 0.0, scale, causal, -1, -1, 0.0, False, None)
    ro, rl = _reference(q, k, v, bias_raw, scale, causal)
    seen = torch.isfinite(rl)
    assert torch.equal(torch.isfinite(lse), seen)
    assert_close("out", to_np(out), ro.cpu().numpy())
    assert_close("lse", to_np(lse[seen]), rl[seen].cpu().numpy())


def _grads(q, k, v, bias, dout, scale, causal=True):
    """Gradients of one sequence in float64: dq, dk, dv, dbias_raw (None without a bias)."""
    (n, H, _), m = q.shape, k.shape[0]
    g = H // k.shape[1]
    q, k, v, dout = (t.double() for t in (q, k, v, dout))
    dq, dk, dv = (torch.zeros_like(t) for t in (q, k, v))
    db = None if bias is None else torch.zeros_like(bias, dtype=torch.float64)
    hidden = torch.ones(n, m, dtype=torch.bool, device=q.device).triu(1 + m - n)
    for h in range(H):
        kh, vh = k[:, h // g], v[:, h // g]
        z = q[:, h] @ kh.t() * scale
        if bias is not None:
            z = z + bias[h].double() * scale
        p = torch.softmax(z.masked_fill(hidden, float("-inf")) if causal else z, -1)
        dp = dout[:, h] @ vh.t()
        ds = p * (dp - (p * dp).sum(-1, keepdim=True))
        dq[:, h] = scale * (ds @ kh)
        dk[:, h // g] += scale * (ds.t() @ q[:, h])
        dv[:, h // g] += p.t() @ dout[:, h]
        if bias is not None:
            db[h] = scale * ds.sum(0)
    return dq, dk, dv, db


BWD_SHAPES = [
    # B, Sq, Sk, H, Hkv, causal, bias
    (1, 1, 1, 16, 8, True, True), (1, 31, 31, 16, 8, True, True), (1, 33, 33, 2, 2, True, False),
    (1, 129, 129, 16, 8, True, True), (2, 517, 517, 16, 8, True, True), (1, 161, 417, 16, 8, True, True),
    (1, 300, 140, 6, 2, False, True), (1, 777, 777, 8, 8, False, False), (1, 1025, 1025, 6, 2, True, True),
    (1, 2049, 2049, 8, 2, True, True), (3, 1000, 1000, 4, 4, True, True), (1, 3073, 3073, 16, 8, True, True),
]


@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,causal,has_bias", BWD_SHAPES,
                         ids=[f"{s[1]}x{s[2]}h{s[3]}b{s[0]}" for s in BWD_SHAPES])
def test_backward_forms(cuda, B, Sq, Sk, H, Hkv, causal, has_bias):
    """The backward's groups (two or four per workgroup, summed through LDS) and its own D = rowsum(dO * O),
    into buffers full of NaN, twice with the same bits."""
    from tests.attn_util import assert_close_grad
    from tokengate_amd.fa2bias.keybias import ext
    g = torch.Generator(device=cuda).manual_seed(Sq + 3 * Sk + H)
    q, k, v, dout = (torch.randn(B, s, h, 128, generator=g, device=cuda).to(torch.bfloat16)
                     for s, h in ((Sq, H), (Sk, Hkv), (Sk, Hkv), (Sq, H)))
    scale = 128 ** -0.5
    bias = torch.randn(B, H, Sk, generator=g, device=cuda) / scale if has_bias else None
    out, lse, _, _ = ext().fwd(q, k, v, None, bias, 0.0, scale, causal, -1, -1, 0.0, False, None)
    got = []
    for _ in range(2):
        bufs = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        got.append(ext().bwd(dout, q, k, v, out, lse, *bufs, bias, 0.0, scale, causal, -1, -1, 0.0, False, None, None))
    for x, y in zip(*got):
        assert x is None or torch.equal(x, y)
    dq, dk, dv, sd, db = got[0]
    d_ref = (dout.double() * out.double()).sum(-1).transpose(1, 2)
    assert float((sd - d_ref).abs().max()) <= 1e-4      # 128 products of bf16 values summed in fp32
    for b in range(B):
        ref = _grads(q[b], k[b], v[b], None if bias is None else bias[b], dout[b], scale, causal)
        for what, x, r in zip(("dq", "dk", "dv", "db"), (dq[b], dk[b], dv[b], None if db is None else db[b]), ref):
            if r is not None:
                assert_close_grad(f"{what} {b}", to_np(x), r.cpu().numpy())


@pytest.mark.parametrize("n,H,Hkv", [(1, 16, 8), (33, 2, 2), (517, 16, 8), (2049, 6, 2), (4096, 16, 8)])
def test_backward_row_sums_keep_their_order(cuda, n, H, Hkv):
    """A dense backward forms D = rowsum(dO * O) inside the dQ kernel, a packed one in a launch of its own:
    the same products added in the same order, so the same bits."""
    from tokengate_amd.fa2bias.keybias import ext
    g = torch.Generator(device=cuda).manual_seed(n + H)
    q, k, v, dout = (torch.randn(1, n, h, 128, generator=g, device=cuda).to(torch.bfloat16) for h in (H, Hkv, Hkv, H))
    out, lse, _, _ = ext().fwd(q, k, v, None, None, 0.0, 0.1, True, -1, -1, 0.0, False, None)
    dense = ext().bwd(dout, q, k, v, out, lse, None, None, None, None, 0.0, 0.1, True, -1, -1, 0.0, False, None, None)[3]
    cu = torch.tensor([0, n], dtype=torch.int32, device=cuda)
    packed = ext().varlen_bwd(dout[0], q[0], k[0], v[0], out[0], lse[0].contiguous(), None, None, None, cu, cu, None, n, n,
                              0.0, 0.1, False, True, -1, -1, 0.0, False, None, None)[3]
    assert torch.equal(dense[0], packed)


RAGGED = {
    "nine": [0, 1, 63, 64, 65, 300, 0, 129, 700],
    "equal": [512, 512, 512],
    "sixty_four": [17 * (i % 7) for i in range(64)],
    "long": [4500, 0, 333, 2100],                 # more than 64 levels of 32 and of 64 rows
    "sixty_five": [40 + (i % 3) for i in range(65)],
}


@pytest.mark.parametrize("name", list(RAGGED))
@pytest.mark.parametrize("H,Hkv", [(4, 2), (3, 3)])
def test_varlen_tile_order(cuda, name, H, Hkv):
    """Packed sequences through the varlen launches' level order (up to 64 sequences; 65 take the
    sequence-major order), with empty sequences and a max_seqlen longer than any."""
    from tests.attn_util import assert_close_grad
    from tokengate_amd.fa2bias.keybias import ext
    lens = RAGGED[name]
    total, mx, scale = sum(lens), max(lens) + 75, 128 ** -0.5
    g = torch.Generator(device=cuda).manual_seed(total + H)
    q, k, v, dout = (torch.randn(total, h, 128, generator=g, device=cuda).to(torch.bfloat16) for h in (H, Hkv, Hkv, H))
    bias = (torch.randn(len(lens), H, mx, generator=g, device=cuda) / scale).contiguous()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=cuda)
    out, lse, _, _ = ext().varlen_fwd(q, k, v, None, cu, cu, None, None, None, bias, mx, mx, 0.0, scale, False, True,
                                      -1, -1, 0.0, False, None)
    dq, dk, dv, _, db = ext().varlen_bwd(dout, q, k, v, out, lse, None, None, None, cu, cu, bias, mx, mx, 0.0, scale,
                                         False, True, -1, -1, 0.0, False, None, None)
    r0 = 0
    for b, n in enumerate(lens):
        s = slice(r0, r0 + n)
        r0 += n
        assert not db[b, :, n:].any()
        if n == 0:
            continue
        ro, rl = _reference(q[None, s], k[None, s], v[None, s], bias[None, b, :, :n], scale, True)
        assert_close(f"out {b}", to_np(out[s]), ro[0].cpu().numpy())
        assert_close(f"lse {b}", to_np(lse[:, s]), rl[0].cpu().numpy())
        for what, got, ref in zip(("dq", "dk", "dv", "db"), (dq[s], dk[s], dv[s], db[b, :, :n]),
                                  _grads(q[s], k[s], v[s], bias[b, :, :n], dout[s], scale)):
            assert_close_grad(f"{what} {b}", to_np(got), ref.cpu().numpy())


def test_varlen_backward_with_a_far_larger_max_seqlen(cuda):
    """max_seqlen may be any bound on the lengths: the gradients are those of the exact one, and the host does
    not walk over tiles that cannot exist (half a million of them per estimate)."""
    import time
    from tokengate_amd.fa2bias.keybias import ext
    lens = [300, 77, 1200]
    g = torch.Generator(device=cuda).manual_seed(6)
    q, k, v, dout = (torch.randn(sum(lens), h, 128, generator=g, device=cuda).to(torch.bfloat16) for h in (4, 2, 2, 4))
    cu = torch.tensor([0, 300, 377, 1577], dtype=torch.int32, device=cuda)
    out, lse, _, _ = ext().varlen_fwd(q, k, v, None, cu, cu, None, None, None, None, 1200, 1200, 0.0, 0.1, False, True,
                                      -1, -1, 0.0, False, None)
    got, host = [], []
    for mx in (1200, 1 << 24):
        t = time.perf_counter()
        got.append(ext().varlen_bwd(dout, q, k, v, out, lse, None, None, None, cu, cu, None, mx, mx, 0.0, 0.1, False, True,
                                    -1, -1, 0.0, False, None, None)[:3])
        host.append(time.perf_counter() - t)
    torch.cuda.synchronize()
    for x, y in zip(*got):
        assert torch.equal(x, y)
    assert host[1] < 0.1


def _best(f):
    """Time of f in us, best of ten replays of five launches each."""
    graph = torch.cuda.CUDAGraph()
    f()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        for _ in range(5):
            f()
    t = 1e9
    for _ in range(10):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        graph.replay()
        b.record()
        b.synchronize()
        t = min(t, a.elapsed_time(b) * 200)
    return t


def _times(lens, heads, causal, device, heads_k=None):
    """Times of a packed forward and backward in us."""
    from tokengate_amd.fa2bias.keybias import ext
    g = torch.Generator(device=device).manual_seed(sum(lens))
    q, k, v, dout = (torch.randn(sum(lens), h, 128, generator=g, device=device).to(torch.bfloat16)
                     for h in (heads, heads_k or heads, heads_k or heads, heads))
    cu, mx = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=device), max(lens)
    fw = lambda: ext().varlen_fwd(q, k, v, None, cu, cu, None, None, None, None, mx, mx, 0.0, 0.1, False, causal,
                                  -1, -1, 0.0, False, None)
    out, lse, _, _ = fw()
    bw = lambda: ext().varlen_bwd(dout, q, k, v, out, lse, None, None, None, cu, cu, None, mx, mx, 0.0, 0.1, False,
                                  causal, -1, -1, 0.0, False, None, None)
    return [_best(fw), _best(bw)]


@pytest.mark.parametrize("rows", [100, 500])
def test_varlen_tile_order_costs_little(cuda, rows):
    """64 short sequences, which run in level order, take little longer than 65, which run sequence after
    sequence (finding a workgroup's tile by walking over the sequences made the backward 2.6 times and the
    forward 1.5 times as slow)."""
    level, major = _times([rows] * 64, 8, True, cuda), _times([rows] * 65, 8, True, cuda)
    print(f"64 / 65 sequences of {rows}: forward {level[0]:.1f} / {major[0]:.1f} us, backward {level[1]:.1f} / {major[1]:.1f}")
    assert level[0] < 1.3 * major[0] and level[1] < 1.3 * major[1]


def test_varlen_non_causal_runs_sequence_after_sequence(cuda):
    """Without the causal mask the level order gains nothing and interleaves the sequences' K/V, so 64
    sequences take the time of 65, which never ran in level order (there 64 took 1.35 times as long)."""
    short, major = _times([6000, 4000] + [64] * 62, 8, False, cuda), _times([6000, 4000] + [64] * 63, 8, False, cuda)
    print(f"non-causal, 64 / 65 sequences: forward {short[0]:.1f} / {major[0]:.1f} us, backward {short[1]:.1f} / {major[1]:.1f}")
    assert short[0] < 1.1 * major[0] and short[1] < 1.1 * major[1]


def test_varlen_forward_level_order_only_where_it_balances(cuda):
    """Where every query tile has a CU of its own the forward runs sequence after sequence, so the causal
    mask makes no such batch slower (level order, which only causal launches take: 1.15 times).  So do sequences
    of one length with up to three tiles: 64 take the time of 65, which never run in level order (1.1 times).
    Where two tiles share a CU, uneven sequences do run in level order (17.8 us without, 14.1 with)."""
    lens = list(range(21, 81, 4)) + [80]
    causal, full = _times(lens, 16, True, cuda, 8)[0], _times(lens, 16, False, cuda, 8)[0]
    few, major = _times([354] * 64, 16, True, cuda, 8)[0], _times([354] * 65, 16, True, cuda, 8)[0]
    print(f"own CUs, causal / full: {causal:.1f} / {full:.1f} us, 64 / 65 sequences: {few:.1f} / {major:.1f} us")
    assert causal < 1.02 * full and few < 1.08 * major
    lens = [115, 42, 175, 106, 191, 119, 149, 83, 65, 83, 141, 91, 42, 160, 96, 21, 94, 166, 200, 99]
    causal, full = (_times(lens, 16, c, cuda, 8)[0] for c in (True, False))
    print(f"two to a CU, causal / full: {causal:.1f} / {full:.1f} us")
    assert causal < 0.8 * full


def test_varlen_short_rows_keep_one_group(cuda):
    """The backward of short packed sequences takes one group per workgroup, as 65 sequences always do: the
    estimate behind the choice counted a part of a tile as none, and so took four (1.3 to 1.8 times the time)."""
    few, major = _times([91] + [40] * 61, 8, True, cuda), _times([91] + [40] * 64, 8, True, cuda)
    print(f"62 / 65 short sequences: backward {few[1]:.1f} / {major[1]:.1f} us")
    assert few[1] < 1.12 * major[1]


@pytest.mark.parametrize("rows", [16, 32, 48])
def test_few_rows_keep_one_group(cuda, rows):
    """The dense backward of up to 64 rows takes one group, as the packed one does, and so is faster than that by
    the packed one's third launch (four groups, three of them idle, took as long as the packed one)."""
    from tokengate_amd.fa2bias.keybias import ext
    g = torch.Generator(device=cuda).manual_seed(rows)
    q, k, v, dout = (torch.randn(1, rows, h, 128, generator=g, device=cuda).to(torch.bfloat16) for h in (16, 8, 8, 16))
    out, lse, _, _ = ext().fwd(q, k, v, None, None, 0.0, 0.1, True, -1, -1, 0.0, False, None)
    dense = _best(lambda: ext().bwd(dout, q, k, v, out, lse, None, None, None, None, 0.0, 0.1, True, -1, -1, 0.0, False,
                                    None, None))
    packed = _times([rows], 16, True, cuda, 8)[1]
    print(f"{rows} rows: backward dense {dense:.1f}, packed {packed:.1f} us")
    assert dense < 0.96 * packed


def test_packed_non_causal_backward_takes_groups(cuda):
    """Groups are chosen by the batch's size and lengths, not by the order of its tiles: a small batch with one
    long sequence takes them without the mask as well, and so runs faster than 65 sequences, which never do
    (with one group it took as long as they)."""
    lens = [1227] + [44] * 5
    few, many = (_times(x, 32, False, cuda, 8)[1] for x in (lens, lens + [1] * 59))
    print(f"non-causal, 6 / 65 sequences: backward {few:.1f} / {many:.1f} us")
    assert few < 0.85 * many
