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
