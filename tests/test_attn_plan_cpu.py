"""The form that a dense forward takes (tg_keybias_fwd_plan; without a device the plan is that of 256 compute
units): waves per workgroup, key groups, chunks of a split tile.  The shapes are those where the choice was
wrong or is close; the comments give the times in us that speak for it."""
import pytest

from tokengate_amd import _lib


@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,causal,form", [
    # the forms without key groups: other choices were slower
    (1, 3000, 32768, 16, 8, True, (4, 1, 2)),     # 760; unsplit 827
    (1, 3072, 4096, 16, 8, False, (4, 1, 2)),     # 108; unsplit 116
    (1, 3072, 3072, 16, 8, False, (4, 1, 2)),     # 87; unsplit 93
    (8, 1024, 1024, 16, 8, True, (8, 1, 1)),      # 46; four waves 49
    (16, 512, 512, 16, 8, True, (8, 1, 1)),       # 36; four waves 37.4
    (3, 1700, 1700, 12, 4, True, (4, 1, 1)),      # 42; two key groups 44.5
    (16, 225, 225, 8, 2, True, (4, 1, 1)),        # two key groups 1.15 times
    (1, 3510, 5394, 4, 4, True, (4, 1, 4)),       # 43; eight waves 48
    (1, 6000, 6000, 16, 8, True, (4, 1, 1)),      # 145; two key groups 162
    (1, 8192, 8192, 16, 8, True, (8, 1, 1)), (1, 32768, 32768, 16, 8, True, (8, 1, 1)),
    # eight against four waves in two rounds and over
    (16, 1074, 1074, 8, 8, True, (4, 1, 1)),      # 56; eight waves 64
    (16, 626, 626, 12, 4, True, (4, 1, 1)),       # 38; 47
    (4, 3944, 3944, 12, 4, True, (4, 1, 1)),      # 0.89 times
    (64, 287, 446, 12, 4, True, (4, 1, 1)),       # 76; 95
    (64, 112, 112, 8, 8, False, (4, 1, 1)),       # 17; 19
    (1, 8040, 8040, 16, 8, True, (8, 1, 1)),      # 231; four waves 258
    # key groups
    (1, 1024, 1024, 16, 8, True, (8, 4, 1)),      # 18; four waves, split 24
    (1, 2048, 2048, 16, 8, True, (8, 4, 1)),      # 34; 42
    (1, 4096, 4096, 16, 8, True, (8, 2, 1)),      # 76; unsplit 91
    (1, 2320, 2320, 12, 4, True, (8, 4, 1)),      # 35; 41
])
def test_form(B, Sq, Sk, H, Hkv, causal, form):
    assert _lib.fwd_plan(B, Sq, Sk, H, Hkv, causal, 1 << 40)[:3] == form


def split_bytes(s):
    """Fewest workspace bytes with which a launch that splits does (found by bisection), else 0."""
    full, lo, hi = _lib.fwd_plan(*s, 1 << 40), 0, 1 << 30
    if full[2] == 1:
        return 0
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if _lib.fwd_plan(*s, mid) == full else (mid, hi)
    return hi


def test_a_launch_splits_as_planned_or_not_at_all():
    """tg_keybias_fwd_workspace_size holds the split of the launch's plan, and with fewer bytes than that split
    needs the launch is the one without a workspace, never the split of another form."""
    size = _lib.load().tg_keybias_fwd_workspace_size
    split = set()
    for Sq in (1, 3, 64, 200, 700, 1024, 1500, 2320, 3000, 4096):
        for Sk in (Sq, 3000, 9000, 32768, 131072):
            for H, Hkv in ((16, 8), (8, 8), (6, 2), (1, 1)):
                for causal in (True, False):
                    s = (1, Sq, Sk, H, Hkv, causal)
                    n, full, none = size(*s[:5], int(causal)), _lib.fwd_plan(*s, 1 << 40), _lib.fwd_plan(*s, 0)
                    need = split_bytes(s)
                    assert n >= need and none[2] == 1 and _lib.fwd_plan(*s, n) == full, s
                    if need > 0:
                        split.add(full[:2])
                        for w in (need - 1, need // 2, 16):
                            assert _lib.fwd_plan(*s, w) == none, (s, w)
    assert split == {(4, 1), (8, 1), (8, 2), (8, 4)}       # every form has launches that split


def test_plan_rejects_bad_sizes():
    for a in ((0, 8, 8, 2, 1, 1, 0), (1, 0, 8, 2, 1, 1, 0), (1, 8, -1, 2, 1, 1, 0), (1, 8, 8, 3, 2, 1, 0), (1, 8, 8, 2, 1, 1, -1)):
        with pytest.raises(RuntimeError, match="bad sizes"):
            _lib.fwd_plan(*a)
