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
    (1, 6000, 6000, 16, 8, True, (4, 1, 1)),      # 145; two key groups 162
    (1, 8192, 8192, 16, 8, True, (8, 1, 1)), (1, 32768, 32768, 16, 8, True, (8, 1, 1)),
    # key groups
    (1, 1024, 1024, 16, 8, True, (8, 4, 1)),      # 18; four waves, split 24
    (1, 2048, 2048, 16, 8, True, (8, 4, 1)),      # 34; 42
    (1, 4096, 4096, 16, 8, True, (8, 2, 1)),      # 76; unsplit 91
    (1, 2320, 2320, 12, 4, True, (8, 4, 1)),      # 35; 41
])
def test_form(B, Sq, Sk, H, Hkv, causal, form):
    assert _lib.fwd_plan(B, Sq, Sk, H, Hkv, causal, 1 << 40)[:3] == form


def test_workspace_is_what_the_plan_needs():
    """tg_keybias_fwd_workspace_size is 0 exactly where the launch does not split, and with any fewer bytes the
    launch is the one without a workspace."""
    size = _lib.load().tg_keybias_fwd_workspace_size
    split = set()
    for Sq in (1, 3, 64, 200, 700, 1024, 1500, 2320, 3000, 4096):
        for Sk in (Sq, 3000, 9000, 32768, 131072):
            for H, Hkv in ((16, 8), (8, 8), (6, 2), (1, 1)):
                for causal in (True, False):
                    s = (1, Sq, Sk, H, Hkv, causal)
                    n, full, none = size(*s[:5], int(causal)), _lib.fwd_plan(*s, 1 << 40), _lib.fwd_plan(*s, 0)
                    assert (n > 0) == (full[2] > 1) and none[2] == 1, s
                    assert _lib.fwd_plan(*s, n) == full
                    if n > 0:
                        split.add(full[:2])
                        assert _lib.fwd_plan(*s, n - 1) == _lib.fwd_plan(*s, 16) == none
    assert split == {(4, 1), (8, 1), (8, 2), (8, 4)}       # every form has launches that split


def test_plan_rejects_bad_sizes():
    for a in ((0, 8, 8, 2, 1, 1, 0), (1, 0, 8, 2, 1, 1, 0), (1, 8, -1, 2, 1, 1, 0), (1, 8, 8, 3, 2, 1, 0), (1, 8, 8, 2, 1, 1, -1)):
        with pytest.raises(RuntimeError, match="bad sizes"):
            _lib.fwd_plan(*a)
