"""gate._row_elems (the pack's row check by shape and stride) against what the view t[0] says, over
shapes, permutations, slices and expanded axes."""
import itertools

import torch

from tokengate_amd.gate import _row_elems


def test_row_elems_matches_the_view():
    n = 0
    for shape in [(3,), (1,), (4, 8), (4, 1), (4, 0), (2, 3, 8), (2, 1, 8), (2, 3, 1), (3, 2, 4, 8), (2, 1, 1, 5)]:
        base = torch.zeros(*(max(1, 2 * s) for s in shape))
        for perm in itertools.permutations(range(len(shape))):
            for cut in itertools.product((1, 2), repeat=len(shape)):
                t = base.permute(perm)[tuple(slice(0, shape[d] * c, c) for d, c in enumerate(cut))]
                for u in (t, t.contiguous(), t[:1].expand(2, *t.shape[1:])):
                    if u.shape[0] == 0:
                        continue
                    want = u[0].numel() if u[0].is_contiguous() else -1
                    assert _row_elems(u.shape, u.stride()) == want, (u.shape, u.stride())
                    n += 1
    assert n > 1000
