"""Which form of the gradient tiles by pairs the GPU tests' shapes take, read from the backward pass's workspace (no GPU needed): a plane of
partial sums per tile of negatives, 128, 64 or 32 of them by the number of phases, and one per range of positives."""
import ctypes as C

import pytest

from cuke_amd import _lib
from test_gpu_pair_tiles import SHAPES


def plan(model, p, batch, chunk, n_neg, dim):
    """(phases, ranges of positives) of the tiles by pairs, every number of phases that fits; empty: the other tiles."""
    def query(name, norm):
        tab = _lib.Tables(_lib.MODELS[name], norm, 0.0, 0, dim, dim // 2 if model == "RotatE" else dim, 10, 3, 0x10000, 0x10000, 0x10000)
        bat = _lib.Batch(batch, 0x10000, 0x10000, 0x10000, 0x10000, chunk, n_neg, None, None, None, 0, 0)
        return _lib.lib().kge_score_bwd_workspace(C.byref(tab), C.byref(bat))

    def up(floats):
        return (4 * max(floats, 1) + 255) // 256 * 256

    sides = 2 if model == "TransH" else 1
    one = query("TransH", 2) if model == "TransH" else query("DistMult", 2)  # the same rows, tiles without planes
    more, row = query(model, p) - one, batch // chunk * n_neg * dim
    if more == 0:
        return []
    return [(ph, splits) for ph in (1, 2, 4) for splits in range(1, -(-chunk // 16) + 1)
            if sides * (up(-(-n_neg * ph // 128) * batch * dim) - up(batch * dim)) + up((splits - 1) * row) - up(0) == more]


@pytest.mark.parametrize("model,p", [("RotatE", 2), ("TransE", 1), ("TransE", 2), ("TransH", 1)])
def test_every_form_is_reached(model, p):
    plans = {s: plan(model, p, *s) for s in SHAPES}
    known = [q[0] for q in plans.values() if len(q) == 1]
    assert {ph for ph, _ in known} == {1, 2, 4}, plans
    assert any(splits > 1 for _, splits in known)
    assert model == "RotatE" or any(not q for q in plans.values())  # (and the other side of the rule)
