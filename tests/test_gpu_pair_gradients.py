"""TransR against shared negatives, gradients of the pairs: negative counts around the register blocks, rows of one and two column blocks,
groups inside a block of positions, across two and over many."""
import numpy as np
import pytest
import torch

from cuke_amd import synth
from helpers import assert_close, gpu_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rel", [1, 4, 60])
@pytest.mark.parametrize("dim", [48, 260])
@pytest.mark.parametrize("n_neg", [1, 15, 16, 17, 32, 33, 64, 65, 130])
def test_pair_gradients(oracle, n_neg, dim, n_rel):
    w = synth.custom_workload("TransR", seed=n_neg, n_ent=80, n_rel=n_rel, dim=dim, batch=66, chunk=33, n_neg=n_neg, norm_p=2, sigma=0.25)
    a = w.arrays
    m, ix = gpu_model(w)
    rng = np.random.default_rng(n_neg)
    dpos, dneg = rng.standard_normal(66).astype(np.float32), rng.standard_normal((66, n_neg)).astype(np.float32)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], 33)
    tabs = (a["E"], a["R"], a["A"], a["h"], a["r"], a["t"])
    g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
    ref = oracle.backward("TransR", *tabs, a["neg"], 33, dpos, dneg, p=2)
    for name in ("ent_rows", "rel_rows", "aux_rows"):
        assert_close(getattr(g, name).cpu().numpy(), getattr(ref, name), what=name, rows=True)
    g = m.backward(fw, torch.from_numpy(dpos).cuda(), None)  # no gradient of the pairs: their rows are zero
    ref = oracle.backward("TransR", *tabs, dpos=dpos, p=2)
    assert_close(g.rel_rows.cpu().numpy(), ref.rel_rows, what="relation rows alone", rows=True)
    assert_close(g.aux_rows.cpu().numpy(), ref.aux_rows, what="projection rows alone", rows=True)
