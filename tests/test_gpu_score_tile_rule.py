"""Score tiles of the vector ALUs on both sides of the size rule: RotatE in small tiles at every size, chunks that half fill the large
tiles, chunks that fill them; rows whose last slice is ragged, whole, or the only one."""
import numpy as np
import pytest
import torch

from cuke_amd import synth
from helpers import assert_close, gpu_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,chunk,n_neg", [(4096, 32, 500),    # 1024 large tiles, half of each empty
                                               (4480, 20, 257),    # 1120 of them, two thirds empty, a ragged last column
                                               (4096, 64, 1000)])  # 1024 full ones
@pytest.mark.parametrize("model,p,dim", [("TransE", 1, 98), ("TransE", 2, 96), ("TransE", 2, 31), ("TransH", 1, 96), ("TransH", 2, 98),
                                         ("RotatE", 2, 60), ("RotatE", 2, 64), ("RotatE", 2, 196)])
def test_scores_and_gradients_of_large_batches(oracle, model, p, dim, batch, chunk, n_neg):
    w = synth.custom_workload(model, n_ent=3000, n_rel=11, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, norm_p=p, sigma=0.2, gamma=4.0,
                              seed=dim + n_neg, lattice=(p == 1))
    a = w.arrays
    m, ix = gpu_model(w)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], chunk)
    tabs = (a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], a["neg"], chunk)
    pos, neg = oracle.score(model, *tabs, p=p, gamma=4.0, fast="omp")
    assert_close(fw.pos.cpu().numpy(), pos, what="positives")
    assert_close(fw.neg.cpu().numpy(), neg, what="negatives")
    if model == "TransH":                   # (its tiles save what the gradients are formed from)
        rng = np.random.default_rng(dim)
        dpos, dneg = rng.standard_normal(batch).astype(np.float32), rng.standard_normal((batch, n_neg)).astype(np.float32)
        g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
        ref = oracle.backward(model, *tabs, dpos, dneg, p=p, fast="omp")
        for what in ("ent_rows", "rel_rows", "aux_rows"):
            assert_close(getattr(g, what).cpu().numpy(), getattr(ref, what), what=what, rows=True)
