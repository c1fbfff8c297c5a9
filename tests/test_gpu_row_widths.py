"""Row widths and negative counts that are no multiple of four, and rows off the 16-byte grid: the last quad of a row ends with
it and overlaps the one before (score tiles, gradient tiles, per-row kernels, coefficient rows)."""
import numpy as np
import pytest
import torch

from cuke_amd import synth
from cuke_amd.kge import KGEModel, inspect, margin_loss, sparse_adagrad, sparse_sgd
from helpers import assert_close, gpu_model

pytestmark = pytest.mark.gpu

FORMS = [("TransE", 1), ("TransE", 2), ("TransH", 1), ("TransH", 2), ("DistMult", 2), ("ComplEx", 2), ("RotatE", 2), ("TransF", 2)]
# one row of tiles with ragged edges | as many tiles as the 64 x 64 forms want, of a few pairs each
BATCHES = [dict(batch=140, chunk=70, n_neg=67), dict(batch=3 * 1024, chunk=3, n_neg=5)]


@pytest.mark.parametrize("batch", BATCHES, ids=["edges", "many"])
@pytest.mark.parametrize("dim", [5, 66, 131, 150, 262])
@pytest.mark.parametrize("model,p", FORMS)
def test_forward_and_backward(oracle, model, p, dim, batch):
    if model in ("ComplEx", "RotatE"):
        dim *= 2  # (halves of these widths)
    lattice = p == 1
    w = synth.custom_workload(model, seed=dim, n_ent=90, n_rel=5, dim=dim, norm_p=p, sigma=0.3, gamma=2.0, lattice=lattice, **batch)
    a = w.arrays
    m, ix = gpu_model(w)
    if batch["chunk"] == 70:  # tables that start 4 bytes off the grid
        off = lambda x: None if x is None else torch.cat((x.new_zeros(1), x.reshape(-1)))[1:].view(x.shape)
        m = KGEModel(model, off(m.E), off(m.R), off(m.A), norm_p=p, gamma=2.0)
    rng = np.random.default_rng(dim)
    dpos, dneg = rng.standard_normal(w.batch).astype(np.float32), rng.standard_normal((w.batch, w.n_neg)).astype(np.float32)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], w.chunk)
    g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
    tabs, ids = (a["E"], a["R"], a["A"]), (a["h"], a["r"], a["t"], a["neg"])
    pos, negs = oracle.score(model, *tabs, *ids, w.chunk, p=p, gamma=2.0)
    ref = oracle.backward(model, *tabs, *ids, w.chunk, dpos, dneg, p=p)
    assert_close(fw.pos.cpu().numpy(), pos, what="pos")
    assert_close(fw.neg.cpu().numpy(), negs, what="neg")
    floor = 0.1 if dim <= 10 else 0.0  # (few columns: no scale of their own, as in the random shapes)
    for name in ("ent_rows", "rel_rows", "aux_rows"):
        want = getattr(ref, name)
        if want is not None:
            # RotatE: among the up to 2 M pair elements of a call the smallest |u| is about 1e-3 of its operands, whose rounding
            # (1e-7) turns its unit vector by 1e-4; times an upstream gradient of up to 4 in a bound of 1e-4: a few elements
            out = (max(1e-5, 2 / want.size), 4.0) if model == "RotatE" else None
            assert_close(getattr(g, name).cpu().numpy(), want, what=name, rows=True, outliers=out, global_floor=floor)


@pytest.mark.parametrize("dim", [4, 5, 255, 257, 259, 1027])
def test_optimizer_rows(oracle, dim):
    """(a last quad that overlaps one of the turn before: its elements are updated once)"""
    rng = np.random.default_rng(dim)
    table, state = rng.standard_normal((9, dim)).astype(np.float32), rng.random(9).astype(np.float32)
    ins = inspect(torch.tensor([7, 2, 2, 5, 0, 7], device="cuda"), 9)
    rows = rng.standard_normal((6, dim)).astype(np.float32)
    u = ins.ids().cpu().numpy()
    t, s, g = torch.from_numpy(table).cuda(), torch.from_numpy(state).cuda(), torch.from_numpy(rows).cuda()
    sparse_sgd(t, ins, g, 0.1)
    assert_close(t.cpu().numpy(), oracle.sparse_sgd(table, u, rows[:4], 0.1), what="sgd")
    t = torch.from_numpy(table).cuda()
    sparse_adagrad(t, s, ins, g, 0.1)
    wt, ws = oracle.sparse_adagrad(table, state, u, rows[:4], 0.1)
    assert_close(t.cpu().numpy(), wt, what="adagrad")
    assert_close(s.cpu().numpy(), ws, what="state")


@pytest.mark.parametrize("n_neg", [3, 4, 5, 255, 257, 258, 515])
def test_margin_rows(n_neg):
    rng = np.random.default_rng(n_neg)
    pos, neg = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda() for s in ((7,), (7, n_neg)))
    loss, dpos, dneg = margin_loss(pos, neg, 0.5, 1.0)
    v = 0.5 - (pos.double()[:, None] - neg.double())
    on = (v > 0).double() / v.numel()
    assert torch.allclose(loss.double().reshape(()), (v.clamp(min=0)).mean(), rtol=1e-6)
    assert torch.equal(dneg, on.float()) and torch.allclose(dpos.double(), -on.sum(1), rtol=1e-6)
