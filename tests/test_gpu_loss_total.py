"""The margin loss whose last sum rides in the backward pass: the same bits as the loss call, from one partial to all 1024 of them, with one to
three reduction jobs and the sums of split relations beside it, in plain, staged and captured steps."""
import ctypes as C

import pytest
import torch

from cuke_amd import _lib, synth
from cuke_amd.kge import TrainStep, margin_loss
from helpers import gpu_model

pytestmark = pytest.mark.gpu


def _step(model, batch, chunk, n_neg, dim=16, n_rel=7):
    w = synth.custom_workload(model, n_ent=300, n_rel=n_rel, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, sigma=0.2, seed=batch)
    m, ix = gpu_model(w)
    return TrainStep(m, ix["h"], ix["r"], ix["t"], ix["neg"], chunk, loss="margin")


def _same(st):
    want = margin_loss(st.pos, st.neg, st.margin, st.sign)
    torch.cuda.synchronize()
    assert torch.equal(st.loss.view(-1), want[0].view(-1))
    assert torch.equal(st.dpos, want[1]) and torch.equal(st.dneg.view_as(want[2]), want[2])


@pytest.mark.parametrize("model", ["DistMult", "TransE", "TransH", "TransR", "RESCAL"])
@pytest.mark.parametrize("batch,chunk,n_neg,dim", [(1, 1, 1, 16), (5, 5, 3, 15), (1029, 343, 4, 16), (4100, 4100, 1, 18), (5000, 1000, 8, 16)])
def test_same_as_the_loss_call(model, batch, chunk, n_neg, dim):
    if model in ("TransR", "RESCAL"):
        dim = 16  # (shared negatives take rows of whole quads there)
    st = _step(model, batch, chunk, n_neg, dim)
    for fused in (None, False):
        st.loss.fill_(float("nan"))
        st.run(fused=fused)
        _same(st)


def test_one_call_staged_and_captured_steps():
    st = _step("DistMult", 4096, 1024, 16)
    st.loss.fill_(float("nan"))
    st.run(pipeline=True)
    _same(st)
    st = _step("ComplEx", 4096, 1024, 16)
    st.capture()
    for _ in range(3):
        st.loss.fill_(float("nan"))
        st.replay()
        _same(st)
    st = _step("TransE", 4096, 1024, 16)
    st.loss.fill_(float("nan"))
    st.run_native(None, 0), st.run_native(0, None)
    _same(st)


@pytest.mark.parametrize("model", ["TransR", "RESCAL"])
@pytest.mark.parametrize("batch,dim,n_rel", [(1024, 1024, 2), (2048, 1024, 7), (4096, 512, 15), (8192, 200, 20), (2048, 1022, 7)])
def test_beside_the_sums_of_split_relations(model, batch, dim, n_rel):
    """Explicit triples, where level 1 of the reduction rides with dM and level 2 carries the split relations' sums and the loss: more pieces of
    sums than the grid has workgroups, (8192 x 200) fewer, (1022) rows that are padded first."""
    w = synth.custom_workload(model, n_ent=300, n_rel=n_rel, dim=dim, batch=batch, sigma=0.2, seed=batch)
    m, ix = gpu_model(w)
    r = torch.arange(batch, device="cuda") % n_rel
    st = TrainStep(m, ix["h"], r, ix["t"], dpos=torch.randn(batch, device="cuda"))
    parts, loss = torch.rand(1000, device="cuda", dtype=torch.float64), torch.empty(1, device="cuda")
    total = _lib.LossTotal(parts.data_ptr(), parts.numel(), 0.25, loss.data_ptr())
    rows = [x for x in (st.ent_rows, st.rel_rows, st.aux_rows) if x is not None]
    for fused in (None, False):
        got = []
        for p in (None, C.addressof(total)):
            for x in (*rows, loss):
                x.fill_(float("nan"))
            st.bat.loss_total = p
            st.run(fused=fused)
            torch.cuda.synchronize()
            got.append([x.clone() for x in rows])
        st.bat.loss_total = None
        assert not torch.isnan(got[1][-1][:n_rel]).any()
        assert all(torch.equal(x.view(torch.int32), y.view(torch.int32)) for x, y in zip(*got))
        assert abs(loss.item() - 0.25 * parts.sum().item()) <= 1e-6 * abs(loss.item())
