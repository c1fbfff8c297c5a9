"""The margin loss whose last sum rides in the backward pass: the same bits as the loss call, from one partial to all 1024 of them, with one to
three reduction jobs beside it, in plain, staged and captured steps."""
import pytest
import torch

from cuke_amd import synth
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
