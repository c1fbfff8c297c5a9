"""TransR against shared negatives: the (relation, chunk) groups over more than one workgroup's positions, chunks of one positive and of all,
one relation and hundreds, chunks of more than 256 positives (the list of a chunk's groups in several turns), workgroups behind one, four and more others."""
import pytest

from cuke_amd import synth
from test_gpu_backward import compare, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["tail", "head"])
@pytest.mark.parametrize("batch,chunk,n_rel", [(4096, 512, 1), (4100, 41, 300), (8193, 2731, 40), (8200, 8200, 700), (5000, 1, 7), (1, 1, 3), (4097, 241, 5),
                                               (20501, 20501, 900), (36900, 9, 2), (70000, 7000, 1)])
def test_scores_and_gradients(oracle, batch, chunk, n_rel, mode):
    w = synth.custom_workload("TransR", n_ent=400, n_rel=n_rel, dim=16, batch=batch, chunk=chunk, n_neg=5, sigma=0.2, ent_zipf=0.8, seed=batch + n_rel)
    g, ref = run_both(oracle, w, seed=1, neg_mode=mode, fast=True)
    compare(g, ref, f"{batch} / {chunk}, {n_rel} relations, {mode}")
