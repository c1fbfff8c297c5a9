"""Gradient tiles that evaluate every pair once (TransE, RotatE, TransH L1): one, two and four phases, several tiles of negatives and ranges of
positives, their ragged edges, widths that end inside a quad, rows of one to three coefficients; head and tail negatives; the forms on
both sides of the rule."""
import pytest

import test_gpu_transe_distances

from cuke_amd import synth
from test_gpu_backward import compare, run_both

pytestmark = pytest.mark.gpu

# (batch, chunk, negatives, dim)
SHAPES = [
    (64, 64, 1, 16), (66, 33, 3, 20),          # coefficient rows of fewer than four
    (200, 200, 25, 50), (340, 17, 33, 70),     # four and two phases
    (256, 16, 129, 36), (512, 512, 130, 66),   # a second tile of one negative; ranges of positives that end inside a step
    (2048, 1024, 128, 8), (514, 257, 300, 264),
    (4096, 64, 257, 130),
    (1000, 25, 250, 98),                       # one phase and two tiles, for each model
]


@pytest.mark.parametrize("mode", ["tail", "head"])
@pytest.mark.parametrize("model,p", [("RotatE", 2), ("TransE", 1), ("TransE", 2), ("TransH", 1)])
@pytest.mark.parametrize("batch,chunk,n_neg,dim", SHAPES)
def test_gradients(oracle, model, p, batch, chunk, n_neg, dim, mode):
    # (L1: lattice tables, where every residual is exact and no sign is ambiguous)
    w = synth.custom_workload(model, n_ent=500, n_rel=7, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, norm_p=p, sigma=0.2, gamma=4.0,
                              ent_zipf=0.8, seed=dim + n_neg, lattice=(p == 1))
    g, ref = run_both(oracle, w, seed=2, neg_mode=mode, fast=True)
    # RotatE: unit vectors of residuals a thousand times smaller than their operands, where the 32-bit oracle itself leaves the bar: one
    # complex element of the 32500 of 4096 x 257 x 130 head lies 2.3 bars from 64 bits there, the kernel's 0.25
    compare(g, ref, f"{model} L{p} {batch}x{n_neg}x{dim} {mode}", outliers=(4e-5, 4.0) if model == "RotatE" else None)


@pytest.mark.parametrize("dim", [5, 34, 65, 96, 97, 150])
@pytest.mark.parametrize("mode", ["tail", "head"])
def test_last_column_tile_of_the_64_bit_products(dim, mode):
    """One to 32 columns left over (and 33, where the whole tile takes them)."""
    test_gpu_transe_distances.test_gradients_of_close_rows(8192, 256, 200, dim, "matrix_cores", "offset 0.25", mode)
