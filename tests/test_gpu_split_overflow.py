"""Three-part bf16 products whose leading parts overflow, and operands that are not finite: the results are those of fp32, at the ragged
edges of tiles too."""
import numpy as np
import pytest
import torch

from cuke_amd import kge, synth
from cuke_amd.kge import KGEModel
from helpers import assert_close, gpu_model

pytestmark = pytest.mark.gpu

BIG = 0.9985 * 2.0 ** 64  # the square is below FLT_MAX, the square of its bf16 rounding (2^64) is not


def _same(got, want, what):
    got, want = got.cpu().numpy(), want.numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)), what
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(got.dtype)), what
    fine = np.isfinite(want)
    # (what surrounds a large term is rounded at its size, in both)
    assert np.allclose(got[fine], want[fine], rtol=1e-5, atol=1e-5 * np.abs(want[fine & (np.abs(want) < 1e30)]).max()), what


# 128 x 128 and 64 x 128 tiles, ragged in rows, negatives and columns
@pytest.mark.parametrize("dim,chunk,n_neg,chunks", [(128, 512, 12288, 1), (101, 130, 129, 96), (131, 33, 513, 205)])
@pytest.mark.parametrize("model", ["DistMult", "ComplEx", "TransF"])
def test_scores(model, dim, chunk, n_neg, chunks):
    dim += dim % 2 if model == "ComplEx" else 0
    rng = np.random.default_rng(dim)
    E = rng.random((4000, dim)).astype(np.float32)
    R = np.ones((3, dim), np.float32)
    if model == "ComplEx":
        R[:, dim // 2:] = 0
    if model == "TransF":
        R[:] = 0
    h, t, neg = (rng.integers(10, 4000, n) for n in (chunk * chunks, chunk * chunks, n_neg * chunks))
    E[0], E[1] = 0.0, 0.0
    E[0, dim - 1], E[1, dim - 1] = BIG * (0.5 if model == "TransF" else 1.0), BIG   # their product: a finite score
    E[2, 3], E[3, dim - 2], E[4, 0] = np.inf, np.nan, -np.inf
    h[[0, 1, chunk - 1]], neg[[0, 1, n_neg - 1]] = (0, 2, 3), (1, 3, 4)             # first chunk: every kind, on the tiles' edges
    h[-1], neg[-1] = 0, 1                                                           # last chunk: the finite one in its last row and column
    fw = KGEModel(model, torch.from_numpy(E).cuda(), torch.from_numpy(R).cuda()).score(
        *(torch.from_numpy(x).cuda() for x in (h, np.zeros_like(h), t, neg)), chunk)
    for c, rows, cols in ((0, slice(0, chunk), slice(0, n_neg)), (chunks - 1, slice((chunks - 1) * chunk, None), slice((chunks - 1) * n_neg, None))):
        q, x = torch.from_numpy(E[h[rows]]).double(), torch.from_numpy(E[neg[cols]]).double()
        rel, shift = torch.from_numpy(R[0]).double(), 0.0
        if model == "ComplEx":
            (hr, hi), (qr, qi) = q.chunk(2, 1), rel.chunk(2)
            q = torch.cat((hr * qr - hi * qi, hr * qi + hi * qr), 1)
        elif model == "TransF":
            q, shift = 2 * q + rel, -(rel * q).sum(1, keepdim=True)
        want = torch.stack([(q[i] * x).sum(1) for i in range(q.shape[0])]) + shift
        _same(fw.neg[rows], want, f"{model}, chunk {c}")


@pytest.mark.parametrize("dim", [128, 132])
def test_grouped_products(dim):
    rng = np.random.default_rng(dim)
    sizes = [70, 33, 40] * 100
    r = np.repeat(np.arange(300), sizes)
    E, A = rng.random((700, dim)).astype(np.float32), rng.random((300, dim, dim)).astype(np.float32)
    h, t = rng.integers(10, 350, r.size), rng.integers(350, 700, r.size)
    E[0], E[1], E[2, 5] = 0.0, 0.0, np.inf
    E[0, dim - 1] = BIG
    A[[0, 1], dim - 1, dim - 1] = BIG
    h[[0, 69, 75]], t[[0, 69]] = (0, 0, 2), 1
    score = kge.transR(r.size, dim, 700, *(torch.from_numpy(x).cuda() for x in (E, h, t)), 300, torch.from_numpy(A).cuda(), torch.from_numpy(r).cuda(),
                       torch.zeros(300, dim, device="cuda"))
    x = torch.from_numpy(E[h]).double() - torch.from_numpy(E[t]).double()
    for u in range(3):
        m = torch.from_numpy(r == u)
        want = (x[m][:, :, None] * torch.from_numpy(A[u]).double()).sum(1)
        fits = want.abs() < 3.4e38
        _same(score[m.cuda()], torch.where(fits | ~want.isfinite(), want, want.sign() * np.inf), f"relation {u}")
        assert u or bool(fits[0].all()) and float(want[0, dim - 1]) > 3.3e38


# (items of 128 x 128 as in the listed projection gradients' own test: one, and ragged second ones)
@pytest.mark.parametrize("dim,batch,n_rel,chunk,n_neg", [(60, 512, 600, 512, 63), (132, 256, 150, 128, 64), (196, 256, 150, 16, 64)])
@pytest.mark.parametrize("value", [BIG, np.inf])
def test_listed_projection_gradients(oracle, dim, batch, n_rel, chunk, n_neg, value):
    w = synth.custom_workload("TransR", seed=dim, n_ent=3000, n_rel=n_rel, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, norm_p=1, sigma=0.25)
    a = w.arrays
    rng = np.random.default_rng(dim)
    neg = a["neg"].reshape(-1)
    a["h"][:], a["t"][:], neg[:] = rng.integers(10, 3000, batch), rng.integers(10, 3000, batch), rng.integers(10, 3000, neg.size)
    neg[n_neg - 1] = 0                      # one negative of the first chunk has the value in its last column
    a["E"][0, dim - 1] = value
    dneg = np.zeros((batch, n_neg), np.float32)
    dneg[:chunk] = 1e-4 * (1 + rng.random((chunk, n_neg)))
    if np.isfinite(value):                  # one pair's gradient makes upstream rows whose products with the value are below FLT_MAX
        dneg[:chunk, n_neg - 1] = 0
        dneg[0, n_neg - 1] = BIG
    m, ix = gpu_model(w)
    dpos = np.zeros(batch, np.float32)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], chunk)
    g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
    ref = oracle.backward("TransR", a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], a["neg"], chunk, dpos, dneg, p=1)
    got, want = g.aux_rows.cpu().numpy().reshape(-1, dim, dim), ref.aux_rows.reshape(-1, dim, dim)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    last = np.abs(want[:, dim - 1])
    if np.isfinite(value):
        assert last.max() > 3.3e38
        rows = last.max(1) > 1e38
        assert_close(got[rows, dim - 1], want[rows, dim - 1], what="the column with the value", rows=True)
    else:
        assert np.isinf(last).any()
    small = last.max(1) < 1.0               # relations without it
    assert_close(got[small], want[small], what="projection gradients", rows=True)
