"""TransR against shared negatives, projection gradients in 128 x 128 items: result widths around the tiles and their 32-column blocks,
groups of one chunk, of several and of a few rows more than a slice; values beyond bf16's range."""
import numpy as np
import pytest
import torch

from cuke_amd import synth
from helpers import assert_close, gpu_model

pytestmark = pytest.mark.gpu


# (rows, relations, negatives and widths chosen so that batches can hold 512 items: (relations + rows / 256) * tiles^2)
@pytest.mark.parametrize("dim,batch,n_rel,chunk,n_neg", [
    (8, 512, 600, 128, 48), (60, 512, 600, 512, 63), (128, 512, 600, 64, 64), (132, 256, 150, 128, 64), (160, 256, 150, 256, 49),
    (196, 256, 150, 16, 64), (256, 256, 150, 128, 48), (260, 128, 60, 64, 64), (388, 64, 40, 32, 64),
])
@pytest.mark.parametrize("zipf", [False, True])
def test_listed_projection_gradients(oracle, dim, batch, n_rel, chunk, n_neg, zipf):
    w = synth.custom_workload("TransR", seed=dim, n_ent=300, n_rel=n_rel, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, norm_p=2, sigma=0.25)
    a = w.arrays
    rng = np.random.default_rng(dim)
    if zipf:  # one relation of many rows, many of one triple
        a["r"][:] = np.where(rng.random(batch) < 0.5, 0, a["r"])
    m, ix = gpu_model(w)
    dpos, dneg = rng.standard_normal(batch).astype(np.float32), rng.standard_normal((batch, n_neg)).astype(np.float32)
    tabs = (a["E"], a["R"], a["A"], a["h"], a["r"], a["t"])
    ref = oracle.backward("TransR", *tabs, a["neg"], chunk, dpos, dneg, p=2)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], chunk)
    for _ in range(2):  # (a second pass hands out the items again)
        g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
        assert_close(g.aux_rows.cpu().numpy(), ref.aux_rows, what="projection rows", rows=True)


def test_listed_projection_gradients_beyond_bf16(oracle):
    w = synth.custom_workload("TransR", seed=5, n_ent=40, n_rel=600, dim=48, batch=512, chunk=128, n_neg=48, norm_p=1, sigma=0.25)
    a = w.arrays
    a["E"][a["neg"].reshape(-1)[3], 7] = 3.395e38  # rounds to infinity in bf16
    m, ix = gpu_model(w)
    rng = np.random.default_rng(5)
    dpos, dneg = np.zeros(512, np.float32), (1e-4 * rng.random((512, 48))).astype(np.float32)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], 128)
    g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
    ref = oracle.backward("TransR", a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], a["neg"], 128, dpos, dneg, p=1)
    got, want = g.aux_rows.cpu().numpy().reshape(-1, 48, 48), ref.aux_rows.reshape(-1, 48, 48)
    assert np.isfinite(want).all() and np.isfinite(got).all() and np.abs(want[:, 7]).max() > 1e30
    rows = np.abs(want[:, 7]).max(1) > 1e30  # the relations that meet the value
    assert_close(got[rows, 7], want[rows, 7], what="the column with the value", rows=True)


@pytest.mark.parametrize("dim,batch,n_rel,chunk,n_neg", [(128, 1024, 1100, 128, 64), (60, 1024, 1100, 512, 48), (200, 512, 300, 64, 64)])
def test_listed_projection_gradients_against_64_bits(dim, batch, n_rel, chunk, n_neg):
    """L1, upstream gradients that are multiples of 2^-12: every upstream row is an exact sum of signs, so what differs from 64 bits
    is the product of the rows alone.  Half of the triples share a relation (items of 256 positions and their partial sums)."""
    from cuke_amd.kge import KGEModel
    g = torch.Generator(device="cuda")
    g.manual_seed(dim)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda") * 0.05
    E, R, A = rand(3000, dim), rand(n_rel, dim), rand(n_rel, dim, dim)
    ids = lambda n, k: torch.randint(0, n, (k,), generator=g, device="cuda")
    h, t, neg, r = ids(3000, batch), ids(3000, batch), ids(3000, batch // chunk * n_neg), ids(n_rel, batch)
    r[torch.rand(batch, generator=g, device="cuda") < 0.5] = 0
    dpos, dneg = (ids(2048, k).float().add_(1).div_(4096) for k in (batch, batch * n_neg))
    dneg = dneg.view(batch, n_neg)
    m = KGEModel("TransR", E, R, A, norm_p=1)
    fw = m.score(h, r, t, neg, chunk)
    grads = m.backward(fw, dpos, dneg)
    rows = {int(u): i for i, u in enumerate(grads.rel_ids.tolist())}
    D = lambda x: x.double()
    for u in [0] + r.unique()[1:8].tolist():
        M, want, size, n = D(A[u]), torch.zeros(dim, dim, dtype=torch.float64, device="cuda"), 0.0, 0
        sure = torch.ones(dim, dtype=torch.bool, device="cuda")  # columns in which no residual is within rounding of zero
        for c in range(batch // chunk):
            b = torch.arange(c * chunk, (c + 1) * chunk, device="cuda")
            b = b[r[b] == u]
            if b.numel() == 0:
                continue
            hx, tx, nx = D(E[h[b]]), D(E[t[b]]), D(E[neg.view(-1, n_neg)[c]])
            yp = (hx - tx) @ M + D(R[u])
            a = hx @ M + D(R[u])
            pair = a[:, None, :] - (nx @ M)[None]
            sure &= (pair.abs().amin((0, 1)) > 1e-6) & (yp.abs().amin(0) > 1e-6)
            cs = D(dneg[b])[:, :, None] * pair.sign()
            for x, q in (((D(E[h[b]] - E[t[b]])), D(dpos[b])[:, None] * yp.sign()), (hx, cs.sum(1)), (nx, -cs.sum(0))):
                want += x.t().contiguous() @ q
                size = size + x.abs().t().contiguous() @ q.abs()
                n += x.shape[0]
        got = D(grads.aux_rows.view(-1, dim, dim)[rows[u]])
        err = ((got - want).abs() / size)[:, sure] * 2 ** 24
        assert sure.float().mean() > 0.5
        # each product and each addition rounds once: sqrt(n) half ulps of the terms' total, at most
        assert float(err.max()) <= 4 + n ** 0.5, (u, n, float(err.max()))
