"""TransE L2 gradients of rows that lie close together compared with their own size, against 64 bits: tables with a common offset,
negatives beside the translated positives.  Every form of the gradient tiles, in both negative modes."""
import numpy as np
import pytest
import torch

from cuke_amd.kge import KGEModel

pytestmark = pytest.mark.gpu

# (batch, chunk, n_neg, dim): the 64-bit products' side of the rule and the differences' 16-, 32- and 64-owner tiles, with and without
# a narrow last column tile; odd widths and counts
SHAPES = [
    (1536, 256, 200, 150, "matrix_cores"),   # 3 x 6 x 200 owners are too few: 16-owner differences
    (1024, 256, 256, 400, "matrix_cores"),   # 7 x 4 x 256: products
    (2000, 500, 130, 801, "matrix_cores"),   # products, odd rows and a last tile of 33 columns
    (8192, 128, 1, 130, "matrix_cores"),     # 576 tiles of single owners: 32-owner differences
    (1100, 100, 77, 200, "vector_alus"),     # 16 owners
    (2048, 128, 128, 550, "vector_alus"),    # 32 owners
    (4096, 256, 256, 523, "vector_alus"),    # 64 owners, 11 columns in narrow tiles
    (4096, 64, 300, 500, "vector_alus"),     # 64 owners, no narrow tile, a ragged last coefficient quad
]


@pytest.mark.parametrize("batch,chunk,n_neg,dim,unit", SHAPES)
@pytest.mark.parametrize("rows", ["centred", "offset 0.25", "offset 5", "near 1e-2", "near 1e-5"])
@pytest.mark.parametrize("mode", ["tail", "head"])
def test_gradients_of_close_rows(batch, chunk, n_neg, dim, unit, rows, mode):
    rng = np.random.default_rng(dim)
    dev = torch.device("cuda:0")
    n_chunks, n_rel, sign = batch // chunk, 7, (1.0 if mode == "tail" else -1.0)
    E = (rng.standard_normal((2 * batch + n_chunks * n_neg, dim)) * 0.05).astype(np.float32)
    R = (rng.standard_normal((n_rel, dim)) * 0.05).astype(np.float32)
    ids = rng.permutation(E.shape[0])        # every entity occurs once: a row's gradient is one sum
    kept, other, neg = ids[:batch], ids[batch:2 * batch], ids[2 * batch:]
    r = rng.integers(0, n_rel, batch)
    if rows.startswith("offset"):
        E += np.float32(rows.split()[1])
    if rows.startswith("near"):              # negative k of a chunk beside the translated positive k of it
        k = np.arange(min(n_neg, chunk))
        for c in range(n_chunks):
            b = c * chunk + k
            E[neg[c * n_neg + k]] = E[kept[b]] + sign * R[r[b]] + rng.standard_normal((len(k), dim)) * float(rows.split()[1])
    E, R, kept, other, neg, r = (torch.from_numpy(x).to(dev) for x in (E, R, kept, other, neg, r))
    m = KGEModel("TransE", E, R, norm_p=2, pair_sums=unit)
    h, t = (kept, other) if mode == "tail" else (other, kept)
    fw = m.score(h, r, t, neg, chunk, neg_mode=mode)
    dneg = -torch.rand(fw.neg.shape, device=dev, generator=torch.Generator(dev).manual_seed(1))
    g = m.backward(fw, None, dneg)
    got = torch.zeros(E.shape, dtype=torch.float64, device=dev)
    got[g.ent_ids.long()] = g.ent_rows.double()

    q = (E[kept] + sign * R[r]).double().view(n_chunks, chunk, dim)  # the translated rows, rounded to fp32 as every form has them
    x = E[neg].double().view(n_chunks, n_neg, dim)
    coef = torch.where(fw.neg > 0, dneg.double() / fw.neg.double(), torch.zeros_like(fw.neg, dtype=torch.float64)).view(n_chunks, chunk, n_neg)
    for c in range(n_chunks):
        u = q[c][:, None, :] - x[c][None]
        for what, idx, ref in (("positive's", kept.view(n_chunks, chunk)[c], (coef[c][:, :, None] * u).sum(1)),
                               ("negative's", neg.view(n_chunks, n_neg)[c], -(coef[c][:, :, None] * u).sum(0))):
            # A difference, a quotient and each level of the two-level sum round once by at most 2^-24 of what they form, whatever the
            # rows' size (differences: 1.0 to 1.5 times 2^-24 over a chunk's rows; products in 64 bits: 0.4).  Sums of products in fp32
            # round by 2^-24 of the rows: 5 to 120 times 2^-24 for all but the centred rows.
            err = (got[idx] - ref).norm() / ref.norm()
            assert err <= 4 * 2.0 ** -24, f"chunk {c}, the {what} gradients: {err:.2e} of their norm"
