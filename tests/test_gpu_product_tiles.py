"""TransR / RESCAL: the 64-row tiles of the grouped product and the rule between them and the 32-row tiles."""
import numpy as np
import pytest
import torch

from cuke_amd import synth
from helpers import assert_close, gpu_model

pytestmark = pytest.mark.gpu

EDGES = (1, 4, 5, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65, 129)  # rows of a group around one to four row blocks and one to three tiles


@pytest.mark.parametrize("model", ["TransR", "RESCAL"])
@pytest.mark.parametrize("dim,singles", [(4, 0), (36, 0), (124, 0), (128, 0), (132, 0), (260, 0), (388, 0), (512, 0), (1000, 0),
                                         # (many groups of one row beside them: the 32-row tiles)
                                         (4, 900), (36, 900), (132, 300), (260, 600)])
def test_groups_at_the_edges_of_a_tile(oracle, model, dim, singles):
    sizes = EDGES + (1,) * singles
    w = synth.custom_workload(model, n_ent=300, n_rel=len(sizes) + 1, dim=dim, batch=sum(sizes), norm_p=2, sigma=0.2, seed=dim)
    a = w.arrays
    a["r"][:] = np.random.default_rng(dim).permutation(np.repeat(np.arange(len(sizes)), sizes))
    m, ix = gpu_model(w)
    from cuke_amd.kge import inspect
    fw = m.score(ix["h"], ix["r"], ix["t"], rel_insp=inspect([ix["r"]], m.n_rel))
    pos, _ = oracle.score(model, a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], p=2)
    assert_close(fw.pos.cpu().numpy(), pos, what="scores")
    dpos = np.random.default_rng(1).standard_normal(w.batch).astype(np.float32)
    g = m.backward(fw, torch.from_numpy(dpos).to(fw.pos.device))
    ref = oracle.backward(model, a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], dpos=dpos, p=2)
    assert_close(g.ent_rows.cpu().numpy(), ref.ent_rows, what="entity rows", rows=True)
    assert_close(g.aux_rows.cpu().numpy(), ref.aux_rows, what="projection gradients", rows=True)


@pytest.mark.parametrize("n_rel,dim", [(3, 36), (3, 132), (3, 260), (60, 36), (200, 12)])
@pytest.mark.parametrize("model", ["TransR", "RESCAL"])
def test_shared_negatives_by_both_tiles(oracle, model, n_rel, dim):
    w = synth.custom_workload(model, n_ent=400, n_rel=n_rel, dim=dim, batch=384, chunk=96, n_neg=21, norm_p=2, sigma=0.2, seed=n_rel)
    a = w.arrays
    m, ix = gpu_model(w)
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], 96)
    kw = dict(p=2, neg=a["neg"], chunk=96)
    pos, neg = oracle.score(model, a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], **kw)
    assert_close(fw.pos.cpu().numpy(), pos, what="scores")
    assert_close(fw.neg.cpu().numpy(), neg, what="negatives' scores")
    rng = np.random.default_rng(2)
    dpos, dneg = rng.standard_normal(384).astype(np.float32), rng.standard_normal((384, 21)).astype(np.float32)
    g = m.backward(fw, torch.from_numpy(dpos).cuda(), torch.from_numpy(dneg).cuda())
    ref = oracle.backward(model, a["E"], a["R"], a["A"], a["h"], a["r"], a["t"], dpos=dpos, dneg=dneg, **kw)
    assert_close(g.ent_rows.cpu().numpy(), ref.ent_rows, what="entity rows", rows=True)
    assert_close(g.aux_rows.cpu().numpy(), ref.aux_rows, what="projection gradients", rows=True)


@pytest.mark.parametrize("model", ["TransR", "RESCAL"])
@pytest.mark.parametrize("dim", [36, 132, 200, 260, 1000])
def test_an_infinite_weight_in_the_last_row_stays_in_its_column(model, dim):
    """Widths that are no multiple of 16: where a tile's last step reaches past the row, the projection's last row is read in its
    place.  Few groups, so the 64-row tiles take them; one to four rows each, which streaming also kept clean."""
    w = synth.custom_workload(model, n_ent=50, n_rel=3, dim=dim, batch=8, norm_p=2, sigma=0.2, seed=dim)
    w.arrays["r"][:] = [0, 0, 0, 0, 1, 1, 2, 2]
    w.arrays["t"][:] = (w.arrays["h"] + 1) % 50  # (no zero difference: 0 * inf is a NaN of the product itself)
    w.arrays["A"][1, dim - 1, dim - 2] = np.inf
    a = {k: torch.from_numpy(v) for k, v in w.arrays.items() if v is not None}
    m, ix = gpu_model(w)
    from cuke_amd.kge import inspect
    got = m.score(ix["h"], ix["r"], ix["t"], rel_insp=inspect([ix["r"]], m.n_rel)).residual.cpu()
    x = (a["E"][a["h"]] - (a["E"][a["t"]] if model == "TransR" else 0)).double()
    want = torch.bmm(x[:, None, :], a["A"][a["r"]].double())[:, 0] + (a["R"][a["r"]].double() if model == "TransR" else 0)
    assert torch.isinf(want).sum() == 2 and not torch.isnan(want).any()
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)].double(), want[torch.isinf(want)])
    assert not torch.isnan(got).any()


@pytest.mark.parametrize("n_rel,dim,kw,form", [(3, 48, {}, "tall"), (900, 144, {}, "gemm"), (3, 48, dict(chunk=32, n_neg=4), "tall"),
                                               (900, 144, dict(chunk=32, n_neg=4), "gemm")])
def test_the_timeline_names_the_form_that_ran(n_rel, dim, kw, form):
    from cuke_amd.kge import TrainStep
    w = synth.custom_workload("TransR", n_ent=300, n_rel=n_rel, dim=dim, batch=256, sigma=0.2, seed=1, **kw)
    m, ix = gpu_model(w)
    st = TrainStep(m, ix["h"], ix["r"], ix["t"], ix.get("neg"), w.chunk or None, back_rows=False)
    names = [name for name, _ in st.kernel_times(2)]
    first = "list>" if kw else "fwd>"
    assert any(n.endswith(f"transr_{form}_kernel<{first}") for n in names) and f"transr_{form}_kernel<dX>" in names, names


@pytest.mark.parametrize("dim,n_rel,batch,tiles", [
    (200, 20, 5600, "tall"),    # at most 200 short tiles
    (132, 20, 6400, "gemm"),    # more, and too few 64-row tiles for the bf16 matrix cores
    (200, 100, 4500, "gemm"),
    (200, 20, 8192, "tall"),    # 276 items of 64 rows x 128 columns on average
    (256, 237, 7500, "gemm"),   # fewer than 32 rows a relation
])
def test_the_rule_between_the_tiles(dim, n_rel, batch, tiles):
    from cuke_amd.kge import KGEModel, TrainStep
    g = torch.Generator(device="cuda")
    g.manual_seed(dim)
    E, A = (torch.randn(*s, generator=g, device="cuda") * 0.05 for s in ((3000, dim), (n_rel, dim, dim)))
    h, t = (torch.randint(0, 3000, (batch,), generator=g, device="cuda") for _ in range(2))
    r = torch.arange(batch, device="cuda") % n_rel
    st = TrainStep(KGEModel("RESCAL", E, None, A), h, r, t, dpos=torch.randn(batch, generator=g, device="cuda"))
    names = [k for k, _ in st.kernel_times(steps=1)]
    assert any(f"transr_{tiles}_kernel<fwd>" in k for k in names), names
    want = torch.empty(batch, dtype=torch.float64, device="cuda")
    for u in range(n_rel):
        m = r == u
        want[m] = ((E[h[m]].double() @ A[u].double()) * E[t[m]].double()).sum(1)
    assert_close(st.pos.cpu().numpy(), want.cpu().numpy(), what="scores")
