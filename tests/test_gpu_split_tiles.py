"""Dot-product scores on the bf16 matrix cores (three-part splits): tile edges, widths, shapes on both sides of the rule, no worse than
fp32 against 64 bits, infinities and NaNs as fp32 gives them."""
import numpy as np
import pytest
import torch

from cuke_amd.kge import KGEModel

pytestmark = pytest.mark.gpu


def _case(model, n_ent, dim, batch, n_neg, chunks, seed, scale=0.05):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    E, R = (torch.randn(n, dim, generator=g, device="cuda") * scale for n in (n_ent, 7))
    ids = lambda n, k: torch.randint(0, n, (k,), generator=g, device="cuda")
    return E, R, ids(n_ent, batch), ids(7, batch), ids(n_ent, batch), ids(n_ent, chunks * n_neg)


def _exact(model, E, R, h, r, t, neg, chunk, head):
    """64-bit scores and, per pair, the sum of the products' magnitudes (the scale of fp32 rounding)."""
    x, r = (E[t] if head else E[h]).double(), R[r].double()
    n = E[neg].double().view(-1, neg.numel() // (x.shape[0] // chunk), E.shape[1])
    s = -1.0 if head else 1.0
    if model == "DistMult":
        q, shift = x * r, 0
    elif model == "TransF":
        q, shift = 2 * x + s * r, -s * (r * x).sum(1, keepdim=True)
    else:
        a, b = torch.complex(*x.chunk(2, 1)), torch.complex(r.chunk(2, 1)[0], s * r.chunk(2, 1)[1])
        q = torch.view_as_real(a * b)
        q, shift = torch.cat((q[..., 0], q[..., 1]), 1), 0
    q3 = q.view(-1, chunk, E.shape[1])
    return (torch.bmm(q3, n.transpose(1, 2).contiguous()).view(x.shape[0], -1) + shift,
            torch.bmm(q3.abs(), n.abs().transpose(1, 2).contiguous()).view(x.shape[0], -1) + (shift.abs() if torch.is_tensor(shift) else 0))


# (dim, chunk, negatives, chunks): 128 x 128 tiles with ragged edges, one chunk against many, 64 x 128 tiles; then below the rule
SHAPES = [(96, 130, 129, 96), (101, 65, 384, 128), (400, 257, 20481, 1), (131, 128, 127, 384), (200, 33, 513, 205), (98, 64, 512, 256),
          (95, 130, 129, 96), (128, 130, 129, 32), (200, 33, 300, 205)]


@pytest.mark.parametrize("head", [False, True], ids=["tail", "head"])
@pytest.mark.parametrize("model", ["DistMult", "ComplEx", "TransF"])
@pytest.mark.parametrize("dim,chunk,n_neg,chunks", SHAPES)
def test_scores_against_64_bits(model, dim, chunk, n_neg, chunks, head):
    if model == "ComplEx":
        dim += dim % 2
    E, R, h, r, t, neg = _case(model, 3000, dim, chunk * chunks, n_neg, chunks, dim + n_neg)
    fw = KGEModel(model, E, R).score(h, r, t, neg, chunk, neg_mode="head" if head else "tail")
    want, size = _exact(model, E, R, h, r, t, neg, chunk, head)
    # fp32: the query's own rounding (up to 3 roundings) and the sum's, sqrt(dim) half ulps of the terms' total at most
    err = (fw.neg.double() - want).abs()
    assert bool((err <= 2.0 ** -24 * (4 + dim ** 0.5) * size).all()), float((err / size).max() * 2 ** 24)


def test_infinities_and_nans_as_fp32_has_them():
    E, R, h, r, t, neg = _case("DistMult", 3000, 128, 512, 12288, 1, 3, scale=1.0)
    R.fill_(1.0), E.abs_()
    E[5, 7], E[6, 8], E[9, 3], E[11, 100], E[12, 127] = float("inf"), float("nan"), 3.4e38, -float("inf"), 1e-30
    E[13].zero_()
    h[:6] = torch.tensor([5, 6, 9, 11, 12, 13], device="cuda")
    neg[:6] = h[:6]
    fw = KGEModel("DistMult", E, R).score(h, r, t, neg, 512)
    q, n = E[h].cpu(), E[neg].cpu()
    want = torch.stack([(q[i] * n[:200]).sum(1) for i in range(200)])
    got = fw.neg[:200, :200].cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    assert torch.equal(got[~fine].nan_to_num(nan=0.0), want[~fine].nan_to_num(nan=0.0))
    assert torch.allclose(got[fine], want[fine], rtol=1e-5)


def _grouped(sizes, dim, seed, scale=0.05):
    """Triples in groups of the given sizes (one relation each), shuffled."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = torch.repeat_interleave(torch.arange(len(sizes), device="cuda"), torch.tensor(sizes, device="cuda"))
    r = r[torch.randperm(r.numel(), generator=g, device="cuda")]
    E, R = (torch.randn(n, dim, generator=g, device="cuda") * scale for n in (700, len(sizes)))
    A = torch.randn(len(sizes), dim, dim, generator=g, device="cuda") * scale
    h, t = (torch.randint(0, 700, (r.numel(),), generator=g, device="cuda") for _ in range(2))
    return E, R, A, h, r, t


# groups on both sides of a tile's 64 rows and of its row blocks; more items than one per CU (and one launch of fewer, in fp32)
@pytest.mark.parametrize("dim,copies", [(128, 30), (132, 20), (200, 20), (256, 20), (260, 12), (388, 12), (128, 3)])
def test_grouped_products_against_64_bits(dim, copies):
    from cuke_amd import kge
    sizes = [1, 15, 16, 17, 31, 32, 33, 47, 63, 64, 65, 100, 129] * copies
    E, R, A, h, r, t = _grouped(sizes, dim, dim)
    B, bound = r.numel(), 2.0 ** -24 * (4 + dim ** 0.5)
    x = (E[h] - E[t]).double()
    want, size = torch.empty_like(x), torch.empty_like(x)
    head, tail = E[h].double(), E[t].double()
    proj, psize = torch.empty_like(x), torch.empty_like(x)
    back = torch.empty_like(x)
    for u in range(len(sizes)):
        m = r == u
        M = A[u].double()
        want[m], size[m] = x[m] @ M + R[u].double(), x[m].abs() @ M.abs() + R[u].abs().double()
        proj[m], psize[m] = head[m] @ M, head[m].abs() @ M.abs()
        back[m] = tail[m] @ M.t().contiguous()
    score = kge.transR(B, dim, 700, E, h, t, len(sizes), A, r, R)
    err = (score.double() - want).abs() / size
    assert bool((err <= bound).all()), float(err.max() / bound)
    m = KGEModel("RESCAL", E, None, A)
    fw = m.score(h, r, t)
    err = (fw.pos.double() - (proj * tail).sum(1)).abs() / (psize * tail.abs()).sum(1)
    assert bool((err <= 2 * bound).all()), float(err.max() / bound)  # (two sums of dim terms, one after the other)
    g = m.backward(fw, torch.ones(B, device="cuda"))
    rows = torch.zeros(700, dim, dtype=torch.float64, device="cuda").index_add_(0, h, back).index_add_(0, t, proj)
    rows = rows[g.ent_ids]
    assert bool(((g.ent_rows.double() - rows).norm(dim=1) <= 1e-6 * rows.norm(dim=1)).all())


def test_grouped_infinities_and_nans_as_fp32_has_them():
    from cuke_amd import kge
    E, R, A, h, r, t = _grouped([70, 33, 40] * 100, 128, 1, scale=1.0)
    E[3, 5], E[4, 6], A[0, 9, 17], A[1, 100, 3], A[200, 127, 127], E[8, 0] = float("inf"), float("nan"), -float("inf"), float("inf"), 3.4e38, 0.0
    h[:4], t[:4] = 3, torch.tensor([4, 5, 3, 6], device="cuda")
    got = kge.transR(r.numel(), 128, 700, E, h, t, 300, A, r, R).cpu()
    x, want, size = (E[h] - E[t]).cpu(), torch.empty(r.numel(), 128), torch.empty(r.numel(), 128, dtype=torch.float64)
    for u in range(300):
        m = (r == u).cpu()
        want[m] = (x[m][:, :, None] * A[u].cpu()).sum(1) + R[u].cpu()
        size[m] = (x[m][:, :, None].double() * A[u].cpu().double()).abs().sum(1) + R[u].cpu().abs().double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    # both sides round: 2 (4 + sqrt(128)) half ulps of the terms' total
    assert bool(((got.double() - want.double()).abs() <= 2.0 ** -23 * (4 + 128 ** 0.5) * size)[fine].all())


@pytest.mark.parametrize("model", ["DistMult", "ComplEx", "TransF"])
def test_a_step_whose_split_tiles_host_the_inspection(model):
    """(65536 ids beside 384 tiles: the riding form gives the bits of the inspection beside the step, and of a call without workspace's
    general tiles within rounding)"""
    import ctypes as C
    from cuke_amd import _lib
    from cuke_amd.kge import TrainStep
    E, R, h, r, t, neg = _case(model, 5000, 96, 8192, 768, 64, 7)
    st = TrainStep(KGEModel(model, E, R), h, r, t, neg, 128, loss="margin", sign=1.0)
    assert st.fusable
    outs = []
    for fused in (True, False):
        st.run(fused=fused)
        g = st.sparse_grads()
        outs.append([x.clone() for x in (st.pos, st.neg, st.loss, g.ent_ids, g.ent_rows, g.rel_rows)])
    assert all(torch.equal(x, y) for x, y in zip(*outs))
    neg2, side = torch.empty_like(st.neg), torch.empty(8192, device="cuda")
    p = lambda x: C.c_void_p(x.data_ptr())
    assert _lib.lib().kge_score_fwd(C.byref(st.m._tab), C.byref(st.bat), p(st.pos), p(neg2), p(side) if model == "TransF" else None, None, None, None, 0,
                                    C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert not torch.equal(neg2, st.neg) and torch.allclose(neg2, st.neg, rtol=1e-5, atol=1e-5 * float(st.neg.std()))
