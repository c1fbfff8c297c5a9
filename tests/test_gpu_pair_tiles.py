"""Gradient tiles that evaluate every pair once (TransE, RotatE, TransH L1): one, two and four phases, several tiles of negatives and ranges of
positives, their ragged edges, widths that end inside a quad, rows of one to three coefficients; head and tail negatives; the forms on
both sides of the rule; batches whose tiles take several launches, by the planes' bytes and by a workspace's."""
import ctypes as C

import pytest
import torch

import test_gpu_transe_distances

from cuke_amd import _lib, synth
from cuke_amd.kge import TrainStep
from helpers import assert_close, gpu_model
from test_gpu_backward import compare, run_both

pytestmark = pytest.mark.gpu

# (batch, chunk, negatives, dim); test_pair_plans.py holds them to reach every form
SHAPES = [
    (64, 64, 1, 16), (66, 33, 3, 20),          # coefficient rows of fewer than four
    (200, 200, 25, 50),                        # one tile, few negatives
    (340, 17, 33, 70), (256, 16, 129, 36), (512, 512, 130, 66),  # four phases, a last tile of one or two; ranges of positives that end inside a step
    (2048, 1024, 128, 8),                      # many ranges
    (514, 257, 300, 264), (4096, 64, 257, 130),  # two phases
    (1000, 25, 250, 98), (320, 320, 256, 702),  # one phase and two tiles: TransE L1 and TransH; all
]


@pytest.mark.parametrize("mode", ["tail", "head"])
@pytest.mark.parametrize("model,p", [("RotatE", 2), ("TransE", 1), ("TransE", 2), ("TransH", 1)])
@pytest.mark.parametrize("batch,chunk,n_neg,dim", SHAPES)
def test_gradients(oracle, model, p, batch, chunk, n_neg, dim, mode):
    # (L1: lattice tables, where every residual is exact and no sign is ambiguous)
    w = synth.custom_workload(model, n_ent=500, n_rel=7, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, norm_p=p, sigma=0.2, gamma=4.0,
                              ent_zipf=0.8, seed=dim + n_neg, lattice=(p == 1))
    if model == "RotatE":  # (unit vectors of residuals a thousand times smaller than their operands, where the 32-bit oracle leaves the bar)
        return compare_64(w, mode, f"{batch}x{n_neg}x{dim} {mode}")
    g, ref = run_both(oracle, w, seed=2, neg_mode=mode, fast=True)
    compare(g, ref, f"{model} L{p} {batch}x{n_neg}x{dim} {mode}")


@pytest.mark.parametrize("dim", [5, 34, 65, 96, 97, 150])
@pytest.mark.parametrize("mode", ["tail", "head"])
def test_last_column_tile_of_the_64_bit_products(dim, mode):
    """One to 32 columns left over (and 33, where the whole tile takes them)."""
    test_gpu_transe_distances.test_gradients_of_close_rows(8192, 256, 200, dim, "matrix_cores", "offset 0.25", mode)


def in_64_bits(w, rotated, dpos, dneg, mode, block):
    """Dense gradients of a workload's entity, relation and normal tables: scores in 64 bits on the GPU, a block of negatives of a chunk at a
    time, differentiated by autograd.  rotated: RotatE's rows h e^{i theta} (t e^{-i theta}) rounded to fp32, as the pair differences take them."""
    a, dev = w.arrays, torch.device("cuda:0")
    E, R, A = tabs = [torch.from_numpy(a[k]).to(dev).double().requires_grad_() if a[k] is not None and a[k].size else None for k in ("E", "R", "A")]
    h, r, t, neg = (torch.from_numpy(a[k]).to(dev) for k in ("h", "r", "t", "neg"))
    half = E.shape[1] // 2

    def turn(x, theta):
        c, s = torch.cos(theta), torch.sin(theta)
        return torch.cat((x[..., :half] * c - x[..., half:] * s, x[..., :half] * s + x[..., half:] * c), -1)

    def score(x, rel, y):
        if w.model == "RotatE":  # (x: turned)
            u = x - y
            return w.gamma - torch.sqrt(u[..., :half] ** 2 + u[..., half:] ** 2).sum(-1)
        u = x - y + R[rel]
        if w.model == "TransH":
            u = u - ((x - y) * A[rel]).sum(-1, keepdim=True) * A[rel]
        return u.abs().sum(-1) if w.norm_p == 1 else (u * u).sum(-1).sqrt()

    (score(turn(E[h], R[r]) if w.model == "RotatE" else E[h], r, E[t]) * dpos).sum().backward()
    C, N, tail = w.chunk, w.n_neg, mode == "tail"
    for c in range(w.batch // C):
        b = slice(c * C, (c + 1) * C)
        for k0 in range(0, N, block):
            other = E[neg[c * N + k0:c * N + min(k0 + block, N)]][None]
            kept = E[(h if tail else t)[b]]
            if w.model == "RotatE":
                kept = turn(kept, R[r[b]] if tail else -R[r[b]])
                kept = kept + (rotated[b].double() - kept).detach()
            kept, rel = kept[:, None], r[b][:, None]
            s = score(kept, rel, other) if tail or w.model == "RotatE" else score(other, rel, kept)
            (s * dneg[b, k0:k0 + block]).sum().backward()
    return [x.grad if x is not None else None for x in tabs]


def compare_64(w, mode, what, block=1024, global_floor=0.0):
    m, ix = gpu_model(w)
    gen = torch.Generator("cuda:0").manual_seed(2)
    dpos, dneg = (torch.randn(n, device="cuda:0", generator=gen) for n in (w.batch, (w.batch, w.n_neg)))
    fw = m.score(ix["h"], ix["r"], ix["t"], ix["neg"], w.chunk, neg_mode=mode)
    g = m.backward(fw, dpos, dneg)
    want = in_64_bits(w, fw.residual, dpos.double(), dneg.double(), mode, block)
    for name, ids, rows, ref in (("entity", g.ent_ids, g.ent_rows, want[0]), ("relation", g.rel_ids, g.rel_rows, want[1]),
                                 ("normal", g.rel_ids, g.aux_rows, want[2])):
        if rows is not None:
            assert_close(rows.cpu().numpy(), ref[ids.long()].cpu().numpy(), what=f"{what} {name} rows", rows=True,
                         global_floor=global_floor)


@pytest.mark.parametrize("model,p", [("RotatE", 2), ("TransE", 1), ("TransH", 1)])
def test_many_negatives_take_several_launches(model, p):
    """Planes of the positives' sums, one per tile of negatives, of more bytes than a batch may have: the tiles' launches add to each other's."""
    w = synth.custom_workload(model, n_ent=30000, n_rel=7, dim=1000, batch=1100, chunk=1100, n_neg=20500, norm_p=p, sigma=0.2, gamma=4.0,
                              seed=3, lattice=(p == 1))
    compare_64(w, "tail", f"{model} L{p}", block=128)


@pytest.mark.parametrize("mode", ["tail", "head"])
@pytest.mark.parametrize("model,p", [("RotatE", 2), ("TransE", 1), ("TransE", 2), ("TransH", 1)])
@pytest.mark.parametrize("batch,chunk,n_neg,dim", [(600, 300, 450, 70), (200, 200, 350, 50), (1600, 400, 700, 264)])  # (two, four and one phase)
def test_a_smaller_workspace(model, p, batch, chunk, n_neg, dim, mode):
    """A workspace queried for a larger batch of the same chunks may hold fewer planes than this batch would take, down to one of either side:
    the gradients are the same sums, and nothing past its end is written.  Less than that is refused."""
    from cuke_amd._lib import KgeError
    w = synth.custom_workload(model, n_ent=500, n_rel=7, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, norm_p=p, sigma=0.2, gamma=4.0,
                              ent_zipf=0.8, seed=dim, lattice=(p == 1))
    m, ix = gpu_model(w)
    st = TrainStep(m, ix["h"], ix["r"], ix["t"], ix["neg"], chunk, neg_mode=mode, dpos=torch.randn(batch, device="cuda:0"),
                   dneg=torch.randn((batch, n_neg), device="cuda:0"))
    st.run()
    want = in_64_bits(w, st.residual, st.dpos.double(), st.dneg.double(), mode, 1024)
    like = _lib.Tables.from_buffer_copy(m._tab)  # the same rows without planes: dot products, or TransH's L2 tiles
    like.model, like.norm_p = (m._tab.model, 2) if model == "TransH" else (_lib.MODELS["DistMult"], 2)
    one, full = int(_lib.lib().kge_score_bwd_workspace(C.byref(like), C.byref(st.bat))), st._ws_b_bytes
    plane = 4 * batch * dim
    assert full > one + 3 * plane or model == "TransE" and p == 2
    for size in sorted({one, one + plane + 1000, one + 2 * plane + 1000, one + 3 * plane + 1000, full - 1, full}):
        if not one <= size <= full:
            continue
        room = torch.full((size + 4096,), 0x7f, dtype=torch.uint8, device="cuda:0")
        st._ws_b, st._ws_b_bytes = room, size
        for x in (st.ent_rows, st.rel_rows, st.aux_rows):
            if x is not None:
                x.fill_(float("nan"))
        for fused in (None, False):
            st.run(fused=fused)
            g = st.sparse_grads()
            for name, ids, rows, ref in (("entity", g.ent_ids, g.ent_rows, want[0]), ("relation", g.rel_ids, g.rel_rows, want[1]),
                                         ("normal", g.rel_ids, g.aux_rows, want[2])):
                if rows is not None:
                    assert_close(rows.cpu().numpy(), ref[ids.long()].cpu().numpy(), what=f"{model} {size - one} bytes of planes, {name} rows", rows=True)
            assert (room[size:] == 0x7f).all()
    st._ws_b_bytes = one - 1
    with pytest.raises(KgeError):
        st.run()


@pytest.mark.parametrize("mode", ["tail", "head"])
@pytest.mark.parametrize("dim", [2, 4, 6])
@pytest.mark.parametrize("batch,chunk,n_neg", [(8192, 16, 5), (2048, 8, 4), (130, 65, 33)])  # 64, 32 and 16 owners
def test_rotate_rows_of_less_than_a_quad(batch, chunk, n_neg, dim, mode):
    """These have no pair tiles."""
    w = synth.custom_workload("RotatE", n_ent=4000, n_rel=7, dim=dim, batch=batch, chunk=chunk, n_neg=n_neg, sigma=0.2, gamma=4.0, seed=dim)
    # (rows of two to six floats, each the sum of a few unit vectors that may nearly cancel: a tenth of the array's scale)
    compare_64(w, mode, f"{batch}x{n_neg}x{dim} {mode}", global_floor=0.1)
