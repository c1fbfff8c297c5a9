"""What users have this library do, as cases that can be timed and compared.

Four ways of using it, named by a case's ``kind``:

  call   the positional score functions ``transE`` ... ``RESCAL`` on a batch of triples (the reference's surface)
  loop   a training loop over the eager surface: sampler -> score -> margin loss -> backward -> row-wise Adagrad
  step   a preallocated ``TrainStep`` plus the optimizer steps: what a loop that cares about its speed runs
  eval   link prediction: every entity of the table scored as a candidate for a batch of queries, forward only

Tables are N(0, 0.05) fp32 (TransH normals of unit length, RotatE phases uniform), ids Zipf or uniform as in
``cuke_amd.synth``; everything is drawn on the GPU from the seed.
"""
from __future__ import annotations

import math

import torch

from cuke_amd import kge
from cuke_amd.data import TrainSampler
from cuke_amd.kge import KGEModel, TrainStep, margin_loss, sparse_adagrad, sparse_adagrad_factored

LR = 0.05
CALLS = ("TransE", "TransH", "TransR", "TransF", "RESCAL")
PROJECTED = ("TransR", "RESCAL")           # one dim x dim matrix per relation
HIGHER_IS_BETTER = ("DistMult", "ComplEx", "RotatE", "TransF", "RESCAL")
# flop per pair and element of the row: multiply-add; difference, square, sum; two multiply-adds more for the
# hyperplane; complex difference and modulus (per complex element, half as many as the row has floats)
PAIR_FLOPS = {"DistMult": 2, "ComplEx": 2, "TransF": 2, "RESCAL": 2, "TransE": 3, "TransR": 3, "TransH": 6, "RotatE": 3.5}


def _case(name, kind, model, batch, dim, n_ent, n_rel, chunk=0, n_neg=0, norm_p=2, mode="tail", ent_zipf=0.0, rel_zipf=0.0,
          index="int64"):
    c = dict(kind=kind, model=model, batch=batch, dim=dim, n_ent=n_ent, n_rel=n_rel, chunk=chunk, n_neg=n_neg,
             norm_p=norm_p, mode=mode, ent_zipf=ent_zipf, rel_zipf=rel_zipf, index=index)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The reference's smallest score call: a kilotriple of TransE, where the call itself is what costs.
        _case("call_transe_1024x128", "call", "TransE", 1024, 128, 16384, 1024),
        # The reference's sweep of the projection models: batch 4096 / 8192, width 512 / 1024.
        _case("call_transr_4096x512", "call", "TransR", 4096, 512, 14541, 237, rel_zipf=1.0),
        _case("call_rescal_8192x1024", "call", "RESCAL", 8192, 1024, 40943, 51, rel_zipf=1.0),
        # A first experiment: small batches, row width 50, both sides corrupted in turn.  Host work and launches.
        _case("loop_transe_l1_500x50", "loop", "TransE", 500, 50, 14951, 1345, chunk=100, n_neg=25, norm_p=1, mode="both",
              rel_zipf=1.0),
        # The usual experiment on a benchmark graph, through the eager surface; 32-bit ids as data loaders hand them out.
        _case("loop_complex_1024x200", "loop", "ComplEx", 1024, 200, 14951, 1345, chunk=128, n_neg=128, mode="both",
              ent_zipf=0.8, rel_zipf=1.0, index="int32"),
        # The benchmark's shared-negative step over a million entities.
        _case("step_distmult_4096x256", "step", "DistMult", 4096, 256, 1_000_000, 2000, chunk=256, n_neg=256, ent_zipf=1.1),
        # The benchmark's projection step: triples with upstream gradients of their own, most relations seen once or twice.
        _case("step_transr_8192x200", "step", "TransR", 8192, 200, 40000, 1345, rel_zipf=1.2),
        # Wide complex rows, a small batch, few relations, margin loss.
        _case("step_rotate_1024x1000", "step", "RotatE", 1024, 1000, 40943, 11, chunk=256, n_neg=256, ent_zipf=1.1),
        # TransR against shared negatives, heads corrupted.
        _case("step_transr_neg_4096x200", "step", "TransR", 4096, 200, 14951, 1345, chunk=512, n_neg=64, mode="head", rel_zipf=1.2),
        # A large batch: more ids than the small-set inspector takes; a width that is no multiple of the tiles.
        _case("step_transe_30000x150", "step", "TransE", 30000, 150, 1_000_000, 2000, chunk=600, n_neg=200, ent_zipf=1.1,
              rel_zipf=1.0),
        # Link prediction over a whole benchmark graph.
        _case("eval_complex_512x400", "eval", "ComplEx", 512, 400, 14951, 1345),
        # The largest: sixteen million pair scores and their gradients over a 6.4 GB table.
        _case("step_transh_l1_16384x400", "step", "TransH", 16384, 400, 4_000_000, 10000, chunk=1024, n_neg=1024, norm_p=1,
              ent_zipf=1.05),
    ]


# ---- drawn cases -----------------------------------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi, model):
    d = _log(rng, lo, hi)
    if rng.random() < 0.75:                # most people take a round width
        d = max(lo, d // 4 * 4)
    return max(2, d // 2 * 2) if model in ("ComplEx", "RotatE") else d


def draw(rng):
    while True:
        kind = rng.choice(["call", "loop", "step", "step", "eval"])
        mode = "tail"
        chunk = n_neg = 0
        norm_p = rng.choice([1, 2])
        n_rel = _log(rng, 10, 2000)
        if kind == "call":
            model = rng.choice(CALLS)
            batch, dim = _log(rng, 256, 8192), _dim(rng, 32, 1024, model)
            n_ent = _log(rng, 10_000, 100_000)
            norm_p = 2
        elif kind == "eval":
            model = rng.choice(["TransE", "DistMult", "ComplEx", "RotatE", "TransF"])
            batch, dim, n_ent = _log(rng, 64, 1024), _dim(rng, 48, 500, model), _log(rng, 5000, 50_000)
        else:
            model = rng.choice(["TransE", "TransH", "DistMult", "ComplEx", "RotatE", "TransF", "TransR", "RESCAL"])
            dim = _dim(rng, 48, 256, model) if model in PROJECTED else _dim(rng, 48, 1000, model)
            if model in PROJECTED and kind == "step" and rng.random() < 0.5:
                batch = _log(rng, 512, 8192)
            else:
                chunk, n_neg = _log(rng, 16, 1024), _log(rng, 16, 1024 if model not in PROJECTED else 64)
                if model in PROJECTED:
                    dim = dim // 4 * 4     # (a TrainStep takes TransR's negatives in this form only)
                batch = chunk * max(1, _log(rng, 256, 16384 if model not in PROJECTED else 4096) // chunk)
            mode = rng.choice(["tail", "head"]) if kind == "step" else rng.choice(["tail", "head", "both"])
            n_ent = _log(rng, 5000, 50_000) if kind == "loop" else _log(rng, 10_000, 1_000_000)
        c = _case(None, kind, model, batch, dim, n_ent, n_rel, chunk, n_neg, norm_p, mode,
                  ent_zipf=rng.choice([0.0, 0.8, 1.1]), rel_zipf=rng.choice([0.0, 1.0, 1.2]),
                  index=rng.choice(["int64", "int64", "int32"]) if kind in ("loop", "eval") else "int64")
        if kind != "call" and not n_neg and kind != "eval":
            c["mode"] = "tail"
        floats = n_ent * dim + (n_rel * dim * dim if model in PROJECTED else 0)
        if chunk and batch // chunk * n_neg * dim > 40_000_000:
            continue
        if floats <= 400_000_000 and _pairs(c) * c["dim"] * PAIR_FLOPS[model] <= 1.2e10:
            return c


# ---- inputs ----------------------------------------------------------------------------------------
def _dev():
    return torch.device("cuda:0")


def _ids(g, n_rows, count, zipf):
    if not zipf:
        return torch.randint(0, n_rows, (count,), generator=g, device=_dev(), dtype=torch.int64)
    cdf = torch.arange(1, n_rows + 1, device=_dev(), dtype=torch.float64).pow_(-zipf).cumsum_(0)
    u = torch.rand(count, generator=g, device=_dev(), dtype=torch.float64) * cdf[-1]
    rank = torch.searchsorted(cdf, u).clamp_(max=n_rows - 1)
    return torch.randperm(n_rows, generator=g, device=_dev())[rank]


def _tables(case, g):
    f32 = dict(generator=g, device=_dev(), dtype=torch.float32)
    model, dim, n_rel = case["model"], case["dim"], case["n_rel"]
    E = torch.randn((case["n_ent"], dim), **f32).mul_(0.05)
    R = A = None
    if model == "RotatE":
        R = torch.rand((n_rel, dim // 2), **f32).mul_(2 * math.pi).sub_(math.pi)
    elif model != "RESCAL":
        R = torch.randn((n_rel, dim), **f32).mul_(0.05)
    if model == "TransH":
        A = torch.nn.functional.normalize(torch.randn((n_rel, dim), **f32), dim=1)
    elif model in PROJECTED:
        A = torch.randn((n_rel, dim, dim), **f32).mul_(0.05)
    return E, R, A


class _State:
    pass


def prepare(case, seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed))
    s = _State()
    s.case = case
    s.E, s.R, s.A = _tables(case, g)
    B, n_ent, n_rel = case["batch"], case["n_ent"], case["n_rel"]
    kind, model = case["kind"], case["model"]
    if kind == "loop":
        n = max(50_000, 4 * B)             # training triples of a small benchmark graph, in host memory as a reader leaves them
        triples = tuple(_ids(g, rows, n, z).cpu().numpy() for rows, z in
                        ((n_ent, case["ent_zipf"]), (n_rel, case["rel_zipf"]), (n_ent, case["ent_zipf"])))
        s.sampler = TrainSampler(triples, n_ent, B, case["n_neg"], case["chunk"], seed=int(seed), device=_dev(), mode=case["mode"])
    else:
        s.h, s.t = _ids(g, n_ent, B, case["ent_zipf"]), _ids(g, n_ent, B, case["ent_zipf"])
        s.r = _ids(g, n_rel, B, case["rel_zipf"])
    if kind == "call":
        return s
    gamma = 12.0 if model == "RotatE" else 0.0
    s.model = KGEModel(model, s.E, s.R, s.A, norm_p=case["norm_p"], gamma=gamma)
    s.sign = 1.0 if model in HIGHER_IS_BETTER else -1.0
    if kind == "eval":
        s.neg = torch.arange(n_ent, device=_dev(), dtype=torch.int64)
        if case["index"] == "int32":
            s.h, s.r, s.t, s.neg = (x.to(torch.int32) for x in (s.h, s.r, s.t, s.neg))
        return s
    zeros = dict(device=_dev(), dtype=torch.float32)
    s.sE = torch.zeros(n_ent, **zeros)
    s.sR = torch.zeros(n_rel, **zeros) if s.R is not None else None
    s.sA = torch.zeros(n_rel, **zeros) if s.A is not None else None
    if kind == "step":
        if case["n_neg"]:
            s.neg = _ids(g, n_ent, B // case["chunk"] * case["n_neg"], case["ent_zipf"])
            s.step = TrainStep(s.model, s.h, s.r, s.t, s.neg, case["chunk"], loss="margin", margin=1.0, sign=s.sign,
                               neg_mode=case["mode"])
        else:
            # every triple carries an upstream gradient (a label's), small groups' projection gradients stay factored
            up = torch.randn(B, generator=g, **zeros)
            s.step = TrainStep(s.model, s.h, s.r, s.t, dpos=up, factor_max=4 if case["dim"] % 4 == 0 else 0)
    return s


# ---- one pass --------------------------------------------------------------------------------------
def _call(s):
    c = s.case
    B, d, ne, nr = c["batch"], c["dim"], c["n_ent"], c["n_rel"]
    model = c["model"]
    if model == "TransE":
        return kge.transE(B, d, ne, s.E, s.h, s.t, nr, s.R, s.r)
    if model == "TransH":
        return kge.transH(B, d, ne, s.E, s.h, s.t, nr, s.R, s.r, s.A)
    if model == "TransR":
        return kge.transR(B, d, ne, s.E, s.h, s.t, nr, s.A, s.r, s.R)
    if model == "TransF":
        return kge.transF(B, d, ne, s.E, s.h, nr, s.R, s.r, s.t)
    return kge.RESCAL(B, d, ne, s.E, s.h, nr, s.A, s.r, s.t)


def _loop(s):
    h, r, t, neg = next(s.sampler)
    if s.case["index"] == "int32":         # (a caller's own 32-bit ids, as far as the score call sees)
        h, r, t, neg = (x.to(torch.int32) for x in (h, r, t, neg))
    fw = s.model.score(h, r, t, neg, s.case["chunk"], neg_mode=s.sampler.neg_mode)
    loss, dpos, dneg = margin_loss(fw.pos, fw.neg, 1.0, s.sign)
    g = s.model.backward(fw, dpos, dneg)
    sparse_adagrad(s.E, s.sE, fw.ent_insp, g.ent_rows, LR)
    if s.R is not None:
        sparse_adagrad(s.R, s.sR, fw.rel_insp, g.rel_rows, LR)
    if s.A is not None:
        A = s.A.view(s.A.shape[0], -1)
        sparse_adagrad(A, s.sA, fw.rel_insp, g.aux_rows, LR)
    return [x for x in (loss, fw.pos, fw.neg, s.E, s.R, s.A, s.sE, s.sR, s.sA) if x is not None]


def _step(s):
    st = s.step
    st.run()
    sparse_adagrad(s.E, s.sE, st.ent_insp, st.ent_rows, LR)
    if s.R is not None:
        sparse_adagrad(s.R, s.sR, st.rel_insp, st.rel_rows, LR)
    if st.factor_max:
        sparse_adagrad_factored(s.A, s.sA, st.sparse_grads(), LR)
    elif s.A is not None:
        sparse_adagrad(s.A.view(s.A.shape[0], -1), s.sA, st.rel_insp, st.aux_rows, LR)
    return [x for x in (st.loss, st.pos, st.neg, s.E, s.R, s.A, s.sE, s.sR, s.sA) if x is not None]


def run(state):
    kind = state.case["kind"]
    if kind == "call":
        return _call(state)
    if kind == "loop":
        return _loop(state)
    if kind == "step":
        return _step(state)
    fw = state.model.score(state.h, state.r, state.t, state.neg, state.case["batch"])
    return [fw.pos, fw.neg]


# ---- what a pass cannot do without -------------------------------------------------------------------
def _pairs(case):
    if case["kind"] == "eval":
        return case["batch"] * (1 + case["n_ent"])
    return case["batch"] * (1 + case["n_neg"])


def work(case):
    B, d, ne, nr, kind, model = (case[k] for k in ("batch", "dim", "n_ent", "n_rel", "kind", "model"))
    rd = {"RotatE": d // 2, "RESCAL": 0}.get(model, d)
    n_neg = B // case["chunk"] * case["n_neg"] if case["chunk"] else (ne if kind == "eval" else 0)
    width = 4 if case["index"] == "int32" else 8
    ent, rel = min(ne, 2 * B + n_neg), min(nr, B)
    aux = {"TransH": d, "TransR": d * d, "RESCAL": d * d}.get(model, 0)
    rows = 4 * (ent * d + rel * (rd + aux))                        # every distinct row once
    ids = width * (3 * B + n_neg)
    flops = PAIR_FLOPS[model] * _pairs(case) * d
    if model in PROJECTED:
        flops += 2 * B * d * d
        if model == "TransR":
            flops += 2 * min(n_neg, ne) * d * d
    if kind == "call":
        return {"bytes": rows + ids + 4 * B * (1 if model in ("TransF", "RESCAL") else d), "flops": flops}
    scores = 4 * _pairs(case)
    if kind == "eval":
        return {"bytes": rows + ids + scores, "flops": flops}
    states = 2 * 4 * (ent + rel * (1 if rd else 0) + rel * (1 if aux else 0))
    return {"bytes": 2 * rows + ids + scores + states, "flops": 3 * flops}


def tolerance(case):
    """fp32 throughout: 1e-5 for values that are one sum.  A training pass also holds decisions that rounding can
    turn -- a pair on the margin's edge, the sign of an L1 residual element within an ulp of zero -- and Adagrad
    scales every row's first update to the learning rate however small its gradient is, so there a few rows out of
    thousands may differ visibly: 1e-4 over an array and a fraction of the typical element in the worst place."""
    if case["kind"] in ("call", "eval"):
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 1e-4, "max": 0.2}
