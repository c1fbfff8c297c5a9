"""The native host path: what it takes gives the results of the general path, and what it does not take falls
through to it (other integer widths, non-contiguous inputs, host-side batches)."""
import gc

import numpy as np
import pytest
import torch

from cuke_amd import synth
from helpers import gpu_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,kw", [("ComplEx", dict(chunk=32, n_neg=17)), ("TransH", dict(chunk=64, n_neg=8, norm_p=1)),
                                      ("TransR", dict(chunk=32, n_neg=5)), ("TransR", dict()), ("RESCAL", dict(chunk=128, n_neg=3))])
def test_narrow_ids_and_strided_inputs_give_the_same_bits(model, kw):
    w = synth.custom_workload(model, n_ent=200, n_rel=9, dim=24, batch=128, sigma=0.3, seed=4, **kw)
    m, ix = gpu_model(w)
    forms = [ix, {k: v.to(torch.int32) for k, v in ix.items()},
             {k: torch.stack((v, v), 1)[:, 0] for k, v in ix.items()}]  # the last one is not contiguous
    dpos = torch.randn(w.batch, device="cuda")
    dneg = torch.randn((w.batch, w.n_neg), device="cuda") if w.chunk else None
    out = []
    for f in forms:
        fw = m.score(f["h"], f["r"], f["t"], f.get("neg"), w.chunk or None)
        g = m.backward(fw, dpos, dneg)
        assert g.ent_rows.shape[0] == g.ent_ids.numel() == fw.ent_insp.num_unique == int(fw.ent_insp.num_unique_dev.item())
        ei = fw.ent_insp
        assert int(ei.offsets()[-1]) == ei.n and torch.equal(ei.inverse[ei.perm.long()], ei.sorted_seg)
        out.append([x for x in (fw.pos, fw.neg, g.ent_ids, g.ent_rows, g.rel_ids, g.rel_rows, g.aux_rows) if x is not None])
    # (the third form goes through the general path where it is not contiguous and through the native one after that)
    for other in out[1:]:
        assert len(other) == len(out[0]) and all(torch.equal(x, y) for x, y in zip(out[0], other))


def test_sampler_equals_the_host_batches_over_epochs(oracle):
    from cuke_amd.data import TrainSampler
    rng = np.random.default_rng(3)
    triples = tuple(rng.integers(0, n, 103) for n in (50, 7, 50))
    kw = dict(n_entities=50, batch_size=20, neg_sample_size=3, neg_chunk_size=5, seed=9, mode="both")
    a, b = TrainSampler(triples, **kw), TrainSampler(triples, **kw)
    b._dev_index = torch.cuda.device_count()  # (not the current device: the native path declines)
    for step in range(13):  # five batches an epoch
        x, y = next(a), next(b)
        assert a.neg_mode == b.neg_mode
        assert all(torch.equal(p, q) and p.dtype == torch.int64 for p, q in zip(x, y)), step


def test_train_step_in_one_call_equals_the_call_by_call_issue():
    from cuke_amd.kge import TrainStep
    for model, kw in (("DistMult", dict(chunk=64, n_neg=32)), ("TransR", dict()), ("TransR", dict(chunk=32, n_neg=8))):
        w = synth.custom_workload(model, n_ent=400, n_rel=12, dim=48, batch=256, sigma=0.2, rel_zipf=1.1, seed=20, **kw)
        m, ix = gpu_model(w)
        loss = dict(loss="margin") if w.chunk else {}
        st = TrainStep(m, ix["h"], ix["r"], ix["t"], ix.get("neg"), w.chunk or None, **loss)

        def outputs():
            g = st.sparse_grads()
            return [x.clone() for x in (st.pos, st.neg, st.loss, g.ent_ids, g.ent_rows, g.rel_rows, g.aux_rows) if x is not None]

        _one_call_step(st, fused=int(st.fusable))
        one = outputs()
        st.run()
        assert all(torch.equal(x, y) for x, y in zip(one, outputs())), model
        if st.fusable:
            st.run(fused=False)
            assert all(torch.equal(x, y) for x, y in zip(one, outputs())), model


@pytest.mark.parametrize("dim", [4096, 4100, 4 * 1024 * 4 + 4, 40000, 65536, 65540, 100004])
@pytest.mark.parametrize("opt", ["sgd", "adagrad"])
def test_optimizer_rows_of_thousands_of_floats(oracle, dim, opt):
    """A workgroup per row: widths on both sides of the register-resident variants' edges."""
    from cuke_amd.kge import inspect, sparse_adagrad, sparse_sgd
    from helpers import assert_close
    rng = np.random.default_rng(dim)
    table, state = rng.standard_normal((9, dim)).astype(np.float32), rng.random(9).astype(np.float32)
    ids = np.array([7, 2, 2, 5, 0, 7], dtype=np.int64)
    rows = rng.standard_normal((6, dim)).astype(np.float32)
    ins = inspect(torch.from_numpy(ids).cuda(), 9)
    t, s, g = torch.from_numpy(table).cuda(), torch.from_numpy(state).cuda(), torch.from_numpy(rows).cuda()
    u = ins.ids().cpu().numpy()
    if opt == "sgd":
        sparse_sgd(t, ins, g, 0.1)
        assert_close(t.cpu().numpy(), oracle.sparse_sgd(table, u, rows[:len(u)], 0.1), what="table")
    else:
        sparse_adagrad(t, s, ins, g, 0.1)
        wt, ws = oracle.sparse_adagrad(table, state, u, rows[:len(u)], 0.1)
        assert_close(t.cpu().numpy(), wt, what="table")
        assert_close(s.cpu().numpy(), ws, what="state")


@pytest.mark.parametrize("capacity", [3, (1 << 22) - 1, 1 << 22, 5_000_000])
def test_optimizer_rows_of_thousands_of_floats_in_arrays_of_millions(capacity):
    """The row array's capacity (rows past the distinct ids are not read) on both sides of what a workgroup per row can launch."""
    import ctypes as C
    from cuke_amd import _lib
    dim = 4096
    table, state, rows = torch.ones(5, dim, device="cuda"), torch.zeros(5, device="cuda"), torch.full((3, dim), 2.0, device="cuda")
    ids, count = torch.tensor([0, 2, 3], device="cuda"), torch.tensor([3], dtype=torch.int32, device="cuda")
    p = lambda x: C.c_void_p(x.data_ptr())
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert _lib.lib().kge_sparse_sgd(p(table), dim, p(ids), p(count), capacity, p(rows), 0.25, st) == 0
    want = torch.ones(5, dim, device="cuda")
    want[ids] = 0.5
    assert torch.equal(table, want)
    assert _lib.lib().kge_sparse_adagrad(p(table), p(state), dim, p(ids), p(count), capacity, p(rows), 0.25, 0.0, st) == 0
    want[ids] = 0.25  # state 4, a step of 0.25 * 2 / 2
    assert torch.equal(state, torch.tensor([4.0, 0, 4, 4, 0], device="cuda")) and torch.equal(table, want)


def test_adagrad_without_a_state_raises_and_updates_nothing():
    """(it is not SGD)"""
    from cuke_amd.kge import inspect, sparse_adagrad
    table, rows = torch.ones(5, 8, device="cuda"), torch.ones(2, 8, device="cuda")
    insp = inspect(torch.tensor([3, 1], device="cuda"), 5)
    with pytest.raises(TypeError):
        sparse_adagrad(table, None, insp, rows, 0.1)
    assert torch.equal(table, torch.ones_like(table))


def test_optimizer_steps_without_an_inspection_raise_and_update_nothing():
    """Forward.ent_insp / rel_insp are None until backward() has run: an easy mistake that must not end the process."""
    from cuke_amd.kge import sparse_adagrad, sparse_sgd
    table, rows, state = torch.ones(5, 8, device="cuda"), torch.ones(2, 8, device="cuda"), torch.zeros(5, device="cuda")
    with pytest.raises(TypeError):
        sparse_adagrad(table, state, None, rows, 0.1)
    with pytest.raises(TypeError):
        sparse_sgd(table, None, rows, 0.1)
    assert torch.equal(table, torch.ones_like(table)) and not state.any()


def _hip():
    """The HIP runtime this process runs on (torch may carry its own copy: never load a second one)."""
    import ctypes
    for line in open("/proc/self/maps"):
        path = line.split()[-1]
        if "libamdhip64" in path:
            return ctypes.CDLL(path)
    raise AssertionError("no HIP runtime in the process")


def _one_call_step(st, fused):
    import ctypes as C
    batches, buf = st._native_state()
    assert st.L.kge_train_step(C.byref(st.m._tab), C.byref(batches[0]), C.byref(buf), fused,
                               C.c_void_p(torch.cuda.current_stream().cuda_stream), C.c_void_p(st.side.cuda_stream)) == 0


def test_one_call_step_inspects_the_entities_beside_the_relations():
    """fused == 0, TransR: the entity inspection depends on what came before the step, not on the relation inspection
    in front of the forward pass.  Captured, the step then starts with two nodes that wait for nothing."""
    import ctypes as C
    from cuke_amd.kge import TrainStep
    w = synth.custom_workload("TransR", n_ent=400, n_rel=12, dim=48, batch=256, chunk=32, n_neg=8, sigma=0.2, seed=20)
    m, ix = gpu_model(w)
    st = TrainStep(m, ix["h"], ix["r"], ix["t"], ix["neg"], 32)

    _one_call_step(st, fused=0)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        _one_call_step(st, fused=0)
    n = C.c_size_t(0)
    assert _hip().hipGraphGetRootNodes(C.c_void_p(g.raw_cuda_graph()), None, C.byref(n)) == 0
    assert n.value == 2


def _two_batches(model, **kw):
    from cuke_amd.kge import TrainStep
    w = synth.custom_workload(model, n_ent=300, n_rel=9, dim=24, batch=128, sigma=0.3, seed=4, **kw)
    m, ix = gpu_model(w)
    b0 = [ix["h"], ix["r"], ix["t"], ix.get("neg")]
    b1 = [ix["t"].flip(0), ix["r"].flip(0), ix["h"].flip(0), ix["neg"].flip(0) if "neg" in ix else None]
    return m, (b0, b1), lambda b: TrainStep(m, *b, w.chunk or None)


def _step_outputs(st):
    torch.cuda.synchronize()
    g = st.sparse_grads()
    return [x.clone() for x in (st.pos, st.neg, g.ent_ids, g.rel_ids, g.ent_rows, g.rel_rows, g.aux_rows) if x is not None]


@pytest.mark.parametrize("model,kw", [("DistMult", dict(chunk=32, n_neg=8)), ("TransR", dict())])
def test_fresh_upstream_gradients_and_a_new_batch_between_staged_steps(model, kw, monkeypatch):
    """dpos bound anew for every step, and a batch added when another is staged: the steps follow them, what has been
    staged stays staged, and nothing waits for the device."""
    from helpers import assert_close
    m, batches, make = _two_batches(model, **kw)
    order, ups = [0, 1, 0, 1], [torch.randn(128, device="cuda") for _ in range(4)]
    want = []
    for b, up in zip(order, ups):
        ref = make(batches[b])
        ref.dpos = up
        ref.run()
        want.append(_step_outputs(ref))
    st = make(batches[0])
    sync, waits = torch.cuda.synchronize, []
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: waits.append(1))
    st.run_native(None, 0)
    assert st.add_batch(*batches[1]) == 1
    got = []
    for k, b in enumerate(order):
        st.dpos = ups[k].clone()
        st.run_native(b, order[k + 1] if k + 1 < len(order) else None)
        assert not waits
        sync()
        got.append(_step_outputs(st))
        waits.clear()
    for k in range(len(order)):
        for x, y in zip(got[k], want[k]):
            assert_close(x.cpu().numpy(), y.cpu().numpy(), what=f"step {k}", rows=x.dim() > 1)


@pytest.mark.parametrize("model,kw", [("DistMult", dict(chunk=32, n_neg=8)), ("TransR", dict())])
def test_forms_of_issue_follow_each_other(model, kw):
    """A step of one form, then new ids in the same tensors, then a step of another: the second waits for the first on
    both streams, however far the host is ahead."""
    m, batches, make = _two_batches(model, **kw)
    busy = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")

    def load(tensors, b):
        for x, y in zip(tensors, batches[b]):
            if x is not None:
                x.copy_(y)

    def native(st):
        st.run_native(None, 0), st.run_native(0, None)

    def staged(st):
        st.stage(batch=0), st.run(pipeline=True)

    forms = [lambda st: st.run(), native, staged]
    want = []
    for b in (0, 1):
        st = make(batches[b])
        st.run()
        want.append(_step_outputs(st))
    at = 1 if batches[0][3] is None else 2  # of the entity ids among the outputs
    n0 = want[0][at].numel()
    for first in forms:
        for second in forms:
            if first is second:
                continue
            mine = [x.clone() if x is not None else None for x in batches[0]]
            st = make(mine)
            for _ in range(20):  # (milliseconds of work in front of the steps)
                busy.zero_()
            first(st)
            pos, ids, rows = st.pos.clone(), st.ent_insp.unique_ids.clone(), st.ent_rows.clone()
            load(mine, 1)
            second(st)
            got = _step_outputs(st)
            assert torch.equal(pos, want[0][0]) and torch.equal(ids[:n0], want[0][at])
            assert torch.allclose(rows[:n0], want[0][at + 2], rtol=1e-4, atol=1e-6)
            assert torch.equal(got[0], want[1][0]) and torch.equal(got[at], want[1][at]) and torch.equal(got[at + 1], want[1][at + 1])
            assert torch.allclose(got[at + 2], want[1][at + 2], rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("fused", [0, 1])
def test_one_call_step_leaves_a_staged_batch_staged(fused):
    """TransR without negatives: staging plans the batch; a step that plans for itself in between does not undo that."""
    m, batches, make = _two_batches("TransR")
    st = make(batches[0])
    assert st.fusable
    st.run_native(None, 0)
    torch.cuda.synchronize()
    _one_call_step(st, fused)
    one = _step_outputs(st)
    st.run_native(0, None)
    assert all(torch.equal(x, y) for x, y in zip(one, _step_outputs(st)))


@pytest.mark.parametrize("fused", [0, 1])
@pytest.mark.parametrize("model,kw", [("DistMult", dict(chunk=32, n_neg=8)), ("RotatE", dict(chunk=64, n_neg=8)), ("TransH", dict(chunk=32, n_neg=8)),
                                      ("TransR", dict()), ("TransR", dict(chunk=32, n_neg=8)), ("RESCAL", dict(chunk=32, n_neg=8))])
def test_one_call_step_gives_the_results_of_run(model, kw, fused):
    m, batches, make = _two_batches(model, **kw)
    st, ref = make(batches[0]), make(batches[0])
    ref.run(fused=bool(fused) and ref.fusable)
    want = _step_outputs(ref)
    for _ in range(2):
        for x in (st.pos, st.ent_rows):
            x.fill_(7.0)
        _one_call_step(st, fused and st.fusable)
        assert all(torch.equal(x, y) for x, y in zip(_step_outputs(st), want))


def test_a_replaced_stage_is_called():
    """A loss of one's own, as a subclass or on the object."""
    from cuke_amd.kge import TrainStep
    m, batches, make = _two_batches("DistMult", chunk=32, n_neg=8)

    class Own(TrainStep):
        def loss_grad(self, st):
            self.dpos = 2.0 * self.pos

    a, b = Own(m, *batches[0], 32), make(batches[0])
    b.loss_grad = lambda st: setattr(b, "dpos", 2.0 * b.pos)
    ref = make(batches[0])
    ref.run()
    ref.dpos = 2.0 * ref.pos.clone()
    ref.run()
    for st in (a, b):
        st.run()
        assert all(torch.equal(x, y) for x, y in zip(_step_outputs(st), _step_outputs(ref)))


def test_gradients_of_a_step_keep_their_row_counts_past_the_next_run():
    """sparse_grads() does not wait, and what is read from it later has the counts of its own step: the views of one
    object never mix two steps (the rows themselves are overwritten)."""
    from cuke_amd.kge import sparse_adagrad_factored
    m, batches, make = _two_batches("TransR")
    mine = [x.clone() if x is not None else None for x in batches[0]]
    from cuke_amd.kge import TrainStep
    st = TrainStep(m, *mine, factor_max=4)
    state = torch.zeros(m.n_rel, device="cuda")
    st.run()
    want = [len(torch.unique(torch.cat((mine[0], mine[2])))), len(torch.unique(mine[1]))]
    torch.cuda.set_sync_debug_mode("error")
    try:
        read, later = st.sparse_grads(), st.sparse_grads()
        sparse_adagrad_factored(m.A, state, later, 0.0)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    assert read.ent_ids.numel() == want[0]
    mine[0].fill_(3), mine[2].fill_(5), mine[1].fill_(1)  # two entities, one relation
    st.run()
    assert st.sparse_grads().ent_ids.tolist() == [3, 5] and st.sparse_grads().rel_rows.shape[0] == 1
    for g in (read, later):
        assert [g.ent_ids.numel(), g.rel_ids.numel()] == want == [g.ent_rows.shape[0], g.rel_rows.shape[0]]
        assert g.aux_rows.shape[0] == want[1] and g.rel_seg_offsets.numel() == want[1] + 1


def _sampler(n=700, **kw):
    from cuke_amd.data import TrainSampler
    rng = np.random.default_rng(3)
    triples = [rng.integers(0, m, n) for m in (90, 7, 90)]
    kw = dict(dict(batch_size=128, neg_sample_size=5, neg_chunk_size=32, seed=11, mode="both"), **kw)
    return triples, TrainSampler(triples, 90, **kw)


@pytest.mark.parametrize("device", ["cuda:0", "cuda"])
@pytest.mark.parametrize("shuffle", [True, False])
def test_sampler_batches_are_the_host_arrays_in_the_epochs_order(device, shuffle):
    triples, s = _sampler(device=device, shuffle=shuffle)
    _, plain = _sampler(device=device, shuffle=shuffle)
    for step in range(13):  # five batches an epoch
        got = next(s)
        want = plain._host_batch(plain._next_ids(), 20)
        plain.step += 1
        assert all(torch.equal(x, y) and x.dtype == torch.int64 for x, y in zip(got, want)), step
        order = np.random.default_rng([11, step // 5]).permutation(700) if shuffle else np.arange(700)
        ids = order[step % 5 * 128:][:128]
        assert all(np.array_equal(x.cpu().numpy(), y[ids]) for x, y in zip(got, triples)), step


def test_sampler_reads_its_arrays_as_they_are_at_each_batch():
    """Changed in place, rebound, strided: the next batch has it.  An order that points outside raises."""
    triples, s = _sampler(shuffle=False)
    first = next(s)
    s.h[128:256] = 17
    assert (next(s)[0] == 17).all()
    s.t = np.arange(1400)[::2]
    assert torch.equal(next(s)[2], torch.arange(256, 384, device="cuda") * 2)
    s.r = np.arange(400)
    with pytest.raises(IndexError):
        next(s)
    assert torch.equal(first[0], torch.from_numpy(triples[0][:128]).cuda())


@pytest.mark.parametrize("batch", [1, 255, 256, 257, 64 * 256, 64 * 256 + 1, 50000])
def test_sampler_batches_of_every_size_reuse_their_pinned_memory(batch):
    """Around one id per thread, one workgroup, and one and two turns of the whole grid; three epochs of three batches."""
    import copy
    triples, s = _sampler(3 * batch, batch_size=batch, neg_chunk_size=batch, neg_sample_size=3)
    kept = [next(s) for _ in range(5)]
    again = copy.deepcopy(s)
    kept += [next(s) for _ in range(4)]
    for k, got in enumerate(kept):
        ids = np.random.default_rng([11, k // 3]).permutation(3 * batch)[k % 3 * batch:][:batch]
        assert all(np.array_equal(x.cpu().numpy(), y[ids]) for x, y in zip(got, triples)), k
    for k in range(5, 9):
        assert all(torch.equal(x, y) for x, y in zip(next(again), kept[k])), k


def test_batches_of_a_resident_triple_list():
    """kge_sample_batch, for hosts that keep the triples on the device."""
    import ctypes as C
    from cuke_amd import _lib
    rng = np.random.default_rng(5)
    cols = [torch.from_numpy(rng.integers(0, 50, 600)).cuda() for _ in range(3)]
    order = torch.from_numpy(rng.permutation(600)).cuda()
    h, r, t, neg, neg2 = (torch.empty(n, dtype=torch.int64, device="cuda") for n in (257, 257, 257, 300, 300))
    p = lambda x: C.c_void_p(x.data_ptr())
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert _lib.lib().kge_sample_batch(*map(p, cols), p(order), 257, p(h), p(r), p(t), p(neg), 300, 50, 9, 4, st) == 0
    assert _lib.lib().kge_sample_negatives(p(neg2), 300, 50, 9, 4, st) == 0
    assert all(torch.equal(x, c[order[:257]]) for x, c in zip((h, r, t), cols)) and torch.equal(neg, neg2)


def test_sampler_keeps_nothing_on_the_device_and_waits_for_nothing():
    """200 batches from three streams behind a busy device, the host far ahead: every batch is its own, the sampler holds no
    device memory, and neither a batch nor the end of an epoch (5 batches) synchronises."""
    triples, s = _sampler(shuffle=False)
    next(s), torch.cuda.synchronize()
    gc.collect()  # (tensors that an earlier test's frames hold in a cycle would otherwise go while the batches are drawn)
    before = torch.cuda.memory_allocated()
    busy = torch.empty(1 << 28, dtype=torch.uint8, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(3)]
    kept = []
    torch.cuda.set_sync_debug_mode("error")
    try:
        for k in range(1, 200):
            with torch.cuda.stream(streams[k % 3]):
                if k % 40 < 3:
                    busy.zero_()
                kept.append(next(s))
    finally:
        torch.cuda.set_sync_debug_mode("default")
    torch.cuda.synchronize()
    for k, got in enumerate(kept, 1):
        assert all(np.array_equal(x.cpu().numpy(), y[k % 5 * 128:][:128]) for x, y in zip(got, triples)), k
    del kept, got, busy
    assert torch.cuda.memory_allocated() == before


def test_numbers_are_converted_as_the_general_path_does():
    """Whatever int() / float() takes: a row count as a float, a margin or a rate as text or as a tensor."""
    from cuke_amd.kge import inspect, margin_loss, sparse_sgd
    ids = torch.tensor([4, 2, 4], device="cuda")
    ins = inspect(ids, 9.0)
    assert ins.n_rows == 9 and inspect(ids, np.int64(9)).ids().tolist() == ins.ids().tolist() == [2, 4]
    with pytest.raises((TypeError, ValueError)):
        inspect(ids, "many")
    pos, neg = torch.randn(8, device="cuda"), torch.randn(8, 4, device="cuda")
    want = margin_loss(pos, neg, 0.5, -1.0)
    for margin in ("0.5", torch.tensor(0.5), torch.tensor([0.5], device="cuda")):
        assert all(torch.equal(x, y) for x, y in zip(margin_loss(pos, neg, margin, "-1"), want))
    with pytest.raises((TypeError, ValueError)):
        margin_loss(pos, neg, None)
    table = torch.ones(9, 4, device="cuda")
    sparse_sgd(table, ins, torch.ones(3, 4, device="cuda"), "0.25")
    assert table[:, 0].tolist() == [1, 1, 0.75, 1, 0.75, 1, 1, 1, 1]


def test_empty_batches():
    """Positional calls, scores, losses and inspections of nothing."""
    from cuke_amd import kge
    E, R = torch.ones(9, 8, device="cuda"), torch.ones(4, 8, device="cuda")
    A = torch.ones(4, 8, 8, device="cuda")
    e = torch.zeros(0, dtype=torch.int64, device="cuda")
    assert kge.transE(0, 8, 9, E, e, e, 4, R, e).shape == (0, 8)
    assert kge.transR(0, 8, 0, E, e, e, 0, A, e, R).shape == (0, 8)
    assert kge.RESCAL(0, 8, 0, E, e, 0, A, e, e).shape == (0,)
    assert kge.inspect(e, 9).num_unique == 0
    loss, dpos, dneg = kge.margin_loss(torch.zeros(0, device="cuda"), torch.zeros(0, 5, device="cuda"), 1.0)
    assert loss.item() == 0.0 and dpos.shape == (0,) and dneg.shape == (0, 5)


@pytest.mark.parametrize("model,kw", [("DistMult", dict(chunk=32, n_neg=8)), ("TransR", dict())])
def test_a_staged_set_is_not_rewritten_before_what_follows_its_step(model, kw):
    """The ring of next_inputs(): index tensors refilled on a stream of their own, the next batches staged while the device is
    still busy behind a step; what the caller has put there (an optimizer step, say) reads that step's inspection."""
    m, batches, make = _two_batches(model, **kw)
    batches = batches[0], [x // 2 if x is not None and i != 1 else x for i, x in enumerate(batches[0])]  # (other entities)
    st, copies = make(batches[0]), torch.cuda.Stream()
    busy = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    want = [torch.unique(torch.cat([x for x in (b[0], b[2], b[3]) if x is not None])) for b in batches]
    read = []

    def stage(k):
        tensors = st.next_inputs(copies)
        with torch.cuda.stream(copies):
            for x, y in zip(tensors, batches[k % 2]):
                if x is not None:
                    x.copy_(y)
            ready = copies.record_event()
        st.stage(ready)

    stage(0)
    for k in range(6):
        stage(k + 1)
        st.run(pipeline=True)
        for _ in range(10):  # (milliseconds)
            busy.zero_()
        read.append((st.ent_insp.unique_ids.clone(), st.ent_insp.num_unique_dev.clone()))
    torch.cuda.synchronize()
    for k, (ids, n) in enumerate(read):
        assert torch.equal(ids[:int(n)], want[k % 2]), k


@pytest.mark.parametrize("model,kw", [("DistMult", dict(chunk=32, n_neg=8)), ("TransR", dict()), ("RESCAL", dict())])
@pytest.mark.parametrize("step", [dict(), dict(overlap=False), dict(backward=False)])
def test_a_set_is_not_refilled_under_a_plain_step(model, kw, step):
    """run() between staged steps, in each of its forms, on a device that is still busy in front of it: the stream that refills the set's index
    tensors waits for that step too.  While a batch is staged a plain step is refused."""
    from cuke_amd._lib import KgeError
    m, batches, make = _two_batches(model, **kw)
    st, copies = make(batches[0]), torch.cuda.Stream()
    busy = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    st.run(**step)
    torch.cuda.synchronize()
    want = st.pos.clone()

    def stage(b):
        tensors = st.next_inputs(copies)
        with torch.cuda.stream(copies):
            for x, y in zip(tensors, b):
                if x is not None:
                    x.copy_(y)
            st.stage(copies.record_event())
        return tensors

    first = stage(batches[0])
    if step.get("backward", True) and "overlap" not in step:
        with pytest.raises(KgeError):
            st.run()
    st.run(pipeline=True)
    for _ in range(20):  # (milliseconds)
        busy.zero_()
    st.run(**step)
    got = st.pos.clone()
    for _ in range(2):
        stage(batches[0])
        st.run(pipeline=True)
    again = stage(batches[1])
    assert again[0] is first[0]
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("batch,up_front", [(2000, True), (32768, True), (32769, False)])
def test_large_explicit_batches_inspect_on_the_side_stream(batch, up_front):
    """Explicit TransR triples: up to 65536 entity ids both sets in front of the step in one call, the entities of more beside the forward pass."""
    from cuke_amd.kge import TrainStep
    w = synth.custom_workload("TransR", n_ent=500, n_rel=9, dim=16, batch=batch, sigma=0.3, seed=4)
    m, ix = gpu_model(w)
    st, calls = TrainStep(m, ix["h"], ix["r"], ix["t"]), []
    st.inspect = lambda *a: (calls.append(1), TrainStep.inspect(st, *a))
    st.run()
    got = _step_outputs(st)
    assert calls == ([1] if up_front else [])
    st.run(fused=False)
    assert all(torch.equal(x, y) for x, y in zip(got, _step_outputs(st)))
    assert calls == ([1] if up_front else [])
