"""Inspector parity: bit-exact against numpy unique + stable argsort."""
import numpy as np
import pytest
import torch

from cuke_amd import synth

pytestmark = pytest.mark.gpu


def check(oracle, parts, n_rows):
    from cuke_amd.kge import inspect
    dev = torch.device("cuda:0")
    ins = inspect([torch.from_numpy(p).to(dev) for p in parts], n_rows)
    ref = oracle.inspect(np.concatenate(parts))
    U = ins.num_unique
    assert U == ref.unique_ids.shape[0]
    assert np.array_equal(ins.ids().cpu().numpy(), ref.unique_ids)
    assert np.array_equal(ins.offsets().cpu().numpy().astype(np.int64), ref.seg_offsets)
    assert np.array_equal(ins.perm[: ins.n].cpu().numpy().astype(np.int64), ref.perm)
    assert np.array_equal(ins.inverse[: ins.n].cpu().numpy().astype(np.int64), ref.inverse)
    assert np.array_equal(ins.sorted_seg[: ins.n].cpu().numpy().astype(np.int64), ref.inverse[ref.perm])


@pytest.mark.parametrize("n,n_rows", [(0, 10), (1, 10), (37, 1), (64, 64), (2048, 2000), (2049, 5),
                                      (5000, 1 << 11), (5000, (1 << 11) + 1), (12288, 1_000_000),
                                      (49152, 4_000_000), (70000, 1 << 22), (300_000, 40_000),
                                      # block size (1024 keys) and the mid / large path switch (65536 keys)
                                      (1023, 50), (1024, 50), (1025, 50), (65535, 70_000), (65536, 1000),
                                      (65537, 1000), (65537, 1 << 30)])
def test_inspect_uniform(oracle, n, n_rows):
    rng = np.random.default_rng(n + n_rows)
    check(oracle, [rng.integers(0, n_rows, n, dtype=np.int64)], n_rows)


def test_inspect_all_equal_and_all_distinct(oracle):
    check(oracle, [np.full(5000, 123, np.int64)], 1000)
    check(oracle, [np.random.default_rng(0).permutation(6000).astype(np.int64)], 6000)
    check(oracle, [np.arange(4096, dtype=np.int64)[::-1].copy()], 4096)
    check(oracle, [np.array([(1 << 32) - 1, 0, (1 << 32) - 1, 7], np.int64)], 1 << 32)


@pytest.mark.parametrize("name", ["cfg2_distmult", "cfg3_transr", "cfg4_rotate", "cfg5_transh"])
def test_inspect_benchmark_index_sets(oracle, name):
    w = synth.make_workload(name, tables=False)
    a = w.arrays
    parts = [a["h"], a["t"]] + ([a["neg"]] if "neg" in a else [])
    check(oracle, parts, w.n_ent)
    check(oracle, [a["r"]], w.n_rel)


def test_inspect_multi_part_ragged(oracle):
    rng = np.random.default_rng(3)
    parts = [rng.integers(0, 777, k, dtype=np.int64) for k in (5, 0, 2047, 1)]
    check(oracle, parts, 777)


@pytest.mark.parametrize("n_rows", [1, 2, 128, 512, 513, 129 << 7, 1 << 21, 1 << 32])
@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 2047, 2048, 2049, 3071, 4095, 4096, 4097])
def test_inspect_in_one_workgroup_and_past_it(oracle, n, n_rows):
    """Edges of the one-workgroup kernel: keys per thread, digits of one to five passes, what goes to the launches behind it."""
    rng = np.random.default_rng(n * 7 + n_rows)
    ids = rng.integers(0, n_rows, n, dtype=np.int64)
    check(oracle, [ids], n_rows)
    check(oracle, [ids[:n // 3], np.minimum(ids[n // 3:], n_rows // 5)], n_rows)
    check(oracle, [np.full(n, n_rows - 1, np.int64)], n_rows)


@pytest.mark.parametrize("n,n_rows", [(1024, 1 << 20), (2048, 40), (2047, 1345), (4096, 1345), (4095, 14951)])
def test_inspect_ids_that_follow_each_other(oracle, n, n_rows):
    """(the one-workgroup kernel scatters them a power of two apart)"""
    ids = np.arange(n, dtype=np.int64)
    check(oracle, [ids % n_rows], n_rows)
    check(oracle, [(n_rows - 1 - ids % n_rows)], n_rows)
    check(oracle, [(ids * 64) % n_rows, (ids * 2048) % n_rows], n_rows)


@pytest.mark.parametrize("n,n_rows", [((5000, 5001), (3000, 64)), ((8192, 16384), (65, 14951)), ((4097, 60000), (2048, 5000)),
                                      ((0, 9000), (1345, 4000)), ((6000, 6000), (2047, 1 << 23))])
def test_a_narrow_set_beside_a_wide_one(oracle, n, n_rows):
    """Two sets in one batch of launches: a set of one digit pass takes two beside a set of two or three (from 65 rows on)."""
    import ctypes as C

    from cuke_amd import _lib
    from cuke_amd.kge import inspect
    rng = np.random.default_rng(n[0] + n_rows[0])
    ids = [rng.integers(0, r, k, dtype=np.int64) for k, r in zip(n, n_rows)]
    dev = [torch.from_numpy(x).cuda() for x in ids]
    got = [inspect([x], r) for x, r in zip(dev, n_rows)]
    L, jobs, ws = _lib.lib(), (_lib.InspectJob * 2)(), []
    for j, g, x, r in zip(jobs, got, dev, n_rows):
        for a in (g.num_unique_dev, g.unique_ids, g.seg_offsets, g.perm, g.inverse, g.sorted_seg):
            a.fill_(-1)
        size = int(L.kge_inspect_workspace(x.numel(), r))
        ws.append(torch.empty(max(size, 1), dtype=torch.uint8, device="cuda"))
        j.parts[0], j.part_len[0], j.n_parts, j.n_rows, j.out = x.data_ptr(), x.numel(), 1, r, g._c
        j.workspace, j.workspace_bytes = ws[-1].data_ptr(), size
    assert L.kge_inspect_batch(jobs, 2, C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    for g, x in zip(got, ids):
        ref, k, u = oracle.inspect(x), x.size, int(g.num_unique_dev.item())
        assert u == ref.unique_ids.shape[0]
        for a, want in ((g.unique_ids[:u], ref.unique_ids), (g.seg_offsets[:u + 1], ref.seg_offsets), (g.perm[:k], ref.perm),
                        (g.inverse[:k], ref.inverse), (g.sorted_seg[:k], ref.inverse[ref.perm])):
            assert np.array_equal(a.cpu().numpy().astype(np.int64), want)


def test_an_empty_set_without_arrays_beside_another():
    """Nothing to inspect beside a set of the mid-size launches: the empty set has no more than its count and its one offset."""
    import ctypes as C

    from cuke_amd import _lib
    from cuke_amd.kge import inspect
    L, ids = _lib.lib(), torch.arange(9000, device="cuda") * 7 % 4000
    full = inspect([ids], 4000)
    want = [x.clone() for x in (full.unique_ids[:full.num_unique], full.perm, full.inverse)]
    full.perm.fill_(-1)
    count, offset = torch.full((1,), -1, dtype=torch.int32, device="cuda"), torch.full((1,), -1, dtype=torch.int32, device="cuda")
    for at in (0, 1):
        jobs, ws = (_lib.InspectJob * 2)(), []
        for j, n, rows, out in ((jobs[at], 0, 1345, _lib.Inspection(0, 1345, count.data_ptr(), None, offset.data_ptr(), None, None, None)),
                                (jobs[1 - at], ids.numel(), 4000, full._c)):
            ws.append(torch.empty(int(L.kge_inspect_workspace(n, rows)), dtype=torch.uint8, device="cuda"))
            j.parts[0], j.part_len[0], j.n_parts, j.n_rows, j.out = ids.data_ptr() if n else None, n, 1, rows, out
            j.workspace, j.workspace_bytes = ws[-1].data_ptr(), ws[-1].numel()
        count.fill_(-1), offset.fill_(-1), full.perm.fill_(-1)
        assert L.kge_inspect_batch(jobs, 2, C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        assert int(count) == 0 and int(offset) == 0
        assert all(torch.equal(x, y) for x, y in zip(want, (full.unique_ids[:full.num_unique], full.perm, full.inverse)))
