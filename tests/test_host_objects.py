"""The objects the native host path returns, without a GPU."""
import copy

import pytest
import torch


def packed(n, seg_offsets, parts):
    """A _PackedInspection as csrc/host.cpp lays it out: one block, each part on a 256-byte boundary."""
    from cuke_amd import _lib
    from cuke_amd.kge import _PackedInspection

    def part(x):
        bytes_ = torch.tensor(x, dtype=torch.int32).view(torch.uint8)
        return torch.cat((bytes_, torch.zeros(-len(bytes_) % 256, dtype=torch.uint8)))

    block = torch.cat([part([len(seg_offsets) - 1]), part(list(seg_offsets) + [0] * (n + 1 - len(seg_offsets)))] + [part(x) for x in parts])
    return _PackedInspection(torch.arange(n), block, bytes(_lib.Inspection(n, 9)))


def test_packed_inspection_names_its_parts_and_can_be_copied():
    n = 100
    perm, inverse, sorted_seg = ([k * i for i in range(n)] for k in (1, 2, 3))
    ins = packed(n, [0, 60, 100], [perm, inverse, sorted_seg])
    for x in (copy.copy(ins), ins):
        assert (x.n, x.n_rows, x.num_unique) == (n, 9, 2)
        assert x.offsets().tolist() == [0, 60, 100] and x.ids().tolist() == [0, 1]
        assert x.perm.tolist() == perm and x.inverse.tolist() == inverse and x.sorted_seg.tolist() == sorted_seg
        with pytest.raises(AttributeError):
            x.no_such_part


def test_staged_batches_are_validated_on_the_host():
    import ctypes as C
    from cuke_amd import _lib
    f, fake = _lib.lib().kge_sample_staged_batch, C.c_void_p(0x1000)
    ok = [fake, 8, fake, fake, fake, fake, 4, 10, 1, 0, fake, 1, None]

    def call(**kw):
        return f(*[kw.get(f"a{i}", x) for i, x in enumerate(ok)])
    assert call(a1=-1) == call(a6=-1) == call(a7=0) == -2
    for null in (0, 2, 3, 4, 5, 10):
        assert call(**{f"a{null}": None}) == -1
    assert call(a1=0, a6=0) == 0  # empty work: nothing is launched
