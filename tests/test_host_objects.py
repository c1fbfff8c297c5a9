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
