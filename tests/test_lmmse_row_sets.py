"""Row lists per SNR point: one launch serves them only while they are the disjoint lists they were made as."""

import copy
import pickle

import numpy as np
import pytest
import torch

from hermespy_amd.lmmse import RowSets


def _sets():
    return RowSets([torch.tensor([0, 1]), None, torch.tensor([2])])


def test_as_made():
    s = _sets()
    assert s.disjoint and len(s) == 3 and s[1] is None and isinstance(s, list)
    assert copy.copy(s).disjoint
    assert pickle.loads(pickle.dumps(s)).disjoint


@pytest.mark.parametrize("change", [lambda s: s.__setitem__(1, s[0]), lambda s: s.append(s[0]), lambda s: s.insert(0, s[2]),
                                    lambda s: s.extend([s[0]]), lambda s: s.pop(), lambda s: s.reverse(),
                                    lambda s: s.__imul__(2)])
def test_changed(change):
    s = _sets()
    change(s)
    assert not s.disjoint


@pytest.mark.gpu
def test_changed_sets_apply_in_order(cuda):
    """A set added by the caller overrides the rows it shares, as in a list of the caller's own."""

    from hermespy_amd.configs import mimo2x2_512_pilots
    from hermespy_amd.lmmse import LMMSEChannelEstimation

    lm = LMMSEChannelEstimation(mimo2x2_512_pilots())
    g = torch.Generator(device=cuda).manual_seed(2)
    point = np.arange(40) % 3
    ls = torch.view_as_complex(torch.randn(2, 40, 2, lm.num_pilots, 2, generator=g, device=cuda))
    sets = lm.rows_by_set(point)
    sets[5] = sets[1]
    assert torch.equal(lm.apply(ls, point, rows_by_set=sets), lm.apply(ls, point, rows_by_set=list(sets)))
