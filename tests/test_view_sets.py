"""View subsets prepared on first use: as if prepared when the object was made, whatever happens to the caller's arrays
or to the object's geometry in between."""
import copy

import numpy as np
import pytest

from tigre_amd.algorithms import ViewSets
from tigre_amd.geometry import cone_geometry


def _geo():
    geo = cone_geometry((5, 6, 7), (5.0, 3.0, 14.0), (8, 9), (0.5, 0.25), 100.0, 170.0)
    geo.offOrigin = np.arange(18.0).reshape(6, 3)
    return geo


def _same(a, b):
    (ia, ga, ca, aa), (ib, gb, cb, ab) = a, b
    assert np.array_equal(ia, ib) and np.array_equal(aa, ab) and np.array_equal(ca._keep, cb._keep)
    assert np.array_equal(ga.offOrigin, gb.offOrigin) and ga.nVoxel.tolist() == gb.nVoxel.tolist()


def test_sets_are_those_of_the_construction():
    geo, angles = _geo(), np.linspace(0, 3, 6)
    blocks = [np.array([0, 2, 4]), np.array([1, 3]), [5]]
    want = ViewSets(geo, angles, copy.deepcopy(blocks)).sets
    assert len(want) == 3 and [len(s[0]) for s in want] == [3, 2, 1]
    late = ViewSets(geo, angles, blocks)
    blocks[0][:] = [5, 4, 3]
    geo.offOrigin[:] = 0
    angles[:] = 0
    late.geo.offOrigin[:] = -1
    late.geo.nVoxel = np.array([1, 1, 1])
    late.angles[:] = 7
    for j in range(3):
        _same(late.set(j), want[j])
        assert late.set(j) is late.set(j) and late.sets[j] is late.set(j)


def test_index_out_of_range_is_refused_at_once():
    with pytest.raises(IndexError):
        ViewSets(_geo(), np.linspace(0, 3, 6), [[0, 1], [6]])
