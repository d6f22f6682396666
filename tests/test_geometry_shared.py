"""Geometry copies keep the sharing of arrays between fields, as copy.deepcopy does."""
import copy

import numpy as np

from tigre_amd.geometry import cone_geometry, duplicate


def _geo():
    geo = cone_geometry((5, 6, 7), (5.0, 3.0, 14.0), (8, 9), (0.5, 0.25), 100.0, 170.0)
    geo.offOrigin = np.arange(18.0).reshape(6, 3)
    return geo


def test_duplicate_keeps_shared_arrays_shared():
    geo = _geo()
    geo.first = geo.second = np.arange(3.0)
    geo.third = [geo.first, np.arange(2)]
    for got in (duplicate(geo), copy.deepcopy(geo)):
        assert got.first is got.second and got.third[0] is got.first and got.first is not geo.first
    geo = _geo()
    geo.before = [geo.offOrigin]
    geo.__dict__["offOrigin"] = geo.__dict__.pop("offOrigin")  # after the list that holds it
    for got in (duplicate(geo), copy.deepcopy(geo)):
        assert got.before[0] is got.offOrigin
