"""The geometry copies behind every operator call: ``duplicate`` against copy.deepcopy, and the C struct against the
values it is filled from, over the forms a geometry's fields take."""
import copy
import ctypes

import numpy as np
import pytest

from tigre_amd import _native
from tigre_amd.geometry import Geometry, cone_geometry, duplicate, geometry, prepared


class Own(Geometry):
    """A subclass with a copy protocol of its own."""

    def __deepcopy__(self, memo):
        g = Own()
        g.__dict__.update(copy.deepcopy(self.__dict__, memo), marked=True)
        return g


def _case(name):
    geo = cone_geometry((5, 6, 7), (5.0, 3.0, 14.0), (8, 9), (0.5, 0.25), 100.0, 170.0)
    if name == "per view":
        rng = np.random.default_rng(1)
        geo.DSO, geo.DSD, geo.COR = rng.uniform(90, 99, 4), rng.uniform(150, 160, 4).astype(np.float32), np.arange(4)
        geo.offOrigin, geo.offDetector = rng.normal(size=(4, 3)), rng.normal(size=(4, 2))
        geo.rotDetector = np.asfortranarray(rng.normal(size=(4, 3)))
    elif name == "scalars":
        geo.DSO, geo.DSD, geo.COR, geo.accuracy = np.float32(100.0), 170, 0.1, 1
        geo.note, geo.more, geo.nested = "text", [1, {"a": np.zeros(2)}], np.array([None, "x"], dtype=object)
    elif name == "preset":
        geo = geometry(default=True, high_resolution=False)
    elif name == "subclass":
        own = Own()
        own.__dict__.update(geo.__dict__)
        geo = own
    return geo


def _same(a, b):
    assert type(a) is type(b)
    if isinstance(a, np.ndarray):
        assert a.dtype == b.dtype and a.shape == b.shape and a.strides == b.strides and np.array_equal(a, b)
    else:
        assert repr(a) == repr(b)


@pytest.mark.parametrize("name", ["plain", "per view", "scalars", "preset", "subclass"])
def test_duplicate(name):
    geo = _case(name)
    got, want = duplicate(geo), copy.deepcopy(geo)
    assert type(got) is type(want) and list(got.__dict__) == list(want.__dict__)
    for k, v in want.__dict__.items():
        _same(got.__dict__[k], v)
        if isinstance(v, np.ndarray):
            assert not np.shares_memory(got.__dict__[k], geo.__dict__[k])
    if name == "scalars":
        assert got.more is not geo.more and got.more[1]["a"] is not geo.more[1]["a"]


@pytest.mark.parametrize("name", ["plain", "per view", "scalars"])
def test_c_geometry(name):
    n = 4
    g = prepared(_case(name), np.linspace(0, 1, n))
    c = _native.CGeometry(g, n)
    s = c.struct
    f32 = np.float32
    for axis, k in (("X", 2), ("Y", 1), ("Z", 0)):
        assert getattr(s, "nVoxel" + axis) == g.nVoxel[k]
        assert f32(getattr(s, "sVoxel" + axis)) == f32(g.sVoxel[k]) and f32(getattr(s, "dVoxel" + axis)) == f32(g.dVoxel[k])
        assert getattr(s, "unit" + axis) == 1.0
        assert getattr(s, "offOrig" + axis)[:n] == g.offOrigin[:, k].astype(f32).tolist()
    for axis, k in (("U", 1), ("V", 0)):
        assert getattr(s, "nDetec" + axis) == g.nDetector[k]
        assert f32(getattr(s, "sDetec" + axis)) == f32(g.sDetector[k]) and f32(getattr(s, "dDetec" + axis)) == f32(g.dDetector[k])
        assert getattr(s, "offDetec" + axis)[:n] == g.offDetector[:, k].astype(f32).tolist()
    for field, k in (("dRoll", 2), ("dPitch", 1), ("dYaw", 0)):
        assert getattr(s, field)[:n] == g.rotDetector[:, k].astype(f32).tolist()
    for field in ("DSO", "DSD", "COR"):
        assert getattr(s, field)[:n] == np.asarray(getattr(g, field), f32).tolist()
    assert f32(s.accuracy) == f32(g.accuracy) and s.alpha == s.theta == s.psi == s.maxLength == 0.0
    assert _native._PACK.size <= ctypes.sizeof(_native.TigreGeometry)
    g.DSO = np.asarray(g.DSO).reshape(1, n)  # refused as before
    with pytest.raises(ValueError):
        _native.CGeometry(g, n)
