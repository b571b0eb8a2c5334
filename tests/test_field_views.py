"""The htr_fields that FieldSet.c() packs in one go, on the CPU: the views of the
struct, one by one, whatever members the struct has."""
import ctypes as C

import pytest

import htr_amd
from htr_amd import Fields, View, api


@pytest.mark.parametrize("kw", [dict(), dict(layout="aos", bounds_lo=(3, -2, 5)), dict(layout="padded", profiles=True)])
def test_packed_views_are_the_tensors_views(kw):
    fs = htr_amd.FieldSet((5, 4, 3), 5, device="cpu", **kw)
    f = fs.c()
    for name, kind in Fields._fields_:
        for d in range(1 if kind is View else 3):
            got = getattr(f, name) if kind is View else getattr(f, name)[d]
            key = name if kind is View else "%s%d" % (name, d)
            want = fs.view(key) if key in fs.t else View()
            assert bytes(got) == bytes(want), key


def test_order_follows_the_struct():
    i = [k for k, _ in Fields._fields_].index("rho")

    class More(C.Structure):
        _fields_ = Fields._fields_[:i] + [("added", View), ("pair", View * 2)] + Fields._fields_[i:]

    order = api.field_order(More)
    assert [k for k in order if k not in ("added", "pair0", "pair1")] == list(api.FIELD_ORDER)
    for k in ("added", "rho", "shockSensor2", "DucrosSensor"):
        name, d = (k[:-1], int(k[-1])) if k[-1].isdigit() else (k, 0)
        assert getattr(More, name).offset // C.sizeof(View) + d == order.index(k)

    class Other(C.Structure):
        _fields_ = [("count", C.c_int64)] + Fields._fields_

    with pytest.raises((TypeError, AttributeError)):
        api.field_order(Other)
