"""The C view that a TensorView hands to the library: every field, whatever was asked for before."""
import copy
import pickle

import emel_hip as eh


def fields(v):
    return v.data, v.dtype, v.reserved, list(v.ne), list(v.nb), v.data_bytes


def test_view_fields_follow_the_view():
    lay = eh.Layout(12, [4096, 7, 3, 2], [1, 2304, 16128, 48384])
    for ptr, size in ((0x1000, 96768), (2**63 + 8, 2**40)):
        v = eh.TensorViewMut(ptr, lay, size)
        for _ in range(2):
            assert fields(v.c()) == (ptr, 12, 0, [4096, 7, 3, 2], [1, 2304, 16128, 48384], size)
    first, second = v.c(), v.c()
    first.ne[0] = 5  # each call's view is its own
    assert second.ne[0] == 4096 and v.c().ne[0] == 4096
    v.ptr, v.data_bytes, v.layout = 64, 16, eh.Layout.dense(0, [4, 1, 1, 1])
    assert fields(v.c()) == (64, 0, 0, [4, 1, 1, 1], [4, 16, 16, 16], 16)


def test_layout_stays_a_value():
    a, b = eh.Layout.dense(0, [4, 2, 1, 1]), eh.Layout.dense(0, [4, 2, 1, 1])
    a.wire()
    assert a == b and hash(a) == hash(b) and "_wire" not in repr(a)
    for c in (copy.deepcopy(a), pickle.loads(pickle.dumps(a)), pickle.loads(pickle.dumps(b))):
        assert c == a and c.wire() == b.wire()
