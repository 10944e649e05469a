"""The calls that bypass ctypes against the ctypes route: the same descriptors reach the library, the same errors come back."""
import ctypes as C

import pytest

import moye_hip as mh
from moye_hip import _lib, device

calls = _lib.calls
pytestmark = pytest.mark.skipif(calls is None, reason="built without Python.h")

PTR = 1 << 40


class Recorder:
    """Stands where the library's functions are: keeps the bytes each argument pointed to, launches nothing."""

    def __init__(self):
        self.seen = []
        T, P, vp, d = _lib.Tensor, C.POINTER, C.c_void_p, C.c_double

        def record(*kinds):
            def f(*args):
                self.seen.append([None if (k is not None and not a) else bytes(a.contents) if k is not None else a for k, a in zip(kinds, args)])
                return 0
            return f
        t, m, tc, e = P(T), P(_lib.TiledMMA), P(_lib.TiledCopy), P(_lib.GemmEpilogue)
        self.keep = []

        def make(sig, kinds):
            self.keep.append(C.CFUNCTYPE(C.c_int32, *sig)(record(*kinds)))
            return C.cast(self.keep[-1], vp).value
        self.addresses = [make([m, t, t, t, t, C.c_float, vp], [1, 1, 1, 1, 1, None, None]),
                          make([m, t, t, t, t, e, vp, C.c_size_t, vp], [1, 1, 1, 1, 1, 1, None, None, None]),
                          make([tc, t, t, vp], [1, 1, 1, None]), make([t, t, t, vp], [1, 1, 1, None]),
                          make([d, t, d, t, vp], [None, 1, None, 1, None]), make([C.c_int32, t, t, t, d, vp], [None, 1, 1, 1, None, None])]


@pytest.fixture
def recorder():
    _lib.lib()
    r = Recorder()
    calls.bind(mh.MoYeArray, _lib.Tensor, _lib.TiledMMA, _lib.TiledCopy, _lib.GemmEpilogue, *r.addresses)
    yield r
    _lib._bind_calls(_lib.lib())


def array(rows, cols, dt=mh.F16, at=PTR):
    return mh.MoYeArray(at, dt, mh.Layout((rows, cols), (cols, 1)))


def test_arrays_and_descriptors_arrive_as_ctypes_hands_them_over(recorder):
    D, A, B, C_ = array(8, 4), array(8, 2, at=PTR + 64), array(4, 2), array(8, 4, mh.F32)
    mma = mh.tiled_mma_desc(mh.MFMA_F32_16x16x32_F16, split_k=-1)
    ep = mh.gemm_epilogue(alpha=0.5, op=_lib.MAP_MAX, scalar=2.0)
    raw = [x.tensor() for x in (D, A, B, C_)]
    tc = mh.tiled_copy_desc(vec_bits=128)
    for d, a, b, c in ((D, A, B, C_), raw, (D, raw[1], B, None)):
        mh.gemm_(mma, d, a, b, c, alpha=0.25, stream=77)
        assert recorder.seen[-1] == [bytes(mma)] + [bytes(x) for x in raw[:3]] + [None if c is None else bytes(raw[3]), 0.25, 77]
        device.gemm_ex_(mma, d, a, b, c, ep, 4096, 512, None)
        assert recorder.seen[-1] == [bytes(mma)] + [bytes(x) for x in raw[:3]] + [None if c is None else bytes(raw[3]), bytes(ep), 4096, 512, None]
        mh.copyto_(d, a, tc if c is None else None)
        assert recorder.seen[-1] == [bytes(tc) if c is None else None, bytes(raw[0]), bytes(raw[1]), None]
        mh.copyto_if_(d, a, b, stream=5)
        assert recorder.seen[-1] == [bytes(x) for x in raw[:3]] + [5]
        mh.axpby_(2, a, 0.5, d)
        assert recorder.seen[-1] == [2.0, bytes(raw[1]), 0.5, bytes(raw[0]), None]
        mh.map_("add", d, a, None if c is None else b, scalar=3)
        assert recorder.seen[-1] == [_lib.MAP_ADD, bytes(raw[0]), bytes(raw[1]), None if c is None else bytes(raw[2]), 3.0, None]
    # an array that is changed, and a layout made from its text alone, as an old pickle leaves it
    A.ptr += 2
    A.dtype = mh.BF16
    bare = mh.Layout.__new__(mh.Layout)
    bare.text = A.layout.text
    A.layout = bare
    mh.copyto_(D, A)
    assert recorder.seen[-1][2] == bytes(A.tensor()) != bytes(raw[1])


def test_an_array_s_own_descriptor_is_asked_for(recorder, monkeypatch):
    """A subclass of MoYeArray that says what its descriptor is (it takes ctypes), and a subclass of Layout that does."""
    class Library:
        @staticmethod
        def moye_copy(tc, dst, src, stream):
            recorder.seen.append([tc, bytes(dst._obj), bytes(src._obj), stream])
            return 0
    monkeypatch.setattr(device, "lib", Library)

    class Shifted(mh.MoYeArray):
        def tensor(self):
            t = super().tensor()
            t.ptr += 128
            return t

    class Halved(mh.Layout):
        def descriptor(self):
            return mh.Layout((4, 4), (8, 1)).descriptor()

    D, A = array(4, 4), Shifted(PTR, mh.F16, mh.Layout((4, 4), (4, 1)))
    mh.copyto_(D, A)
    assert recorder.seen[-1][2] == bytes(A.tensor()) != bytes(array(4, 4).tensor())
    B = mh.MoYeArray(PTR, mh.F16, Halved((8, 4), (4, 1)))
    B.layout._descriptor = mh.Layout((8, 4), (4, 1)).descriptor()
    mh.copyto_(D, B)
    assert recorder.seen[-1][2] == bytes(B.tensor())


@pytest.mark.parametrize("bad", [None, object(), 3.5, "x"])
def test_what_ctypes_refuses_stays_refused(recorder, bad):
    D, A = array(8, 4), array(8, 4)
    mma = mh.tiled_mma_desc(mh.MFMA_F32_16x16x32_F16)
    for f in (lambda: mh.copyto_(D, bad), lambda: mh.copyto_(bad, A), lambda: device.gemm_(bad, D, A, A), lambda: mh.gemm_(mma, D, bad, A), lambda: mh.axpby_(1.0, bad, 1.0, D),
              lambda: mh.map_("add", D, bad), lambda: mh.copyto_if_(D, A, bad)):
        with pytest.raises((TypeError, AttributeError, C.ArgumentError)):
            f()
    for f in (lambda: mh.copyto_(D, A, stream=object()), lambda: mh.axpby_("1", A, 1.0, D)):
        with pytest.raises((TypeError, C.ArgumentError)):
            f()
    assert not recorder.seen


def test_the_library_s_errors_come_back():
    with pytest.raises(mh.MoyeError) as e:
        mh.gemm_(mh.tiled_mma_desc(mh.MFMA_F32_16x16x32_F16), array(8, 4), array(8, 2), array(4, 3))
    assert e.value.status == _lib.ERR_SHAPE and "differ" in str(e.value)
