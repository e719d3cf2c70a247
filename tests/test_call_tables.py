"""Tables the operator wrappers hand to the library: as many entries as the call says it reads, whatever the lengths of
the lists a caller passes.  A stand-in takes the library's place and reads every table as the library would."""

import dataclasses
import types

import pytest

from modelexpress_amd import engine as E
from modelexpress_amd.manifest import TensorRecord, _record, build_manifest

BASE = 0x7F0000000000


class Library:
    """Records (pointers, sizes) of each call, n entries of every table."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            tables = [a for a in args if hasattr(a, "_length_")]
            n = next(a for a in args[1:] if type(a) is int)
            words = [t for t in tables if t._type_ in (E.C.c_void_p, E.C.c_uint64) and t._length_ != 7 * n]
            assert all(t._length_ >= n for t in words), f"{name} reads {n} entries of {[t._length_ for t in words]}"
            self.calls.append((name, n, [[int(t[i] or 0) for i in range(n)] for t in words]))
            return 0

        if name.startswith("mxp_"):
            return call
        raise AttributeError(name)


@pytest.fixture
def lib(monkeypatch):
    standin = Library()
    monkeypatch.setattr(E.L, "lib", lambda: standin)
    return standin


@pytest.fixture
def engine():
    eng = object.__new__(E.PlacementEngine)
    eng._h = None
    return eng


BUFFERS = [BASE, BASE + 4096, BASE + 8192]
CALLS = {
    "checksum32": lambda e, b, s: e.checksum32(b, s),
    "checksum32_static": lambda e, b, s: e.checksum32_static(b, s),
    "digest": lambda e, b, s: e.digest(b, s),
    "fingerprint": lambda e, b, s: e.fingerprint(b, s),
    "copy_batch": lambda e, b, s: e.copy_batch(b, [x + (1 << 20) for x in b], s),
    "verify_plan": lambda e, b, s: e.verify_plan(b, s),
    "build_manifest": lambda e, b, s: build_manifest(e, [types.SimpleNamespace(name=str(i), dtype="U8", nbytes=n) for i, n in enumerate(s)], b),
}


@pytest.mark.parametrize("name", CALLS)
def test_missing_sizes_are_zero(lib, engine, name):
    CALLS[name](engine, BUFFERS, [100, 200])
    _, n, tables = lib.calls[0]
    assert n == 3 and tables[0] == BUFFERS and tables[-1] == [100, 200, 0]


@pytest.mark.parametrize("name", CALLS)
def test_extra_sizes_are_refused(lib, engine, name):
    with pytest.raises(IndexError):
        CALLS[name](engine, BUFFERS, [100, 200, 300, 400])
    assert not lib.calls


def test_missing_destinations_are_null(lib, engine):
    engine.copy_batch(BUFFERS, BUFFERS[:1], [16])
    assert lib.calls[0][2] == [BUFFERS, [BASE, 0, 0], [16, 0, 0]]


@pytest.mark.parametrize("strides", [(64, 8), [64, 8], "iterator"])
def test_view_shapes_and_strides_from_any_iterable(strides):
    it = iter([64, 8]) if strides == "iterator" else strides
    arr = E.PlacementEngine.views_array([{"src": BASE, "dst": BASE + 4096, "shape": iter([3, 5]), "elem_size": 2, "src_strides": it}])
    v = arr[0]
    assert (v.ndim, v.elem_size, list(v.shape[:3]), list(v.src_strides[:3])) == (2, 2, [3, 5, 0], [64, 8, 0])
    assert (v.contiguous_src, v.contiguous_dst) == (0, 1)


def test_manifest_records_are_the_dataclass():
    """``_record`` fills the fields by hand: all of them, in their order, wherever the dataclass keeps them."""
    fields = ("name", 24, "BF16", "0badf00d", "00" * 16)
    assert len(dataclasses.fields(TensorRecord)) == len(fields)
    made, plain = _record(*fields), TensorRecord(*fields)
    assert made == plain and vars(made) == vars(plain) and hash(made) == hash(plain)
