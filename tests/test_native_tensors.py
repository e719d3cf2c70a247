"""The native readers of tensor containers (csrc/mxp_tensors.cpp) against the Python functions beside their callers: the
same tables for what they take, and hands off - the Python function decides - for everything else."""

import dataclasses
import random

import pytest
import torch
from torch import nn

from modelexpress_amd import _lib, engine as E, mla, reshard
from modelexpress_amd.engine import ParamSpec, PlacementEngine
from modelexpress_amd.manifest import TensorRecord, build_manifest

N = _lib.tensors()


class Tagged(torch.Tensor):
    """A tensor subclass."""


def _general(monkeypatch, f):
    with monkeypatch.context() as m:
        m.setattr(_lib, "tensors", lambda: None)
        return f()


def _words(arr, n):
    return bytes(memoryview(arr).cast("B"))[: n * 224]


# ---- views --------------------------------------------------------------------------------------------------------
def _random_view(rng, tensors):
    def side():
        t = rng.choice(tensors)
        return t if rng.random() < 0.5 else t.data_ptr() + rng.randrange(64)

    nd = rng.randrange(9)
    seq = rng.choice([tuple, list, torch.Size])
    v = {"src": side(), "dst": side(), "shape": seq([rng.randrange(1 << 20) for _ in range(nd)]), "elem_size": rng.choice([1, 2, 4, 8])}
    for key in ("src_strides", "dst_strides"):
        pick = rng.random()
        if pick < 0.5:
            v[key] = rng.choice([tuple, list])([rng.randrange(-5, 1 << 40) for _ in range(rng.choice([nd, nd, rng.randrange(9)]))])
        elif pick < 0.7:
            v[key] = None
    if rng.random() < 0.5:
        v["cast"] = rng.randrange(8)
    odd = rng.random()
    if odd < 0.05:
        v["shape"] = iter(list(v["shape"]))
    elif odd < 0.1:
        v["elem_size"] = True
    elif odd < 0.15:
        v["src"] = torch.zeros(3).as_subclass(Tagged)
    elif odd < 0.2:
        v["cast"] = 1.0
    return v


@pytest.mark.parametrize("seed", range(40))
def test_views(monkeypatch, seed):
    rng = random.Random(seed)
    tensors = [torch.zeros(16), nn.Parameter(torch.zeros(5, 7)), torch.zeros(4, 6)[1:, 2:]]
    state = rng.getstate()
    views = [_random_view(rng, tensors) for _ in range(rng.randrange(30))]
    for k, v in enumerate(views):  # an iterator can be read once: each side gets its own
        if not hasattr(v["shape"], "__len__"):
            views[k] = dict(v, shape=list(v["shape"]))
            views[k]["iterate"] = True

    def fresh():
        return [{**{a: b for a, b in v.items() if a != "iterate"}, **({"shape": iter(v["shape"])} if "iterate" in v else {})} for v in views]

    got = PlacementEngine.views_array(fresh())
    want = _general(monkeypatch, lambda: PlacementEngine.views_array(fresh()))
    assert _words(got, len(views)) == _words(want, len(views))
    assert _words(PlacementEngine.views_array(tuple(fresh())), len(views)) == _words(want, len(views))
    rng.setstate(state)


def test_views_of_another_kind_are_not_asked_for_one_by_one(monkeypatch):
    t, asked = torch.zeros(4), []
    odd, plain = {"src": t.as_subclass(Tagged), "dst": 64, "shape": (4,), "elem_size": 4}, {"src": t, "dst": 64, "shape": (4,), "elem_size": 4}
    native = type("N", (), {"put_views": staticmethod(lambda views, words, k: (asked.append(k), N.put_views(views, words, k))[1])})
    for views, want in (([odd] * 50, 4), ([plain] * 50, 1), ([odd, odd, odd, plain] * 12, 4 * 12), ([odd] * 3 + [plain] * 40, 4)):
        asked.clear()
        with monkeypatch.context() as m:
            m.setattr(_lib, "tensors", lambda: native)
            got = PlacementEngine.views_array(views)
        assert _words(got, len(views)) == _words(_general(monkeypatch, lambda: PlacementEngine.views_array(views)), len(views))
        assert len(asked) == want, (len(views), asked)


@pytest.mark.parametrize("bad", [{"src": "x"}, {"shape": (1,) * 9}, {"src_strides": (1,) * 9}, {"shape": (1.5, "y")}, {"elem_size": None},
                                 {"src": 1 << 70}, {"shape": (1 << 70,)}, {"cast": None}, {"shape": None}])
def test_views_that_are_refused_stay_refused(monkeypatch, bad):
    good = {"src": 4096, "dst": 8192, "shape": (2, 3), "elem_size": 2}
    views = [good, {**good, **bad}]

    def outcome():
        try:
            return _words(PlacementEngine.views_array(views), 2)
        except Exception as exc:  # noqa: BLE001
            return type(exc)

    assert outcome() == _general(monkeypatch, outcome)
    missing = [{k: x for k, x in good.items() if k != "dst"}]
    with pytest.raises(KeyError):
        PlacementEngine.views_array(missing)


def test_pointers(monkeypatch):
    t = torch.zeros(3, 4)
    for bufs in ([t, 4096, t[1:]], (t, nn.Parameter(t)), [], [t.as_subclass(Tagged), 7], [True, 0]):
        assert list(E._addrs(bufs)) == _general(monkeypatch, lambda: E._addrs(bufs))
    with pytest.raises(AttributeError):
        E._addrs(["x"])


# ---- recorded copies ------------------------------------------------------------------------------------------------
def test_addresses(monkeypatch):
    held = {"a": torch.zeros(3, 4), "b": torch.zeros(5, dtype=torch.bfloat16), "c": nn.Parameter(torch.zeros(())), "d": torch.zeros(0, 2)}
    meta = {n: (tuple(t.shape), t.dtype) for n, t in held.items()}
    run = reshard.ReslicePlan._addresses
    quick = N.addresses(held, meta, True)
    monkeypatch.setattr(reshard.L, "tensors", lambda: type("No", (), {"addresses": staticmethod(lambda *a: None)}))
    assert quick is not None and quick == run(held, meta, True)
    plain = dict(held)
    for change in ({"a": None}, {"a": held["a"].double()}, {"a": torch.zeros(4, 3)}, {"a": torch.zeros(4, 3).t()}, {"a": torch.zeros(12)},
                   {"a": "x"}, {"a": held["a"].as_subclass(Tagged)}):
        assert N.addresses({**plain, **change}, meta, True) is None
    assert N.addresses({k: v for k, v in plain.items() if k != "b"}, meta, True) is None
    strided = {**plain, "a": torch.zeros(4, 3).t()}
    assert N.addresses(strided, meta, False) == run(strided, meta, False)  # a parameter may be strided
    assert N.addresses(type("D", (dict,), {})(plain), meta, True) is None
    assert N.addresses({**plain, "extra": 1}, meta, True) == quick


# ---- modules ----------------------------------------------------------------------------------------------------------
def _mla(heads=2, nope=3, v=4, lora=8, w=torch.bfloat16, out=torch.bfloat16, linear=True):
    m = nn.Module()
    m.num_heads, m.qk_nope_head_dim, m.v_head_dim = heads, nope, v
    if linear:
        m.kv_b_proj = nn.Linear(lora, heads * (nope + v), bias=False).to(w)
    else:
        m.kv_b_proj = nn.Module()
        m.kv_b_proj.weight = torch.zeros(heads * (nope + v), lora, dtype=w)
    m.W_UV, m.W_UK_T = torch.zeros(v, heads, lora, dtype=out), torch.zeros(nope, lora, heads, dtype=out)
    return m


def _model():
    model = nn.Module()
    shared = _mla(linear=False)
    model.layers = nn.ModuleList([_mla(), _mla(3, 2, 5, 6, torch.float32, torch.bfloat16), shared, nn.Linear(2, 2)])
    model.again = shared
    model.late = nn.ModuleDict({"x": _mla(w=torch.float16, out=torch.float32)})
    model.none = None
    model.register_module("hole", None)
    model.layers[0].W_UK_T = None
    model.layers[1].register_buffer("W_X", torch.zeros(1))
    del model.late["x"].W_UV
    model.late["x"].register_buffer("W_UV", torch.zeros(5, 4, 8)[1:].transpose(0, 1)[:2].transpose(0, 1))
    return model


def test_modules(monkeypatch):
    model = _model()
    quick = N.mla_views(model, nn.Module)
    assert quick is not None and bytes(quick) == mla._views_of_modules(model, False).tobytes() and len(quick) == 7 * 224
    assert N.mla_views(nn.Linear(2, 2), nn.Module) == b""


class OwnGetattr(nn.Module):
    def __getattr__(self, name):
        return super().__getattr__(name)


class OwnWalk(nn.Module):
    def named_modules(self, *a, **k):
        return iter(())


class ClassHeads(nn.Module):
    num_heads = 2


class Property(nn.Module):
    W_UV = property(lambda self: None)


@pytest.mark.parametrize("cls", [OwnGetattr, OwnWalk, ClassHeads, Property])
def test_modules_that_look_attributes_up_their_own_way_are_left_alone(cls):
    model = _model()
    model.special = cls()
    assert N.mla_views(model, nn.Module) is None


@pytest.mark.parametrize("spoil", [lambda m: setattr(m, "num_heads", 3), lambda m: setattr(m, "num_heads", 2.0), lambda m: delattr(m, "v_head_dim"),
                                   lambda m: setattr(m, "W_UV", torch.zeros(4, 2, 9, dtype=torch.bfloat16)),
                                   lambda m: setattr(m, "W_UV", torch.zeros(4, 2, 8, dtype=torch.int32)),
                                   lambda m: setattr(m, "W_UV", torch.zeros(4, 2, 8).as_subclass(Tagged)),
                                   lambda m: setattr(m.kv_b_proj, "weight", nn.Parameter(torch.zeros(8, 14).t().bfloat16())),
                                   lambda m: setattr(m, "kv_b_proj", None)])
def test_modules_that_may_be_refused_are_left_alone(spoil):
    m = _mla()
    spoil(m)
    assert N.mla_views(m, nn.Module) is None


# ---- snapshots and manifests --------------------------------------------------------------------------------------------
def test_state_key():
    a, b = torch.zeros(4, 6), torch.zeros(3, dtype=torch.float16)
    key = N.state_key({"a": a, "b": b})
    assert key == N.state_key({"a": a, "b": b}) == N.state_key({"x": a.view(4, 6), "y": b})  # names are the caller's to compare
    for other in ({"a": a}, {"b": b, "a": a}, {"a": a.view(6, 4), "b": b}, {"a": a.clone(), "b": b}, {"a": a.as_strided((4, 6), (1, 4)), "b": b},
                  {"a": a, "b": b.view(torch.bfloat16)}, {"a": a, "b": b[:2]}):
        assert N.state_key(other) != key
    for other in ({"a": a, "n": torch.tensor(3)}, {"a": a.as_subclass(Tagged)}, {"a": 1}, [a]):
        assert N.state_key(other) is None


class Sizes:
    def fingerprint(self, buffers, sizes):
        return [f"{n:08x}" for n in sizes], [f"{n:032x}" for n in sizes]


def test_manifest_records(monkeypatch):
    class Odd(ParamSpec):
        @property
        def nbytes(self):
            return 77

    params = [ParamSpec("a", "BF16", (3, 5)), ParamSpec("b", "F32", ()), ParamSpec("c", "U8", (0, 4)), Odd("d", "U8", (1,)),
              ParamSpec("e", "F8_E4M3", [2, 3]), ParamSpec("f", "F64", torch.Size([2, 2]))]
    got = build_manifest(Sizes(), params, [0] * 6)
    want = _general(monkeypatch, lambda: build_manifest(Sizes(), params, [0] * 6))
    assert got == want and [vars(r) for r in got] == [vars(r) for r in want] and [type(r) for r in got] == [TensorRecord] * 6
    assert [r.nbytes for r in got] == [30, 4, 0, 77, 6, 32] and hash(got[0]) == hash(want[0])
    assert [list(vars(r)) for r in got] == [[f.name for f in dataclasses.fields(TensorRecord)]] * 6
    with pytest.raises(KeyError):
        build_manifest(Sizes(), [ParamSpec("x", "NOPE", (1,))], [0])


def test_the_module_has_no_thread_local_storage():
    """Loaded after other libraries, it would slow their thread-local accesses down."""
    import struct

    elf = (_lib.PKG_DIR / "_tensors.so").read_bytes()
    phoff, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    assert 7 not in [struct.unpack_from("<I", elf, phoff + k * size)[0] for k in range(count)]  # PT_TLS


def test_lists_that_change_under_the_readers(monkeypatch):
    """A parameter's own attribute may run any code, such as one that shortens the list it is in."""
    class Shortens:
        def __init__(self, params, name):
            self.params, self._name, self.dtype = params, name, "U8"

        @property
        def nbytes(self):
            self.params[:] = []
            return 7

        @property
        def name(self):
            self.params[:] = []
            return self._name

    def outcome():
        out = []
        for _ in range(20):
            params = []
            params.extend(Shortens(params, f"name {k}") for k in range(300))
            out.append([(r.name, r.nbytes) for r in build_manifest(Sizes(), params, [])])
            params.extend(Shortens(params, f"name {k}") for k in range(300))
            out.append([r.name for r in build_manifest(Sizes(), [*params], [])])
            params.clear()
            params.extend(Shortens(params, f"name {k}") for k in range(300))
            out.append([(r.name, r.nbytes) for r in (N.records if _lib.tensors() else _plain_records)(TensorRecord, params, [7] * 300, ["c"] * 300, [None] * 300)])
        return out

    assert outcome() == _general(monkeypatch, outcome)


def _plain_records(cls, params, sizes, sums, digests):
    return [cls(p.name, n, p.dtype, s, d) for p, n, s, d in zip(params, sizes, sums, digests)]
