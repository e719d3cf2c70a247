"""The walk over a model's modules for the refresh of absorbed weights: a module that the native walk cannot read itself is
asked in Python, by itself, and the rest of the model is read natively; the views are those of the Python walk, in its order."""

import ctypes as C

import pytest
import torch
from torch import nn

from modelexpress_amd import _lib, mla


class Engine:
    def copy_views_array(self, arr, n, *, stream=0):
        self.words, self.n = bytes(memoryview(arr).cast("B"))[: n * C.sizeof(_lib.ViewCopy)], n


class Plain(nn.Module):
    def __init__(self, heads=2, nope=3, v=4, lora=8):
        super().__init__()
        self.num_heads, self.qk_nope_head_dim, self.v_head_dim = heads, nope, v
        self.kv_b_proj = nn.Linear(lora, heads * (nope + v), bias=False)
        self.W_UV, self.W_UK_T = torch.zeros(v, heads, lora), torch.zeros(nope, lora, heads)


class OwnGetattr(Plain):
    """What a compiled module does: attributes come from somewhere else."""

    def __getattr__(self, name):
        if name == "num_heads":
            return 2
        return super().__getattr__(name)


class ClassHeads(Plain):
    qk_nope_head_dim = 3


class Wrapper(nn.Module):
    def __init__(self, inner):
        super().__init__()
        self._orig_mod = inner

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(super().__getattr__("_orig_mod"), name)


class OwnWalk(nn.Module):
    def named_modules(self, *a, **k):
        return iter([("x", self.hidden)])


def _own_walk():
    m = OwnWalk()
    object.__setattr__(m, "hidden", Plain())
    return m


def _spoiled(**changes):
    m = Plain()
    for k, v in changes.items():
        setattr(m, k, v)
    return m


def _outcome(monkeypatch, model, native):
    eng = Engine()
    with monkeypatch.context() as ctx:
        if not native:
            ctx.setattr(_lib, "tensors", lambda: None)
        try:
            n = mla.update_mla_absorbed_weights(eng, model, quantized=False)
        except Exception as exc:  # noqa: BLE001
            return type(exc), str(exc)
    return n, getattr(eng, "words", None)


SHARED = Plain()
MODELS = {
    "own getattr among plain ones": lambda: [Plain(), OwnGetattr(), Plain(3, 2, 5, 6)],
    "class attribute": lambda: [Plain(), ClassHeads(), nn.Linear(2, 2)],
    "wrapped": lambda: [Wrapper(Plain()), Plain(), Wrapper(nn.Sequential(Plain(), Wrapper(SHARED))), SHARED],
    "numbers of another type": lambda: [Plain(), _spoiled(num_heads=2.0)],
    "own walk": lambda: [Plain(), _own_walk()],
    "wrong heads": lambda: [Plain(), Wrapper(_spoiled(num_heads=3))],
    "wrong shape": lambda: [_spoiled(W_UV=torch.zeros(4, 2, 9)), Plain()],
    "no conversion": lambda: [Plain(), _spoiled(W_UK_T=torch.zeros(3, 8, 2, dtype=torch.int32))],
    "no projection": lambda: [_spoiled(kv_b_proj=None)],
    "no number": lambda: [_spoiled(v_head_dim="x")],
    "no views": lambda: [nn.Linear(2, 2), Wrapper(nn.Linear(2, 2))],
}


@pytest.mark.parametrize("name", MODELS)
def test_the_views_are_those_of_the_python_walk(monkeypatch, name):
    torch.manual_seed(0)
    model = nn.ModuleList(MODELS[name]())
    got, want = _outcome(monkeypatch, model, True), _outcome(monkeypatch, model, False)
    assert got == want
    if name in ("own getattr among plain ones", "class attribute", "wrapped"):
        assert got[0] >= 4


def test_only_the_odd_modules_are_asked(monkeypatch):
    asked = []
    one = mla._views_of_module
    monkeypatch.setattr(mla, "_views_of_module", lambda m, *a: (asked.append(m), one(m, *a))[1])
    odd = OwnGetattr()
    model = nn.ModuleList([Plain(), odd, Plain()])
    eng = Engine()
    assert mla.update_mla_absorbed_weights(eng, model, quantized=False) == 6 and asked == [odd]
