"""The native readers of tensor containers are an option: without them, or with ones built for another torch or interpreter,
every caller does the same work in Python."""

import logging
import sys

import pytest
import torch
from torch import nn

import modelexpress_amd
from modelexpress_amd import _lib, build, engine as E, manifest, mla, publisher, reshard


@pytest.fixture(params=["missing", "other torch", "no tag"])
def without(request, monkeypatch, caplog):
    """tensors() as it answers in a process whose _tensors.so is missing or was built for something else."""
    _lib.tensors()
    native = sys.modules.get("modelexpress_amd._tensors")
    assert native is not None and native.built_for == _lib.tensors_tag(torch)
    monkeypatch.setattr(_lib, "_tensors", None)
    monkeypatch.setattr(_lib, "_tensors_refused", False)
    if request.param == "missing":
        monkeypatch.setitem(sys.modules, "modelexpress_amd._tensors", None)
        monkeypatch.delattr(modelexpress_amd, "_tensors", raising=False)
    elif request.param == "other torch":
        monkeypatch.setattr(_lib, "tensors_tag", lambda t: "another")
    else:
        monkeypatch.delattr(native, "built_for")
    with caplog.at_level(logging.WARNING, logger="modelexpress_amd"):
        for _ in range(3):
            assert _lib.tensors() is None
    assert len([r for r in caplog.records if "_tensors.so" in r.getMessage()]) == 1


class Engine:
    """What the callers ask of an engine, on tensors in host memory."""

    def fingerprint(self, buffers, sizes):
        return [f"{n:08x}" for n in sizes], [f"{n:032x}" for n in sizes]

    def view_plan(self, arr, n):
        plan = type("Plan", (), {"run": lambda self, stream=0: None, "run_digests": lambda self, stream=0: ["d"] * n, "close": lambda self: None})()
        plan.bytes = 0
        return plan

    def copy_views_array(self, arr, n, *, stream=0):
        self.n = n


def test_every_caller_works_without_them(without):
    t = torch.zeros(3, 4)
    assert list(E._addrs([t, 4096])) == [t.data_ptr(), 4096]
    arr = E.PlacementEngine.views_array([{"src": t, "dst": 8192, "shape": (3, 4), "elem_size": 4}])
    assert arr[0].src == t.data_ptr() and arr[0].shape[1] == 4
    [record] = manifest.build_manifest(Engine(), [E.ParamSpec("a", "F32", (3, 4))], [t])
    assert (record.name, record.nbytes) == ("a", 48)
    m = nn.Module()
    m.num_heads, m.qk_nope_head_dim, m.v_head_dim = 2, 3, 4
    m.kv_b_proj = nn.Linear(8, 14, bias=False)
    m.W_UV, m.W_UK_T = torch.zeros(4, 2, 8), torch.zeros(3, 8, 2)
    assert mla.update_mla_absorbed_weights(Engine(), m, quantized=False) == 2
    stager = publisher.WireStager(Engine(), publish_digests=True)
    for _ in range(3):
        out = stager.stage({"a": t, "step": torch.tensor(1)})
        assert out["digests"] == {"a": "d"} and out["total_bytes"] == 24 and stager.skipped == ["step"]
    held = {"a": t}
    assert reshard.ReslicePlan._addresses(held, {"a": ((3, 4), torch.float32)}, True) == t.data_ptr().to_bytes(8, sys.byteorder)


def test_stale_readers_are_built_again(monkeypatch, tmp_path):
    assert build.tensors_built()
    monkeypatch.setattr(_lib, "tensors_tag", lambda t: "another torch")
    assert not build.tensors_built()
    monkeypatch.undo()
    monkeypatch.setattr(build, "TENSORS_PATH", tmp_path / "_tensors.so")
    assert not build.tensors_built()


def test_the_library_builds_without_torch(monkeypatch, capsys, tmp_path):
    monkeypatch.setattr(build, "TENSORS_PATH", tmp_path / "_tensors.so")
    monkeypatch.setitem(sys.modules, "torch", None)
    assert build.build_tensors() is None and "no torch here" in capsys.readouterr().err
    assert not build.tensors_built()
