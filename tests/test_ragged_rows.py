"""Boxes whose destination rows abut off the 16-byte grid (ragged segments): the lowering against the plain form on
the CPU, the kernel against the conversions of torch on the GPU, at rows from one unit to several tiles, every
remainder of the grid, with the checksum and the digest taken on the way."""

import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

ROOT = Path(__file__).resolve().parent.parent
SRC = ROOT / "tests" / "c" / "ragged_check.cpp"
CASTS = {("F32", "BF16"): 1, ("BF16", "F32"): 2, ("F16", "F32"): 3, ("F32", "F16"): 4, ("F8_E4M3", "BF16"): 5,
         ("F16", "BF16"): 6, ("BF16", "F16"): 7}
TORCH = {"BF16": torch.bfloat16, "F16": torch.float16, "F32": torch.float32, "F8_E4M3": torch.float8_e4m3fn}


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    out = tmp_path_factory.mktemp("ragged") / "ragged_check"
    cmd = ["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT / 'include'}",
           f"-I{ROOT / 'modelexpress_amd' / 'csrc'}", "-I/opt/rocm/include", str(SRC), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("first", [0, 1000])
def test_ragged_tables_take_every_byte_from_where_the_plain_form_does(checker, first):
    r = subprocess.run([str(checker), str(first), "1000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert int(r.stdout.split()[0]) > 500


@pytest.mark.gpu
@pytest.mark.parametrize("src_dtype,dst_dtype", [("BF16", "BF16"), ("F8_E4M3", "F8_E4M3")] + list(CASTS))
@pytest.mark.parametrize("rows,cols,extra,first", [(700, 357, 357, 1), (3000, 17, 3, 0), (2, 100003, 5, 3), (5, 8191, 1, 7),
                                                   (999, 131, 2000, 2), (40000, 9, 1, 5)])
def test_ragged_boxes_on_the_device(gpu_engine, oracle, src_dtype, dst_dtype, rows, cols, extra, first):
    gen = torch.Generator("cuda").manual_seed(rows + cols)
    full = (torch.randn(rows, cols + extra, generator=gen, device="cuda") * 0.5).to(TORCH[src_dtype])
    want = full[:, extra:].to(TORCH[dst_dtype]).contiguous().view(torch.uint8).flatten()
    es, ed = full.element_size(), torch.empty(0, dtype=TORCH[dst_dtype]).element_size()
    n = rows * cols * ed
    lead = first * ed  # where in the 16-byte grid the destination starts
    buf = torch.full((lead + n + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    box = {"src": full.data_ptr() + extra * es, "dst": buf.data_ptr() + lead, "rows": rows, "row_bytes": cols * ed,
           "src_pitch": (cols + extra) * es, "dst_pitch": cols * ed, "cast": CASTS.get((src_dtype, dst_dtype), 0)}
    sums = gpu_engine.place_boxes([box], 1)
    assert torch.equal(buf[lead:lead + n], want)
    assert bool((buf[:lead] == 0xA5).all()) and bool((buf[lead + n:] == 0xA5).all())
    assert sums == [oracle.safe_checksum_bytes(want.cpu().numpy())]


@pytest.mark.gpu
@pytest.mark.parametrize("ckpt_dtype,param_dtype", [("BF16", "BF16"), ("F32", "BF16"), ("F16", "F32"), ("F32", "F32")])
@pytest.mark.parametrize("ffn", [714, 2 * 5003])
def test_ragged_parameters_with_digests(gpu_engine, oracle, tmp_path, ckpt_dtype, param_dtype, ffn):
    """Row-parallel slices of odd width placed out of device memory: bytes, checksums and digests of every parameter."""
    from modelexpress_amd import models, synth
    from modelexpress_amd.engine import Checkpoint, PlacementPlan

    m = models.Llama(layers=1, hidden=322, ffn=ffn, q_heads=6, kv_heads=2, head_dim=32, vocab=1002)
    synth.write_checkpoint(m.checkpoint(ckpt_dtype), tmp_path, seed=3)
    view = m.rank_view(2, 1, param_dtype=param_dtype)
    ck = Checkpoint(str(tmp_path))
    plan = PlacementPlan(ck, view.params, tp_size=2, tp_rank=1, stacked_params_mapping=view.stacked_params_mapping,
                         allow_cast=ckpt_dtype != param_dtype)
    dst = gpu_engine.allocate(plan, fill=0xCD)
    staged = [torch.from_numpy(np.fromfile(f["path"], dtype=np.uint8)).cuda() for f in ck.files()]
    gpu_engine.execute(plan, dst)  # the ring kernel, which takes none of these tables
    want = [t.clone() for t in dst]
    gpu_engine.set_fused_digests(True)
    try:
        for t in dst:
            t.fill_(0xCD)
        torch.cuda.synchronize()
        gpu_engine.execute_resident(plan, staged, dst)
        sums, digests = gpu_engine.checksums(plan), gpu_engine.digests(plan)
    finally:
        gpu_engine.set_fused_digests(False)
    for p, t, w, s, d in zip(plan.params, dst, want, sums, digests):
        assert torch.equal(t, w), p.name
        host = t.cpu().numpy()
        assert (s, d) == (oracle.safe_checksum_bytes(host), oracle.tensor_digest_bytes(host)), p.name
