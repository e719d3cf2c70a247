"""Digests and checksums taken by the launch that places the bytes, at the edges of what a tile sums up in steps: tiles
that end with, before and after a buffer's last whole row of 1024 words, words that carry the largest 32-bit sums a tile
can reach, and tiles whose destination rows do not abut."""

import numpy as np
import pytest
import torch
from safetensors.torch import save_file

from modelexpress_amd.engine import Checkpoint, ParamSpec, PlacementEngine, PlacementPlan, VirtualTensor

pytestmark = pytest.mark.gpu

ROW = 2048  # 2-byte elements of a digest row
SIZES = [16 * ROW, 16 * ROW - 4, 16 * ROW + 4, 32 * ROW, 32 * ROW + 8, 64 * ROW, 64 * ROW - 8, 65 * ROW + 1, 129 * ROW, 8, ROW, ROW - 1, 3 * ROW + 5]


def _words(kind, n, gen):
    if kind == "random":
        return torch.randint(-32768, 32768, (n,), generator=gen, device="cuda", dtype=torch.int32).to(torch.int16)
    return torch.full((n,), kind, dtype=torch.int16, device="cuda")


@pytest.mark.parametrize("kind", ["random", -1, 0x7F7F, -32768, 0x7FFF])
def test_tiles_around_the_last_whole_row(gpu_engine, oracle, kind):
    gen = torch.Generator("cuda").manual_seed(3)
    src = [_words(kind, n, gen) for n in SIZES]
    dst = [torch.zeros_like(t) for t in src]
    views = [{"src": s, "dst": d, "shape": (s.numel(),), "elem_size": 2} for s, d in zip(src, dst)]
    plan = gpu_engine.view_plan(PlacementEngine.views_array(views), len(views))
    sums = gpu_engine.copy_batch(src, [torch.zeros_like(t) for t in src])
    for _ in range(2):
        digests = plan.run_digests()
        for s, d, c, g in zip(src, dst, sums, digests):
            raw = s.cpu().numpy().view(np.uint8)
            assert torch.equal(s, d)
            assert (c, g) == (oracle.safe_checksum_bytes(raw), oracle.tensor_digest_bytes(raw)), s.numel()
    plan.close()


@pytest.mark.parametrize("src_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,left,right", [(64, 1024, 1024), (640, 64, 192), (33, 4096, 8), (200, 24, 1000)])
def test_tiles_of_rows_that_do_not_abut(gpu_engine, oracle, tmp_path, src_dtype, rows, left, right):
    gen = torch.Generator().manual_seed(rows)
    a, b = (torch.randn(rows, c, generator=gen).to(src_dtype) for c in (left, right))
    save_file({"a": a, "b": b}, str(tmp_path / "model.safetensors"))
    whole = VirtualTensor("w", (rows, left + right), (("a", (0, 0), (0, 0), (rows, left)), ("b", (0, 0), (0, left), (rows, right))))
    ck = Checkpoint(str(tmp_path))
    plan = PlacementPlan(ck, [ParamSpec("w", "BF16", (rows, left + right))], virtual_tensors=[whole], skip_prefixes=["a", "b"],
                         allow_cast=True, allow_unmapped=True)
    want = torch.cat([a, b], 1).to(torch.bfloat16).view(torch.uint8).reshape(-1).numpy()
    staged = [torch.from_numpy(np.fromfile(f["path"], dtype=np.uint8)).cuda() for f in ck.files()]
    dst = gpu_engine.allocate(plan, fill=0xCD)
    gpu_engine.set_fused_digests(True)
    try:
        for run in (lambda: gpu_engine.execute_resident(plan, staged, dst), lambda: gpu_engine.execute(plan, dst)):
            dst[0].fill_(0xCD)
            torch.cuda.synchronize()
            run()
            assert gpu_engine.checksums(plan) == [oracle.safe_checksum_bytes(want)]
            assert gpu_engine.digests(plan) == [oracle.tensor_digest_bytes(want)]
            assert np.array_equal(dst[0].cpu().numpy(), want)
    finally:
        gpu_engine.set_fused_digests(False)
