"""Digests taken by the launch that runs a view plan: against the oracle and against the pass over the finished
buffers, for the views one launch can digest and for those that need the second pass."""

import numpy as np
import pytest
import torch

from modelexpress_amd.engine import PlacementEngine
from modelexpress_amd.publisher import COPY_TO_DEVICE, WireStager

pytestmark = pytest.mark.gpu

SHAPES = [(1,), (3,), (1024,), (2, 1024), (2048, 1), (33, 2048), (700, 357), (0, 5), (), (65, 4099), (3, 1025)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("strided", [False, "rows", "transposed"])
def test_snapshot_digests(gpu_engine, oracle, dtype, strided):
    gen = torch.Generator("cuda").manual_seed(5)
    state = {}
    for k, shape in enumerate(SHAPES):
        t = torch.randn(shape, generator=gen, device="cuda").to(dtype)
        if strided and len(shape) == 2:
            wide = torch.randn(shape[0], shape[1] + 3, generator=gen, device="cuda").to(dtype)
            t = wide[:, 3:] if strided == "rows" else torch.randn(shape[::-1], generator=gen, device="cuda").to(dtype).t()
        state[f"t{k}"] = t
    stager = WireStager(gpu_engine, publish_digests=True)
    for step in range(3):  # the accumulators are clear again for every run
        out = stager.stage(state, COPY_TO_DEVICE)
        for n, t in state.items():
            served = out["served"][n]
            want = t.to(torch.bfloat16).contiguous()
            assert torch.equal(served.view(torch.int16), want.view(torch.int16)), n
            raw = served.reshape(-1).view(torch.uint8).cpu().numpy() if served.numel() else np.zeros(0, np.uint8)
            assert out["digests"][n] == oracle.tensor_digest_bytes(raw), n
        assert list(out["digests"]) == list(out["served"])
        for t in state.values():
            t.mul_(-1.5)
    stager.close()


def test_destinations_that_one_pass_cannot_digest(gpu_engine):
    src = torch.randn(64, 64, device="cuda").bfloat16()
    dst = torch.zeros(64 * 64 + 8, dtype=torch.bfloat16, device="cuda")

    def view(**kw):
        return {"src": src, "dst": dst, "shape": (64, 64), "elem_size": 2, **kw}

    def run(views):
        plan = gpu_engine.view_plan(PlacementEngine.views_array(views), len(views))
        got = plan.run_digests()
        torch.cuda.synchronize()
        return got

    whole = [dst[: 64 * 64]]
    assert run([view()]) == gpu_engine.digest(whole)
    off_grid = [dst[1: 64 * 64 + 1]]
    assert run([view(dst=off_grid[0])]) == gpu_engine.digest(off_grid)
    twice = run([view(), view()])  # the same bytes into the same buffer
    assert twice == gpu_engine.digest(whole + whole)
    with pytest.raises(Exception, match="not contiguous"):
        run([view(shape=(32, 64), dst_strides=(128, 1))])
    assert run([]) == []
