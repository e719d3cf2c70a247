"""Checksums and digests delivered by the execute that placed the bytes (fused digests on): in either order, asked for
more than once, after a second execute on another stream, around a captured launch, and with a plan that goes away
before anybody asked."""

import numpy as np
import pytest
import torch
from safetensors.torch import save_file

from modelexpress_amd.engine import Checkpoint, ParamSpec, PlacementEngine, PlacementPlan

pytestmark = pytest.mark.gpu

N = [5, 4096 * 3 + 2, 70001]


@pytest.fixture
def setup(tmp_path, mxp):
    def data(seed):
        g = torch.Generator().manual_seed(seed)
        return [torch.randint(0, 256, (n,), generator=g, dtype=torch.uint8) for n in N]

    save_file({f"p{k}": t for k, t in enumerate(data(0))}, str(tmp_path / "model.safetensors"))
    ck = Checkpoint(str(tmp_path))
    offsets = {t.name: t.file_offset for t in ck.tensors()}
    base = np.fromfile(ck.files()[0]["path"], dtype=np.uint8)

    def staged(seed):
        raw = base.copy()
        for k, t in enumerate(data(seed)):
            raw[offsets[f"p{k}"]:offsets[f"p{k}"] + N[k]] = t.numpy()
        return torch.from_numpy(raw).cuda()

    eng = PlacementEngine(0, ring_slots=4, slot_bytes=1 << 16)
    eng.set_fused_digests(True)
    yield eng, (lambda: PlacementPlan(ck, [ParamSpec(f"p{k}", "U8", (n,)) for k, n in enumerate(N)])), staged, data
    eng.close()


def _want(oracle, parts):
    raws = [t.numpy() for t in parts]
    return [oracle.safe_checksum_bytes(r) for r in raws], [oracle.tensor_digest_bytes(r) for r in raws]


def test_results_in_any_order(setup, oracle):
    eng, make, staged, data = setup
    plan = make()
    dst = eng.allocate(plan, fill=0)
    files = [staged(s) for s in range(4)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for step in range(1, 4):
        eng.execute_resident(plan, [files[step - 1]], dst, stream=streams[0].cuda_stream)  # nobody asks for these
        eng.execute_resident(plan, [files[step]], dst, stream=streams[step % 2].cuda_stream)
        sums, digests = _want(oracle, data(step))
        if step == 2:
            assert eng.digests(plan) == digests
        for _ in range(2):
            assert eng.checksums(plan) == sums
            assert eng.digests(plan) == digests
    eng.execute(plan, dst)
    assert (eng.checksums(plan), eng.digests(plan)) == _want(oracle, data(0))
    eng.execute_resident(plan, [files[1]], dst, stream=streams[1].cuda_stream)
    assert (eng.checksums(plan), eng.digests(plan)) == _want(oracle, data(1))
    eng.set_fused_digests(False)
    eng.execute_resident(plan, [files[2]], dst)
    assert eng.checksums(plan) == _want(oracle, data(2))[0]
    with pytest.raises(Exception, match="did not accumulate digests"):
        eng.digests(plan)


def test_a_captured_launch_is_asked_anew(setup, oracle):
    eng, make, staged, data = setup
    plan = make()
    dst = eng.allocate(plan, fill=0)
    src = staged(1)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    eng.execute_resident(plan, [src], dst, stream=stream.cuda_stream)
    assert (eng.checksums(plan), eng.digests(plan)) == _want(oracle, data(1))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        eng.execute_resident(plan, [src], dst, stream=stream.cuda_stream)
    for seed in (2, 3, 1, 2):
        src.copy_(staged(seed))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert (eng.checksums(plan), eng.digests(plan)) == _want(oracle, data(seed))
    src.copy_(staged(3))
    torch.cuda.synchronize()
    eng.execute_resident(plan, [src], dst)  # and an eager run of a plan that has been captured
    assert (eng.checksums(plan), eng.digests(plan)) == _want(oracle, data(3))


def test_a_plan_goes_away_with_its_results_under_way(setup):
    eng, make, staged, _ = setup
    src = staged(1)
    for _ in range(8):
        plan = make()
        dst = eng.allocate(plan)
        eng.execute_resident(plan, [src], dst)
        plan.close()
    torch.cuda.synchronize()
