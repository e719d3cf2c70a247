"""The kernel that reads the pinned ingest ring: a launch walks its work list with at most eight workgroups, so the
lists that can go wrong are those around a multiple of that, with a last tile that is short."""

import numpy as np
import pytest

from modelexpress_amd import models, synth
from modelexpress_amd.engine import Checkpoint, ParamSpec, PlacementEngine, PlacementPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("digests", [False, True])
@pytest.mark.parametrize("src,dst", [("F16", "F16"), ("F32", "BF16")])
@pytest.mark.parametrize("tiles,rest", [(1, 0), (7, 4), (8, 0), (8, 2), (9, 0), (16, 6), (17, 0), (40, 1022)])
def test_ring_launches_around_their_workgroup_count(mxp, oracle, tmp_path, tiles, rest, src, dst, digests):
    n = (tiles * 1024 + rest) // 2  # tiles of 1 KiB of destination bytes, then `rest` more
    n += rest % 2
    tensors = [models.TensorSpec("w", src, (n,)), models.TensorSpec("b", src, (3,))]
    synth.write_checkpoint(tensors, str(tmp_path), seed=tiles)
    eng = PlacementEngine(0, ring_slots=2, slot_bytes=1 << 16, reader_threads=2, streams=2, tile_bytes=1024 * (2 if src == "F32" else 1))
    ck = Checkpoint(str(tmp_path))
    plan = PlacementPlan(ck, [ParamSpec(t.name, dst, t.shape) for t in tensors], allow_cast=True)
    bufs = eng.allocate(plan, fill=0xEE)
    eng.set_fused_digests(digests)
    eng.execute(plan, bufs)
    sums = eng.checksums(plan)
    got_digests = eng.digests(plan) if digests else None
    raw = np.fromfile(tmp_path / "model.safetensors", dtype=np.uint8)
    for k, e in enumerate(ck.tensors()):
        want = raw[e.file_offset:e.file_offset + e.nbytes]
        if src == "F32":
            want = oracle.cast_f32_bf16_bits(want.view(np.uint32)).view(np.uint8)
        i = [p.name for p in plan.params].index(e.name)
        assert np.array_equal(bufs[i].cpu().numpy(), want)
        assert sums[i] == oracle.safe_checksum_bytes(want)
        if digests:
            assert got_digests[i] == oracle.tensor_digest_bytes(want)
    eng.close()
