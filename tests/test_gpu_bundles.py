"""Segments that one wavefront of a bundle moves: edges of runs off the 16-byte grid, buffers and last pieces of around
one unit a lane, one to a few bundles of them, beside full tiles and alone; copies, every conversion, checksums and
digests, and nothing written around them.  Moves and conversions have one correct answer."""

import pytest
import torch

from modelexpress_amd.engine import PlacementEngine

pytestmark = pytest.mark.gpu

CASTS = {("F32", "BF16"): 1, ("BF16", "F32"): 2, ("F16", "F32"): 3, ("F32", "F16"): 4, ("F8_E4M3", "BF16"): 5,
         ("F16", "BF16"): 6, ("BF16", "F16"): 7}
TORCH = {"U8": torch.uint8, "BF16": torch.bfloat16, "F16": torch.float16, "F32": torch.float32, "F8_E4M3": torch.float8_e4m3fn}
TILE, UNIT = 128 * 1024, 16
SIZES = [1, 15, 16, 17, 63 * UNIT, 64 * UNIT, 64 * UNIT + 1, 65 * UNIT, TILE, TILE + UNIT, TILE + 64 * UNIT, TILE + 64 * UNIT + 9,
         TILE + 65 * UNIT, 2 * TILE + 31, 4096, 74296]


def _buffers(sizes, lead, gen):
    """Sources of those sizes at odd places, guarded destinations `lead` bytes past the 16-byte grid."""
    srcs = [torch.randint(0, 256, (n + 19,), generator=gen, device="cuda", dtype=torch.uint8)[3:3 + n] for n in sizes]
    holds = [torch.full((32 + lead + n + 32,), 0xA5, dtype=torch.uint8, device="cuda") for n in sizes]
    return srcs, holds, [h[32 + lead:32 + lead + n] for h, n in zip(holds, sizes)]


def _guarded(holds, dsts):
    for h, d in zip(holds, dsts):
        at = d.data_ptr() - h.data_ptr()
        assert bool((h[:at] == 0xA5).all()) and bool((h[at + d.numel():] == 0xA5).all()), d.numel()


@pytest.mark.parametrize("lead", [0, 1, 8])
@pytest.mark.parametrize("count", [1, 2, 15, 16, 17, 33, len(SIZES)])
def test_copies_and_checksums(gpu_engine, oracle, lead, count):
    gen = torch.Generator("cuda").manual_seed(lead + count)
    sizes = SIZES if count == len(SIZES) else [(5 + 61 * k) % 1025 for k in range(count)]
    srcs, holds, dsts = _buffers(sizes, lead, gen)
    boxes = [{"src": s, "dst": d, "rows": 1, "row_bytes": n, "csum_group": k} for k, (s, d, n) in enumerate(zip(srcs, dsts, sizes))]
    sums = gpu_engine.place_boxes(boxes, len(boxes))
    for s, d, c in zip(srcs, dsts, sums):
        assert torch.equal(s, d)
        assert c == oracle.safe_checksum_bytes(s.cpu().numpy()), s.numel()
    _guarded(holds, dsts)
    assert gpu_engine.checksum32(srcs) == sums
    verify = gpu_engine.verify_plan(srcs)
    assert verify.checksums() == verify.checksums() == sums
    verify.close()


@pytest.mark.parametrize("src_dtype,dst_dtype", list(CASTS))
def test_conversions(gpu_engine, oracle, src_dtype, dst_dtype):
    gen = torch.Generator("cuda").manual_seed(7)
    es, ed = TORCH[src_dtype].itemsize, TORCH[dst_dtype].itemsize
    elems = [1, 3, 64 * 8 // ed, 64 * 16 // ed, 64 * 16 // ed + 1, TILE // ed + 5, TILE // max(es, ed) + 64 * 8 // ed] + [37 * k + 1 for k in range(20)]
    srcs = [(torch.randn(n + 3, generator=gen, device="cuda") * 0.5).to(TORCH[src_dtype])[3:] for n in elems]
    holds = [torch.full((32 + ed + n * ed + 32,), 0xA5, dtype=torch.uint8, device="cuda") for n in elems]
    dsts = [h[32 + ed:32 + ed + n * ed] for h, n in zip(holds, elems)]
    boxes = [{"src": s, "dst": d, "rows": 1, "row_bytes": d.numel(), "csum_group": k, "cast": CASTS[src_dtype, dst_dtype]}
             for k, (s, d) in enumerate(zip(srcs, dsts))]
    sums = gpu_engine.place_boxes(boxes, len(boxes))
    for s, d, c in zip(srcs, dsts, sums):
        want = s.to(TORCH[dst_dtype]).view(torch.uint8)
        assert torch.equal(d, want), s.numel()
        assert c == oracle.safe_checksum_bytes(want.cpu().numpy())
    _guarded(holds, dsts)


def test_digests(gpu_engine, oracle):
    gen = torch.Generator("cuda").manual_seed(9)
    sizes = SIZES + [2 * k + 1 for k in range(40)] + [4096 * 3 + 2, 4096 - 2]
    srcs, holds, dsts = _buffers(sizes, 0, gen)
    views = [{"src": s, "dst": d, "shape": (n,), "elem_size": 1} for s, d, n in zip(srcs, dsts, sizes)]
    plan = gpu_engine.view_plan(PlacementEngine.views_array(views), len(views))
    for _ in range(2):
        for s, d, g in zip(srcs, dsts, plan.run_digests()):
            assert torch.equal(s, d) and g == oracle.tensor_digest_bytes(s.cpu().numpy()), s.numel()
    _guarded(holds, dsts)
    plan.close()
