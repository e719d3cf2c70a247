"""Transposed views recorded into a HIP graph: every replay moves what the call described, whatever the engine ran between
the replays, and the engine's other calls go on working after the capture."""

import pytest
import torch

from modelexpress_amd.engine import PlacementEngine

pytestmark = pytest.mark.gpu


# one shape in the wavefront form, several shapes, the staged and the woven form alike and mixed
@pytest.mark.parametrize("shapes", [((300, 70),), ((300, 70), (41, 65), (520, 130)), ((16, 65536),) * 3, ((12, 60000), (24, 50000), (300, 70)),
                                    ((512, 640),) * 5])
def test_replays_stand_on_their_own(shapes):
    gen = torch.Generator(device="cuda").manual_seed(7)
    eng = PlacementEngine(0, ring_slots=2, slot_bytes=1 << 16, reader_threads=1, streams=1)
    srcs = [torch.randn(ni, nj, generator=gen, device="cuda").bfloat16() for ni, nj in shapes]
    outs = [torch.empty(nj, ni, dtype=torch.bfloat16, device="cuda") for ni, nj in shapes]
    views = [{"src": s, "dst": o, "shape": tuple(o.shape), "src_strides": (1, s.shape[1]), "elem_size": 2} for s, o in zip(srcs, outs)]
    other = torch.randn(70, 90, generator=gen, device="cuda")
    across = [torch.empty(90, 70, device="cuda") for _ in range(3)]
    others = [{"src": other, "dst": a, "shape": (90, 70), "src_strides": (1, 90), "elem_size": 4} for a in across]
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    eng.copy_views(views, stream=stream.cuda_stream)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        eng.copy_views(views, stream=stream.cuda_stream)
    for _ in range(3):
        for s in srcs:
            s.copy_(torch.randn(s.shape, generator=gen, device="cuda"))
        for o in [*outs, *across]:
            o.zero_()
        for _ in range(3):
            eng.copy_views(others)
            eng.checksum32([other])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for s, o in zip(srcs, outs):
            assert torch.equal(o, s.t())
        for a in across:
            assert torch.equal(a, other.t())
    eng.close()
