"""Views of three and four dimensions that move as row boxes: the rows of a box run along the longest outer dimension
where the destination is whole 16-byte units, along the last one otherwise.  Extents on both sides of that choice,
destinations with and without gaps, conversions, and the checksum's positions."""

import pytest
import torch

pytestmark = pytest.mark.gpu
CASTS = {(torch.float32, torch.bfloat16): 1, (torch.bfloat16, torch.float32): 2, (torch.float16, torch.bfloat16): 6}


@pytest.mark.parametrize("src_dtype,dst_dtype", [(torch.bfloat16, torch.bfloat16), (torch.uint8, torch.uint8)] + list(CASTS))
@pytest.mark.parametrize("shape", [(37, 5, 64), (5, 37, 64), (6, 6, 64), (200, 3, 24), (3, 40, 7, 48), (40, 3, 7, 48), (2, 3, 90, 16), (9, 4, 21)])
@pytest.mark.parametrize("gap", [0, 16, 3])
def test_row_boxes_of_many_dimensions(gpu_engine, oracle, src_dtype, dst_dtype, shape, gap):
    gen = torch.Generator("cuda").manual_seed(sum(shape))
    nd = len(shape)
    order = list(range(nd - 1))[::-1] + [nd - 1]  # the source holds the outer dimensions the other way round
    base = (torch.randn([shape[d] for d in order], generator=gen, device="cuda") * 50).to(src_dtype)
    src = base.permute([order.index(d) for d in range(nd)])
    dst_strides, n = [], 1
    for d in reversed(range(nd)):
        dst_strides.insert(0, n)
        n = n * shape[d] + (gap if d == nd - 1 else 0)
    room = torch.full((n + 64,), 0x5A, dtype=torch.uint8, device="cuda").repeat(torch.empty(0, dtype=dst_dtype).element_size()).view(dst_dtype)
    want = room.clone()
    want.as_strided(shape, dst_strides).copy_(src.to(dst_dtype))
    views = dict(src=src.data_ptr(), dst=room, shape=shape, elem_size=room.element_size(), src_strides=src.stride(),
                 dst_strides=dst_strides, cast=CASTS.get((src_dtype, dst_dtype), 0))
    got_sum = gpu_engine.copy_view(**views)
    assert torch.equal(room.view(torch.uint8), want.view(torch.uint8))
    # the checksum of the stored bytes at their distance from the view's first element
    mask = torch.zeros_like(room.view(torch.uint8)).view(dst_dtype)
    mask.view(torch.uint8).zero_()
    mask.as_strided(shape, dst_strides).copy_(want.as_strided(shape, dst_strides))
    assert got_sum == oracle.safe_checksum_bytes(mask.view(torch.uint8).cpu().numpy())
    room.view(torch.uint8).fill_(0x5A)
    gpu_engine.copy_views([views])
    torch.cuda.synchronize()
    assert torch.equal(room.view(torch.uint8), want.view(torch.uint8))
