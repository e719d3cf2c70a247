"""Every bit pattern through the woven transposes, NaN, infinities and subnormals among them: the bytes are those of the
wavefront-autonomous form, which the conversion tests hold against torch."""

import pytest
import torch

from modelexpress_amd.engine import set_transpose_form

pytestmark = pytest.mark.gpu

# source / destination element bytes, conversion
TYPES = [(1, 1, 0), (2, 2, 0), (4, 4, 0), (4, 2, 1), (2, 4, 2), (2, 4, 3), (4, 2, 4), (1, 2, 5), (2, 2, 6), (2, 2, 7)]


@pytest.mark.parametrize("es, ed, cast", TYPES)
@pytest.mark.parametrize("rows, cols, batch", [(12, 4099, 50), (40, 2053, 30)])
def test_any_bits(gpu_engine, es, ed, cast, rows, cols, batch):
    gen = torch.Generator("cuda").manual_seed(es + 10 * cast)
    src = torch.randint(0, 256, (batch * rows * cols * es,), generator=gen, device="cuda", dtype=torch.uint8)
    if es > 1:  # exponents of all ones and of zero as often as the rest
        top = src.view(-1, es)[:, -2:]
        pick = torch.randint(0, 4, (top.shape[0],), generator=gen, device="cuda")
        top[pick == 0] |= torch.tensor([0x80, 0x7F], dtype=torch.uint8, device="cuda")
        top[pick == 1] &= torch.tensor([0x7F, 0x80], dtype=torch.uint8, device="cuda")
    out = [torch.zeros(batch * rows * cols * ed, dtype=torch.uint8, device="cuda") for _ in range(2)]
    made = [{"src": src, "dst": o, "shape": (batch, cols, rows), "elem_size": ed, "src_strides": (rows * cols, 1, cols), "cast": cast} for o in out]
    assert gpu_engine.describe_views(made[:1])[0][:2] == ("staged_tile", rows)
    gpu_engine.copy_views(made[:1])
    set_transpose_form(1)
    try:
        assert gpu_engine.describe_views(made[1:])[0][0] == "transpose"
        gpu_engine.copy_views(made[1:])
    finally:
        set_transpose_form(0)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
