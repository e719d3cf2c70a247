"""Transposed views whose rows start anywhere and end anywhere: every remainder of the 16-byte chunk on both sides,
views narrower than a chunk, sub-tiles with and without columns before them, pitches and offsets of odd elements,
each element size and conversion, guard bytes around the destination, and the checksum's positions."""

import pytest
import torch

pytestmark = pytest.mark.gpu
TYPES = {"b1": (torch.uint8, torch.uint8, 0), "b2": (torch.int16, torch.int16, 0), "b4": (torch.int32, torch.int32, 0),
         "b8": (torch.int64, torch.int64, 0), "narrow": (torch.float32, torch.bfloat16, 1), "widen": (torch.bfloat16, torch.float32, 2),
         "recode": (torch.float16, torch.bfloat16, 6), "fp8": (torch.float8_e4m3fn, torch.bfloat16, 5)}


@pytest.mark.parametrize("kind", list(TYPES))
@pytest.mark.parametrize("ni,nj", [(2, 2), (3, 7), (9, 3), (63, 17), (64, 64), (65, 130), (130, 65), (591, 70), (70, 591), (128, 33), (200, 1027)])
@pytest.mark.parametrize("lead,gap", [(0, 0), (1, 3), (3, 1), (8, 8)])
def test_transposed_view_at_any_edge(gpu_engine, oracle, kind, ni, nj, lead, gap):
    src_dtype, dst_dtype, cast = TYPES[kind]
    gen = torch.Generator("cuda").manual_seed(ni * 7 + nj)
    pitch = nj + gap
    raw = torch.randint(0, 200, (lead + ni * pitch + 8,), generator=gen, device="cuda")
    src_all = raw.to(src_dtype) if cast == 0 else (raw / 7 - 14).to(src_dtype)
    src = src_all.as_strided((nj, ni), (1, pitch), lead)
    es, ed = src_all.element_size(), torch.empty(0, dtype=dst_dtype).element_size()
    n = lead + nj * (ni + gap) + 64
    room = torch.full((n * ed,), 0x5A, dtype=torch.uint8, device="cuda").view(dst_dtype)
    want = room.clone()
    want.as_strided((nj, ni), (ni + gap, 1), lead).copy_(src.to(dst_dtype))
    got = gpu_engine.copy_view(src_all.data_ptr() + lead * es, room.data_ptr() + lead * ed, (nj, ni), ed, src_strides=(1, pitch),
                               dst_strides=(ni + gap, 1), cast=cast)
    assert torch.equal(room.view(torch.uint8), want.view(torch.uint8))
    stored = torch.zeros(n * ed, dtype=torch.uint8, device="cuda").view(dst_dtype)
    stored.as_strided((nj, ni), (ni + gap, 1), lead).copy_(src.to(dst_dtype))
    assert got == oracle.safe_checksum_bytes(stored.view(torch.uint8)[lead * ed:].cpu().numpy())
