"""Transposes into short destination rows that abut (a layer's heads): every element type and conversion, rows from two
elements to past the last length that goes through the woven form, source rows from 16 bytes to several tiles with
every kind of remainder, odd pitches, destinations off the 16-byte grid, batch dimensions, batches alike and mixed, and
nothing written around them.  Moves and conversions have one correct answer."""

import pytest
import torch

from modelexpress_amd.engine import PlacementEngine

pytestmark = pytest.mark.gpu

T = {"U8": torch.uint8, "F8_E4M3": torch.float8_e4m3fn, "BF16": torch.bfloat16, "F16": torch.float16, "F32": torch.float32}
PAIRS = [("U8", "U8", 0), ("BF16", "BF16", 0), ("F32", "F32", 0), ("F32", "BF16", 1), ("BF16", "F32", 2), ("F16", "F32", 3), ("F32", "F16", 4),
         ("F8_E4M3", "BF16", 5), ("F16", "BF16", 6), ("BF16", "F16", 7)]
# rows, columns, spare columns of the source pitch, elements the destination starts off the grid, batch dimensions
# (a call of less than 2 MB stays with the other forms: the first dozen are woven when all go out in one call)
CASES = [(2, 64, 0, 0, ()), (3, 17, 1, 0, (5,)), (5, 401, 3, 3, (2, 3)), (7, 16, 0, 0, ()), (8, 4096, 0, 0, (3,)), (16, 8192, 16, 0, (2, 2)),
         (17, 1031, 5, 7, ()), (24, 640, 0, 0, (7,)), (48, 1000, 24, 0, (2,)), (81, 257, 1, 0, ()), (88, 22, 242, 0, (6,)), (89, 300, 4, 1, ()),
         (2, 30001, 3, 1, (70,)), (5, 4001, 3, 3, (2, 60)), (12, 2050, 2, 0, (90,)), (16, 65536, 0, 0, (3,)), (24, 640, 0, 0, (140,)),
         (31, 333, 1, 1, (220,)), (64, 1029, 3, 0, (33,)), (80, 513, 0, 2, (60,)), (88, 300, 4, 1, (90,))]


def _source(dtype, n, gen):
    if dtype == "F32":
        return torch.randn(n, generator=gen, device="cuda")
    if dtype in ("F16", "BF16"):
        return torch.randn(n, generator=gen, device="cuda").to(T[dtype])
    raw = torch.randint(0, 127 if dtype == "F8_E4M3" else 256, (n,), generator=gen, device="cuda", dtype=torch.uint8)
    return raw.view(T[dtype])


def _prod(dims):
    out = 1
    for d in dims:
        out *= d
    return out


def _case(src_dtype, dst_dtype, cast, case, gen):
    ni, nj, spare, off, bdims = case
    es, ed = T[src_dtype].itemsize, T[dst_dtype].itemsize
    nb = _prod(bdims)
    src = _source(src_dtype, nb * ni * (nj + spare) + 64, gen)
    flat = src.view(torch.uint8)
    lead, n = 64 + off * ed, nb * nj * ni * ed
    buf = torch.full((lead + n + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    first = 3 * (spare > 0)  # source rows off the grid too
    b_src = [_prod(bdims[k + 1:]) * ni * (nj + spare) for k in range(len(bdims))]
    view = {"src": flat.data_ptr() + first * es, "dst": buf.data_ptr() + lead, "shape": (*bdims, nj, ni), "elem_size": ed,
            "src_strides": (*b_src, 1, nj + spare), "cast": cast}
    rows = torch.as_strided(src, (nb, ni, nj), (ni * (nj + spare), nj + spare, 1), first)
    want = rows.to(T[dst_dtype]).transpose(1, 2).contiguous().view(torch.uint8).reshape(-1)
    return view, buf, lead, want, src


def _check(buf, lead, want, what):
    n = want.numel()
    assert torch.equal(buf[lead:lead + n], want), what
    assert bool((buf[:lead] == 0xA5).all()) and bool((buf[lead + n:] == 0xA5).all()), what


@pytest.mark.parametrize("src_dtype,dst_dtype,cast", PAIRS)
def test_short_rows_that_abut(gpu_engine, oracle, src_dtype, dst_dtype, cast):
    gen = torch.Generator("cuda").manual_seed(11)
    made = [_case(src_dtype, dst_dtype, cast, c, gen) for c in CASES]
    for c, (view, buf, lead, want, src) in zip(CASES, made):  # one by one, with the checksum
        got = gpu_engine.copy_view(view["src"], view["dst"], view["shape"], view["elem_size"], src_strides=view["src_strides"], cast=cast)
        _check(buf, lead, want, c)
        assert got == oracle.safe_checksum_bytes(want.cpu().numpy()), c
        buf.fill_(0xA5)
    torch.cuda.synchronize()
    views = [m[0] for m in made]
    gpu_engine.copy_views(views)  # all in one call
    for c, (view, buf, lead, want, src) in zip(CASES, made):
        _check(buf, lead, want, c)
        buf.fill_(0xA5)
    torch.cuda.synchronize()
    plan = gpu_engine.view_plan(PlacementEngine.views_array(views), len(views))
    for _ in range(2):
        plan.run()
        for c, (view, buf, lead, want, src) in zip(CASES, made):
            _check(buf, lead, want, c)
    plan.close()


@pytest.mark.parametrize("n_items", [2, 97])
@pytest.mark.parametrize("case", [(16, 2048, 0, 0, (3,)), (12, 1001, 1, 0, ())])
def test_batches_of_one_shape(gpu_engine, n_items, case):
    """Items that share a descriptor travel as kernel arguments, 96 to a launch."""
    gen = torch.Generator("cuda").manual_seed(12)
    made = [_case("BF16", "BF16", 0, case, gen) for _ in range(n_items)]
    torch.cuda.synchronize()
    gpu_engine.copy_views([m[0] for m in made])
    for k, (view, buf, lead, want, src) in enumerate(made):
        _check(buf, lead, want, k)


def test_which_rows_are_woven(gpu_engine):
    """A tile of the woven form holds all the rows of the view."""
    def form(ni, nj, es=2, batch=1):
        view = {"src": 1 << 20, "dst": 1 << 40, "shape": (batch, nj, ni), "elem_size": es, "src_strides": (ni * nj, 1, nj)}
        return gpu_engine.describe_views([view])[0][:2]

    assert form(12, 1 << 17) == form(12, (1 << 17) - 1) == ("staged_tile", 12)
    assert form(88, 300, 2, 80) == ("staged_tile", 88) and form(80, 300, 1, 160) == ("staged_tile", 80)
    assert form(89, 300, 2, 80)[0] == form(81, 300, 1, 160)[0] == "transpose"  # the wavefront form from there on
    assert form(12, 7, 2, 1 << 20)[0] == "transpose"                           # source rows of less than 16 bytes
    assert form(12, 8192)[0] == "transpose"                                    # a call of less than 2 MB
    assert form(16, 1 << 17, 4) == ("staged_tile", 16) and form(64, 1 << 17) == ("staged_tile", 64)  # panels


@pytest.mark.parametrize("small", [1, 3])
@pytest.mark.parametrize("large", [(112, 8000, 0, 0, ()), (700, 900, 3, 1, (2,)), (40, 30, 1, 0, ())])
def test_short_rows_beside_others_in_one_call(gpu_engine, small, large):
    """Transposes of one call are shaped together: a few woven views beside others, in two element types, with row boxes."""
    gen = torch.Generator("cuda").manual_seed(13)
    made = [_case("F32", "F32", 0, (56, 112, 0, 0, ()), gen) for _ in range(small)] + [_case("F32", "F32", 0, large, gen)]
    made += [_case("BF16", "F32", 2, (24, 1000, 0, 0, ()), gen), _case("BF16", "F32", 2, (12, 60000, 1, 0, ()), gen)]
    rows = torch.randn(300, 70, generator=gen, device="cuda")
    flat = torch.zeros(300 * 40, device="cuda")
    box = {"src": rows[:, 3:].data_ptr(), "dst": flat, "shape": (300, 40), "elem_size": 4, "src_strides": (70, 1)}
    torch.cuda.synchronize()
    views = [m[0] for m in made] + [box]
    plan = gpu_engine.view_plan(PlacementEngine.views_array(views), len(views))
    for run in (lambda: gpu_engine.copy_views(views), plan.run, lambda: gpu_engine.copy_views(views)):
        run()
        for k, (view, buf, lead, want, src) in enumerate(made):
            _check(buf, lead, want, k)
            buf.fill_(0xA5)
        assert torch.equal(flat.view(300, 40), rows[:, 3:43])
        flat.zero_()
        torch.cuda.synchronize()
    plan.close()
