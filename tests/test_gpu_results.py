"""Results handed to the host by the kernel that folds accumulators and hashes digests: one record per buffer, at
counts around its four wavefronts per workgroup, the first growth of the result block and the grid's own limit, for
buffers with and without whole rows, words after them and ragged bytes."""

import numpy as np
import pytest
import torch

from modelexpress_amd.engine import digest_from_scalars

pytestmark = pytest.mark.gpu

ROW = 4096  # a tensor_digest row
SIZES = [0, 1, 3, 4, 7, 8, ROW - 1, ROW, ROW + 1, ROW + 4, 2 * ROW + 6, 33 * ROW, 33 * ROW + 12 + 3]


@pytest.mark.parametrize("n", [1, 3, 4, 5, 13, 1024, 1025, 16385 + 4])
def test_checksums_and_digests_of_many_buffers(gpu_engine, oracle, n):
    rng = np.random.default_rng(n)
    small = [s for s in SIZES if s <= 8] if n > 2000 else SIZES
    sizes = [small[(k * 5 + n) % len(small)] for k in range(n)]
    offsets = np.concatenate([[0], np.cumsum([(s + 31) // 16 * 16 for s in sizes])])
    host = rng.integers(0, 256, int(offsets[-1]) + 16, dtype=np.uint8)
    dev = torch.from_numpy(host).cuda()
    ptrs = [dev.data_ptr() + int(o) for o in offsets[:-1]]
    parts = [host[int(o):int(o) + s] for o, s in zip(offsets, sizes)]
    want = [oracle.tensor_digest_bytes(p) for p in parts]
    want_sums = [oracle.safe_checksum_bytes(p) for p in parts]
    assert gpu_engine.digest(ptrs, sizes) == want
    assert gpu_engine.checksum32(ptrs, sizes) == want_sums
    assert gpu_engine.fingerprint(ptrs, sizes) == (want_sums, want)
    plan = gpu_engine.verify_plan(ptrs, sizes)
    for _ in range(2):  # a run leaves the accumulators cleared for the next
        assert plan.digests() == want
        assert plan.checksums() == want_sums
    plan.close()
    got, scalars = gpu_engine.digest(ptrs[:13], sizes[:13], with_scalars=True)
    assert got == want[:13]
    assert [digest_from_scalars(sc) for sc in scalars] == want[:13]


@pytest.mark.parametrize("offset", [0, 2, 3, 8])
@pytest.mark.parametrize("rows", [511 * 32, 512 * 32])  # a workgroup takes 16 rows below 512 x 32, 32 from there on
def test_one_pass_over_large_buffers_at_any_address(gpu_engine, oracle, rows, offset):
    """Both workgroup shapes of the digest pass, whole and short last workgroups, buffers off the 16-byte grid:
    the pass that takes checksum and digest together against the two that take one each, and the smaller buffer
    against the oracle."""
    n = (rows - 33) * ROW
    dev = torch.randint(0, 256, (rows * ROW + 64,), dtype=torch.uint8, device="cuda", generator=torch.Generator("cuda").manual_seed(rows))
    ptrs = [dev.data_ptr() + offset, dev.data_ptr() + n + offset]
    sizes = [n, 33 * ROW + 5]
    sums, digests = gpu_engine.fingerprint(ptrs, sizes)
    assert sums == gpu_engine.checksum32(ptrs, sizes)
    assert digests == gpu_engine.digest(ptrs, sizes)
    small = dev[n + offset: n + offset + sizes[1]].cpu().numpy()
    assert (sums[1], digests[1]) == (oracle.safe_checksum_bytes(small), oracle.tensor_digest_bytes(small))
    shifted = dev[offset: offset + n].clone()  # the same bytes on the grid
    assert gpu_engine.fingerprint([shifted], [n]) == (sums[:1], digests[:1])
