"""No placement kernel keeps scalar registers in lanes of vector registers: what a small launch waits for is the chain of
dependent loads at its start, and spilled registers lengthen it."""

import pytest

from test_kernel_registers import kernels  # noqa: F401


@pytest.mark.parametrize("name", ["place_kernel", "place_ragged_kernel", "place_digest_kernel", "place_digest_ragged_kernel", "checksum_kernel"])
def test_scalar_registers_stay_scalar(kernels, name):  # noqa: F811
    [mine] = [k for mangled, k in kernels.items() if f"{len(name)}{name}E" in mangled]
    assert mine[".sgpr_spill_count"] == 0
