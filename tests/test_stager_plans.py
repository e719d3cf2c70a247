"""The snapshot's lowered plan: closed with the stager, or given up for tensors that are refused, it is not run again."""

import pytest
import torch

from modelexpress_amd.publisher import WireStager


class Plan:
    def __init__(self, n):
        self.n, self.open = n, True
        self.bytes = 0

    def run(self, *, stream=0):
        assert self.open

    def run_digests(self, *, stream=0):
        assert self.open
        return ["d"] * self.n

    def close(self):
        self.open = False


class Engine:
    def __init__(self):
        self.lowered = 0

    def view_plan(self, arr, n):
        self.lowered += 1
        return Plan(n)


@pytest.mark.parametrize("digests", [False, True])
def test_a_closed_stager_lowers_its_plan_anew(digests):
    eng, state = Engine(), {"a": torch.zeros(3, 4), "b": torch.zeros(5, dtype=torch.bfloat16)}
    stager = WireStager(eng, publish_digests=digests)
    for lowered in (1, 2, 3):
        for _ in range(3):
            stager.stage(state)
        assert eng.lowered == lowered
        stager.close()


def test_a_refused_snapshot_leaves_no_closed_plan_behind():
    eng, state = Engine(), {"a": torch.zeros(3, 4)}
    stager = WireStager(eng)
    stager.stage(state)
    with pytest.raises(NotImplementedError, match="no conversion"):
        stager.stage({"a": torch.zeros(3, 4, dtype=torch.float64)})
    stager.stage(state)
    assert eng.lowered == 2
