"""The waits that staged kernels rely on, checked in the instructions of the built library: a
missing one would show in results only now and then."""
import re

import pytest

from device_code import kernels, waits


@pytest.fixture(scope="module")
def stationary():
    return kernels("gemm_bf16_ws_kernel")


def barrier_waits(code):
    """Per barrier that follows LDS reads: the waits between the last read and the barrier."""
    out, reads, since = [], 0, []
    for _, op, args, _ in code:
        if op.startswith("ds_read"):
            reads, since = reads + 1, []
        elif op == "s_waitcnt":
            since.append(waits(args))
        elif op == "s_barrier":
            if reads:
                out.append((reads, since))
            reads, since = 0, []
    return out


def test_stationary_stage_slots(stationary):
    """A stage is loaded into the slot that was read two stages before: at its barrier no more
    reads may be outstanding than the last stage's eight."""
    assert len(stationary) == 42
    for name, code in stationary.items():
        stages = barrier_waits(code)
        assert len(stages) >= int(re.search(r"ELi(\d)ELi\dE", name)[1]) - 1, name
        for reads, since in stages:
            assert reads == 8, name
            assert any(lgkm is not None and lgkm <= 8 for _, lgkm in since), name
