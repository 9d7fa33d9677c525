"""The waits that staged kernels rely on, checked in the instructions of the built library: a
missing one would show in results only now and then."""
import heapq
import re

import pytest

from device_code import kernels, resources, waits


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


VMEM = re.compile(r"(global|buffer|flat)_(load|store|atomic)")


def to_lds(c):
    return c[2].endswith(" lds") or "load_lds" in c[1]


def predecessors(code):
    """Per instruction: the instructions that control can come from."""
    by_address = {c[0]: i for i, c in enumerate(code)}
    before = [[] for _ in code]
    for i, (_, op, _, to) in enumerate(code):
        if to in by_address:
            before[by_address[to]].append(i)
        if op not in ("s_branch", "s_endpgm") and i + 1 < len(code):
            before[i + 1].append(i)
    return before


def fewest_after(code, at, behind):
    """Fewest vector memory operations that a wave has issued, on any path to code[at], after
    its last-but-`behind` stage load; None where no path holds so many stage loads."""
    before = predecessors(code)
    best, queue = {}, [(0, at, 0)]
    while queue:
        ops, i, stages = heapq.heappop(queue)
        if best.setdefault((i, stages), ops) < ops:
            continue
        for j in before[i]:
            n, s = ops, stages
            if VMEM.match(code[j][1]):
                if to_lds(code[j]):
                    s += 1
                    if s > behind:
                        return ops
                n += 1
            if (j, s) not in best or best[j, s] > n:
                best[j, s] = n
                heapq.heappush(queue, (n, j, s))
    return None


def test_stationary_stage_arrival(stationary):
    """A stage's load has landed at its barrier: memory operations complete in order, so the
    wave may leave outstanding only as many as it has issued after that load, on every path.
    Operand loads that are counted there must not be merged, dropped or moved past the wait."""
    for name, code in stationary.items():
        waves = int(re.search(r"ILi(\d)ELi\dELi\dE", name)[1])
        slots, loads = (15, 1) if waves == 8 else (9, 2)
        checked = 0
        for i, (_, op, args, _) in enumerate(code):
            if op != "s_waitcnt" or "s_barrier" not in [c[1] for c in code[i:i + 5]]:
                continue
            allowed = waits(args)[0]
            if not allowed:
                continue
            issued = fewest_after(code, i, (slots - 3) * loads)
            assert issued is not None and allowed <= issued, (name, i, allowed, issued)
            checked += 1
        assert checked >= int(re.search(r"ELi(\d)ELi\dE", name)[1]) - 1, name


@pytest.mark.parametrize("kernel", ["gemm_bf16_nn_kernel", "gemm_bf16_nn_persist_kernel",
                                    "gemm_bf16_wgrad_kernel"])
def test_refilled_stage_was_read(kernel):
    """These kernels refill the slot of the stage before: its reads have returned when a wave
    arrives at the barrier in front of the stage loads, by the wait ahead of it."""
    for name, code in kernels(kernel).items():
        before, stages = predecessors(code), set()
        queue = [i for i, c in enumerate(code) if to_lds(c)]
        seen = set(queue)
        while queue:  # back from the stage loads to the barriers ahead of them
            i = queue.pop()
            if code[i][1] == "s_barrier":
                stages.add(i)
                continue
            new = [j for j in before[i] if j not in seen]
            seen.update(new)
            queue += new
        assert stages, name
        for i in stages:
            wait = [waits(c[2]) for c in code[max(i - 4, 0):i] if c[1] == "s_waitcnt"]
            assert any(vm is not None and lgkm == 0 for vm, lgkm in wait), name


def test_narrow_backward_keeps_its_sums_in_registers():
    """No variant of the narrow layer's backward spills (its tail once held every partial sum
    of a workgroup in one wave)."""
    for name, r in resources("narrow_bwd_vec_kernel").items():
        assert r["vgpr_spill_count"] == 0 and r["private_segment_fixed_size"] == 0, name
