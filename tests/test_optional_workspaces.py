"""Choice of the optional, larger workspaces against the HBM that is there (no GPU).

The split launches take more workspace than a call needs.  It is asked for only
where it fits, because an allocation that does not fit makes the caching
allocator release every block it holds before it raises.
"""

import pytest
import torch

import gemma4_fa4_amd as g
from gemma4_fa4_amd import attention as att

CPU = torch.device("cpu")


class _Hbm:
    """Stands for the device: free bytes, allocator's bytes, and the sizes asked of it."""

    def __init__(self, monkeypatch, free, reserved=0, allocated=0, refuse_above=None):
        self.asked = []
        empty = torch.empty

        def recorded(size, **kw):
            self.asked.append(size)
            if refuse_above is not None and size > refuse_above:
                raise torch.OutOfMemoryError("no room")
            return empty(0, **kw)

        monkeypatch.setattr(att, "_free_hbm", self.free_hbm)
        monkeypatch.setattr(torch.cuda, "memory_reserved", lambda _d: reserved)
        monkeypatch.setattr(torch.cuda, "memory_allocated", lambda _d: allocated)
        monkeypatch.setattr(torch, "empty", recorded)
        self.free, self.readings = free, 0

    def free_hbm(self, _device):
        self.readings += 1
        return self.free


def _forward_plan(new=16, keys=4096):
    q = torch.empty(1, new, 32, 512, dtype=torch.bfloat16)
    k = torch.empty(1, keys, 4, 512, dtype=torch.bfloat16)
    plan = att._fixed_plan(q, k, g.GLOBAL_ATTENTION)
    need, most = plan.workspace_bytes(0), plan.workspace_bytes(3)
    assert most > need, "the problem is not split"
    return plan, need, most


def test_forward_takes_the_larger_workspace_that_fits(monkeypatch):
    plan, _, most = _forward_plan()
    hbm = _Hbm(monkeypatch, free=most)
    _, nbytes = plan._forward_workspace(plan.problem(), CPU)
    assert nbytes == most and hbm.asked == [most]


@pytest.mark.parametrize("new,keys", [(16, 4096), (1, 8192)])
def test_forward_on_a_full_device_asks_only_for_what_it_needs(monkeypatch, new, keys):
    plan, need, most = _forward_plan(new, keys)
    hbm = _Hbm(monkeypatch, free=most - 1, reserved=1 << 38, allocated=(1 << 38) - most + 1)
    _, nbytes = plan._forward_workspace(plan.problem(), CPU)
    assert nbytes == need and hbm.asked == ([need] if need else [])


def test_forward_counts_the_blocks_that_the_allocator_holds(monkeypatch):
    plan, _, most = _forward_plan()
    hbm = _Hbm(monkeypatch, free=0, reserved=1 << 38, allocated=(1 << 38) - most)
    _, nbytes = plan._forward_workspace(plan.problem(), CPU)
    assert nbytes == most and hbm.asked == [most]


def test_forward_falls_back_and_reads_afresh_when_the_reading_was_stale(monkeypatch):
    plan, need, most = _forward_plan()
    hbm = _Hbm(monkeypatch, free=most, refuse_above=need)
    _, nbytes = plan._forward_workspace(plan.problem(), CPU)
    assert nbytes == need and hbm.asked[0] == most and hbm.readings == 2


# ---- backward: the split dK/dV launch ----------------------------------------


def _backward_plan():
    q = torch.empty(1, 1000, 32, 512, dtype=torch.bfloat16)
    k = torch.empty(1, 1000, 4, 512, dtype=torch.bfloat16)
    plan = att._fixed_plan(q, k, g.GLOBAL_ATTENTION)
    plan.global_backward = True
    need, most = plan.workspace_bytes(1), plan.workspace_bytes(2)
    assert most > need, "the problem is not split"
    return plan, q, k, need, most


def _free_for(budget):  # free bytes whose guarded budget is `budget`
    return max(budget * 5 // 4 + 4, budget + 2 * 1024 ** 3)


def _refit_and_ask(monkeypatch, beyond, **hbm_kw):
    """Sizes asked for with ``beyond`` bytes free past what the backward needs."""
    plan, q, k, need, most = _backward_plan()
    free = _free_for(att._backward_additional_bytes(plan, q, k, k) + beyond)
    hbm = _Hbm(monkeypatch, free=free, **hbm_kw)
    att._refit_backward(plan, q, k, k)
    plan._workspace(1, CPU)
    return hbm.asked, need, most


def test_backward_is_split_where_its_workspace_fits(monkeypatch):
    _, _, _, need, most = _backward_plan()
    asked, _, _ = _refit_and_ask(monkeypatch, most - need)
    assert asked == [most]


def test_backward_is_not_split_on_a_full_device(monkeypatch):
    _, _, _, need, most = _backward_plan()
    asked, _, _ = _refit_and_ask(monkeypatch, most - need - 1, reserved=most, allocated=1)
    assert asked == [need]


def test_backward_counts_the_blocks_that_the_allocator_holds(monkeypatch):
    # A training process's allocator has taken nearly all of the HBM.
    _, _, _, _, most = _backward_plan()
    asked, _, _ = _refit_and_ask(monkeypatch, 0, reserved=most + 5, allocated=5)
    assert asked == [most]


def test_backward_falls_back_when_the_larger_workspace_is_refused(monkeypatch):
    _, _, _, need, most = _backward_plan()
    asked, _, _ = _refit_and_ask(monkeypatch, most, refuse_above=need)
    assert asked == [most, need]


@pytest.mark.parametrize("pin", [-1, 0, 1 << 34])
def test_pinned_backward_is_never_split(monkeypatch, pin):
    previous = g.pin_backward_ds_budget(pin)
    try:
        plan, q, k, _, most = _backward_plan()
        hbm = _Hbm(monkeypatch, free=1 << 50, reserved=1 << 50)
        att._refit_backward(plan, q, k, k)
        plan._workspace(1, CPU)
        assert hbm.asked == [plan.workspace_bytes(1)] and hbm.asked[0] < most
    finally:
        g.pin_backward_ds_budget(previous)
