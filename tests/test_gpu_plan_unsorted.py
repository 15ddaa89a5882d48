"""Schedules of graphs whose rows do not ascend, built on the device: rows that are cut are ordered in the
schedule's own copy of the indices (stably), the others keep their order, and the item list equals the
host scheduler's."""
import ctypes

import numpy as np
import pytest
import torch

from neutronbench_amd import abi
from neutronbench_amd.abi import call, ptr
from neutronbench_amd.layout import SpmmPlan
from test_plan_schedule import power_law_block, schedule

pytestmark = pytest.mark.gpu


def _arrays(co, ri, device, base=0):
    return (torch.from_numpy(co.view(np.int32)).to(device), torch.from_numpy((ri + np.uint32(base)).view(np.int32)).to(device))


@pytest.mark.parametrize("chunk,slabs", [(512, 32), (64, 8), (16, 3)])
@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("base", [0, 5000])
def test_unsorted_rows(device, chunk, slabs, mixed, base):
    """mixed = 1: only every third row is out of order; Vs = 257 makes most neighbours parallel edges."""
    Vd, Vs, F = 700, 257 if mixed else 3000, 20
    co, ri, deg = power_law_block(Vd, Vs, 5, sort_rows=False, hubs=(70000, 9000, chunk, chunk + 1, chunk // 4, chunk // 4 + 1))
    if mixed:
        for r in range(Vd):
            if r % 3:
                ri[co[r]:co[r + 1]].sort()
    want, n_splits, n_partials = schedule(co, ri, Vs, chunk, slabs)
    co_d, ri_d = _arrays(co, ri, device, base)
    handle, s = ctypes.c_void_p(), torch.cuda.current_stream().cuda_stream
    call("nts_spmm_plan_create_slabs", ctypes.byref(handle), ptr(co_d), ptr(ri_d), base, Vs, Vd, int(co[-1]), chunk, slabs, s)
    items = np.zeros((want.shape[0], 4), dtype=np.uint32)
    call("nts_spmm_plan_copy_schedule", handle, items.ctypes.data, items.shape[0], None, 0)
    assert np.array_equal(items, want)
    # parallel edges are counted in the index array that the schedule gathers through
    cut_above, repeated = (chunk // 4 if slabs >= 8 else chunk), 0
    for r in range(Vd):
        row = ri[co[r]:co[r + 1]]
        row = np.sort(row) if row.size > cut_above else row
        repeated += int((row[1:] == row[:-1]).sum())
    rep = ctypes.c_uint64()
    call("nts_spmm_plan_scratch_info", handle, F, None, None, ctypes.byref(rep), None)
    assert rep.value == repeated
    # the gather through the copy, weights in the caller's order: integers, so that any order gives the same sums
    x = torch.randint(-8, 9, (Vs, F), device=device).float()
    w = torch.randint(1, 4, (int(co[-1]),), device=device).float()
    out = torch.empty(Vd, F, device=device)
    call("nts_spmm_gather_planned", handle, ptr(x), ptr(out), ptr(w), ptr(co_d), ptr(ri_d), base, F, 0, s)
    own = torch.repeat_interleave(torch.arange(Vd, device=device), torch.from_numpy(deg).to(device))
    ref = torch.zeros(Vd, F, device=device).index_add_(0, own, x[torch.from_numpy(ri.astype(np.int64)).to(device)] * w[:, None])
    assert torch.equal(out, ref)
    call("nts_spmm_plan_destroy", handle)


def test_offsets_are_checked_before_they_are_followed(device):
    ri = torch.zeros(7, dtype=torch.int32, device=device)
    for off in ([0, 3, 2, 6, 7], [0, 1, 2, 3, 6]):
        co = torch.tensor(off, dtype=torch.int32, device=device)
        handle = ctypes.c_void_p()
        assert abi.status("nts_spmm_plan_create_slabs", ctypes.byref(handle), ptr(co), ptr(ri), 0, 9, 4, 7, 16, 4,
                          torch.cuda.current_stream().cuda_stream) == abi.NTS_ERR_INVALID
        assert not handle.value and "offsets" in abi.last_error()


def test_edges_before_the_first_row_stay_out_of_it(device):
    """offsets[0] > 0: those edges belong to no row and carry a source that no row has; row 0 is a hub."""
    Vd, Vs, F = 700, 3000, 20
    co, ri, deg = power_law_block(Vd + 3, Vs, 5, sort_rows=False, hubs=(9000, 600))
    co, deg = co[3:].copy(), deg[3:]
    lead = int(co[0])
    assert lead and deg[0] == 9000
    ri %= np.uint32(Vs - 1)
    ri[:lead] = Vs - 1
    want, _, _ = schedule(co, ri, Vs, 64, 8)
    co_d, ri_d = _arrays(co, ri, device)
    handle, s = ctypes.c_void_p(), torch.cuda.current_stream().cuda_stream
    call("nts_spmm_plan_create_slabs", ctypes.byref(handle), ptr(co_d), ptr(ri_d), 0, Vs, Vd, int(co[-1]), 64, 8, s)
    items = np.zeros((want.shape[0], 4), dtype=np.uint32)
    call("nts_spmm_plan_copy_schedule", handle, items.ctypes.data, items.shape[0], None, 0)
    assert np.array_equal(items, want)
    x = torch.randint(-8, 9, (Vs, F), device=device).float()
    x[Vs - 1] = 1e9
    out = torch.empty(Vd, F, device=device)
    call("nts_spmm_gather_planned", handle, ptr(x), ptr(out), 0, ptr(co_d), ptr(ri_d), 0, F, 0, s)
    own = torch.repeat_interleave(torch.arange(Vd, device=device), torch.from_numpy(deg).to(device))
    ref = torch.zeros(Vd, F, device=device).index_add_(0, own, x[torch.from_numpy(ri[lead:].astype(np.int64)).to(device)])
    assert torch.equal(out, ref)
    call("nts_spmm_plan_destroy", handle)


def test_one_row_of_many_edges(device):
    n = 300000
    ri = torch.randperm(n, device=device).to(torch.int32)
    co = torch.tensor([0, n], dtype=torch.int32, device=device)
    plan = SpmmPlan(co, 1, n, 512, ri, n, 32)
    x, out = torch.ones(n, 4, device=device), torch.empty(1, 4, device=device)
    call("nts_spmm_gather_planned", plan.handle, ptr(x), ptr(out), 0, ptr(co), ptr(ri), 0, 4, 0,
         torch.cuda.current_stream().cuda_stream)
    assert out.tolist() == [[float(n)] * 4]
    plan.close()


def test_memory_of_destroyed_schedules_is_reused_and_given_back(device):
    """Schedules made and dropped over and over: the same results, and nts_scratch_trim frees what lies idle."""
    Vd, Vs, F = 700, 3000, 20
    co, ri, deg = power_law_block(Vd, Vs, 5, sort_rows=False, hubs=(200000,))
    co_d, ri_d = _arrays(co, ri, device)
    x = torch.randint(-8, 9, (Vs, F), device=device).float()
    out, first, s = torch.empty(Vd, F, device=device), None, torch.cuda.current_stream().cuda_stream
    for k in range(6):
        plan = SpmmPlan(co_d, Vd, int(co[-1]), 64, ri_d, Vs, 8)
        call("nts_spmm_gather_planned", plan.handle, ptr(x), ptr(out), 0, ptr(co_d), ptr(ri_d), 0, F, 0, s)
        plan.close()
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
        if k % 2:
            call("nts_scratch_trim")
