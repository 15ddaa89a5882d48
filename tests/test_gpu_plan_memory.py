"""Memory that a destroyed schedule leaves to the next one: not before the work that uses it has ended, and not
at the cost of a capture that runs meanwhile."""
import ctypes

import numpy as np
import pytest
import torch

from neutronbench_amd import abi
from neutronbench_amd.abi import call, ptr
from neutronbench_amd.layout import SpmmPlan
from test_plan_schedule import power_law_block

pytestmark = pytest.mark.gpu


def _graph(device, seed):
    co, ri, deg = power_law_block(20000, 5000, seed, hubs=(60000, 9000))
    return torch.from_numpy(co.view(np.int32)).to(device), torch.from_numpy(ri.view(np.int32)).to(device), int(co[-1])


def _gather(plan, x, out, co, ri, stream):
    call("nts_spmm_gather_planned", plan.handle, ptr(x), ptr(out), 0, ptr(co), ptr(ri), 0, x.shape[1], 0, stream)


@pytest.mark.parametrize("slabs", [0, 8])
def test_destroyed_with_work_in_flight_on_another_stream(device, slabs):
    """The next schedule is of the same size and overwrites what the first one's calls read, if they still run."""
    F, rows, n_src = 64, 20000, 5000
    graphs = [_graph(device, s) for s in (3, 4)]
    x = torch.randint(-8, 9, (n_src, F), device=device).float()
    side, main = torch.cuda.Stream(), torch.cuda.current_stream()

    def plan_of(g):
        p = SpmmPlan(g[0], rows, g[2], 64, g[1], n_src, slabs) if slabs else SpmmPlan(g[0], rows, g[2], 64)
        p.reserve(F)
        return p

    want = []
    for g in graphs:
        p, out = plan_of(g), torch.empty(rows, F, device=device)
        _gather(p, x, out, g[0], g[1], main.cuda_stream)
        want.append(out)
        p.close()
    for _ in range(3):
        first = plan_of(graphs[0])
        outs = [torch.empty(rows, F, device=device) for _ in range(40)]
        done = torch.cuda.Event()
        side.wait_stream(main)
        for out in outs:
            _gather(first, x, out, graphs[0][0], graphs[0][1], side.cuda_stream)
        done.record(side)
        first.close()
        assert done.query()
        second, out2 = plan_of(graphs[1]), torch.empty(rows, F, device=device)
        _gather(second, x, out2, graphs[1][0], graphs[1][1], main.cuda_stream)
        assert torch.equal(out2, want[1])
        assert all(torch.equal(o, want[0]) for o in outs)
        second.close()


def test_destroyed_while_a_stream_is_captured(device):
    """In the relaxed mode, where freeing memory does not end a capture."""
    co, ri, edges = _graph(device, 5)
    plan = SpmmPlan(co, 20000, edges, 64)
    plan.reserve(16)
    x, y = torch.arange(1000.0, device=device), torch.zeros(1000, device=device)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        y.copy_(x * 2)
        assert abi.status("nts_spmm_plan_destroy", plan.handle) == 0
        plan.handle = None
    for k in range(3):
        x.fill_(k)
        graph.replay()
        torch.cuda.synchronize()
        assert bool((y == 2.0 * k).all())


def test_idle_memory_is_free_to_the_library_and_given_back(device):
    """A schedule with 1 GiB of partial sums: destroyed, it leaves nts_mem_info what it was, the next one of its size
    takes the same memory, and nts_scratch_trim returns it to the driver."""
    co = torch.arange(0, (1 << 21) + 1, 64, dtype=torch.int32, device=device)
    rows, edges = co.numel() - 1, int(co[-1])
    torch.cuda.synchronize()
    call("nts_scratch_trim")

    def library_free():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        call("nts_mem_info", ctypes.byref(free), ctypes.byref(total))
        return free.value

    before, slack = library_free(), 64 << 20
    for k in range(3):
        plan = SpmmPlan(co, rows, edges, 32)
        plan.reserve(1 << 12)
        used = before - library_free()
        assert used > (1 << 30) - slack
        driver = torch.cuda.mem_get_info()[0]
        plan.close()
        assert abs(library_free() - before) < slack
        assert abs(torch.cuda.mem_get_info()[0] - driver) < slack  # kept: the next schedule takes it
    call("nts_scratch_trim")
    assert torch.cuda.mem_get_info()[0] - driver > (1 << 30) - slack


def test_ordering_falls_back_to_the_host_without_memory_for_the_sort(device):
    """30 M edges in rows that do not ascend, with 640 MiB left on the device: the sort alone takes over 900 MB, the
    ordered copies 240.  The same schedule, and the same sums, as with all of the memory."""
    rows, n_src, edges, F = 3000, 100000, 30000000, 4
    g = torch.Generator(device=device).manual_seed(6)
    ri = torch.randint(0, n_src, (edges,), generator=g, device=device, dtype=torch.int32)
    co = torch.arange(0, edges + 1, edges // rows, dtype=torch.int32, device=device)
    x = torch.randint(-8, 9, (n_src, F), generator=g, device=device).float()

    def schedule_and_sums():
        plan = SpmmPlan(co, rows, edges, 512, ri, n_src, 8)
        items = np.zeros((plan.info()["items"], 4), dtype=np.uint32)
        call("nts_spmm_plan_copy_schedule", plan.handle, items.ctypes.data, items.shape[0], None, 0)
        out = torch.empty(rows, F, device=device)
        _gather(plan, x, out, co, ri, torch.cuda.current_stream().cuda_stream)
        plan.close()
        call("nts_scratch_trim")
        return items, out

    want, sums = schedule_and_sums()
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    fill = torch.empty(torch.cuda.mem_get_info()[0] - (640 << 20), dtype=torch.uint8, device=device)
    try:
        items, out = schedule_and_sums()
    finally:
        del fill
        torch.cuda.empty_cache()
    assert np.array_equal(items, want) and torch.equal(out, sums)
