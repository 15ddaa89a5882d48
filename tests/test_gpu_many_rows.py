"""Schedules of 2^28 rows and more: several threads a row or work item would be 2^32 of them, which no launch can have.
Nearly all rows are empty; the first and the last ones have edges, two of them enough to be cut."""
import pytest
import torch

from neutronbench_amd.abi import call, ptr
from neutronbench_amd.layout import SpmmPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F", [4, 16])
def test_rows_beyond_what_several_threads_each_can_cover(device, F):
    rows, V = (1 << 28) + 3, 1000
    if torch.cuda.mem_get_info(device)[0] < (rows * (120 + 4 * F)):
        pytest.skip("not enough memory free")
    g = torch.Generator(device=device).manual_seed(F)
    some = torch.tensor([0, 1, 5, 1 << 27, rows - 3, rows - 2, rows - 1], device=device)
    deg = torch.tensor([3, 700, 1, 40, 64, 65, 900], device=device)
    E = int(deg.sum())
    off = torch.zeros(rows + 1, dtype=torch.int32, device=device)
    off[some + 1] = deg.to(torch.int32)
    off.cumsum_(0)
    own = torch.repeat_interleave(torch.arange(len(some), device=device), deg)
    idx = torch.randint(V, (E,), generator=g, device=device)
    idx = idx[torch.argsort(own * V + idx)].to(torch.int32)  # ascending within a row
    x, w = torch.randn(V, F, generator=g, device=device), torch.rand(E, generator=g, device=device)
    plan = SpmmPlan(off, rows, E, 64, idx, V, 2)
    out = torch.full((rows, F), float("nan"), device=device)
    call("nts_spmm_gather_planned", plan.handle, ptr(x), ptr(out), ptr(w), ptr(off), ptr(idx), 0, F, 0,
         torch.cuda.current_stream().cuda_stream)
    terms = x.double()[idx.long()] * w.double()[:, None]
    want, size = (torch.zeros(len(some), F, dtype=torch.float64, device=device).index_add_(0, own, t) for t in (terms, terms.abs()))
    assert bool(((out[some].double() - want).abs() <= 902 * 2.0 ** -24 * size).all())
    out[some] = 0
    step = 1 << 26
    assert not any(bool(out[r:r + step].any()) for r in range(0, rows, step))
