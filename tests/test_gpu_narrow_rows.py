"""Aggregation of narrow rows: widths that are no multiple of four and rows off 16-byte boundaries, whose last lane
shares columns with the lane before it; both sides of the lines between lanes of one and of four floats."""
import pytest
import torch

from neutronbench_amd import synth
from neutronbench_amd.abi import call, ptr
from neutronbench_amd.layout import SpmmPlan

pytestmark = pytest.mark.gpu


def graph(rows, edges, seed, device):
    src, dst = synth.rmat_edges(rows, edges, seed=seed, device=device, sort=True)
    order = torch.sort(dst, stable=True).indices
    off = torch.zeros(rows + 1, dtype=torch.int64, device=device)
    off[1:] = torch.bincount(dst, minlength=rows).cumsum(0)
    return off.to(torch.int32), src[order].to(torch.int32).contiguous(), dst[order]


def shifted(t, by):
    """The same values, `by` floats off the start of an allocation, NaN on both sides."""
    buf = torch.full((t.numel() + 8,), float("nan"), device=t.device)
    out = buf[by:by + t.numel()].view(t.shape)
    out.copy_(t)
    return buf, out


def check(device, rows, off, idx, dst, H, Fh, by, run):
    """Each element is a chain of at most `longest` multiply-adds: off by at most longest * 2^-24 of the sum of its
    terms' sizes (and one more rounding with what was there)."""
    g = torch.Generator(device=device).manual_seed(17 * H + Fh)
    F, E = H * Fh, idx.numel()
    x, w = torch.randn(rows, F, generator=g, device=device), torch.rand(E, H, generator=g, device=device)
    longest = int((off[1:] - off[:-1]).max())
    want = torch.zeros(rows, F, dtype=torch.float64, device=device)
    size = torch.zeros_like(want)
    terms = (x.double()[idx.long()].view(E, H, Fh) * w.double()[:, :, None]).view(E, F)
    want.index_add_(0, dst, terms)
    size.index_add_(0, dst, terms.abs())
    _, xs = shifted(x, by)
    for accumulate in (0, 1):
        old = torch.randn(rows, F, generator=g, device=device) if accumulate else torch.zeros(rows, F, device=device)
        buf, out = shifted(old, (by + 1) % 4)
        run(xs, out, w, accumulate)
        bound = (longest + 2) * 2.0 ** -24 * (size + old.double().abs()) + 1e-30
        assert bool(((out.double() - want - old.double()).abs() <= bound).all())
        at = (by + 1) % 4
        assert bool(buf[:at].isnan().all()) and bool(buf[at + rows * F:].isnan().all())


# items: 16,384, 32,768 and 65,536 are lines of calls without a schedule; the widths are both sides of every group's
@pytest.mark.parametrize("rows,edges", [(60, 900), (16384, 30000), (16385, 30000), (32769, 66000), (66000, 70000)])
@pytest.mark.parametrize("F", [1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 47, 64, 65, 127, 129, 255, 257])
def test_rows(device, rows, edges, F):
    off, idx, dst = graph(rows, edges, 3, device)
    s = torch.cuda.current_stream().cuda_stream
    check(device, rows, off, idx, dst, 1, F, F % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather", ptr(x), ptr(y), ptr(w), ptr(off), ptr(idx), 0, rows, edges, F, acc, s))


# 131,072 items are a line of the schedules; pieces with and without source ranges, six million edges beyond the other one
@pytest.mark.parametrize("rows,edges,ranges", [(60, 900, 1), (5000, 90000, 8), (131000, 140000, 1), (140000, 150000, 1)])
@pytest.mark.parametrize("F", [2, 5, 16, 17, 32, 33, 47, 127, 129, 255, 257])
def test_scheduled_rows(device, rows, edges, ranges, F):
    off, idx, dst = graph(rows, edges, 4, device)
    s = torch.cuda.current_stream().cuda_stream
    plan = SpmmPlan(off, rows, edges, 64, idx, rows, ranges) if ranges > 1 else SpmmPlan(off, rows, edges, 64)
    check(device, rows, off, idx, dst, 1, F, F % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_planned", plan.handle, ptr(x), ptr(y), ptr(w), ptr(off), ptr(idx), 0, F, acc, s))


@pytest.mark.parametrize("F", [16, 31, 32])
def test_scheduled_rows_of_many_edges(device, F):
    rows, edges = 4000, 6100000
    off, idx, dst = graph(rows, edges, 5, device)
    s = torch.cuda.current_stream().cuda_stream
    plan = SpmmPlan(off, rows, edges, 512)
    check(device, rows, off, idx, dst, 1, F, F % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_planned", plan.handle, ptr(x), ptr(y), ptr(w), ptr(off), ptr(idx), 0, F, acc, s))


@pytest.mark.parametrize("rows,edges", [(60, 900), (17000, 66000), (66000, 70000)])
@pytest.mark.parametrize("H,Fh", [(1, 1), (3, 1), (1, 47), (2, 3), (16, 3), (11, 5), (4, 13), (8, 9), (5, 25), (3, 31), (4, 41),
                                  (7, 33), (8, 41)])
def test_heads(device, rows, edges, H, Fh):
    off, idx, dst = graph(rows, edges, 6, device)
    s = torch.cuda.current_stream().cuda_stream
    check(device, rows, off, idx, dst, H, Fh, Fh % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_heads", ptr(x), ptr(y), ptr(w), 0, ptr(off), ptr(idx), rows, edges, H, Fh, acc, s))
    plan = SpmmPlan(off, rows, edges, 64, idx, rows, 4)
    check(device, rows, off, idx, dst, H, Fh, Fh % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_heads_planned", plan.handle, ptr(x), ptr(y), ptr(w), 0, ptr(off), ptr(idx), H, Fh, acc, s))


def even_graph(rows, edges, seed, device):
    """Rows of about as many edges each, none of 256."""
    g = torch.Generator(device=device).manual_seed(seed)
    dst = torch.randint(rows, (edges,), generator=g, device=device).sort().values
    off = torch.zeros(rows + 1, dtype=torch.int64, device=device)
    off[1:] = torch.bincount(dst, minlength=rows).cumsum(0)
    idx = torch.randint(rows, (edges,), generator=g, device=device).to(torch.int32)
    return off.to(torch.int32), idx, dst


# 2,048, 16,384, 32,768 and 65,536 rows are lines of calls that bound their rows, 16 edges a row another
@pytest.mark.parametrize("rows,edges", [(2048, 40000), (2049, 9000), (16385, 90000), (32768, 100000), (32769, 100000), (65537, 200000)])
@pytest.mark.parametrize("F", [3, 4, 7, 8, 15, 16, 17, 32, 47, 64, 129, 201])
def test_bounded_rows(device, rows, edges, F):
    off, idx, dst = even_graph(rows, edges, 8, device)
    s = torch.cuda.current_stream().cuda_stream
    check(device, rows, off, idx, dst, 1, F, F % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_bounded", ptr(x), ptr(y), ptr(w), ptr(off), ptr(idx), 0, rows, edges, F, acc, 256, s))


# 8, 12, 16, 32, 64 and 128 edges a row, 32,768 and 65,536 rows and 2^20 edges are lines of the schedules
@pytest.mark.parametrize("rows,edges", [(65537, 500000), (65536, 500000), (120000, 1100000), (90000, 1100000), (33000, 1100000),
                                        (16400, 1100000), (8000, 1100000), (3000, 200000), (32768, 262144)])
@pytest.mark.parametrize("F", [3, 7, 8, 13, 16, 17, 31, 32, 47, 65, 127, 201])
def test_scheduled_rows_by_their_length(device, rows, edges, F):
    off, idx, dst = even_graph(rows, edges, 9, device)
    s = torch.cuda.current_stream().cuda_stream
    plan = SpmmPlan(off, rows, edges, 64)
    check(device, rows, off, idx, dst, 1, F, F % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_planned", plan.handle, ptr(x), ptr(y), ptr(w), ptr(off), ptr(idx), 0, F, acc, s))


# source ranges, without and with repeated edges in a row, on both sides of 32,768 rows and of 32 and 64 edges a row
@pytest.mark.parametrize("rows,edges,repeats", [(16400, 1100000, False), (33000, 1000000, False), (33000, 2300000, False),
                                                (16400, 1100000, True), (33000, 2300000, True)])
@pytest.mark.parametrize("F", [31, 33, 47, 64, 101, 127])
def test_scheduled_rows_with_source_ranges(device, rows, edges, repeats, F):
    off, idx, dst = even_graph(rows, edges, 10, device)
    if repeats:
        idx = idx // 512 * 512
    s = torch.cuda.current_stream().cuda_stream
    plan = SpmmPlan(off, rows, edges, 64, idx, rows, 8)
    check(device, rows, off, idx, dst, 1, F, F % 4, lambda x, y, w, acc: call(
        "nts_spmm_gather_planned", plan.handle, ptr(x), ptr(y), ptr(w), ptr(off), ptr(idx), 0, F, acc, s))
