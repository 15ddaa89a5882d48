"""Sums of edge rows over few vertex rows (fewer than 16,384), whose hub rows the launch's first blocks find and add up a
column tile at a time: rows of at most 1,024 edges are the running sum in edge order, bit for bit; longer ones are added by at
most n / 2 chains in a fixed tree, off by at most n 2^-24 of the sum of the magnitudes."""
import pytest
import torch

from neutronbench_amd.abi import call, ptr

pytestmark = pytest.mark.gpu


def running_sums(msg, off, rows):
    """Sums of the given rows, each of at most 1,024 edges, in 32 bits, one edge after the other (a zero more changes no sum that
    starts at zero)."""
    longest = int((off[rows + 1] - off[rows]).max())
    k = torch.arange(longest, device=msg.device)
    there = (off[rows, None] + k < off[rows + 1, None])[:, :, None]
    terms = torch.where(there, msg[(off[rows, None] + k).clamp(max=msg.shape[0] - 1)], 0.0)
    out = torch.zeros(rows.numel(), msg.shape[1], device=msg.device)
    for i in range(longest):
        out += terms[:, i]
    return out


# rows on both sides of 64 (below it no row is a hub), 4,096 (another kernel from there on) and 16,384
@pytest.mark.parametrize("rows", [1, 63, 64, 4095, 4096, 16383, 16384])
@pytest.mark.parametrize("F", [1, 4, 32, 47, 128, 260])
@pytest.mark.parametrize("dense", [False, True])
def test_sums_over_few_rows(device, rows, F, dense):
    print(f"case rows={rows} F={F} dense={dense}", flush=True)
    g = torch.Generator(device=device).manual_seed(rows + F)
    deg = torch.randint(0, 4 if not dense else max(4, 400000 // rows), (rows,), generator=g, device=device)
    marks = torch.tensor([1025, 1024, 5000, 0, 20001, 1023, 1, 3000], device=device)[:rows]
    deg[torch.randperm(rows, generator=g, device=device)[:len(marks)]] = marks
    off = torch.cat([deg.new_zeros(1), deg.cumsum(0)])
    E = int(off[-1])

    def per_row(v):
        total = torch.cat([v.new_zeros(1, F), v.cumsum(0)])
        return total[off[1:]] - total[off[:-1]]

    msg = torch.randn(E, F, generator=g, device=device)
    perm = torch.randperm(E, generator=g, device=device)
    co, s = off.to(torch.int32), torch.cuda.current_stream().cuda_stream
    init = torch.randn(rows, F, generator=g, device=device)
    for order in (None, perm):
        terms = msg if order is None else msg[order]
        chains = torch.nonzero((deg <= 1024) & (deg > 0)).flatten()
        chains = chains[deg[chains].argsort(descending=True)][:40]
        want = running_sums(terms, off, chains) if chains.numel() else None
        exact, size = per_row(terms.double()), per_row(terms.double().abs())
        for accumulate in (0, 1):
            out = init.clone() if accumulate else torch.full((rows, F), float("nan"), device=device)
            if order is None:
                call("nts_gather_edge_to_dst", ptr(out), ptr(msg), ptr(co), rows, F, accumulate, s)
            else:
                call("nts_gather_edge_to_src", ptr(out), ptr(msg), ptr(co), ptr(order.to(torch.int32)), rows, F, accumulate, s)
            if want is not None:
                assert torch.equal(out[chains], want + init[chains] if accumulate else want)
            assert torch.equal(out[deg == 0], init[deg == 0] if accumulate else torch.zeros_like(out[deg == 0]))
            full = exact + init.double() if accumulate else exact
            bound = (deg.double()[:, None] + 1) * 2.0 ** -24 * (size + init.double().abs() * accumulate) + 1e-8  # (64-bit prefix sums)
            assert ((out.double() - full).abs() <= bound).all()
