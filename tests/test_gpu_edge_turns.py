"""Copies to edges whose messages outgrow the caches (128 MiB): wavefronts take 32 KB turns, so steps of 64 edges, turns and
the spans of 32,768 wavefronts all end somewhere inside; every edge row equals the row it is a copy of."""
import pytest
import torch

from neutronbench_amd.abi import call, ptr

pytestmark = pytest.mark.gpu


# rows of 16 floats (8 steps a turn), 64 (two), 128 (one) and 300 (one, two rounds a row); a little above the line,
# last steps of 1 and 63 edges, few vertices (a small grid: several turns) and many; a hub whose edges fill many turns
@pytest.mark.parametrize("V,E,F", [(300, 2200001, 16), (40000, 2200063, 16), (5000, 530001, 64), (700, 270049, 128),
                                   (200000, 1000001, 128), (3000, 120001, 300), (5000, 530001, 62)])
def test_copies_in_turns(device, V, E, F):
    g = torch.Generator(device=device).manual_seed(F)
    src = torch.randint(0, V, (E,), generator=g, device=device)
    dst = torch.randint(0, V, (E,), generator=g, device=device)
    dst[:E // 5] = V // 3
    dst = dst.sort().values
    co = torch.zeros(V + 1, dtype=torch.int64, device=device)
    co[1:] = torch.bincount(dst, minlength=V).cumsum(0)
    co, ri = co.to(torch.int32), src.to(torch.int32)
    x = torch.randn(V, F, generator=g, device=device)
    s = torch.cuda.current_stream().cuda_stream
    msg = torch.full((E + 1, F), float("nan"), device=device)
    call("nts_scatter_src_to_edge", ptr(msg), ptr(x), ptr(ri), ptr(co), 0, V, F, s)
    assert torch.equal(msg[:E], x[src]) and bool(msg[E].isnan().all())
    call("nts_scatter_dst_to_edge", ptr(msg), ptr(x), ptr(co), V, F, s)
    assert torch.equal(msg[:E], x[dst]) and bool(msg[E].isnan().all())
    call("nts_scatter_grad_to_edge", ptr(msg), ptr(x), ptr(co), V, F, s)  # adds
    assert torch.equal(msg[:E], x[dst] + x[dst]) and bool(msg[E].isnan().all())
