"""Edge sums where hundreds to thousands of rows are cut into pieces: more rows than the plan kernel has threads, close
to the 4,096 that it lists, and a hub that makes the pieces longer than the shortest.  A row of n edges, added in fp32
in any order, is off its exact sum by at most n * 2^-24 times the sum of its terms' magnitudes."""
import numpy as np
import pytest
import torch

from neutronbench_amd.abi import call, ptr

pytestmark = pytest.mark.gpu


# F = 256 takes the launch that sums the long rows in its first blocks, 257 launches of their own; both cut rows
# above 1,024 edges
@pytest.mark.parametrize("F", [256, 257])
@pytest.mark.parametrize("giants,hub", [(1, 0), (256, 0), (300, 2000000), (1100, 0), (3990, 0)])
def test_many_rows_in_pieces(device, F, giants, hub):
    V = 16500
    rng = np.random.default_rng(giants)
    deg = np.zeros(V, dtype=np.int64)
    at = rng.permutation(V)
    deg[at[:giants]] = 1025 + rng.integers(0, 3, giants)
    deg[at[giants:giants + 200]] = rng.integers(0, 1026, 200)  # rows of a block and rows of a wavefront beside them
    if hub:
        deg[at[-1]] = hub
    E = int(deg.sum())
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(deg)])).to(device)
    co = off.to(torch.int32)
    g = torch.Generator(device=device).manual_seed(F + giants)
    msg = torch.randn(E, F, generator=g, device=device)
    perm = torch.randperm(E, generator=g, device=device)
    n = torch.from_numpy(deg).to(device).double()[:, None]
    s = torch.cuda.current_stream().cuda_stream
    own = torch.repeat_interleave(torch.arange(V, device=device), off[1:] - off[:-1])
    for order in (None, perm):
        out, again = (torch.full((V, F), 3.0, device=device) for _ in range(2))
        for o in (out, again):
            if order is None:
                call("nts_gather_edge_to_dst", ptr(o), ptr(msg), ptr(co), V, F, 0, s)
            else:
                call("nts_gather_edge_to_src", ptr(o), ptr(msg), ptr(co), ptr(order.to(torch.int32)), V, F, 0, s)
        assert torch.equal(out, again)
        for c in (0, F - 65):  # the first columns and the last ones, odd widths among them
            terms = (msg if order is None else msg[order])[:, c:c + 65].double()
            want, size = (torch.zeros(V, 65, dtype=torch.float64, device=device) for _ in range(2))
            lo, hi = (int(off[at[-1]]), int(off[at[-1] + 1])) if hub else (E, E)
            for part in (slice(0, lo), slice(hi, E)):  # the hub's edges, all for one row, are summed apart
                want.index_add_(0, own[part], terms[part])
                size.index_add_(0, own[part], terms[part].abs())
            if hub:
                want[at[-1]], size[at[-1]] = terms[lo:hi].sum(0), terms[lo:hi].abs().sum(0)
            assert ((out[:, c:c + 65].double() - want).abs() <= n * 2.0 ** -24 * size).all()
