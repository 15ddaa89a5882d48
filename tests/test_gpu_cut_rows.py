"""Rows cut into 256-edge pieces without a plan, around the sizes where the cutting can go wrong: 1,024 rows a block, rows
of one edge either side of the piece length, rows of more pieces than a wavefront has lanes, blocks without any.  A row
of n edges summed in fp32 in any order is off its exact sum by at most n 2^-24 times the sum of its terms' magnitudes."""
import pytest
import torch

from neutronbench_amd.abi import call, ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("F", [3, 16])
def test_rows_around_the_piece_length(device, rows, F):
    marks = [256, 257, 512, 513, 64 * 256, 64 * 256 + 1, 20000, 255, 0, 1]
    deg = torch.zeros(rows, dtype=torch.int64)
    at = torch.randperm(rows, generator=torch.Generator().manual_seed(rows))[:len(marks)]
    deg[at] = torch.tensor(marks[:len(at)])
    deg[at[0]] += max(0, 65536 - int(deg.sum()))  # calls of fewer edges are not cut
    if rows == 1025:
        deg[1024] = 700  # the only row of its block
    deg = deg.to(device)
    E, V = int(deg.sum()), 4000
    off = torch.cat([deg.new_zeros(1), deg.cumsum(0)])
    g = torch.Generator(device=device).manual_seed(F)
    x, w = torch.randn(V, F, generator=g, device=device), torch.rand(E, generator=g, device=device)
    idx = torch.randint(V, (E,), generator=g, device=device)
    off32, idx32 = off.to(torch.int32), idx.to(torch.int32)
    own = torch.repeat_interleave(torch.arange(rows, device=device), deg)
    terms = x[idx].double() * w[:, None].double()
    want, size = (torch.zeros(rows, F, dtype=torch.float64, device=device).index_add_(0, own, t) for t in (terms, terms.abs()))
    outs = []
    for _ in range(2):
        out = torch.full((rows, F), float("nan"), device=device)
        call("nts_spmm_gather", ptr(x), ptr(out), ptr(w), ptr(off32), ptr(idx32), 0, rows, E, F, 0,
             torch.cuda.current_stream().cuda_stream)
        assert ((out.double() - want).abs() <= (deg.double()[:, None] + 1) * 2.0 ** -24 * size).all()
        outs.append(out)
    assert torch.equal(*outs)


ENTRIES = {
    "plain": lambda x, y, w, off, idx, rows, E, F, s: call("nts_spmm_gather", ptr(x), y, ptr(w), ptr(off), ptr(idx), 0, rows, E, F, 0, s),
    "static": lambda x, y, w, off, idx, rows, E, F, s: call("nts_spmm_gather_static_scratch", ptr(x), y, ptr(w), ptr(off), ptr(idx),
                                                            0, rows, E, F, 0, s),
    "heads": lambda x, y, w, off, idx, rows, E, F, s: call("nts_spmm_gather_heads", ptr(x), y, ptr(w), 0, ptr(off), ptr(idx), rows, E,
                                                           1, F, 0, s),
}


@pytest.mark.parametrize("entry", list(ENTRIES))
@pytest.mark.parametrize("rows,each", [(1000, 1000), (100, 20000), (5000, 300), (3000, 257)])
def test_fewer_edges_stated_than_there_are(device, entry, rows, each):
    """65,536 edges stated: slots for 256 pieces and one more per possible row.  Rows that got all their slots are right, at
    most one got some of them, the others keep what they held; nothing is written anywhere else."""
    F, V, stated = 8, 4000, 65536
    print(f"case {entry} {rows} {each}", flush=True)
    g = torch.Generator(device=device).manual_seed(rows)
    E = rows * each
    x, w = torch.randn(V, F, generator=g, device=device), torch.rand(E, generator=g, device=device)
    idx = torch.randint(V, (E,), generator=g, device=device)
    off = torch.arange(0, E + 1, each, dtype=torch.int32, device=device)
    terms = (x[idx].double() * w[:, None].double()).view(rows, each, F)
    n_slots, per_row = stated // 256 + min(rows, stated // 256) + 1, -(-each // 256)
    for _ in range(3):
        buf = torch.full((rows + 64, F), 7.0, device=device)
        ENTRIES[entry](x, buf.data_ptr() + 32 * F * 4, w, off, idx.to(torch.int32), rows, stated, F,
                       torch.cuda.current_stream().cuda_stream)
        out = buf[32:32 + rows].double()
        assert bool((buf[:32] == 7).all()) and bool((buf[32 + rows:] == 7).all())
        right = ((out - terms.sum(1)).abs() <= (each + 1) * 2.0 ** -24 * terms.abs().sum(1)).all(1)
        kept = (out == 7).all(1)
        some = ~right & ~kept
        assert int(right.sum()) == n_slots // per_row and int(some.sum()) == (1 if n_slots % per_row else 0)
        part = min(each, n_slots % per_row * 256)
        assert bool(((out[some] - terms[some, :part].sum(1)).abs() <= (each + 1) * 2.0 ** -24 * terms[some].abs().sum(1)).all())
