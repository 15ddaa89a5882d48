"""The work that a user of this framework has it do, as cases that can be timed and compared.

Seven kinds of work, each through the package's public classes, on seeded R-MAT graphs:

  gcn     full-graph training step of a two-layer GCN: `ForwardSingleGPUfuseOp` forward and backward at
          the width of the features and at the hidden width, over a chunk resident in HBM
  batch   one mini-batch of sampled GCN training: `BatchBuilder`, feature and label gather, aggregation
          forward and backward of every layer, into arrays that the program keeps (the entry points of
          the C interface, called as the epoch driver calls them)
  gatb    the same with attention layers, through `GATAttentionOp` and `GATAggregateOp`
  gat     one attention layer on the whole graph, forward and backward
  edges   the edge-tensor operators that an attention layer is composed of when it is not fused
          (scatter to edges, edge softmax, edge sums), forward and backward
  build   from an edge list to a chunk: CSC, CSR, weights and both aggregation schedules
  rows    assembling the input of a prediction request: feature rows and labels by vertex id

The dense layers between the aggregations are not part of the framework: where a pass needs the tensor
that a dense layer would hand over, `prepare` holds one of that shape.
"""
import math

import torch

from neutronbench_amd import synth
from neutronbench_amd.abi import call, ptr
from neutronbench_amd.batch import (BatchBuilder, FeatureCache, MappedHostTable, load_feature_gpu,
                                    load_feature_gpu_cache, load_label_gpu)
from neutronbench_amd.layout import FullGraphChunk, SampledLayer, as_u32
from neutronbench_amd.ops import (ForwardSingleGPUfuseOp, GATAggregateOp, GATAttentionOp, SingleGPUAggregateDst,
                                  SingleGPUEdgeSoftMax, SingleGPUScatterDst, SingleGPUScatterSrc)
from neutronbench_amd.stream import CudaStream

DEVICE = "cuda:0"


def listed():
    return [
        # Cora-shaped full-graph GCN: the smallest graph in use, wide binary features, a hidden layer of
        # 16; a pass is four launches' worth of latency.
        dict(name="gcn_cora", kind="gcn", V=2708, E=10556, F=1433, hidden=16, ranges=1, simple=True),
        # Arxiv-shaped full-graph GCN: an ordinary graph whose features fit the caches in part.
        dict(name="gcn_arxiv", kind="gcn", V=169343, E=2480000, F=128, hidden=128, ranges=1, simple=False),
        # Products-shaped full-graph GCN: the most vertices; full-batch training and full-graph evaluation.
        dict(name="gcn_products", kind="gcn", V=2449029, E=126200000, F=100, hidden=128, ranges=32, simple=False),
        # Reddit-shaped full-graph GCN: the headline; the densest graph, rows of 602 floats (8-byte aligned).
        dict(name="gcn_reddit", kind="gcn", V=232965, E=114800000, F=602, hidden=128, ranges=32, simple=True),
        # A training batch of the Arxiv-shaped configuration: features in mapped host memory, a wait
        # after every operator, as the reference's operators have.
        dict(name="batch_arxiv", kind="batch", V=169343, E=2480000, F=128, hidden=128, fanout="25,10", batch=1024,
             table="host", waits=True),
        # A training batch of the Products-shaped configuration: three hops, the features of the top 20 %
        # of the vertices cached in HBM, the others in host memory, no waits between the operators.
        dict(name="batch_products", kind="batch", V=2449029, E=126200000, F=100, hidden=128, fanout="15,10,5",
             batch=6000, table="cache", waits=False),
        # A batch of attention layers, four heads of 32.
        dict(name="batch_gat", kind="gatb", V=2449029, E=126200000, F=100, hidden=128, heads=4, fanout="10,10",
             batch=4096, table="cache", waits=False),
        # Attention output layer (one head, 47 classes: rows of 188 bytes) on an Arxiv-shaped graph.
        dict(name="gat_arxiv", kind="gat", V=169343, E=2480000, heads=1, width=47),
        # Attention hidden layer (four heads of 32) on the whole Products-shaped graph.
        dict(name="gat_products", kind="gat", V=2449029, E=126200000, heads=4, width=32),
        # The unfused attention operators on an Arxiv-shaped graph: [E, 128] messages, [E, 4] scores.
        dict(name="edges_arxiv", kind="edges", V=169343, E=2480000, heads=4, width=128),
        # Loading a graph: a Reddit-shaped edge list, in the order in which its edges were added, to a chunk
        # ready for training.
        dict(name="build_reddit", kind="build", V=232965, E=114800000, ranges=32, sorted=False),
        # A prediction request for 4,096 vertices, features in HBM: a call that is little but its launch.
        dict(name="rows_arxiv", kind="rows", V=169343, F=128, n=4096),
    ]


def _between(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _graph(rng, vertices, edges):
    """Vertices and edges between the two ends of each range, 2 to 600 edges a vertex."""
    V = _between(rng, *vertices)
    return V, min(edges[1], max(edges[0], int(V * math.exp(rng.uniform(math.log(2), math.log(600))))))


def draw(rng):
    kind = rng.choice(["gcn", "gcn", "batch", "gatb", "gat", "edges", "build", "rows"])
    if kind == "gcn":
        V, E = _graph(rng, (2000, 2449029), (8000, 40000000))
        simple = rng.random() < 0.5 and E < V * V // 16
        return dict(kind=kind, V=V, E=E, F=rng.choice([16, 50, 100, 128, 256, 300, 500, 602, rng.randint(8, 700)]),
                    hidden=rng.choice([7, 16, 41, 47, 64, 128, 256, rng.randint(4, 256)]),
                    ranges=32 if E > 8000000 else 1, simple=simple)
    if kind in ("batch", "gatb"):
        V, E = _graph(rng, (20000, 2000000), (100000, 40000000))
        fanout = rng.choice(["25,10", "10,10", "15,10,5", "5,5", "10,25", "%d,%d" % (rng.randint(2, 30), rng.randint(2, 30))])
        case = dict(kind=kind, V=V, E=E, F=rng.choice([100, 128, 50, rng.randint(16, 300)]), hidden=rng.choice([64, 128, 256]),
                    fanout=fanout, batch=_between(rng, 64, 6000), table=rng.choice(["hbm", "host", "cache"]),
                    waits=rng.random() < 0.3)
        return dict(case, heads=rng.choice([1, 2, 4, 8])) if kind == "gatb" else case
    if kind == "gat":
        V, E = _graph(rng, (2000, 2000000), (20000, 30000000))
        return dict(kind=kind, V=V, E=E, heads=rng.choice([1, 2, 4, 8]), width=rng.choice([8, 16, 32, 41, rng.randint(4, 48)]))
    if kind == "edges":
        V, E = _graph(rng, (2000, 1000000), (20000, 8000000))
        return dict(kind=kind, V=V, E=E, heads=rng.choice([1, 2, 4, 8]), width=rng.choice([32, 64, 128, rng.randint(7, 128)]))
    if kind == "build":
        V, E = _graph(rng, (2000, 2449029), (20000, 60000000))
        return dict(kind=kind, V=V, E=E, ranges=32 if E > 8000000 else 1, sorted=rng.random() < 0.5)
    return dict(kind="rows", V=_between(rng, 20000, 2449029), F=rng.choice([100, 128, 602, rng.randint(16, 700)]),
                n=_between(rng, 256, 400000))


# -- what a program has in hand ---------------------------------------------------------------------


def _edges(case, seed, simple=False):
    return synth.rmat_edges(case["V"], case["E"], seed=seed, device=DEVICE, sort=True, distinct=simple)


def _floats(seed, *shape):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float32)


def _whole_graph_layer(case, seed):
    """The whole graph as one layer, a self loop at every vertex among its edges (so every vertex is a
    source and a destination); the CSR permutation is kept."""
    V = case["V"]
    src, dst = synth.rmat_edges(V, case["E"] - V, seed=seed, device=DEVICE)
    everyone = torch.arange(V, device=DEVICE)
    co, ri = synth.build_csc(torch.cat([src, everyone]), torch.cat([dst, everyone]), V)
    del src, dst
    return SampledLayer.from_device_hop(as_u32(co), as_u32(ri), everyone.to(torch.int32), V, want_perm=True)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_gcn(case, seed):
    V, F, hidden = case["V"], case["F"], case["hidden"]
    src, dst = _edges(case, seed, case["simple"])
    chunk = FullGraphChunk.from_edges(src, dst, V, chunk_edges=512 if case["ranges"] > 1 else 0, n_slabs=case["ranges"])
    del src, dst
    for plan in (chunk.plan_forward, chunk.plan_backward):
        plan.reserve(F)
        plan.reserve(hidden)
    return dict(kind="gcn", op=ForwardSingleGPUfuseOp(chunk), x=_floats(seed + 1, V, F), h=_floats(seed + 2, V, hidden),
                gh=_floats(seed + 3, V, hidden), gx=_floats(seed + 4, V, F))


def _prepare_batch(case, seed):
    V, F, batch, hidden = case["V"], case["F"], case["batch"], case["hidden"]
    heads = case.get("heads", 0)
    fanout = [int(f) for f in case["fanout"].split(",")]
    src, dst = _edges(case, seed)
    co, ri = synth.build_csc(src, dst, V)
    out_degree = torch.bincount(src, minlength=V)
    del src, dst
    builder = BatchBuilder(as_u32(co), as_u32(ri), fanout, batch, want_perm=heads > 0, graph=3)
    del co, ri
    features = _floats(seed + 1, V, F)
    state = dict(kind=case["kind"], builder=builder, F=F, heads=heads, waits=case["waits"], pick=seed,
                 stream=CudaStream(synchronize=case["waits"]), cache=None,
                 labels=synth.uniform_labels(V, 47, seed=seed + 2, device=DEVICE),
                 ids=as_u32(synth.permutation(V, seed + 3, DEVICE)[:batch]))
    if case["table"] == "hbm":
        state["table"] = features
    else:
        features_cpu = features.cpu()
        state["host"] = MappedHostTable(features_cpu)
        state["table"] = state["host"].dev_ptr
        if case["table"] == "cache":
            state["cache"] = FeatureCache(features_cpu, out_degree.cpu(), V // 5, torch.device(DEVICE))
        del features
    caps = [batch]  # no hop has more destinations than caps[k], no layer more sources than caps[k + 1]
    for f in fanout:
        caps.append(min(V, caps[-1] * f))
    caps.reverse()  # input side first, as the layers come
    state["x"] = torch.empty(caps[0], F, device=DEVICE).zero_()
    state["label"] = torch.empty(batch, dtype=torch.int64, device=DEVICE).zero_()
    if heads:
        state["h"] = _floats(seed + 4, caps[0], hidden)  # what the dense layer before the attention hands over
        state["el"], state["er"] = _floats(seed + 5, caps[0], heads), _floats(seed + 6, caps[1], heads)
        state["g"] = _floats(seed + 7, batch, hidden)
        # the arrays from which the dense layers take their gradients
        state["gh"] = torch.zeros(caps[0], hidden, device=DEVICE)
        state["gel"] = [torch.zeros(c, heads, device=DEVICE) for c in caps[:-1]]
        state["ger"] = [torch.zeros(c, heads, device=DEVICE) for c in caps[1:]]
        return state
    state["h"] = _floats(seed + 4, caps[1], hidden)  # what a dense layer hands over to the next aggregation
    state["g"] = _floats(seed + 5, caps[1], max(F, hidden))  # and the gradient that it hands back
    widths = [F] + [hidden] * (len(fanout) - 1)
    state["widths"] = widths
    state["gx"] = [state["g"].view(-1)[:c * w].view(c, w) for c, w in zip(caps[1:], widths)]
    state["y"] = [torch.zeros(c, w, device=DEVICE) for c, w in zip(caps[1:], widths)]
    state["gin"] = [torch.zeros(c, w, device=DEVICE) for c, w in zip(caps[:-1], widths)]
    return state


def _prepare_gat(case, seed):
    layer = _whole_graph_layer(case, seed)
    H, F = case["heads"], case["heads"] * case["width"]
    return dict(kind="gat", layer=layer, heads=H, x=_floats(seed + 1, layer.src_size, F),
                el=_floats(seed + 2, layer.src_size, H), er=_floats(seed + 3, layer.v_size, H),
                g=_floats(seed + 4, layer.v_size, F))


def _prepare_edges(case, seed):
    layer = _whole_graph_layer(case, seed)
    H, F = case["heads"], case["width"]
    return dict(kind="edges", layer=layer, x=_floats(seed + 1, layer.src_size, F), xd=_floats(seed + 2, layer.v_size, F),
                scores=_floats(seed + 3, layer.e_size, H), gscores=_floats(seed + 4, layer.e_size, H),
                g=_floats(seed + 5, layer.v_size, F))


def _prepare_build(case, seed):
    # edge files come sorted by source, and in the order in which edges were added
    src, dst = synth.rmat_edges(case["V"], case["E"], seed=seed, device=DEVICE, sort=case["sorted"])
    return dict(kind="build", pairs=torch.stack([src, dst], dim=1).to(torch.int32).contiguous(), V=case["V"],
                ranges=case["ranges"])


def _prepare_rows(case, seed):
    V, n = case["V"], case["n"]
    layer = SampledLayer()
    layer.dev_source = layer.dev_destination = as_u32(synth.permutation(V, seed, DEVICE)[:n] if n <= V else
                                                      synth.uniform24(torch.arange(n, device=DEVICE), seed) % V)
    layer.src_size = layer.v_size = n
    return dict(kind="rows", layer=layer, stream=CudaStream(synchronize=False), table=_floats(seed + 1, V, case["F"]),
                labels=synth.uniform_labels(V, 40, seed=seed + 2, device=DEVICE), F=case["F"])


_PREPARE = dict(gcn=_prepare_gcn, batch=_prepare_batch, gatb=_prepare_batch, gat=_prepare_gat, edges=_prepare_edges,
                build=_prepare_build, rows=_prepare_rows)


# -- one pass -----------------------------------------------------------------------------------------


def run(state):
    return _RUN[state["kind"]](state)


def _run_gcn(s):
    op = s["op"]
    return [op.forward(s["x"]), op.forward(s["h"]), op.backward(s["gh"]), op.backward(s["gx"])]


def _run_batch(s):
    builder, stream, x, F = s["builder"], s["stream"], s["x"], s["F"]
    builder.enqueue(s["ids"], s["pick"])
    layers = builder.collect(join=False)
    hits = None
    if s["cache"] is not None:
        hits = load_feature_gpu_cache(stream, layers[0], x, s["table"], s["cache"])
    else:
        load_feature_gpu(stream, layers[0], x, s["table"])
    load_label_gpu(stream, layers[-1], s["label"], s["labels"])
    builder.join()
    out = [x, s["label"], hits]
    return out + (_attention_layers if s["heads"] else _gcn_layers)(s, layers, stream)


def _gcn_layers(s, layers, stream):
    for layer, width, y, h in zip(layers, s["widths"], s["y"], [s["x"]] + [s["h"]] * (len(layers) - 1)):
        call("nts_spmm_gather_bounded", ptr(h), ptr(y), ptr(layer.dev_ewf()), ptr(layer.dev_c_o()), ptr(layer.dev_r_i()),
             0, layer.v_size, layer.e_size, width, 0, layer.max_in_degree, stream.stream)
        if s["waits"]:
            stream.CUDA_DEVICE_SYNCHRONIZE()
    for layer, width, g, gin in reversed(list(zip(layers, s["widths"], s["gx"], s["gin"]))):
        call("nts_spmm_gather", ptr(g), ptr(gin), ptr(layer.dev_ewb()), ptr(layer.dev_r_o()), ptr(layer.dev_c_i()), 0,
             layer.src_size, layer.e_size, width, 0, stream.stream)
        if s["waits"]:
            stream.CUDA_DEVICE_SYNCHRONIZE()
    return s["y"] + s["gin"]


def _attention_layers(s, layers, stream):
    h, ops = s["h"][:layers[0].src_size], []
    for layer in layers:
        att, agg = GATAttentionOp(layer, 0.2), GATAggregateOp(layer, s["heads"])
        h = agg.forward(h, att.forward(s["el"][:layer.src_size], s["er"][:layer.v_size]))
        ops.append((att, agg))
        if s["waits"]:
            stream.CUDA_DEVICE_SYNCHRONIZE()
    g = s["g"]
    for layer, (att, agg), gel, ger in reversed(list(zip(layers, ops, s["gel"], s["ger"]))):
        g = agg.backward(g)
        gel[:layer.src_size] = att.backward(agg.get_additional_grad())
        ger[:layer.v_size] = att.get_additional_grad()
        if s["waits"]:
            stream.CUDA_DEVICE_SYNCHRONIZE()
    s["gh"][:layers[0].src_size] = g
    return [h, s["gh"]] + s["gel"] + s["ger"]


def _run_gat(s):
    att, agg = GATAttentionOp(s["layer"], 0.2), GATAggregateOp(s["layer"], s["heads"])
    alpha = att.forward(s["el"], s["er"])
    y = agg.forward(s["x"], alpha)
    gx = agg.backward(s["g"])
    gel = att.backward(agg.get_additional_grad())
    return [alpha, y, gx, gel, att.get_additional_grad()]


def _run_edges(s):
    layer = s["layer"]
    src, dst, agg = SingleGPUScatterSrc(layer), SingleGPUScatterDst(layer), SingleGPUAggregateDst(layer)
    softmax = SingleGPUEdgeSoftMax(layer.dev_column_offset, layer.v_size)
    msg = src.forward(s["x"])
    msg_dst = dst.forward(s["xd"])
    alpha = softmax.forward(s["scores"])
    y = agg.forward(msg)
    g_msg = agg.backward(s["g"])
    g_scores = softmax.backward(s["gscores"])
    return [msg_dst, alpha, y, g_msg, g_scores, dst.backward(msg), src.backward(msg_dst)]


def _run_build(s):
    chunk = FullGraphChunk.from_edge_pairs(s["pairs"], s["V"], chunk_edges=512 if s["ranges"] > 1 else 0, n_slabs=s["ranges"])
    return [chunk.column_offset_gpu, chunk.row_indices_gpu, chunk.edge_weight_forward_gpu, chunk.row_offset_gpu,
            chunk.column_indices_gpu, chunk.edge_weight_backward_gpu]


def _run_rows(s):
    layer = s["layer"]
    x = torch.empty(layer.src_size, s["F"], device=DEVICE)
    load_feature_gpu(s["stream"], layer, x, s["table"])
    label = torch.empty(layer.v_size, dtype=torch.int64, device=DEVICE)
    load_label_gpu(s["stream"], layer, label, s["labels"])
    return [x, label]


_RUN = dict(gcn=_run_gcn, batch=_run_batch, gatb=_run_batch, gat=_run_gat, edges=_run_edges, build=_run_build,
            rows=_run_rows)


# -- what a pass cannot do without ------------------------------------------------------------------


def _hops(case):
    """(destinations, edges, sources) that the hops of a batch come to, about: most vertices of a power-law
    graph have fewer neighbours than a fanout, and the hubs among them are drawn again and again."""
    rows, hops = case["batch"], []
    for k, f in enumerate(int(f) for f in case["fanout"].split(",")):
        edges = rows * f * (0.4 if k == 0 else 0.95)
        sources = min(case["V"], edges ** 0.93)
        hops.append((rows, edges, sources))
        rows = sources
    return hops


def work(case):
    kind = case["kind"]
    V, F = case["V"], case.get("F", 0)
    E = case.get("E", 0)
    if kind == "gcn":  # two widths, each forward and backward: structure and weights, rows in, rows out
        widths = F + case["hidden"]
        return {"bytes": 4 * (8.0 * E + 4 * V) + 2 * 8.0 * V * widths, "flops": 4.0 * E * widths}
    if kind in ("batch", "gatb"):
        hidden, hops = case["hidden"], _hops(case)
        nbytes = 8.0 * F * hops[-1][2] + 24.0 * case["batch"]  # features and labels, read and written
        flops = 0.0
        for k, (rows, edges, sources) in enumerate(hops):
            width = F if kind == "batch" and k == len(hops) - 1 else hidden
            nbytes += 32.0 * edges + 8.0 * (rows + sources)  # the structure: picked, relabelled, transposed, weighed
            nbytes += 2 * 4.0 * width * (rows + sources) + 2 * 8.0 * edges  # forward and backward
            flops += 4.0 * edges * width
            if kind == "gatb":
                nbytes += 4.0 * edges * case["heads"] * 6 + 4.0 * hidden * (rows + sources)
                flops += 2.0 * edges * hidden
        return {"bytes": nbytes, "flops": flops}
    if kind == "gat":
        H, F = case["heads"], case["heads"] * case["width"]
        # attention forward, aggregation, its two gradients, attention backward and its sum over the sources
        nbytes = E * (4 + 4 * H) + E * (4 + 4 * H) + E * (8 + 4 * H) + E * (4 + 4 * H) + E * (4 + 12 * H) + E * (4 + 4 * H)
        return {"bytes": float(nbytes) + 4.0 * V * F * 6 + 4.0 * V * H * 6, "flops": 6.0 * E * F}
    if kind == "edges":
        H, F = case["heads"], case["width"]
        # messages written three times and read three times, softmax forward and backward, rows in and out
        return {"bytes": 4.0 * E * F * 6 + 4.0 * E * H * 5 + 8.0 * E + 4.0 * V * F * 6, "flops": 3.0 * E * F}
    if kind == "build":  # pairs in; two index arrays and two weight arrays out
        return {"bytes": 24.0 * E + 8.0 * V, "flops": 0.0}
    return {"bytes": case["n"] * (8.0 * F + 24), "flops": 0.0}


def tolerance(case):
    """Sums in 32 bits whose terms may be added in another order: four times the distance from the same
    sums in 64 bits, the largest over the cases being 3e-7 (gradients of the scores) and 3e-5."""
    if case["kind"] in ("build", "rows"):
        return "exact"
    return {"rel": 1.2e-6, "max": 1e-4}
