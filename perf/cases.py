"""The work that a program built on the sampling server has it do, as cases that can be timed.

A case is one call pattern of the public interface (one mini-batch, a group of mini-batches issued together,
the operators one by one, the call that allocates nothing, presampling and cache construction) on one shape:
graph, batch, fan-outs, feature rows, cache.  The shapes are the configurations that bench.py and the tests
serve -- Cora, ogbn-products, ogbn-papers100M, MAG240M -- with the node counts of the last two cut down so that
a state is made in about a second; batches, fan-outs, rows and the cached share are the real ones.

`prepare` generates a graph in HBM, a feature table, a train set with labels and the cache, and hands over a
server that is ready to serve; `run` serves one pass and returns the output buffers of its mini-batches.  The
buffers are sized for the worst case of a batch and cleared once: a pass writes the same batch into them every
time, so what lies behind a batch's last row stays zero.
"""
import functools
import importlib.util
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch


def _package():
    """The repository's package, whose folder name is no Python identifier."""
    if "legion_ibp_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "legion_ibp_amd", os.path.join(os.getcwd(), "legion-ibp_amd", "__init__.py"))
        module = importlib.util.module_from_spec(spec)
        sys.modules["legion_ibp_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["legion_ibp_amd"]


# ------------------------------------------------------------------------------------------------ the cases
# Graph shapes: degrees follow a shifted Zipf law (alpha > 0) or a Poisson law (alpha 0), neighbours are drawn in
# proportion to their degree (uniformly in the Poisson graph).
_CORA = dict(nodes=2708, mean_deg=7.8, alpha=0.0, d_max=40, dim=1433, dtype="f32")
_PRODUCTS = dict(nodes=2449029, mean_deg=25.27, alpha=2.1, d_max=17000, dim=100, dtype="f32")
_PAPERS = dict(nodes=4000000, mean_deg=14.548, alpha=2.0, d_max=100000, dim=128, dtype="f32")
_MAG = dict(nodes=1000000, mean_deg=7.08, alpha=2.0, d_max=100000, dim=768, dtype="f16")


def _case(name, graph, call, batches, batch, fanout, cache, cached, table, features):
    c = dict(graph, call=call, batches=batches, batch=batch, fanout=fanout, cache=cache, cached=cached, table=table,
             features=features)
    return dict(c, name=name) if name else c


def listed():
    return [
        # Online inference asks for a handful of nodes and waits: nothing but launches and latency.
        _case("inference of 16 nodes", _PRODUCTS, "once", 1, 16, "10,5", "static", 0.30, "rank", "host"),
        # The whole of a small citation graph in the cache, long odd rows (5 732 bytes).
        _case("cora batch", _CORA, "once", 1, 64, "25,10", "static", 1.0, "rank", "host"),
        # A trainer that takes every batch before it asks for the next: ogbn-products as it is usually trained.
        _case("products batch", _PRODUCTS, "once", 1, 800, "25,10", "static", 0.30, "hash", "host"),
        # The same schedule prefetched: groups of six batches, the next group issued while the last is consumed.
        _case("products group", _PRODUCTS, "group", 6, 800, "25,10", "static", 0.30, "rank", "host"),
        # The reference's runner: operators launched one by one, lookups segment by segment; half-precision rows.
        _case("products operators", dict(_PRODUCTS, dtype="f16"), "operators", 1, 800, "25,10", "static", 0.30, "hash",
              "host"),
        # Captured or allocation-free loops: caller-owned buffers, one stream, at the largest server it takes.
        _case("caller's buffers", _PRODUCTS, "static", 1, 800, "25,10", "static", 0.30, "direct", "host"),
        # ogbn-papers100M: batches of 8 000, two thirds of the rows cached, prefetched in groups.
        _case("papers group", _PAPERS, "group", 6, 8000, "25,10", "static", 0.668, "rank", "host"),
        # The same batches from a feature table that lies in HBM whole (288 GB hold it): no cache, no host link.
        _case("papers in HBM", dict(_PAPERS, nodes=20000000), "group", 4, 8000, "25,10", "none", 0.0, "rank", "device"),
        # ... and a trainer that consumes them one at a time from a cache that holds everything.
        _case("papers batch cached", _PAPERS, "once", 1, 8000, "25,10", "static", 1.0, "rank", "host"),
        # Three hops through a dynamic cache: four batches in a row, each filling the cache for the next.
        _case("papers three hops lru", dict(_PAPERS, nodes=2000000), "once", 4, 1024, "15,10,5", "lru", 0.30, "rank",
              "host"),
        # MAG240M: compressed cache, rows dequantised to half precision while they are gathered.
        _case("mag group int8", _MAG, "group", 4, 1024, "25,15", "int8", 0.424, "rank", "host"),
        # Start of a training run: presample part of an epoch, rank by what it touched, fill the cache.
        _case("presample and fill", _PRODUCTS, "presample", 16, 800, "25,10", "static", 0.30, "hash", "host"),
    ]


def draw(rng):
    """Another case of the same ranges: batch sizes from 8 to 8 000 over their logarithm, one to three hops, odd
    row lengths, every cache, table, row type, place of the table and call."""
    limit = max(_cost(c) for c in listed())
    while True:
        call = rng.choice(["once", "once", "group", "group", "operators", "static", "presample"])
        batch = int(round(math.exp(rng.uniform(math.log(8), math.log(8000)))))
        fanout = rng.choice([[25, 10], [10, 5], [25, 15], [15, 10, 5], [5, 4, 3], [20], [64, 2], [33, 7],
                             [rng.randint(1, 40), rng.randint(1, 20)]])
        shape = dict(rng.choice([_PRODUCTS, _PAPERS]))
        shape["nodes"] = int(round(math.exp(rng.uniform(math.log(20000), math.log(2000000)))))
        shape["dim"] = rng.choice([32, 50, 64, 100, 128, 200, 256, 300, 602, 768, 1024, 1433, rng.randint(8, 600)])
        shape["dtype"] = rng.choice(["f32", "f32", "f16"])
        if shape["dtype"] == "f16":
            shape["dim"] += shape["dim"] % 2
        cache = rng.choice(["static", "static", "int8", "lru", "none"])
        features = rng.choice(["host", "host", "device"])
        cached = round(rng.uniform(0.2, 1.0), 3)
        table = rng.choice(["rank", "hash", "direct"])
        batches = 1
        if call == "group":
            batches = rng.randint(2, 6) if len(fanout) < 3 else rng.randint(2, 5)
        elif call == "presample":
            batches = rng.randint(2, 16)
        if cache == "lru" and call == "group":
            call, batches = "once", rng.randint(2, 4)
        if call in ("static", "presample") and cache == "lru":
            cache = "static"
        if call == "presample" and cache == "none":
            cache = "static"
        if cache == "none":
            cached = 0.0
        c = _case(None, shape, call, batches, batch, ",".join(map(str, fanout)), cache, cached, table, features)
        nodes, edges = _worst_case(c)
        if call == "static" and (nodes[-1] > 1 << 18 or max(edges) > 1 << 18):
            continue
        if batch * batches > c["nodes"] // 4 or c["nodes"] * _row_bytes(c) > 2.1e9:
            continue
        if nodes[-1] * _row_bytes(c) > 1.2e9 or _cost(c) > limit:
            continue
        return c


# ------------------------------------------------------------------------------------------- sizes and work
def _fanout(case):
    return [int(f) for f in case["fanout"].split(",")]


def _row_bytes(case):
    return case["dim"] * (2 if case["dtype"] == "f16" else 4)


def _worst_case(case):
    """Rows known after each hop and edges of each hop, were every sampled neighbour a new node."""
    nodes, edges = [case["batch"]], []
    for f in _fanout(case):
        edges.append(nodes[-1] * f)
        nodes.append(nodes[-1] + edges[-1])
    return nodes, edges


@functools.lru_cache(maxsize=None)
def _degree_law(alpha, d_max, mean_deg):
    if alpha == 0.0:
        p = [math.exp(-mean_deg)]
        for d in range(1, d_max + 1):
            p.append(p[-1] * mean_deg / d)
        p = np.array(p)
        return p / p.sum()
    return np.diff(_package().zipf_cdf(alpha, d_max, mean_deg).astype(np.float64) / 2.0 ** 32, prepend=0.0)


def _degrees(case):
    """Probability of each degree 0 .. d_max in the generated graph."""
    return _degree_law(case["alpha"], case["d_max"], case["mean_deg"])


def _expected(case):
    """Expected rows after each hop and edges of each hop of one batch, and the share of its rows that the cache
    holds: neighbours are drawn in proportion to their degree, so a node of degree d has been met by m draws with
    probability 1 - exp(-m d / edges), and the cache holds the nodes of the largest degrees."""
    p = _degrees(case)
    d = np.arange(len(p), dtype=np.float64)
    n_edges = case["nodes"] * float((p * d).sum())
    weight = d if case["alpha"] else np.full(len(d), n_edges / case["nodes"])
    known = np.full(len(p), case["batch"] / case["nodes"])      # share of the nodes of each degree known so far
    nodes, edges = [case["batch"]], []
    for f in _fanout(case):
        e = case["nodes"] * float((p * known * np.minimum(d, f)).sum())
        known = 1.0 - (1.0 - known) * np.exp(-e * weight / n_edges)
        edges.append(e)
        nodes.append(case["nodes"] * float((p * known).sum()))
    above = np.cumsum(p[::-1])[::-1] - p                        # share of the nodes of a larger degree
    held = np.clip((case["cached"] - above) / np.maximum(p, 1e-30), 0.0, 1.0)
    return nodes, edges, float((p * known * held).sum() / (p * known).sum())


def work(case):
    """Bytes that a pass has to read or write, each once.  Rows missing from the cache are counted like all
    others, though they come over the host link, which is two orders of magnitude slower than HBM."""
    nodes, edges, hits = _expected(case)
    rows, row = nodes[-1], _row_bytes(case)
    sampling = 4 * case["batch"] + 16 * nodes[-2] + 4 * sum(edges)   # seeds, row pointers, neighbour ids
    sampling += 4 * rows + 12 * sum(edges) + 4 * sum(nodes[:-1])     # ids, edge lists, block row pointers
    if case["call"] == "presample":
        source = case["dim"] + 4 if case["cache"] == "int8" else row
        fill = case["cached"] * case["nodes"] * (row + source) + 4 * case["nodes"]
        return {"bytes": case["batches"] * (sampling + 8 * rows) + fill, "flops": 0.0}
    source = row
    if case["cache"] == "int8":
        source = hits * (case["dim"] + 4) + (1 - hits) * row
    gather = rows * (4 + 4 + source + row) + 8 * case["batch"]       # table word, slot, row in and out; labels
    flops = rows * case["dim"] if case["cache"] == "int8" else 0.0
    return {"bytes": case["batches"] * (sampling + gather), "flops": case["batches"] * flops}


def _cost(case):
    """Bytes of a pass with the rows that come over the host link weighed by how much slower it is."""
    nodes, _, hits = _expected(case)
    slow = 0.0
    if case["features"] == "host":
        share = case["cached"] if case["call"] == "presample" else 1.0 - hits
        rows = case["nodes"] if case["call"] == "presample" else case["batches"] * nodes[-1]
        slow = 60.0 * share * rows * _row_bytes(case)
    return work(case)["bytes"] + slow


def tolerance(case):
    """Ids, edges and slots are whole numbers; rows are copied, or dequantised by one rounded product."""
    return "exact"


# ------------------------------------------------------------------------------------------------ the state
class _Device:
    """Device memory of the server as an array that torch can lay a tensor over; holds on to its owner."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 2, "strides": None}


class _Owner:
    """A server with the graph and feature table it serves from, given back when nothing refers to it."""

    def __init__(self):
        self.server = self.table = self.graph = None

    def __del__(self):
        lmi = sys.modules.get("legion_ibp_amd")
        if lmi is None:
            return
        torch.cuda.synchronize()
        if self.server is not None:
            self.server.close()
        if isinstance(self.table, lmi.HostBuffer):
            self.table.free()
        for ptr in self.graph or ():
            lmi.check(lmi.lib().lmi_device_free(ptr))


_stream = []


def _the_stream():
    """A program serves all its batches on one stream of its own."""
    if not _stream:
        _stream.append(_package().stream_create())
    return _stream[0]


def _tensor(ptr, shape, typestr, owner):
    return torch.as_tensor(_Device(ptr, shape, typestr, owner), device="cuda")


def prepare(case, seed):
    lmi = _package()
    own = _Owner()
    fanout, n, dim = _fanout(case), case["nodes"], case["dim"]
    half = case["dtype"] == "f16"
    rng = np.random.default_rng(seed)
    # the graph
    p = _degrees(case)
    cdf = np.minimum(np.floor(np.cumsum(p) * 2.0 ** 32), 2.0 ** 32 - 1).astype(np.uint64)
    cdf[-1] = 2 ** 32 - 1
    indptr, indices, n_edges = lmi.synth_graph(seed, cdf.astype(np.uint32), n, 1 if case["alpha"] else 0)
    own.graph = (indptr, indices)
    # the feature table: pinned host memory, or all of it in HBM
    if case["features"] == "host":
        own.table = lmi.HostBuffer((n, dim), np.float16 if half else np.float32)
        lmi.synth_features(seed + 1, own.table)
    else:
        own.table = torch.empty((n, dim), dtype=torch.float16 if half else torch.float32, device="cuda")
        torch.cuda.synchronize()
        lmi.check(lmi.lib().lmi_synth_features(seed + 1, own.table.data_ptr(), n, dim, lmi.F16 if half else lmi.F32))
    # the server
    in_flight = case["batches"] if case["call"] != "presample" else 1
    srv = own.server = lmi.Server(case["batch"], fanout, dim, feat_dtype=lmi.F16 if half else lmi.F32, pipes=in_flight,
                                  seed=seed)
    srv.attach_graph_device(indptr, indices, n, n_edges)
    if case["features"] == "host":
        srv.attach_features(own.table)
    else:
        srv.attach_features_device(own.table.data_ptr(), n)
    train = rng.choice(n, case["batch"] * case["batches"], replace=False).astype(np.int32)
    srv.load_idset(lmi.MODE_TRAIN, train, rng.integers(0, 172, len(train)).astype(np.int32))
    table = {"hash": lmi.TABLE_HASH, "direct": lmi.TABLE_DIRECT, "rank": lmi.TABLE_RANK}[case["table"]]
    rows = max(1, int(case["cached"] * n))
    if case["call"] != "presample":
        if case["cache"] == "static":
            srv.build_static_cache(rows, table)
        elif case["cache"] == "int8":
            srv.build_int8_cache(rows, table)
        elif case["cache"] == "lru":
            srv.build_lru_cache(max(1, rows // 8), 8)
    s = SimpleNamespace(call=case["call"], cache=case["cache"], batches=case["batches"], batch=case["batch"],
                        hops=len(fanout), rows=rows, table=table, nodes=n, server=srv, own=own, stream=_the_stream(),
                        pipes=list(range(in_flight)))
    caps, edge_caps = _worst_case(case)
    f = "<f2" if half else "<f4"
    if s.call == "static":
        # the caller's own buffers
        i32 = dict(dtype=torch.int32, device="cuda")
        out = dict(ids=torch.zeros(caps[-1], **i32), labels=torch.zeros(caps[0], **i32),
                   features=torch.zeros((caps[-1], dim), dtype=torch.float16 if half else torch.float32, device="cuda"),
                   agg_src_ids=torch.zeros(sum(edge_caps), **i32), agg_src_off=torch.zeros(sum(edge_caps), **i32),
                   agg_dst_off=torch.zeros(sum(edge_caps), **i32), node_counter=torch.zeros(16, **i32),
                   edge_counter=torch.zeros(16, **i32), cache_index=torch.zeros(caps[-1], **i32),
                   blk_indptr=[torch.zeros(caps[k] + 1, **i32) for k in range(s.hops)])
        view = lmi.BatchView()
        for key, t in out.items():
            if key == "blk_indptr":
                for k in range(s.hops):
                    view.blk_indptr[k] = t[k].data_ptr()
            else:
                setattr(view, key, t.data_ptr())
        view.max_nodes, view.max_edges, view.row_bytes = caps[-1], sum(edge_caps), _row_bytes(case)
        s.view, s.seeds, s.seed = view, torch.from_numpy(train).to("cuda"), seed
        s.outputs = [dict(out, keep=None)]
    else:
        s.outputs = []
        for pipe in s.pipes:
            v = srv.view(pipe)
            out = dict(ids=_tensor(v.ids, (caps[-1],), "<i4", own), labels=_tensor(v.labels, (caps[0],), "<i4", own),
                       agg_src_ids=_tensor(v.agg_src_ids, (sum(edge_caps),), "<i4", own),
                       agg_src_off=_tensor(v.agg_src_off, (sum(edge_caps),), "<i4", own),
                       agg_dst_off=_tensor(v.agg_dst_off, (sum(edge_caps),), "<i4", own),
                       # both headers: the edge counters follow the node counters
                       headers=_tensor(v.node_counter, (32,), "<i4", own),
                       blk_indptr=[_tensor(v.blk_indptr[k], (caps[k] + 1,), "<i4", own) for k in range(s.hops)])
            if s.call != "presample":
                out["features"] = _tensor(v.features, (caps[-1], dim), f, own)
                if s.cache != "lru":   # where a row lies in the dynamic cache depends on the passes before
                    out["cache_index"] = _tensor(v.cache_index, (caps[-1],), "<i4", own)
            for t in out.values():
                for x in t if isinstance(t, list) else [t]:
                    if x.data_ptr() != v.node_counter:
                        x.zero_()
            s.outputs.append(out)
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------------------------------------- the pass
def run(s):
    lmi, srv, stream = _package(), s.server, s.stream
    if s.call == "once":
        # served one at a time; what consumes a batch follows it on the same stream
        for k in range(s.batches):
            srv.run_once(batch_counter=k, pipe=k, stream=stream)
            srv.batch_wait(k, stream)
    elif s.call == "group":
        # prefetched: whoever takes a batch waits for it then, the next group is issued meanwhile
        srv.run_group(s.pipes, s.pipes, stream=stream)
    elif s.call == "operators":
        for k in range(s.batches):
            srv.op_batch_generate(batch_counter=k, pipe=k, stream=stream)
            srv.op_cache_lookup(0, pipe=k, stream=stream)
            for hop in range(s.hops):
                srv.op_random_sample(hop, pipe=k, stream=stream)
                srv.op_cache_lookup(hop + 1, pipe=k, stream=stream)
            srv.op_io_submit(pipe=k, stream=stream)
            srv.op_io_complete(pipe=k, stream=stream)
            srv.batch_wait(k, stream)
    elif s.call == "static":
        srv.run_once_static(s.seeds.data_ptr(), s.batch, s.view, rng_seed=s.seed + 1, stream=stream)
    else:
        lmi.check(lmi.lib().lmi_presample_reset(srv.h))
        srv.presample(s.batches, stream=stream)
        lmi.check(lmi.lib().lmi_stream_sync(stream))   # the cache is built from the finished counts
        srv.cache_policy(lmi.POLICY_PRESAMPLED)
        if s.cache == "int8":
            srv.build_int8_cache(s.rows, s.table)
        else:
            srv.build_static_cache(s.rows, s.table)
        return {"hotness": srv.hotness(s.nodes), "slots": srv.cache_dump(s.nodes), "last batch": s.outputs}
    return s.outputs
