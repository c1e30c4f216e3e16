"""The selection work that is timed: calls through the package's public entry points over the sizes,
dtypes, value distributions and rank sets that its tests, benchmark and served workload use.

Four kinds of call:
  host    a host k list in, a host array of results out (multiselect, topk): the reference-shaped call
  stream  the stream-ordered entry points: device k list in, device results out, nothing waited for
  batch   many uneven segments of one vector planned once, then replayed (Batch)
  serve   a burst of requests over resident vectors, submitted and drained (Server)

Inputs live in torch tensors; the library gets their addresses.  A result is an order statistic of the
input, so exact() is a full sort of the same input by torch.
"""
from __future__ import annotations

import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package by its path: its folder's name holds a dash."""
    name = "ggks_multiselect_amd"
    if name not in sys.modules:
        here = os.path.join(ROOT, "ggks-multiselect_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(here, "__init__.py"),
                                                      submodule_search_locations=[here])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


NP = {"f32": np.float32, "f64": np.float64, "u32": np.uint32, "i32": np.int32}
TORCH = {"f32": torch.float32, "f64": torch.float64, "u32": torch.int32, "i32": torch.int32}
SIZE = {"f32": 4, "f64": 8, "u32": 4, "i32": 4}
KINDS = {"bucket": 0, "radix": 1, "topk": 2}


# ------------------------------------------------------------------- cases
def listed():
    one = {"call": "host", "kind": "bucket"}
    flow = {"call": "stream", "kind": "bucket"}
    return [
        # the smallest call: a vector that one work-group holds, a few order statistics back on the host
        dict(one, name="tiny_u32", dtype="u32", values="uniform", n=10_007, num_k=16, ranks="uniform"),
        # a latency-bound summary of a column: every percentile of a million floats (the golden fixture's shape)
        dict(one, name="percentiles_f32", dtype="f32", values="uniform", n=1 << 20, num_k=101, ranks="even"),
        # the hundred largest of a ragged column of scores, on the host
        dict(one, name="top100_i32", kind="topk", dtype="i32", values="uniform", n=1_000_003, num_k=100, ranks="top"),
        # doubles inside a pipeline: quantile edges for a histogram, left on the device
        dict(flow, name="edges_f64", dtype="f64", values="normal", n=3_000_017, num_k=256, ranks="uniform"),
        # an ordinary vector of odd length that fits the memory-side cache
        dict(flow, name="ordinary_f32", dtype="f32", values="normal", n=30_000_001, num_k=512, ranks="uniform"),
        # the benchmark's headline: 2^28 floats, 1024 ranks over the whole range
        dict(flow, name="headline_f32", dtype="f32", values="normal", n=1 << 28, num_k=1024, ranks="uniform"),
        # the same bytes in doubles
        dict(flow, name="headline_f64", dtype="f64", values="normal", n=1 << 27, num_k=1024, ranks="uniform"),
        # the largest top-K
        dict(flow, name="top4096_f32", kind="topk", dtype="f32", values="normal", n=1 << 28, num_k=4096, ranks="top"),
        # the radix path on values that a fixed digit window separates badly
        dict(flow, name="radix_f32", kind="radix", dtype="f32", values="normal", n=1 << 27, num_k=1024, ranks="uniform"),
        # heavy tails, ranks close together around the median plus both extremes
        dict(flow, name="cluster_f32", dtype="f32", values="cauchy", n=1 << 27, num_k=258, ranks="cluster"),
        # the benchmark's batch: 4096 uneven segments, half of them top-K, one captured graph
        {"name": "batch_f32", "call": "batch", "dtype": "f32", "segments": 4096, "lo": 10.0, "hi": 22.0,
         "max_k": 64, "max_topk": 4096, "graph": True, "shape": 4096},
        # a burst of requests over resident vectors of three dtypes, continuously batched
        {"name": "serve_burst", "call": "serve", "requests": 48, "lo": 12.0, "hi": 24.0, "max_k": 256,
         "max_topk": 4096, "inflight": 4, "shape": 5000},
    ]


def _between(rng, lo, hi):
    """Spread over the logarithm, ends included, odd numbers among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.random()
    if what < 0.12:
        return {"call": "batch", "dtype": rng.choice(["f32", "f32", "f64", "u32", "i32"]),
                "segments": _between(rng, 16, 1500), "lo": 10.0, "hi": round(rng.uniform(14.0, 22.0), 2),
                "max_k": rng.choice([16, 64, 256]), "max_topk": rng.choice([64, 1024, 4096]),
                "graph": rng.random() < 0.5, "shape": rng.randrange(1, 1 << 20)}
    if what < 0.24:
        return {"call": "serve", "requests": rng.randrange(8, 61), "lo": 12.0, "hi": round(rng.uniform(16.0, 24.0), 2),
                "max_k": rng.choice([16, 256]), "max_topk": rng.choice([64, 4096]), "inflight": rng.choice([2, 4]),
                "shape": rng.randrange(1, 1 << 20)}
    dtype = rng.choice(["f32", "f32", "f64", "u32", "i32"])
    n = _between(rng, 1 << 10, (1 << 28) // (SIZE[dtype] // 4))
    call = "host" if rng.random() < (0.7 if n < 4_000_000 else 0.25) else "stream"
    kind = rng.choice(["bucket", "bucket", "topk", "radix"])
    values = rng.choice(["uniform", "normal", "normal", "cauchy", "plateau", "levels"] if dtype[0] == "f"
                        else ["uniform", "levels"])
    num_k = _between(rng, 1, min(4096, n // 4))
    ranks = "top" if kind == "topk" else rng.choice(["uniform", "uniform", "even", "cluster"])
    return {"call": call, "kind": kind, "dtype": dtype, "values": values, "n": n, "num_k": max(num_k, 3), "ranks": ranks}


# ------------------------------------------------------------------ inputs
class Vec:
    """A torch tensor as the package takes device vectors: an address, a dtype, a length."""

    def __init__(self, t, dtype):
        self.tensor, self.dtype, self.n = t, np.dtype(NP[dtype]), t.numel()
        self.ptr, self.nbytes = t.data_ptr(), t.numel() * t.element_size()

    def __len__(self):
        return self.n


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _values(out, values, dtype, g):
    """Fill a tensor (or a part of one) with a distribution."""
    if dtype[0] != "f":
        if values == "levels":
            return out.random_(0, 1024, generator=g)
        if dtype == "u32":  # all 32 bits
            return out.copy_(torch.randint(0, 1 << 32, out.shape, generator=g, device="cuda").to(torch.int32))
        return out.random_(-(1 << 31), (1 << 31) - 1, generator=g)
    if values == "normal":
        return out.normal_(generator=g)
    if values == "cauchy":
        return out.cauchy_(generator=g).clamp_(-1e30, 1e30)
    if values == "levels":
        return out.random_(0, 1024, generator=g)
    out.uniform_(generator=g)
    if values == "plateau":
        half = torch.rand(out.shape, generator=g, device="cuda") < 0.5
        out.masked_fill_(half, 0.5)
    return out


def _ranks(ranks, n, num_k, rs):
    if ranks == "even":  # percentiles of the vector, both extremes among them
        return (np.rint(np.arange(num_k) / max(1, num_k - 1) * (n - 1)) + 1).astype(np.uint32)
    if ranks == "cluster":  # close together around the median, and both extremes
        width = min(n, max(1000, 4 * num_k))
        near = rs.choice(width, size=max(1, min(width, num_k - 2)), replace=False) + 1 + (n - width) // 2
        return np.concatenate([np.sort(near), [1, n]]).astype(np.uint32)
    return np.sort(rs.randint(1, n + 1, size=num_k)).astype(np.uint32)


def _spec(case):
    """Lengths, kinds and rank counts of a batch's segments or a burst's requests: part of the case."""
    r = np.random.RandomState(case["shape"])
    m = case.get("segments", case.get("requests"))
    lengths = np.floor(2.0 ** r.uniform(case["lo"], case["hi"], m)).astype(np.int64)
    top = r.rand(m) < 0.5
    num_k = 1 + r.randint(0, case["max_k"], m)
    most = np.minimum(lengths, case["max_topk"]).astype(np.float64)
    K = np.clip(np.floor(2.0 ** (r.rand(m) * np.log2(most))), 1, most).astype(np.int64)
    normal = r.rand(m) < 0.5
    dtypes = np.array(["f32", "u32", "f64"])[np.searchsorted([0.6, 0.9], r.rand(m))] if case["call"] == "serve" else \
        np.full(m, case["dtype"])
    return [dict(n=int(n), top=bool(t), num_k=int(k2 if t else k1), dtype=str(d),
                 values="normal" if z and d[0] == "f" else "uniform")
            for n, t, k1, k2, d, z in zip(lengths, top, num_k, K, dtypes, normal)]


def _segments(case, seed):
    """Per dtype one resident tensor holding its segments back to back, and where each lies."""
    spec, rs, g = _spec(case), np.random.RandomState(seed & 0x7FFFFFFF), _gen(seed)
    total = {}
    for s in spec:
        s["offset"] = total.get(s["dtype"], 0)
        total[s["dtype"]] = s["offset"] + s["n"]
    pool = {d: torch.empty(n, dtype=TORCH[d], device="cuda") for d, n in total.items()}
    for s in spec:
        _values(pool[s["dtype"]][s["offset"]:s["offset"] + s["n"]], s["values"], s["dtype"], g)
        s["k"] = None if s["top"] else rs.randint(1, s["n"] + 1, size=s["num_k"]).astype(np.uint32)
    return spec, pool


def _vector(case, seed):
    x = _values(torch.empty(case["n"], dtype=TORCH[case["dtype"]], device="cuda"), case["values"], case["dtype"], _gen(seed))
    k = None
    if case["kind"] != "topk":
        k = _ranks(case["ranks"], case["n"], case["num_k"], np.random.RandomState(seed & 0x7FFFFFFF))
    return x, k


def prepare(case, seed):
    pkg = _package()
    if case["call"] == "batch":
        spec, pool = _segments(case, seed)
        x = pool[case["dtype"]]
        table = pkg.segment_table([s["n"] for s in spec], ["topk" if s["top"] else "bucket" for s in spec],
                                  [s["num_k"] for s in spec])
        ks = [s["k"] for s in spec if s["k"] is not None]
        batch = pkg.Batch(NP[case["dtype"]], table, np.concatenate(ks) if ks else None)
        out = torch.zeros(batch.num_outputs, dtype=x.dtype, device="cuda")
        torch.cuda.synchronize()  # the batch runs on a stream of its own
        return dict(case=case, batch=batch, x=Vec(x, case["dtype"]), out=Vec(out, case["dtype"]))
    if case["call"] == "serve":
        spec, pool = _segments(case, seed)
        torch.cuda.synchronize()
        vecs = {d: Vec(t, d) for d, t in pool.items()}
        server = pkg.Server({NP[d]: v for d, v in vecs.items()}, 4 << 30, max_inflight=case["inflight"])
        outs = [np.zeros(s["num_k"], NP[s["dtype"]]) for s in spec]
        return dict(case=case, server=server, spec=spec, vecs=vecs, outs=outs)
    x, k = _vector(case, seed)
    state = dict(case=case, x=Vec(x, case["dtype"]), k=k)
    state["ctx"] = pkg.Context(0)  # on the null stream, torch's own
    if case["call"] == "stream":
        L = pkg._lib
        count = case["num_k"] if k is None else k.size
        L.check(L.lib().ggks_ctx_reserve(state["ctx"].handle, KINDS[case["kind"]], pkg.api.dtype_code(NP[case["dtype"]]),
                                         case["n"], count))
        state["out"] = Vec(torch.zeros(count, dtype=x.dtype, device="cuda"), case["dtype"])
        if k is not None:
            state["dk"] = Vec(torch.from_numpy(k.view(np.int32)).cuda(), "u32")
    return state


# -------------------------------------------------------------------- runs
def run(state):
    pkg, case = _package(), state["case"]
    if case["call"] == "batch":
        state["batch"].run(state["x"], state["out"], graph=case["graph"])
        state["batch"].sync()
        return state["out"].tensor
    if case["call"] == "serve":
        server = state["server"]
        for i, (s, out) in enumerate(zip(state["spec"], state["outs"])):
            if s["top"]:
                server.submit(NP[s["dtype"]], s["offset"], s["n"], out, K=s["num_k"], kind="topk", tag=i)
            else:
                server.submit(NP[s["dtype"]], s["offset"], s["n"], out, k=s["k"], tag=i)
        server.drain()
        server.poll()
        return state["outs"]
    x, k, ctx, kind = state["x"], state["k"], state["ctx"], case["kind"]
    if case["call"] == "host":
        return pkg.topk(x, case["num_k"], ctx) if kind == "topk" else pkg.multiselect(x, k, ctx, kind=kind)
    out = state["out"]
    if kind == "topk":
        L = pkg._lib
        o = L.Opts()
        L.check(L.lib().ggks_topk_async(ctx.handle, pkg.api.dtype_code(x.dtype), x.ptr, x.n, case["num_k"], out.ptr,
                                        ctypes.byref(o)))
    else:
        pkg.multiselect_async(x, state["dk"], out, ctx, kind=kind)
    return out.tensor


# ------------------------------------------------------------------- model
def work(case):
    if case["call"] in ("batch", "serve"):
        return {"bytes": sum(s["n"] * SIZE[s["dtype"]] + s["num_k"] * (SIZE[s["dtype"]] + (0 if s["top"] else 4))
                             for s in _spec(case)), "flops": 0}
    size = SIZE[case["dtype"]]
    return {"bytes": case["n"] * size + case["num_k"] * (size + (0 if case["kind"] == "topk" else 4)), "flops": 0}


def _select(x, dtype, k, K):
    """The k-th largest values (or the K largest, descending) of a tensor by a full sort."""
    if dtype == "u32":
        x = x.to(torch.int64) & 0xFFFFFFFF
    s = torch.sort(x).values
    v = s[-K:].flip(0) if k is None else s[torch.from_numpy(x.numel() - k.astype(np.int64)).cuda()]
    return v.cpu().numpy().astype(np.float64 if dtype[0] == "f" else NP[dtype])


def exact(case, seed):
    if case["call"] in ("batch", "serve"):
        spec, pool = _segments(case, seed)
        got = [_select(pool[s["dtype"]][s["offset"]:s["offset"] + s["n"]], s["dtype"], s["k"], s["num_k"]) for s in spec]
        if case["call"] == "serve":
            return got
        return torch.from_numpy(np.concatenate(got).view(np.int32) if case["dtype"] == "u32" else np.concatenate(got))
    x, k = _vector(case, seed)
    v = _select(x, case["dtype"], k, case["num_k"])
    if case["call"] == "stream" and case["dtype"] == "u32":
        v = v.view(np.int32)
    return v
