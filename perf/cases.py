"""The performance cases: what a program asks of the framework, through its public entry points.

A case names a kind of work, the graph it is done on and the options of the call:

    count     exact count of a resident graph (``count``), in one of three forms: "stream" (in-lists,
              segment words and the row-aligned streaming copy, the headline path), "split"
              (in-lists and segment words) and "plain" (a bare oriented CSR)
    batch     the mixed-shape batch in one replayed launch (``BatchPlan``)
    prep      raw edge samples to the oriented CSR and what the count reads beside it (``clean_orient``)
    in_lists  in-lists and segment words for a CSR that came without them (``in_lists``)
    halo      all halo parts of a k-way random partition (``halo_extract_parts``)
    support   per-edge and per-vertex triangle counts (``triangle_support``)
    serve     a burst of requests to the count server, prepared and counted (``Server``)

Graphs are the seeded synthetic ones of the benchmark and the tests: RMAT (.57/.19/.19/.05),
Erdos-Renyi, Chung-Lu (gamma 2.1, mean degree 50) and the grid with random cell diagonals.
Counts and preparations take another graph for each seed.  The other kinds return arrays as long as
the graph has edges, so theirs is one graph whose vertices the seed renumbers at random (as graph500
does): every array differs from seed to seed, its length does not.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import trianglecount_amd as tc
from trianglecount_amd import workloads


def listed():
    return [
        # the headline: exact count of RMAT scale 23, edge factor 16
        {"name": "count_rmat_s23", "kind": "count", "form": "stream", "graph": "rmat", "scale": 23, "ef": 16},
        # an ordinary graph of a few million edges, held resident and counted again
        {"name": "count_rmat_s18", "kind": "count", "form": "stream", "graph": "rmat", "scale": 18, "ef": 16},
        # the smallest call: one request-sized uniform graph, where launches and latency count
        {"name": "count_er_1k", "kind": "count", "form": "split", "graph": "er", "n": 1009, "mean": 20.0},
        # the drop-in case: a bare oriented CSR as the text files hold it
        {"name": "count_plain_s21", "kind": "count", "form": "plain", "graph": "rmat", "scale": 21, "ef": 16},
        # 66 graphs of mixed shapes (grid, Chung-Lu, 64 uniform) in one replayed launch
        {"name": "batch_mixed", "kind": "batch", "graphs": 66},
        # preparation of the headline graph: clean, orient, in-lists, segment words, streaming copy
        {"name": "prep_rmat_s23", "kind": "prep", "form": "stream", "graph": "rmat", "scale": 23, "ef": 16},
        # preparation of a request-sized graph
        {"name": "prep_rmat_s12", "kind": "prep", "form": "split", "graph": "rmat", "scale": 12, "ef": 16},
        # preparation with the symmetric CSR kept (what the halo extraction reads), heavy-tailed degrees
        {"name": "prep_sym_cl_1m", "kind": "prep", "form": "symmetric", "graph": "chung_lu", "n": 1000003, "mean": 50.0},
        # drop-in users' step from a bare CSR to the split count
        {"name": "in_lists_s21", "kind": "in_lists", "graph": "rmat", "scale": 21, "ef": 16},
        # the partitioned path: eight halo parts
        {"name": "halo_s21_k8", "kind": "halo", "graph": "rmat", "scale": 21, "ef": 16, "k": 8, "mode": 0},
        # per-edge support and per-vertex counts
        {"name": "support_s21", "kind": "support", "split": True, "graph": "rmat", "scale": 21, "ef": 16},
        # requests that arrive together: raw edges log-uniform in [1e3, 5e6], 70% RMAT, 30% uniform
        {"name": "serve_burst_64", "kind": "serve", "requests": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, max_edges):
    """A graph of 1e3 to max_edges raw samples, with its ragged sizes as they fall."""
    edges = _log_int(rng, 1000, max_edges)
    g = rng.choice(("rmat", "rmat", "er", "chung_lu", "grid"))
    if g == "rmat":
        ef = rng.randint(5, 24)
        scale = max(6, min(23, int(round(math.log2(max(edges / ef, 64))))))
        while (ef << scale) > max_edges:
            scale -= 1
        return {"graph": "rmat", "scale": scale, "ef": ef}
    if g == "grid":
        side = max(8, int(math.sqrt(edges / 3)))
        return {"graph": "grid", "rows": side | 1, "cols": max(8, edges // 3 // (side | 1)), "p": 0.3}
    if g == "er":
        mean = round(rng.uniform(8.0, 40.0), 2)
        return {"graph": "er", "n": max(64, int(edges * 2 / mean)), "mean": mean}
    return {"graph": "chung_lu", "n": max(500, int(edges / 25)), "mean": 50.0}


def draw(rng):
    kind = rng.choice(("count", "count", "count", "batch", "prep", "prep", "in_lists", "halo", "support", "serve"))
    if kind == "batch":
        return {"kind": "batch", "graphs": rng.randint(3, 66)}
    if kind == "serve":
        return {"kind": "serve", "requests": rng.randint(2, 64)}
    case = {"kind": kind}
    if kind == "count":
        case["form"] = rng.choice(("stream", "stream", "split", "plain"))
        return {**case, **_draw_graph(rng, 32 << 20 if case["form"] == "plain" else 96 << 20)}
    if kind == "prep":
        case["form"] = rng.choice(("stream", "split", "symmetric"))
        return {**case, **_draw_graph(rng, 96 << 20)}
    if kind == "halo":
        return {**case, **_draw_graph(rng, 24 << 20), "k": rng.randint(2, 16), "mode": rng.randint(0, 1)}
    if kind == "support":
        return {**case, **_draw_graph(rng, 24 << 20), "split": rng.random() < 0.7}
    return {**case, **_draw_graph(rng, 64 << 20)}


def _raw(case, seed):
    g = case["graph"]
    if g == "rmat":
        return tc.generate_rmat(case["scale"], case["ef"], seed=seed)
    if g == "er":
        return tc.generate_er(case["n"], case["mean"], seed=seed)
    if g == "chung_lu":
        return tc.generate_chung_lu(case["n"], 2.1, case["mean"], 5e4, seed=seed)
    return tc.generate_grid(case["rows"], case["cols"], case["p"], seed=seed)


def _batch_specs(case, seed):
    specs = workloads.mixed_specs(seed)
    return specs[: case["graphs"]]


def _renumbered(case, seed):
    """The case's graph with its vertex ids permuted, and the permutation."""
    n, src, dst = _raw(case, 1)
    gen = torch.Generator(device=src.device).manual_seed(int(seed))
    perm = torch.randperm(n, generator=gen, device=src.device, dtype=torch.int32)
    return n, perm[src.long()], perm[dst.long()], perm


def _halo_parts_of(case, n, src, dst, perm):
    """The k-way random partition of the vertices that the cleaning keeps, one part per vertex
    whatever its id."""
    part = torch.empty_like(perm)
    part[perm.long()] = tc.partition_random(n, case["k"], seed=1)
    real = src != dst
    seen = torch.zeros(n, dtype=torch.bool, device=src.device)
    seen[src[real].long()] = True
    seen[dst[real].long()] = True
    return part[seen].contiguous()


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case, "ws": tc.Workspace()}
    if kind == "serve":
        # a server and the requests it is about to get
        st["requests"] = workloads.serving_stream(case["requests"], seed=seed)
        st["server"] = tc.Server(16 << 30)
        return st
    if kind == "batch":
        # resident graphs and the plan that replays their launch
        graphs = []
        for spec in _batch_specs(case, seed):
            n, s, d = workloads.generate(spec)
            graphs.append(tc.clean_orient(n, s, d, in_lists=True))
        st["plan"] = tc.BatchPlan(graphs)
        return st
    if kind == "prep":
        st["raw"] = _raw(case, seed)
    elif kind == "count":
        form = case["form"]
        st["graph"] = tc.clean_orient(*_raw(case, seed), in_lists=form != "plain", stream_copy=form == "stream")
    else:
        n, src, dst, perm = _renumbered(case, seed)
        st["graph"] = tc.clean_orient(n, src, dst, keep_symmetric=kind == "halo", in_lists=case.get("split", False))
        if kind == "halo":
            st["part"] = _halo_parts_of(case, n, src, dst, perm)
    return st


def _whole(t, used, size=None):
    """A call's output buffer over its whole length, cleared behind the entries that the call wrote."""
    if size is not None and t.numel() < size:  # a view of the buffer's used part
        t = torch.as_strided(t, (size,), (1,))
    if used < t.numel():
        t[used:].zero_()
    return t


def _in_list_outputs(g, entries):
    k = g.meta["in_entries"]
    return {"in_off": _whole(g.in_off, g.n + 1), "in_col": _whole(g.in_col, k), "col_seg": _whole(g.col_seg, g.m),
            "in_seg": _whole(g.in_seg, k, entries)}


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "count":
        return tc.count(st["graph"], ws=st["ws"])
    if kind == "batch":
        st["plan"].launch_graph()
        return np.array(st["plan"].results(), dtype=np.int64)
    if kind == "prep":
        form = case["form"]
        if form == "symmetric":
            g = tc.clean_orient(*st["raw"], keep_symmetric=True, ws=st["ws"])
            more = {"sym_off": _whole(g.sym_off, g.n + 1), "sym_col": _whole(g.sym_col, 2 * g.m)}
        else:
            # (the padding of the streaming copy's rows is unwritten, so the copy itself is not among the outputs:
            # its row starts are, in the segment words, and the counts of the "stream" form read it)
            g = tc.clean_orient(*st["raw"], in_lists=True, stream_copy=form == "stream", ws=st["ws"])
            more = _in_list_outputs(g, st["raw"][1].numel())
        return {"n": g.n, "m": g.m, "off": _whole(g.off, g.n + 1), "col": _whole(g.col, g.m), **more}
    if kind == "in_lists":
        g = tc.in_lists(st["graph"], ws=st["ws"])
        return _in_list_outputs(g, g.m)
    if kind == "halo":
        parts = tc.halo_extract_parts(st["graph"], st["part"], case["k"], mode=case["mode"], ws=st["ws"])
        return {"owned": [h.owned for h in parts], "off": [h.off[: h.n + 1] for h in parts],
                "col": [h.col[: h.m] for h in parts]}
    if kind == "support":
        sup, pv = tc.triangle_support(st["graph"], split=case["split"], ws=st["ws"])
        return {"support": sup, "per_vertex": pv}
    srv = st["server"]
    ids = [srv.submit_rmat(r.a, r.m_raw, r.seed) if r.kind == "rmat" else srv.submit_er(r.a, r.m_raw, r.seed)
           for r in st["requests"]]
    got = [srv.wait(i) for i in ids]
    return {"count": np.array([g["count"] for g in got], dtype=np.int64),
            "edges": np.array([g["edges"] for g in got], dtype=np.int64)}


def _sizes(case):
    """(vertices, edges): the raw samples, a few per cent above the edges that are left after cleaning."""
    g = case["graph"]
    if g == "rmat":
        return 1 << case["scale"], case["ef"] << case["scale"]
    if g == "grid":
        return case["rows"] * case["cols"], int((2 + case["p"]) * case["rows"] * case["cols"])
    return case["n"], int(case["n"] * case["mean"] / 2)


def work(case):
    """Bytes of the inputs read once and the outputs written once; the work is on whole numbers."""
    kind = case["kind"]
    if kind == "serve":  # raw edge samples are made, cleaned and counted on the device
        m = sum(r.m_raw for r in workloads.serving_stream(case["requests"], seed=1))
        return {"bytes": 8 * m + 4 * m, "flops": 0}
    if kind == "batch":
        total = 0
        for s in _batch_specs(case, 1):
            n, m = (s.a * s.b, int(2.3 * s.a * s.b)) if s.kind == "grid" else (s.a, int(s.a * (s.mean or s.p) / 2))
            total += 8 * n + 4 * m
        return {"bytes": total, "flops": 0}
    n, m = _sizes(case)
    csr = 8 * n + 4 * m
    lists = 8 * n + 2 * m  # in-lists hold about half the arcs
    words = 8 * m + 4 * m
    if kind == "count":
        return {"bytes": csr, "flops": 0}
    if kind == "prep":
        out = csr + (8 * n + 8 * m if case["form"] == "symmetric" else lists + words)
        return {"bytes": 8 * m + out + (4 * m if case["form"] == "stream" else 0), "flops": 0}
    if kind == "in_lists":
        return {"bytes": csr + lists + words, "flops": 0}
    if kind == "halo":  # each part holds its owned vertices' rows and their neighbours'
        return {"bytes": 8 * n + 8 * m + 4 * n + csr, "flops": 0}
    return {"bytes": csr + 4 * m + 8 * n, "flops": 0}
