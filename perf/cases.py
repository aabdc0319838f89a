"""Performance cases: what programs built on this framework spend their time on.

A case is a dict of plain values.  `prepare` makes what a program has in hand
before the call (graph, state, batch, selector weights), `run` is one pass
through the public Python entry points (grudon_amd/api.py), the results
included, `work` the bytes and operations a pass cannot do without, `exact`
the FP64 value of the floating-point outputs.

Graphs are made here with torch from the seed alone: RMAT with the benchmark's
a/b/c/d = .57/.19/.19/.05 on any number of vertices (recursive bits, endpoints
beyond n dropped) and Erdos-Renyi, duplicates and self-loops removed; arc
weights uniform in [1, 255], equal in both directions.
"""
import math
import os

import numpy as np
import torch

from grudon_amd import api

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RMAT_A, RMAT_B, RMAT_C = 0.57, 0.19, 0.19

ALGO = {"pr": api.PR, "cc": api.CC, "sssp": api.SSSP, "pr_pull": api.PR_PULL}
SCHED = {"plain": api.SCHED_PLAIN, "heuristic": api.SCHED_HEURISTIC, "learned": api.SCHED_LEARNED,
         "ndp": api.SCHED_NDP_ENGINE}


def _solve(name, **kw):
    c = {"name": name, "kind": "solve", "graph": "rmat", "n": 1 << 10, "ef": 16, "sym": False, "C": 1, "M": 4,
         "algo": "cc", "sched": "heuristic", "weighted": False, "delta": 0, "sources": 1, "value_bytes": 4,
         "mirror": False}
    c.update(kw)
    return c


def listed():
    return [
        # the smoke run's size: connected components of a graph of a thousand
        # vertices, where the launches and the waits of each superstep count
        _solve("cc_1k", n=1 << 10, sym=True, M=2),
        # the command line's defaults (push + sparse sync every superstep) on a
        # small ragged graph over several compute and memory partitions placed
        # by a partition file, with the reference's uint64 vertex properties
        _solve("sssp_hop_20k_parts", graph="er", n=20011, ef=8, sym=True, C=2, M=3, algo="sssp", sched="plain",
               value_bytes=8, mirror=True),
        # the reference's CPU-runnable configuration: delta-push PageRank on
        # RMAT-18, one compute and one memory partition; a hundred supersteps
        _solve("pr_push_rmat18", n=1 << 18, M=1, algo="pr"),
        # the default schedule again on an ordinary graph: connected components
        # by pushes alone
        _solve("cc_plain_rmat20", n=1 << 20, sym=True, sched="plain"),
        # pull PageRank at an ordinary ragged size (a program that ranks one
        # graph of a million vertices)
        _solve("pr_pull_1m", n=1000003, algo="pr_pull"),
        # weighted delta-stepping from several sources under the learned
        # schedule, at the size the selector's gain is tested on
        _solve("sssp_weighted_rmat22", n=1 << 22, sym=True, algo="sssp", sched="learned", weighted=True, delta=256,
               sources=4),
        # connected components at the benchmark's large symmetrized size
        _solve("cc_rmat24", n=1 << 24, sym=True),
        # the largest: pull PageRank on half a billion arcs, the headline's
        # workload one scale down (its preparation takes half the time)
        _solve("pr_pull_rmat25", n=1 << 25, algo="pr_pull"),
        # many graphs of uneven size in one batch, PageRank and components
        {"name": "batch_24", "kind": "batch", "count": 24, "n_lo": 1 << 14, "n_hi": 3 << 17},
        # one graph handed over as a host CSR and solved once, as the command
        # line does: partitioning, state, solve, labels, release
        _solve("whole_call_700k", kind="whole", n=700001, ef=8, sym=True),
        # the selector on its own: logits of a trace's records
        {"name": "selector_infer_2k", "kind": "infer", "rows": 2000},
        # one training batch of the selector: loss and gradients
        {"name": "selector_grad_20k", "kind": "grad", "rows": 20003},
    ]


def draw(rng):
    """One more case of the listed ranges."""
    def loguni(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve"] * 7 + ["whole", "batch", "infer", "grad"])
    if kind in ("infer", "grad"):
        return {"kind": kind, "rows": loguni(1, 4096) if kind == "infer" else loguni(200, 40000)}
    if kind == "batch":
        hi = loguni(1 << 15, 1 << 18)
        return {"kind": "batch", "count": rng.randint(2, 24), "n_lo": loguni(1 << 12, hi), "n_hi": hi}
    algo = rng.choice(["cc", "sssp", "pr", "pr_pull", "pr_pull"]) if kind == "solve" else rng.choice(["cc", "pr_pull"])
    sched = "heuristic" if kind == "whole" else rng.choice(["plain", "heuristic", "heuristic", "learned", "ndp"])
    top = {"cc": 1 << 22, "sssp": 1 << 21, "pr": 1 << 20, "pr_pull": 1 << 23}[algo]
    if kind == "whole" or (sched in ("plain", "ndp") and algo != "pr_pull"):
        top = 1 << 20
    n = loguni(1 << 10, top)
    if rng.random() < 0.5:
        n |= 1
    C, M = rng.choice([(1, 1), (1, 2), (1, 4), (1, 4), (2, 3)])
    # (Erdos-Renyi graphs of these degrees are connected: every label 0)
    c = _solve("", kind=kind, graph="rmat" if algo == "cc" else rng.choice(["rmat", "er"]), n=n, ef=rng.choice([8, 16]),
               sym=rng.random() < 0.5, C=C, M=M, algo=algo, sched=sched,
               weighted=algo == "sssp" and rng.random() < 0.5,
               delta=rng.choice([0, 256]) if algo == "sssp" else 0,
               sources=rng.randint(1, 3) if algo == "sssp" else 1,
               value_bytes=rng.choice([4, 8]) if algo in ("cc", "sssp") else 4, mirror=rng.random() < 0.25)
    del c["name"]
    return c


# ---- inputs ----

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _keys_to_csr(src, dst, n):
    keys = torch.sort(src * n + dst).values
    keep = torch.ones(keys.numel(), dtype=torch.bool, device=keys.device)
    keep[1:] = keys[1:] != keys[:-1]
    keep &= (keys // n) != (keys % n)
    keys = keys[keep]
    rp = torch.searchsorted(keys, torch.arange(n + 1, device=keys.device, dtype=torch.int64) * n)
    return rp, keys % n


def _make_graph(kind, n, ef, sym, seed):
    """Device tensors (row_ptr int64, col int64) of a seeded graph."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    if kind == "er":
        e = max(1, n * ef // 2)
        src = torch.randint(0, n, (e,), device=dev, generator=gen)
        dst = torch.randint(0, n, (e,), device=dev, generator=gen)
        sym = True
    else:
        e, srcs, dsts = max(1, n * ef), [], []
        for lo in range(0, e, 1 << 26):
            k = min(1 << 26, e - lo)
            s = torch.zeros(k, dtype=torch.int64, device=dev)
            d = torch.zeros(k, dtype=torch.int64, device=dev)
            for _ in range(max(1, (n - 1).bit_length())):
                r = torch.rand(k, device=dev, generator=gen)
                s = s * 2 + (r >= RMAT_A + RMAT_B)
                d = d * 2 + (((r >= RMAT_A) & (r < RMAT_A + RMAT_B)) | (r >= RMAT_A + RMAT_B + RMAT_C))
            ok = (s < n) & (d < n)
            srcs.append(s[ok])
            dsts.append(d[ok])
        src, dst = torch.cat(srcs), torch.cat(dsts)
        del srcs, dsts
    if sym:
        src, dst = torch.cat([src, dst]), torch.cat([dst, src])
    return _keys_to_csr(src, dst, n)


def _weights(rp, col, seed):
    """Weights in [1, 255], the same for (u, v) and (v, u)."""
    n = rp.numel() - 1
    src = torch.repeat_interleave(torch.arange(n, device=rp.device), rp[1:] - rp[:-1])
    h = torch.minimum(src, col) * 1000003 + torch.maximum(src, col) * 8191 + seed * 2654435761
    h = (h ^ (h >> 15)) * 2246822519
    h = (h ^ (h >> 13)) & 0x7FFFFFFF
    return h % 255 + 1


def _u32(t):
    return t.to(torch.int32).cpu().numpy().view(np.uint32)


def _host_graph(case, seed):
    rp, col = _make_graph(case["graph"], case["n"], case["ef"], case["sym"], seed)
    w = _u32(_weights(rp, col, seed)) if case["weighted"] else None
    out = (_u32(rp), _u32(col), w)
    del rp, col
    if torch.cuda.is_available():
        torch.cuda.empty_cache()
    return out


def _mirror(case, seed):
    if not case["mirror"] or case["M"] == 1:
        return None
    return np.random.default_rng(seed + 17).integers(0, case["M"], case["n"], dtype=np.uint32)


def _batch_graphs(case, seed):
    """Sizes and degrees belong to the case, the graphs to the seed."""
    rng = np.random.default_rng([case["count"], case["n_lo"], case["n_hi"]])
    out = []
    for i in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        kind, ef = ("rmat", int(rng.integers(8, 33))) if i % 2 == 0 else ("er", int(rng.integers(4, 65)))
        out.append(_make_graph(kind, n, ef, False, seed * 1000 + i))
    return out


def _selector_weights():
    return np.fromfile(os.path.join(ROOT, "grudon_amd", "selector_bf16.bin"), dtype="<u2")


def _features(rows, seed):
    """Records as the traces hold them: sizes and fractions in [0, 1], the
    algorithm as one-hot columns."""
    rng = np.random.default_rng(seed)
    f = rng.random((rows, 16), dtype=np.float32)
    f[:, 13:] = np.eye(3, dtype=np.float32)[rng.integers(0, 3, rows)]
    return f


def _grad_inputs(case, seed):
    rng = np.random.default_rng(seed + 1)
    bits = _selector_weights().astype(np.uint32) << 16
    w = bits.view(np.float32) + rng.normal(0, 1e-3, bits.size).astype(np.float32)
    label = rng.integers(0, 4, case["rows"], dtype=np.uint32)
    sw = rng.uniform(0.1, 10.0, case["rows"]).astype(np.float32)
    return w.astype(np.float32), _features(case["rows"], seed), label, sw


# ---- the pass ----

def prepare(case, seed):
    ctx = api.Context(0)
    st = {"ctx": ctx, "kind": case["kind"]}
    if case["kind"] == "infer":
        ctx.selector_load(_selector_weights(), api.SELECTOR_MARGIN)
        st["feat"] = _features(case["rows"], seed)
    elif case["kind"] == "grad":
        st["args"] = _grad_inputs(case, seed)
    elif case["kind"] == "batch":
        graphs = [(_u32(rp), _u32(col)) for rp, col in _batch_graphs(case, seed)]
        st["batch"] = api.Batch(ctx, graphs)
        st["batch"].tune(tile=1024, grid_per_cu=8, K=8)  # what autotune chooses for such batches
    else:
        rp, col, w = _host_graph(case, seed)
        mirror = _mirror(case, seed)
        st["init"] = [{"sched": SCHED[case["sched"]]}]
        if case["sched"] == "learned":
            ctx.selector_load(_selector_weights(), api.SELECTOR_MARGIN)
        if case["algo"] == "sssp":
            has = np.flatnonzero(np.diff(rp.astype(np.int64)))
            pick = np.random.default_rng(seed + 3).choice(has, size=case["sources"])
            st["init"] = [dict(st["init"][0], source=int(v), weighted=case["weighted"], delta=case["delta"])
                          for v in pick]
        st["algo"], st["value_bytes"] = ALGO[case["algo"]], case["value_bytes"]
        st["csr"] = dict(rp=rp, col=col, w=w, C=case["C"], M=case["M"], mirror=mirror)
        if case["kind"] == "solve":
            g = api.Graph.from_csr(ctx, **st.pop("csr"))
            st["state"] = api.State(g, st["algo"], st["value_bytes"])
    return st


def _solves(S, inits):
    out = []
    for kw in inits:
        S.init(**kw)
        stats = S.run()
        r = {"result": S.result()}
        if S.algo in (api.CC, api.SSSP):
            r["iterations"] = stats["iterations"]
        out.append(r)
    return out


def run(state):
    kind = state["kind"]
    if kind == "infer":
        return state["ctx"].selector_infer(state["feat"])
    if kind == "grad":
        loss, grad = state["ctx"].selector_grad(*state["args"])
        return {"loss": loss, "grad": grad}
    if kind == "batch":
        B = state["batch"]
        B.pagerank(tolerance=1e-6)
        ranks = [B.result(i, api.PR_PULL) for i in range(B.count)]
        it, _ = B.cc()
        return {"ranks": ranks, "labels": [B.result(i, api.CC) for i in range(B.count)], "cc_iterations": it}
    if kind == "solve":
        return _solves(state["state"], state["init"])
    g = api.Graph.from_csr(state["ctx"], **state["csr"])
    S = api.State(g, state["algo"], state["value_bytes"])
    out = _solves(S, state["init"])
    S.free()
    g.free()
    return out


def _arcs(case):
    return case["n"] * case["ef"] * (2 if case["sym"] and case["graph"] == "rmat" else 1)


def work(case):
    """Bytes: a column and a source value per arc and a value per vertex for
    every sweep over the arcs the algorithm needs (PageRank to 1e-6 about 20
    sweeps, the delta form about as many full ones; labels and distances at
    least one), the results once, and the host CSR once where it is handed
    over.  Operations: an add per arc and sweep."""
    k = case["kind"]
    if k == "infer":
        return {"bytes": case["rows"] * 80 + 11016, "flops": 2 * 5376 * case["rows"]}
    if k == "grad":
        return {"bytes": case["rows"] * 72 + 2 * 22032, "flops": 6 * 5376 * case["rows"]}
    if k == "batch":
        n = case["count"] * (case["n_hi"] - case["n_lo"] + 1) / max(1e-9, math.log((case["n_hi"] + 1) / case["n_lo"]))
        m = n * 27
        return {"bytes": int(20 * (8 * m + 8 * n) + 6 * (8 * m + 8 * n)), "flops": int(26 * m)}
    m, n = _arcs(case), case["n"]
    sweeps = 20 if case["algo"] in ("pr", "pr_pull") else case["sources"]
    hand = 4 * (m + n) if k == "whole" else 0
    wb = 1 if case["weighted"] else 0
    return {"bytes": sweeps * ((8 + wb) * m + 8 * n) + case["value_bytes"] * n * case["sources"] + hand,
            "flops": sweeps * m}


# ---- FP64 values ----

def _scatter(rp, col, x):
    """y[v] = sum of x over v's in-neighbours, FP64, arcs in chunks."""
    n = rp.numel() - 1
    y = torch.zeros(n, dtype=torch.float64, device=rp.device)
    rows = 1 << 22
    for a in range(0, n, rows):
        b = min(n, a + rows)
        cnt = rp[a + 1:b + 1] - rp[a:b]
        y.index_add_(0, col[int(rp[a]):int(rp[b])], torch.repeat_interleave(x[a:b], cnt))
    return y


def _pagerank64(rp, col, d=0.85, tol=1e-6):
    n = rp.numel() - 1
    deg = (rp[1:] - rp[:-1]).to(torch.float64)
    sink, inv = deg == 0, torch.where(deg > 0, 1.0 / deg.clamp(min=1.0), torch.zeros_like(deg))
    r = torch.full((n,), 1.0 / n, dtype=torch.float64, device=rp.device)
    for _ in range(1000):
        nr = (1.0 - d) / n + d * (_scatter(rp, col, r * inv) + r[sink].sum() / n)
        res = float((nr - r).abs().sum())
        r = nr
        if res < tol:
            break
    return r.cpu().numpy()


def _delta_pagerank64(rp, col):
    """The reference's delta push: an update above 1e-6 is folded into the
    rank and passed on, what lies below waits for more."""
    deg = (rp[1:] - rp[:-1]).to(torch.float64)
    out = deg > 0
    zero = torch.zeros_like(deg)
    safe = deg.clamp(min=1.0)
    pr, prop = torch.where(out, zero + 0.15, zero), torch.where(out, 0.85 * 0.15 / safe, zero)
    upd, front = zero.clone(), out
    for _ in range(1000):
        upd = upd + _scatter(rp, col, torch.where(front, prop, zero))
        front = upd > 1e-6
        if not bool(front.any()):
            break
        pr = torch.where(front, pr + upd, pr)
        prop = torch.where(front & out, 0.85 * upd / safe, zero)
        upd = torch.where(front, zero, upd)
    return pr.cpu().numpy()


def _mlp64(w, f):
    w, x = w.astype(np.float64), f.astype(np.float64)
    W1, b1, W2 = w[:1024].reshape(64, 16), w[1024:1088], w[1088:5184].reshape(64, 64)
    b2, W3, b3 = w[5184:5248], w[5248:5504].reshape(4, 64), w[5504:5508]
    h1 = np.maximum(x @ W1.T + b1, 0.0)
    h2 = np.maximum(h1 @ W2.T + b2, 0.0)
    return x, W1, W2, W3, h1, h2, h2 @ W3.T + b3


def exact(case, seed):
    k = case["kind"]
    if k == "infer":
        w = (_selector_weights().astype(np.uint32) << 16).view(np.float32)
        return _mlp64(w, _features(case["rows"], seed))[-1]
    if k == "grad":
        w, f, label, sw = _grad_inputs(case, seed)
        x, _, W2, W3, h1, h2, lg = _mlp64(w, f)
        p = np.exp(lg - lg.max(axis=1, keepdims=True))
        p /= p.sum(axis=1, keepdims=True)
        rows = np.arange(len(label))
        loss = float((sw.astype(np.float64) * -np.log(np.maximum(p[rows, label], 1e-30))).sum())
        dl = p.copy()
        dl[rows, label] -= 1.0
        dl *= sw[:, None]
        d2 = (dl @ W3) * (h2 > 0)
        d1 = (d2 @ W2) * (h1 > 0)
        return {"loss": loss, "grad": np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0),
                                                      (dl.T @ h2).ravel(), dl.sum(0)])}
    if k == "batch":
        ranks = [_pagerank64(rp, col) for rp, col in _batch_graphs(case, seed)]
        return {"ranks": ranks, "labels": [None] * case["count"], "cc_iterations": None}
    if case["algo"] in ("cc", "sssp"):
        return None
    rp, col = _make_graph(case["graph"], case["n"], case["ef"], case["sym"], seed)
    return [{"result": _pagerank64(rp, col) if case["algo"] == "pr_pull" else _delta_pagerank64(rp, col)}]
