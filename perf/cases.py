"""The retrieval work that is measured: queries, batches and neighbour searches over a device-resident graph.

A case is one call of the C ABI (include/mars_amd.h) as a serving program makes it: the graph, its reduced-precision row
copies and the query context are in place, query vectors arrive in host memory (single queries) or device memory (batches),
and the answer is in host memory when the call returns. The corpus is the benchmark's: episodes of ten nodes (4 IMAGE,
3 TEXT, 3 AUDIO) around a random centroid, unit rows, timestamps over 600 s; edges within each episode, and from each TEXT and
AUDIO node to four others (on the benchmark corpus an IMAGE node's nearest neighbours lie in its own episode, and about
half of a TEXT or AUDIO node's do). Queries are IMAGE nodes.

Paths: "episode" and "global" (mars_query), "batch" (mars_query_batch), "gbatch" (mars_query_global_batch), "link"
(mars_query_global_batch_knn), "knn" (mars_graph_knn) and "knn_range" (mars_graph_knn_range).
"""
import ctypes as C
import math

import numpy as np
import torch

import mars_amd
from mars_amd import _lib
from mars_amd._lib import check, lib

T_END = 600.0                        # every timestamp lies before it; single queries ask at this time
FMAX = float(np.finfo(np.float32).max)
RESULT = np.dtype([("node", np.int32), ("score", np.float32), ("modality", np.int32), ("hops", np.int32)])


def listed():
    one = dict(k=10, results=15, hops=2, decay=0.1, filter=-1, boost=0.0)
    return [
        # the smallest call: an agent asks for its current episode, ten rows out of 100K
        dict(name="episode_100k", path="episode", n=100_000, d=768, rows="fp32", **{**one, "hops": 0}),
        # a global query over a session's memory with the default context (fp32 rows, stage timers on) and decay
        dict(name="global_10k", path="global", n=10_000, d=768, rows="fp32", timing=True, **{**one, "decay": 1e-8}),
        # a global query over a day's memory; certified over the int8 copy
        dict(name="global_100k", path="global", n=100_000, d=768, rows="int8", timing=False, **one),
        # the headline: a global query over 1M nodes; certified over the int8 copy
        dict(name="global_1m", path="global", n=1_000_000, d=768, rows="int8", timing=False, **one),
        # a boosted query for TEXT nodes alone: fp32 rows, more seeds, narrower rows, a ragged node count
        dict(name="filtered_300k", path="global", n=300_007, d=512, rows="fp32", timing=False,
             **{**one, "k": 32, "results": 32, "filter": 0, "boost": 0.25}),
        # batched scoring for a reranker: 64 queries (HBM-bound), then 256 (MFMA-bound)
        dict(name="batch64_1m", path="batch", n=1_000_000, d=768, q=64, k=10, decay=0.1, filter=-1, mixed=False),
        dict(name="batch256_1m", path="batch", n=1_000_000, d=768, q=256, k=10, decay=0.1, filter=-1, mixed=False),
        # global queries of many agents answered together, BFS included: one int8 pass for 16, one MFMA pass for 100
        dict(name="gbatch16_1m", path="gbatch", n=1_000_000, d=768, q=16, mixed=False, **one),
        dict(name="gbatch100_100k", path="gbatch", n=100_000, d=768, q=100, mixed=True, **one),
        # the streaming server's call: waiting queries, and the neighbours of the nodes inserted since the last one
        dict(name="link_1m", path="link", n=1_000_000, d=768, q=4, nodes=12, knn=8, mixed=False, **one),
        # the 8-NN graph of a small corpus, and a piece of a large one's
        dict(name="knn_10k", path="knn", n=10_000, d=768, knn=8),
        dict(name="knn_range_1m", path="knn_range", n=1_000_000, d=768, nodes=8192, knn=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["episode", "global", "global", "global", "batch", "batch", "gbatch", "gbatch", "link", "knn", "knn_range"])
    n = _log(rng, 2_000, 1_000_000)
    if rng.random() < 0.5:
        n |= 1
    d = rng.choice([256, 512, 768, 768, 768])
    c = dict(path=path, n=n, d=d)
    if path in ("knn", "knn_range"):
        c["knn"] = rng.choice([4, 6, 8, 8, 16])
        if path == "knn":
            c["n"] = _log(rng, 2_000, 60_000) | rng.randint(0, 1)
        else:
            c["nodes"] = min(n, _log(rng, 200, 8_192))
        return c
    c["decay"] = rng.choice([1e-8, 8e-6, 0.1, 0.1])
    c["filter"] = rng.choice([-1, -1, -1, 0, 2])
    if path == "batch":
        c.update(q=_log(rng, 1, 512), k=rng.randint(1, 16), mixed=rng.random() < 0.5)
        return c
    c.update(k=rng.choice([1, 5, 10, 10, 16]), hops=rng.choice([0, 1, 2, 2, 2, 3]), boost=0.0)
    c["results"] = rng.choice([c["k"], 15, 30])
    if path in ("gbatch", "link"):
        c["mixed"] = rng.random() < 0.5
        if path == "gbatch":
            c["q"] = _log(rng, 2, 256)
        else:
            c.update(q=rng.randint(0, 8), nodes=rng.randint(1, 40), knn=8)
        return c
    c["rows"] = rng.choice(["fp32", "fp16", "int8", "int8"])
    if path == "episode":
        c.update(rows="fp32", hops=0, filter=-1, k=min(c["k"], 10), results=15)
        return c
    c["timing"] = rng.random() < 0.3
    if rng.random() < 0.2:
        c.update(k=rng.randint(17, 64), results=rng.choice([40, 200]))
    if c["rows"] == "fp32" and rng.random() < 0.5:
        c["boost"] = 0.25
    return c


# ---- inputs ----------------------------------------------------------------------------------------------------------
class Inputs:
    """Rows, attributes, edges and queries of a case, made on the GPU from the seed alone."""

    def __init__(self, c, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        n, d, dev = c["n"], c["d"], "cuda"
        ne = (n + 9) // 10
        slot = torch.arange(n, device=dev, dtype=torch.int32) % 10
        self.ep = torch.arange(n, device=dev, dtype=torch.int32) // 10
        image = slot < 4
        self.mods = torch.where(image, 2, torch.where(slot < 7, 0, 1)).to(torch.int32)
        emb = torch.randn(n, d, device=dev, generator=g)
        emb *= torch.where(image, 0.3, 1.0)[:, None]
        cent = torch.randn(ne, d, device=dev, generator=g)
        scale = torch.where(image, 1.0, 0.35)
        for lo in range(0, n, 1 << 18):                      # whole episodes need not align: each row adds its own centroid
            hi = min(n, lo + (1 << 18))
            emb[lo:hi].addcmul_(cent[self.ep[lo:hi].long()], scale[lo:hi, None])
        emb /= torch.linalg.vector_norm(emb, dim=1, keepdim=True)
        self.emb = emb
        start = torch.rand(ne, device=dev, generator=g) * 599.0
        self.ts = start[self.ep.long()] + 0.1 * slot.to(torch.float32)
        self.row = self.col = None
        if c["path"] not in ("knn", "knn_range"):
            i = torch.arange(n, device=dev)
            src = [i.repeat_interleave(9)]
            other = torch.arange(9, device=dev).repeat(n)
            other += other >= slot.long().repeat_interleave(9)
            dst = [self.ep.long().repeat_interleave(9) * 10 + other]
            far = i[~image].repeat_interleave(4)
            to = torch.randint(0, n, (far.numel(),), device=dev, generator=g)
            src += [far, to]
            dst += [to, far]
            src, dst = torch.cat(src), torch.cat(dst)
            keep = (dst < n) & (src != dst)
            key = torch.unique(src[keep] * n + dst[keep])
            self.row = torch.zeros(n + 1, dtype=torch.int32, device=dev)
            self.row[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
            self.col = (key % n).to(torch.int32)
        nq = max(1, c.get("q", 1))
        node = (torch.randint(0, max(1, n // 10), (nq,), device=dev, generator=g) * 10
                + torch.randint(0, 4, (nq,), device=dev, generator=g))
        self.node = node.cpu().numpy()
        self.q = emb[node].clone()
        late = torch.rand(nq, device=dev, generator=g).cpu().numpy() * 60.0 if c.get("mixed") else np.zeros(nq)
        self.tq = (T_END - late).astype(np.float32)


def _config(c, inp):
    f = dict(top_k=c.get("k", 10), time_decay_lambda=c.get("decay", 0.0), modality_filter=c.get("filter", -1),
             bfs_max_hops=c.get("hops", 0), max_results_returned=c.get("results", -1))
    if c["path"] == "episode" or c.get("boost"):
        f["query_episode_id"] = int(inp.node[0]) // 10
    if c.get("boost"):
        f["episode_same_boost"] = c["boost"]
    if c["path"] == "episode":
        f.update(retrieval_scope=mars_amd.RetrievalScope.EpisodeScoped,
                 query_episode_member_begin=f["query_episode_id"] * 10, query_episode_member_count=10)
    return mars_amd.RetrievalConfig(**f)


class State:
    """The graph and context that a program keeps, its queries and its result buffers."""

    def __init__(self, c, seed):
        self.dg = self.ctx = self.dq = None
        inp, n, d, path = Inputs(c, seed), c["n"], c["d"], c["path"]
        self.case = c
        torch.cuda.synchronize()
        edges = 0 if inp.col is None else inp.col.numel()
        desc = _lib.GraphDescC(n, edges, d, inp.row.data_ptr() if edges else None, inp.col.data_ptr() if edges else None,
                               inp.emb.data_ptr(), inp.mods.data_ptr(), inp.ts.data_ptr(), 0, 0, _lib.MARS_DESC_DEVICE_POINTERS)
        h = C.c_void_p()
        check(lib.mars_graph_create(C.byref(desc), C.byref(h)), "mars_graph_create")
        self.dg = mars_amd.DeviceMemoryGraph(h, n, edges, d)
        rows = c.get("rows", "")
        if path == "episode" or c.get("boost"):
            ids = inp.ep.cpu().numpy()
            mars_amd.upload_episode_ids(self.dg, ids)
            mars_amd.upload_episode_csr(self.dg, mars_amd.build_episode_csr(ids, n))
        if rows == "fp16" or path in ("batch", "gbatch", "link", "knn", "knn_range"):
            mars_amd.upload_fp16_embeddings(self.dg)
        if rows == "int8" or path in ("gbatch", "link"):
            mars_amd.upload_int8_embeddings(self.dg)
        if path in ("knn", "knn_range"):
            return
        flags = {"fp16": _lib.MARS_CTX_USE_FP16, "int8": _lib.MARS_CTX_CERTIFIED}.get(rows, 0)
        flags |= _lib.MARS_CTX_TIMING if c.get("timing") else 0
        self.ctx = mars_amd.create_query_context(n, d, 64, flags)
        self.cfg = _config(c, inp)
        self.cc = self.cfg.to_c()
        self.tq = inp.tq
        if path in ("episode", "global"):
            self.hq = inp.q[0].cpu().numpy()
            self.out = np.zeros(c["results"], RESULT)
            self.n_out, self.stats = C.c_int32(), _lib.StatsC()
        else:
            self.dq = mars_amd.DeviceBuffer.from_array(inp.q.cpu().numpy())
            self.cap = c.get("results", 1)
            self.out = np.zeros((len(inp.tq), self.cap), RESULT)
            self.n_out, self.stats = np.zeros(len(inp.tq), np.int32), _lib.BatchStatsC()
            if path == "link":
                self.knn = np.full((c["nodes"], c["knn"]), -1, np.int32)

    def __del__(self):
        if self.ctx is not None:
            mars_amd.destroy_query_context(self.ctx)
        if self.dq is not None:
            self.dq.free()
        if self.dg is not None:
            mars_amd.free_device(self.dg)


def prepare(case, seed):
    return State(case, seed)


def _p(a):
    return C.c_void_p(a.ctypes.data)


def run(s):
    c, path = s.case, s.case["path"]
    if path in ("episode", "global"):
        check(lib.mars_query(s.dg.handle, s.ctx.handle, _p(s.hq), float(s.tq[0]), C.byref(s.cc), _p(s.out), len(s.out),
                             C.byref(s.n_out), C.byref(s.stats)), "mars_query")
        return {"n": s.n_out.value, "nodes": s.out["node"], "hops": s.out["hops"], "scores": s.out["score"]}
    if path == "batch":
        ids, scores = mars_amd.query_batch(s.dg, s.ctx, s.dq.ptr, c["q"], s.tq, s.cfg)
        return {"nodes": ids, "scores": scores}
    if path == "gbatch":
        check(lib.mars_query_global_batch(s.dg.handle, s.ctx.handle, C.c_void_p(s.dq.ptr), c["q"], _p(s.tq), C.byref(s.cc),
                                          _p(s.out), s.cap, _p(s.n_out), C.byref(s.stats)), "mars_query_global_batch")
        return {"n": s.n_out, "nodes": s.out["node"], "hops": s.out["hops"], "scores": s.out["score"]}
    if path == "link":
        check(lib.mars_query_global_batch_knn(s.dg.handle, s.ctx.handle, C.c_void_p(s.dq.ptr), c["q"], _p(s.tq),
                                              C.byref(s.cc), _p(s.out), s.cap, _p(s.n_out), C.byref(s.stats),
                                              c["n"] - c["nodes"], c["nodes"], c["knn"], _p(s.knn)),
              "mars_query_global_batch_knn")
        return {"n": s.n_out, "nodes": s.out["node"], "hops": s.out["hops"], "scores": s.out["score"], "knn": s.knn}
    if path == "knn":
        return {"knn": mars_amd.graph_knn(s.dg, c["knn"])}
    return {"knn": mars_amd.graph_knn_range(s.dg, c["knn"], c["n"] // 3 if c["n"] // 3 + c["nodes"] <= c["n"] else 0, c["nodes"])}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def work(case):
    c, path, n, d = case, case["path"], case["n"], case["d"]
    filtered = 4 * n if c.get("filter", -1) >= 0 else 0                # the modalities
    if path == "episode":
        return {"bytes": 10 * (4 * d + 8) + 4 * d, "flops": 20 * d}
    if path == "global":
        row = {"fp32": 4 * d, "fp16": 2 * d, "int8": d + 8}[c["rows"]]  # int8 rows carry a scale and a bound
        return {"bytes": n * (row + 4) + filtered + (4 * n if c["boost"] else 0) + 4 * d, "flops": 2 * n * d}
    if path == "batch":
        return {"bytes": n * (2 * d + 4) + filtered + c["q"] * (4 * d + 8 * c["k"]), "flops": 2 * n * d * c["q"]}
    if path in ("gbatch", "link"):
        q = c["q"] + c.get("nodes", 0)
        row = d + 8 if q <= 16 else 2 * d                               # up to 16 searches are one pass over the int8 rows
        return {"bytes": n * (row + 4) + filtered + 4 * d * q, "flops": 2 * n * d * q}
    q = n if path == "knn" else c["nodes"]
    return {"bytes": 2 * n * d + 4 * d * q + 4 * c["knn"] * q, "flops": 2 * n * d * q}


def tolerance(case):
    if case["path"] in ("knn", "knn_range"):
        return {"differ": 1e-4}                  # neighbours in the exact fp32 order: another order of sums swaps fp32 ties
    if case["path"] == "batch":
        return {"rel": 2e-4, "max": 4e-3, "differ": 5e-3}              # fp16 products, fp32 sums
    if case.get("rows") == "fp16":
        return {"rel": 2e-4, "max": 4e-3}
    return {"rel": 2e-6, "max": 2e-5, "differ": 1e-4}                  # fp32 products and sums


# ---- the same answers in 64 bits, from the definition ----------------------------------------------------------------
def _scores64(c, inp):
    """(n, Q) fused scores: dot times decay; filtered rows -FLT_MAX; the query's episode boosted."""
    n = c["n"]
    q = inp.q.double()
    lam = float(np.float32(c["decay"]))
    tq = torch.from_numpy(inp.tq).cuda()
    out = torch.empty(n, len(q), dtype=torch.float64, device="cuda")
    for lo in range(0, n, 1 << 17):
        hi = min(n, lo + (1 << 17))
        age = torch.clamp_min(tq[None, :] - inp.ts[lo:hi, None], 0.0)
        out[lo:hi] = (inp.emb[lo:hi].double() @ q.T.contiguous()) * torch.exp(-lam * age.double())
    if c["filter"] >= 0:
        out[inp.mods != c["filter"]] = -FMAX
    if c.get("boost"):
        same = (inp.ep == int(inp.node[0]) // 10)[:, None] & (out > -FMAX / 2)
        out = torch.where(same, out * (1.0 + float(np.float32(c["boost"]))), out)
    return out


def _answer64(c, inp, fin, row, col):
    """Sorted scores of one global query: top-k seeds, breadth-first expansion, the best results."""
    val, idx = torch.topk(fin, min(c["k"], len(fin)))
    score = dict(zip(idx.tolist(), val.tolist()))
    front = list(score)
    f = fin.cpu().numpy() if c["hops"] else None
    for _ in range(c["hops"]):
        new = []
        for v in front:
            for u in col[row[v]:row[v + 1]].tolist():
                if u not in score:
                    score[u] = max(0.5 * score[v], 0.8 * float(f[u]))
                    new.append(u)
        front = new
    best = sorted(score.values(), reverse=True)[:c["results"]]
    return np.array(best + [0.0] * (c["results"] - len(best)))


def exact(case, seed):
    c, path = case, case["path"]
    if path in ("knn", "knn_range"):
        return None                              # node numbers alone
    inp = Inputs(c, seed)
    if path == "episode":
        lo = int(inp.node[0]) // 10 * 10
        age = np.maximum(np.float32(0), inp.tq[0] - inp.ts[lo:lo + 10].cpu().numpy()).astype(np.float64)
        dot = (inp.emb[lo:lo + 10].double() @ inp.q[0].double()).cpu().numpy()
        best = np.sort(dot * np.exp(-float(np.float32(c["decay"])) * age))[::-1][:min(c["k"], c["results"])]
        return {"n": None, "nodes": None, "hops": None, "scores": np.concatenate([best, np.zeros(c["results"] - len(best))])}
    fin = _scores64(c, inp)
    if path == "batch":
        return {"nodes": None, "scores": torch.topk(fin, c["k"], dim=0).values.T.contiguous()}
    row, col = inp.row.cpu().numpy(), inp.col.cpu().numpy()
    best = [_answer64(c, inp, fin[:, j].contiguous(), row, col) for j in range(max(1, c.get("q", 1)))]
    if path == "global":
        return {"n": None, "nodes": None, "hops": None, "scores": best[0]}
    if not c["q"]:
        best = [np.zeros(c["results"])]
    out = {"n": None, "nodes": None, "hops": None, "scores": np.stack(best)}
    return {**out, "knn": None} if path == "link" else out
