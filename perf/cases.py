"""Performance cases: the calls a program of this library makes, over the sizes it makes them at.

Five kinds of call (``case["kind"]``):

  keys     one-shot count of an edge list in host memory (``Context.count_keys``): copy, preprocess, count, free.
  build    graph generated in HBM, preprocessed, counted once without judging, freed (``Context.gen_rmat`` + ``count``).
  recount  count of a graph that stays resident (``Graph.count``), as a server or the benchmark repeats it.
  batch    many graphs at once: ``form`` "host" packs host edge lists, preprocesses and counts them in one pass
           (``Context.batch_from_keys`` + ``Batch.count``); "resident" recounts a batch that stays in HBM.
  rank     one rank's task of the multi-GPU decomposition on host chunks (``count_partial_diagonal`` /
           ``count_partial_off_diagonal``).

Edge lists are drawn with torch from the seed alone: R-MAT (0.57, 0.19, 0.19, 0.05), Erdos-Renyi, Chung-Lu and
the stochastic block model, with duplicates, without self-loops, as a file reader hands them over.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tribit_amd as tb

_RMAT = (0.57, 0.19, 0.19)
_CTX = None


def _ctx() -> "tb.Context":
    """The program's one context, with the shipped cost model."""
    global _CTX
    if _CTX is None:
        _CTX = tb.Context(0)
        _CTX.load_cost_model()
    return _CTX


def _dev() -> torch.device:
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------ inputs


def _pack(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    keep = a != b
    a, b = a[keep], b[keep]
    return (torch.minimum(a, b) << 32) | torch.maximum(a, b)


def _draw_keys(family: dict, seed: int) -> torch.Tensor:
    """Packed keys (min << 32) | max (int64, on the GPU) of one random graph."""
    dev = _dev()
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    f, n = family["family"], family["n"]
    if f == "rmat":
        ne, scale = family["samples"], family["n"].bit_length() - 1
        src = torch.zeros(ne, dtype=torch.int64, device=dev)
        dst = torch.zeros(ne, dtype=torch.int64, device=dev)
        a, b, c = _RMAT
        for _ in range(scale):
            r = torch.rand(ne, device=dev, generator=g)
            src = (src << 1) | (r >= a + b)
            dst = (dst << 1) | (((r >= a) & (r < a + b)) | (r >= a + b + c))
        return _pack(src, dst)
    if f == "er":
        e = torch.randint(0, n, (2, family["samples"]), device=dev, generator=g)
        return _pack(e[0], e[1])
    if f == "chung_lu":
        w = torch.arange(1, n + 1, dtype=torch.float64, device=dev) ** (-1.0 / (family["gamma"] - 1.0))
        cdf = torch.cumsum(w, 0)
        r = torch.rand(2, family["samples"], dtype=torch.float64, device=dev, generator=g) * cdf[-1]
        e = torch.searchsorted(cdf, r).clamp_(max=n - 1)
        return _pack(e[0], e[1])
    if f == "sbm":
        size, blocks = family["size"], n // family["size"]
        iu = torch.triu_indices(size, size, 1, device=dev)
        keep = torch.rand(blocks, iu.shape[1], device=dev, generator=g) < family["p_in"]
        blk, pair = torch.nonzero(keep, as_tuple=True)
        inside = _pack(iu[0][pair] + blk * size, iu[1][pair] + blk * size)
        e = torch.randint(0, n, (2, family["cross"]), device=dev, generator=g)
        return torch.cat([inside, _pack(e[0], e[1])])
    raise ValueError(f)


def _host(keys: torch.Tensor) -> np.ndarray:
    return keys.cpu().numpy().view(np.uint64)


def _samples(family: dict) -> int:
    """Edge samples of a family (expected, for the block model)."""
    if family["family"] == "sbm":
        size = family["size"]
        return int(family["n"] // size * (size * (size - 1) // 2) * family["p_in"]) + family["cross"]
    return family["samples"]


def _rmat(scale: int, ef: int) -> dict:
    return {"family": "rmat", "n": 1 << scale, "samples": ef << scale}


def _er(n: int, samples: int) -> dict:
    return {"family": "er", "n": n, "samples": samples}


def _chung_lu(n: int, gamma: float, avg_deg: float) -> dict:
    return {"family": "chung_lu", "n": n, "gamma": gamma, "samples": int(n * avg_deg / 2)}


def _sbm(blocks: int, size: int, p_in: float, cross: int) -> dict:
    return {"family": "sbm", "n": blocks * size, "size": size, "p_in": p_in, "cross": cross}


def _batch_families(case: dict, seed: int) -> list:
    """Chung-Lu graphs of log-uniform size, as the library's batch generator draws its own."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["graphs"]):
        n = int(round(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** rng.random()))
        out.append(_chung_lu(n, 2.1 + 0.7 * rng.random(), 8.0 + 24.0 * rng.random()))
    return out


def _batch_keys(case: dict, seed: int):
    fam = _batch_families(case, seed)
    return [_host(_draw_keys(f, seed * 100003 + j)) for j, f in enumerate(fam)], [f["n"] for f in fam]


def _rank_keys(case: dict, seed: int):
    """(cols, idxs) host chunks of column partition ``part`` of ``parts`` (idxs empty for a diagonal task)."""
    k = _draw_keys(case, seed)
    width = 32 * math.ceil(case["n"] / case["parts"] / 32)
    lo, hi = (k >> 32) // width, (k & 0xFFFFFFFF) // width
    p = case["part"]
    cols = _host(k[hi == p])
    idxs = _host(k[(hi > p) & (lo <= p)]) if case["off"] else np.zeros(0, np.uint64)

    def chunks(a):  # the hosts of such a program hold a partition as a few chunks
        return [c for c in np.array_split(a, 3)]

    return chunks(cols), chunks(idxs)


# ------------------------------------------------------------------- cases


def listed() -> list:
    return [
        # the smallest call: a thousand vertices, all launches and latency
        {"name": "keys_tiny", "kind": "keys", "sched": "learned", **_er(1000, 8000)},
        # the `tribit -i` size of a small real graph
        {"name": "keys_rmat13", "kind": "keys", "sched": "learned", **_rmat(13, 12)},
        # an ordinary skewed graph, its vertex count not a power of two
        {"name": "keys_cl200k", "kind": "keys", "sched": "learned", **_chung_lu(199999, 2.3, 24.0)},
        # a large edge list that comes from host memory
        {"name": "keys_rmat22", "kind": "keys", "sched": "learned", **_rmat(22, 16)},
        # the largest: edges in HBM to an exact count
        {"name": "build_rmat25", "kind": "build", "scale": 25, "ef": 16},
        # a small resident graph counted again: the latency of one count
        {"name": "recount_rmat13", "kind": "recount", "sched": "learned", **_rmat(13, 12)},
        # the benchmark's count: R-MAT scale 25 resident in HBM
        {"name": "recount_rmat25", "kind": "recount", "sched": "learned", "family": "gen_rmat", "scale": 25, "ef": 16},
        # dense communities: blocks for the matrix cores
        {"name": "recount_sbm", "kind": "recount", "sched": "learned", **_sbm(1000, 512, 0.3, 13_000_000)},
        # many small graphs from the host, counted once
        {"name": "batch_host", "kind": "batch", "form": "host", "sched": "learned", "graphs": 96, "n_lo": 600,
         "n_hi": 60000},
        # many graphs kept in HBM, counted by one replay
        {"name": "batch_resident", "kind": "batch", "form": "resident", "sched": "wedge", "graphs": 768, "n_lo": 1024,
         "n_hi": 262144},
        # one rank's tasks of the multi-GPU decomposition
        {"name": "rank_diag", "kind": "rank", "off": False, "parts": 16, "part": 0, **_rmat(21, 16)},
        {"name": "rank_off", "kind": "rank", "off": True, "parts": 16, "part": 0, **_rmat(21, 16)},
    ]


def _log_int(rng, lo: float, hi: float) -> int:
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_family(rng, lo: int, hi: int) -> dict:
    """A graph of lo..hi edge samples (log-uniform), odd vertex counts among them."""
    f = rng.choice(["rmat", "rmat", "er", "chung_lu", "sbm"])
    e = _log_int(rng, lo, hi)
    if f == "rmat":
        ef = rng.choice([8, 12, 16, 24])
        return _rmat(max(8, int(math.log2(e / ef))), ef)
    if f == "er":
        return _er(max(64, int(e / rng.uniform(4, 24))) | 1, e)
    if f == "chung_lu":
        avg = rng.uniform(8, 64)
        return _chung_lu(max(64, int(2 * e / avg)), rng.uniform(2.1, 2.8), avg)
    size = rng.choice([64, 200, 512])
    p_in = rng.uniform(0.15, 0.5)
    per = size * (size - 1) / 2 * p_in
    blocks = max(1, int(0.75 * e / per))
    return _sbm(blocks, size, p_in, max(1, e // 4))


def draw(rng) -> dict:
    kind = rng.choice(["keys", "keys", "build", "recount", "recount", "batch", "rank"])
    sched = rng.choice(["learned", "learned", "wedge", "directed"])
    if kind == "keys":
        return {"kind": kind, "sched": sched, **_draw_family(rng, 4_000, 60_000_000)}
    if kind == "build":
        return {"kind": kind, "scale": rng.randint(12, 24), "ef": rng.choice([8, 16, 16, 24])}
    if kind == "recount":
        return {"kind": kind, "sched": sched, **_draw_family(rng, 4_000, 60_000_000)}
    if kind == "batch":
        if rng.random() < 0.5:
            return {"kind": kind, "form": "host", "sched": "learned", "graphs": _log_int(rng, 5, 160), "n_lo": 300,
                    "n_hi": _log_int(rng, 3000, 60000)}
        return {"kind": kind, "form": "resident", "sched": rng.choice(["wedge", "learned"]),
                "graphs": _log_int(rng, 16, 768), "n_lo": 1024, "n_hi": 262144}
    parts = rng.choice([4, 7, 16])
    off = rng.random() < 0.5
    return {"kind": kind, "off": off, "parts": parts, "part": rng.randrange(parts - 1 if off else parts),
            **_rmat(rng.randint(12, 21), rng.choice([8, 16]))}


# --------------------------------------------------------- prepare and run


class _State:
    """What the program holds between calls; a resident graph or batch is given back with it."""

    def __init__(self, case: dict):
        self.case = case
        self.ctx = _ctx()
        self.held = None

    def __del__(self):
        if self.held is not None:
            self.held.free()


def prepare(case: dict, seed: int) -> _State:
    st = _State(case)
    kind = case["kind"]
    st.seed = seed
    if kind == "keys":
        st.keys = _host(_draw_keys(case, seed))
    elif kind == "recount":
        if case["family"] == "gen_rmat":
            st.held = st.ctx.gen_rmat(case["scale"], case["ef"], seed=seed)
        else:
            st.held = st.ctx.graph_from_keys(_host(_draw_keys(case, seed)), case["n"])
        st.held.count(case["sched"])  # the first count judges the plans, as a program's warm-up does
    elif kind == "batch":
        if case["form"] == "host":
            st.keys, st.n = _batch_keys(case, seed)
        else:
            st.held = st.ctx.batch_gen_chung_lu(seed, 0, case["graphs"])
            st.held.count(case["sched"])  # builds the task lists and the captured launches
    elif kind == "rank":
        st.cols, st.idxs = _rank_keys(case, seed)
    return st


def run(st: _State):
    case, ctx = st.case, st.ctx
    kind = case["kind"]
    if kind == "keys":
        return ctx.count_keys(st.keys, case["n"], case["sched"])[0]
    if kind == "build":
        with ctx.gen_rmat(case["scale"], case["ef"], seed=st.seed) as g:
            return g.count("learned", flags=tb.NO_JUDGE).triangles
    if kind == "recount":
        return st.held.count(case["sched"]).triangles
    if kind == "batch":
        if case["form"] == "host":
            with ctx.batch_from_keys(st.keys, st.n) as b:
                return b.count(case["sched"])[0]
        return st.held.count(case["sched"])[0]
    if case["off"]:
        return tb.count_partial_off_diagonal(ctx, st.cols, st.idxs, case["n"])
    return tb.count_partial_diagonal(ctx, st.cols, case["n"])


# ------------------------------------------------------- work and exact value


def work(case: dict) -> dict:
    """Every input read once, every output written once: 8-byte edge keys, or the resident oriented rows (4 bytes a
    vertex and an edge); the counts written."""
    kind = case["kind"]
    if kind == "keys":
        b = 8 * _samples(case) + 8
    elif kind == "build":
        b = 8 * (case["ef"] << case["scale"]) + 8
    elif kind == "recount":
        if case["family"] == "gen_rmat":
            n, e = 1 << case["scale"], case["ef"] << case["scale"]
        else:
            n, e = case["n"], _samples(case)
        b = 4 * (n + 1) + 4 * e + 8
    elif kind == "batch":
        # mean of a log-uniform size, mean of the average degree
        mean = (case["n_hi"] - case["n_lo"]) / math.log(case["n_hi"] / case["n_lo"])
        if case["form"] == "host":
            b = case["graphs"] * (8 * mean * 20.0 / 2 + 8)
        else:
            b = case["graphs"] * (4 * mean + 4 * mean * 36.0 / 2 + 8)
    else:
        # keys of the task: measured shares of an R-MAT partition vary; the first partitions hold the hubs
        b = 8 * _samples(case) * (0.5 if case["off"] else 1.0 / case["parts"]) + 8
    return {"bytes": int(b), "flops": 0}


def _triangles(keys: torch.Tensor) -> int:
    """Exact triangles of an edge list: every wedge of the degree-ordered rows looked up among the arcs."""
    k = torch.unique(keys)
    if k.numel() == 0:
        return 0
    a, b = k >> 32, k & 0xFFFFFFFF
    n = int(b.max()) + 1
    deg = torch.bincount(torch.cat([a, b]), minlength=n)
    rank = torch.empty_like(deg)
    rank[torch.argsort(deg, stable=True)] = torch.arange(n, device=k.device)
    u, v = torch.minimum(rank[a], rank[b]), torch.maximum(rank[a], rank[b])
    arc = torch.sort(u * n + v).values
    u, v = arc // n, arc % n
    end = torch.cumsum(torch.bincount(u, minlength=n), 0)[u]
    e = torch.arange(arc.numel(), device=k.device)
    after = end - e - 1  # arcs of the row after this one
    tot = torch.cumsum(after, 0)
    count, lo, step = 0, 0, 1 << 26
    while lo < arc.numel():
        before = int(tot[lo - 1]) if lo else 0
        hi = max(lo + 1, int(torch.searchsorted(tot, torch.tensor(before + step, device=k.device))))
        hi = min(hi, arc.numel())
        c = after[lo:hi]
        first = torch.repeat_interleave(e[lo:hi], c)
        off = torch.arange(first.numel(), device=k.device) - torch.repeat_interleave(torch.cumsum(c, 0) - c, c)
        want = v[first] * n + v[first + 1 + off]
        at = torch.searchsorted(arc, want).clamp_(max=arc.numel() - 1)
        count += int((arc[at] == want).sum())
        lo = hi
    return count


def _off_triangles(cols: torch.Tensor, idxs: torch.Tensor, n: int) -> int:
    """Triangles a < b < c with (a, b) in cols and (a, c), (b, c) in idxs."""
    cols, idxs = torch.unique(cols), torch.unique(idxs)
    if not cols.numel() or not idxs.numel():
        return 0
    a, b = cols >> 32, cols & 0xFFFFFFFF
    lo, c = idxs >> 32, idxs & 0xFFFFFFFF
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=cols.device)
    ptr[1:] = torch.cumsum(torch.bincount(lo, minlength=n), 0)
    la, lb = ptr[a + 1] - ptr[a], ptr[b + 1] - ptr[b]
    short, other = torch.where(la <= lb, a, b), torch.where(la <= lb, b, a)
    length = torch.minimum(la, lb)
    tot = torch.cumsum(length, 0)
    count, p, step = 0, 0, 1 << 26
    while p < cols.numel():
        before = int(tot[p - 1]) if p else 0
        q = max(p + 1, int(torch.searchsorted(tot, torch.tensor(before + step, device=cols.device))))
        q = min(q, cols.numel())
        ln = length[p:q]
        row = torch.repeat_interleave(torch.arange(p, q, device=cols.device), ln)
        off = torch.arange(row.numel(), device=cols.device) - torch.repeat_interleave(torch.cumsum(ln, 0) - ln, ln)
        want = (other[row] << 32) | c[ptr[short[row]] + off]
        at = torch.searchsorted(idxs, want).clamp_(max=idxs.numel() - 1)
        count += int((idxs[at] == want).sum())
        p = q
    return count


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("keys", "recount") and case["family"] != "gen_rmat":
        # hubs of the largest R-MAT graphs carry more wedges than 20 seconds of lookups
        if case["family"] in ("rmat", "chung_lu") and _samples(case) > 20_000_000:
            return None
        return _triangles(_draw_keys(case, seed))
    if kind == "batch" and case["form"] == "host":
        keys, _ = _batch_keys(case, seed)
        return np.array([_triangles(torch.from_numpy(k.view(np.int64)).to(_dev())) for k in keys], np.uint64)
    if kind == "rank":
        cols, idxs = _rank_keys(case, seed)
        t = [torch.from_numpy(np.concatenate(x).view(np.int64)).to(_dev()) for x in (cols, idxs)]
        if case["off"]:
            return None if case["n"] > 1 << 18 else _off_triangles(t[0], t[1], case["n"])
        return _triangles(t[0])
    return None
