"""The work that a program using this library has it do, as measured cases.

Each case is one public entry point on inputs of one size: the plain search
(coarse + scan + top-k), the pruned search with exact rerank, one Lloyd step,
the whole index build, exact kNN and the graph search.  Every input comes from
a seed: Gaussian-mixture vectors as the workloads C1-C5 use, and indexes,
codebooks and graphs made from them in plain torch (integer sums only, so the
same seed gives the same bits in every process).
"""
import math

import numpy as np
import torch

import fusiongpu_amd as fg

DEV = "cuda"


def listed():
    return [
        # One interactive query against a small index (C1's): nothing but latency and launches.
        dict(name="search_single", op="search", n=100_000, dim=128, m=16, nlist=256, ncomp=64, sig_lo=0.1, sig_hi=0.1,
             nq=1, nprobe=16, k=10),
        # C1: a modest batch against the small index.
        dict(name="search_c1", op="search", n=100_000, dim=128, m=16, nlist=256, ncomp=64, sig_lo=0.1, sig_hi=0.1,
             nq=1000, nprobe=16, k=10),
        # C2, the headline configuration: offline scoring of a large batch.
        dict(name="search_c2", op="search", n=1_000_000, dim=128, m=32, nlist=1024, ncomp=256, sig_lo=0.08,
             sig_hi=0.08, nq=10_000, nprobe=32, k=10),
        # Nothing round: odd rows, lists, batch, probes and k, C3's geometry (dim 96, two dims a code).
        dict(name="search_ragged", op="search", n=300_007, dim=96, m=48, nlist=601, ncomp=77, sig_lo=0.05, sig_hi=0.15,
             nq=777, nprobe=33, k=37),
        # High recall: many probes, the finest codes, the largest k of the plain search.
        dict(name="search_wide", op="search", n=1_000_000, dim=128, m=64, nlist=2048, ncomp=512, sig_lo=0.05,
             sig_hi=0.15, nq=2000, nprobe=128, k=64),
        # The coarsest codes of dim 96 (six dims a code), a memory-saving index.
        dict(name="search_m16_d96", op="search", n=500_000, dim=96, m=16, nlist=1000, ncomp=128, sig_lo=0.08,
             sig_hi=0.12, nq=4096, nprobe=48, k=10),
        # The reference pipeline's per-batch path at its defaults, on C2's data.
        dict(name="pipeline_b128", op="pipeline", n=1_000_000, dim=128, m=32, nlist=1024, ncomp=256, sig_lo=0.08,
             sig_hi=0.08, nq=128, nprobe=20, k=10, rerank_m=10_000),
        # C3: the pruned scan, compaction to the top 1000 and exact rerank to k = 100, one large batch.
        dict(name="pipeline_c3", op="pipeline", n=10_000_000, dim=96, m=48, nlist=4096, ncomp=1024, sig_lo=0.05,
             sig_hi=0.15, nq=10_000, nprobe=64, k=100, rerank_m=1000),
        # One Lloyd iteration of C4's k-means: the assignment of the 1M sample to 4096 centroids and their update.
        dict(name="lloyd_c4", op="lloyd", n=1_000_000, dim=128, nlist=4096, ncomp=1024, sig_lo=0.05, sig_hi=0.15),
        # A whole index build (k-means++ seeding, Lloyd, PQ training, encoding), half of C2's rows.
        dict(name="build_500k", op="build", n=500_000, dim=128, m=32, nlist=1024, ncomp=256, sig_lo=0.08, sig_hi=0.08,
             init_mode=1, iters=20, pq_iters=8),
        # Ground truth for tuning and recall: exact kNN of a query set over the base.
        dict(name="knn_truth", op="knn", n=1_000_000, dim=128, ncomp=256, sig_lo=0.08, sig_hi=0.08, nq=10_000, k=100),
        # C5's graph search parameters over 2M rows (far beyond the caches).
        dict(name="graph_c5", op="graph", n=2_000_000, dim=128, ncomp=256, sig_lo=0.05, sig_hi=0.15, nq=10_000, k=10,
             degree=32, itopk=64, width=4, max_iter=64),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["search", "search", "search", "pipeline", "pipeline", "lloyd", "build", "knn", "graph"])
    sig = rng.uniform(0.05, 0.12)
    c = dict(op=op, n=log(60_000, 1_000_000), ncomp=log(64, 512), sig_lo=sig, sig_hi=sig * rng.choice([1.0, 1.5, 3.0]))
    if op in ("search", "pipeline"):
        dim, m = rng.choice([(128, 16), (128, 32), (128, 64), (96, 48), (96, 32), (96, 16)])
        c.update(dim=dim, m=m, nlist=int(math.sqrt(c["n"]) * rng.uniform(0.7, 1.6)))
    if op == "search":
        c.update(nq=log(1, 10_000), nprobe=log(8, 128), k=rng.choice([1, 5, 10, 10, 10, 20, 50, 64]))
    elif op == "pipeline":
        c.update(nq=log(16, 10_000), nprobe=rng.choice([20, 20, 32, 50, 64]), k=rng.choice([10, 10, 50, 100]),
                 rerank_m=rng.choice([1000, 3000, 10_000]))
    elif op == "lloyd":
        c.update(dim=rng.choice([64, 96, 100, 128]), nlist=log(256, 4096))
    elif op == "build":
        c.update(n=min(c["n"], 400_000), dim=rng.choice([96, 128]), m=rng.choice([16, 32]), nlist=log(128, 1024),
                 init_mode=rng.choice([0, 1]), iters=rng.choice([10, 20]), pq_iters=rng.choice([8, 15]))
    elif op == "knn":
        c.update(dim=rng.choice([64, 96, 100, 128]), nq=log(64, 8000), k=rng.choice([1, 10, 50, 100, 128]))
    else:
        c.update(dim=rng.choice([96, 128]), nq=log(64, 10_000), k=rng.choice([10, 32]), degree=rng.choice([16, 32]),
                 itopk=64, width=rng.choice([2, 4]), max_iter=64)
    return c


# ---- inputs -------------------------------------------------------------------------------------------------------
# The pruned search's parameters that no case varies: the reference's defaults.
PIPE = dict(p1_lists=12, limit_k=50, threshold_coeff=1.0, mini_batch=128, eps=0.1, beta=2)


def _gen(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1009 + what)
    return g


def _vectors(case, seed, n, what):
    """n rows of the case's Gaussian mixture: centres U[-1, 1], one sigma a component."""
    g = _gen(seed, 1)
    centres = torch.rand((case["ncomp"], case["dim"]), generator=g, device=DEV) * 2 - 1
    sig = case["sig_lo"] + torch.rand((case["ncomp"], 1), generator=g, device=DEV) * (case["sig_hi"] - case["sig_lo"])
    g = _gen(seed, what)
    x = torch.empty((n, case["dim"]), device=DEV)
    for b in range(0, n, 1 << 20):
        comp = torch.randint(case["ncomp"], (min(1 << 20, n - b),), generator=g, device=DEV)
        x[b:b + comp.numel()] = centres[comp] + sig[comp] * torch.randn((comp.numel(), case["dim"]), generator=g,
                                                                        device=DEV)
    return x


def _nearest(x, c):
    """Index of each row's nearest centre."""
    out = torch.empty(x.shape[0], dtype=torch.int64, device=DEV)
    step, cn = max(1, (1 << 29) // c.shape[0]), (c * c).sum(1)
    for b in range(0, x.shape[0], step):
        out[b:b + step] = torch.addmm(cn, x[b:b + step], c.t(), alpha=-2).argmin(1)
    return out


def _update(x, a, c):
    """Means of the rows of each centre (integer sums); a centre without rows stays."""
    s = torch.zeros(c.shape, dtype=torch.int64, device=DEV).index_add_(0, a, (x * 2.0**24).to(torch.int64))
    cnt = torch.bincount(a, minlength=c.shape[0])[:, None]
    return torch.where(cnt > 0, (s.double() / (2.0**24 * cnt.clamp(min=1))).float(), c)


def _kmeans(case, seed, x, k, iters):
    g = _gen(seed, 3)
    x = x[torch.randperm(x.shape[0], generator=g, device=DEV)[:64 * k]]
    c = x[:k].clone()
    for _ in range(iters):
        c = _update(x, _nearest(x, c), c)
    return c


def _pq_nearest(r, cb):
    """Codes [n][m] of the residuals r [n][dim] under the codebook [m][256][s]."""
    m, _, s = cb.shape
    out, cn, t = torch.empty((r.shape[0], m), dtype=torch.uint8, device=DEV), (cb * cb).sum(2)[:, None], None
    step = (1 << 30) // (m * 256)
    for b in range(0, r.shape[0], step):
        v = r[b:b + step].view(-1, m, s).transpose(0, 1).contiguous()
        t = torch.baddbmm(cn, v, cb.transpose(1, 2).contiguous(), alpha=-2)
        out[b:b + step] = t.argmin(2).t().to(torch.uint8)
    return out


def _ivf(case, seed):
    """(base, offsets, ids, codes, centroids, codebook) of the case's index, on the GPU."""
    dim, m, nlist = case["dim"], case["m"], case["nlist"]
    x = _vectors(case, seed, case["n"], 2)
    cent = _kmeans(case, seed, x, nlist, 6)
    a = _nearest(x, cent)
    rows = torch.randperm(x.shape[0], generator=_gen(seed, 4), device=DEV)[:16384]
    r = (x[rows] - cent[a[rows]]).contiguous()
    cb = r[:256].view(256, m, dim // m).transpose(0, 1).contiguous()
    sub = torch.arange(m, device=DEV)[None] * 256
    for _ in range(4):
        flat = (_pq_nearest(r, cb).to(torch.int64) + sub).reshape(-1)
        cb = _update(r.view(-1, dim // m), flat, cb.view(m * 256, -1)).view(m, 256, -1)
    codes = torch.empty((x.shape[0], m), dtype=torch.uint8, device=DEV)
    for b in range(0, x.shape[0], 1 << 20):
        codes[b:b + (1 << 20)] = _pq_nearest(x[b:b + (1 << 20)] - cent[a[b:b + (1 << 20)]], cb)
    order = torch.sort(a, stable=True).indices
    offs = torch.zeros(nlist + 1, dtype=torch.int32, device=DEV)
    offs[1:] = torch.bincount(a, minlength=nlist).cumsum(0).to(torch.int32)
    return x, offs, order.to(torch.int32), codes[order].contiguous(), cent, cb.contiguous()


def _graph(case, seed, x):
    """Fixed out-degree graph: three quarters near rows (within blocks of 256 rows of one cluster order), the rest
    long-range edges, which let a walk reach every component."""
    n, deg = x.shape[0], case["degree"]
    near = deg - deg // 4
    order = torch.sort(_nearest(x, _kmeans(case, seed, x, max(64, n // 512), 3)), stable=True).indices
    graph = torch.randint(n, (n, deg), generator=_gen(seed, 5), device=DEV, dtype=torch.int32)
    for b in range(0, n, 256 * 512):
        rows = order[b:b + 256 * 512]
        nb = rows.numel() // 256
        if nb:  # the rows of a last partial block keep random edges alone
            rows = rows[:nb * 256].view(nb, 256)
            v = x[rows]
            d = torch.baddbmm((v * v).sum(2)[:, None], v, v.transpose(1, 2).contiguous(), alpha=-2)
            d.diagonal(dim1=1, dim2=2).fill_(math.inf)
            idx = d.topk(near, dim=2, largest=False).indices.view(nb, -1)
            graph[rows.reshape(-1), :near] = torch.gather(rows, 1, idx).view(-1, near).to(torch.int32)
    return graph


def _inputs(case, seed):
    """The case's arrays, without the library."""
    op = case["op"]
    if op in ("search", "pipeline"):
        x, offs, ids, codes, cent, cb = _ivf(case, seed)
        return dict(base=x, offs=offs, ids=ids, codes=codes, cent=cent, cb=cb,
                    q=_vectors(case, seed, case["nq"], 6))
    x = _vectors(case, seed, case["n"], 2)
    if op == "lloyd":
        return dict(base=x, cent=_kmeans(case, seed, x, case["nlist"], 2))
    if op == "build":
        return dict(base=x)
    if op == "knn":
        return dict(base=x, q=_vectors(case, seed, case["nq"], 6))
    return dict(base=x, q=_vectors(case, seed, case["nq"], 6), graph=_graph(case, seed, x))


def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device=DEV)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    op, nq = case["op"], case.get("nq")
    if op in ("search", "pipeline"):
        s["index"] = fg.Index.wrap(case["dim"], case["m"], s["offs"], s["ids"], s["codes"], s["cent"], s["cb"])
        s["out"] = (torch.empty((nq, case["k"]), dtype=torch.int32, device=DEV),
                    torch.empty((nq, case["k"]), dtype=torch.float32, device=DEV))
    if op == "search":
        s["ws"] = _bytes(s["index"].search_workspace_bytes(nq, case["nprobe"]))
        del s["base"]
    elif op == "pipeline":
        s["ws"] = _bytes(s["index"].search_rerank_workspace_bytes(nq, case["nprobe"], PIPE["p1_lists"],
                                                                  PIPE["limit_k"], case["rerank_m"]))
    elif op == "lloyd":
        s["shift"] = fg.fixed_shift(float(s["base"].abs().max()), case["n"])
    elif op == "knn":
        s["ws"] = _bytes(fg.lib.fgpu_knn_exact_workspace_bytes(nq, case["n"]))
    return s


def run(s):
    case, op = s["case"], s["case"]["op"]
    if op == "search":
        return s["index"].search(s["q"], case["nprobe"], case["k"], workspace=s["ws"], out=s["out"])
    if op == "pipeline":
        return s["index"].search_rerank(s["q"], s["base"], case["nprobe"], case["k"], rerank_m=case["rerank_m"],
                                        workspace=s["ws"], out=s["out"], **PIPE)
    if op == "lloyd":
        assign, dist = fg.l2_topk(s["base"], s["cent"], 1)
        cent = s["cent"].clone()  # the update works in place
        counts = fg.kmeans_update(s["base"], assign[:, 0], cent, s["shift"])
        return assign, dist, cent, counts
    if op == "build":
        return fg.build_ivfpq(s["base"], case["nlist"], case["m"], kmeans_iters=case["iters"],
                              init_mode=case["init_mode"], pq_iters=case["pq_iters"])
    if op == "knn":
        return fg.knn_exact(s["q"], s["base"], case["k"], workspace=s["ws"])
    return fg.graph_search(s["q"], s["base"], s["graph"], case["k"], itopk=case["itopk"], width=case["width"],
                           max_iter=case["max_iter"])


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    op, n, dim, nq, k = case["op"], case["n"], case["dim"], case.get("nq", 0), case.get("k", 0)
    if op in ("search", "pipeline"):
        m, nlist, nprobe = case["m"], case["nlist"], case["nprobe"]
        rows = n / nlist
        lists = min(nlist, nq * nprobe)
        b = lists * rows * (m + 4) + 4 * nlist * dim + 1024 * dim + 4 * nq * dim + 8 * nq * k
        f = 2 * nq * nlist * dim + nq * nprobe * rows * m  # the centroids' product, one add a probed code
        if op == "pipeline":  # at least beta + 1 mini-batches of rows are reranked
            b += 4 * dim * nq * min(case["rerank_m"], (PIPE["beta"] + 1) * PIPE["mini_batch"])
        return dict(bytes=b, flops=f)
    if op == "lloyd":
        return dict(bytes=4 * n * dim + 8 * n + 8 * case["nlist"] * dim, flops=2 * n * case["nlist"] * dim + n * dim)
    if op == "build":
        sweeps = case["iters"] + 1
        return dict(bytes=4 * n * dim + n * (case["m"] + 4),
                    flops=sweeps * 2 * n * case["nlist"] * dim + 3 * 256 * dim * (n + 50_000 * case["pq_iters"]))
    if op == "knn":
        return dict(bytes=4 * (n + nq) * dim + 8 * nq * k, flops=2 * nq * n * dim)
    rows = case["width"] * case["degree"] * 20  # a walk of about 20 steps
    return dict(bytes=nq * rows * dim * 4 * 0.75, flops=2 * nq * rows * dim * 0.75)


def tolerance(case):
    """Every result is defined to the bit: fp32 chains in a stated order, ties by id, integer k-means sums."""
    return "exact"


# ---- the same in 64 bits, in plain torch ----------------------------------------------------------------------------
def _sq(a, b):
    return ((a * a).sum(1)[:, None] + (b * b).sum(1)[None] - 2.0 * (a @ b.t())).clamp_(min=0.0)


def _decoded(s):
    """(decoded vectors, their lists) in list order."""
    sizes = (s["offs"][1:] - s["offs"][:-1]).to(torch.int64)
    lists = torch.repeat_interleave(torch.arange(sizes.numel(), device=DEV), sizes)
    m = s["cb"].shape[0]
    x = s["cent"].double()[lists]
    for b in range(0, x.shape[0], 1 << 18):
        rows = s["cb"][torch.arange(m, device=DEV)[None], s["codes"][b:b + (1 << 18)].long()]
        x[b:b + (1 << 18)] += rows.reshape(rows.shape[0], -1).double()
    return x, lists, sizes


def _exact_search(case, s):
    x, lists, _ = _decoded(s)
    out = []
    for b in range(0, case["nq"], max(1, (1 << 27) // case["n"])):
        q = s["q"][b:b + max(1, (1 << 27) // case["n"])].double()
        pd, pi = _sq(q, s["cent"].double()).topk(case["nprobe"], dim=1, largest=False)
        probed = torch.zeros((q.shape[0], case["nlist"]), dtype=torch.bool, device=DEV)
        probed.scatter_(1, pi, pd <= 100.0 * pd[:, :1])
        d = _sq(q, x).masked_fill_(~probed[:, lists], math.inf)
        out.append(d.topk(case["k"], dim=1, largest=False).values)
    return None, torch.cat(out)


def _exact_pipeline(case, s):
    x, lists, sizes = _decoded(s)
    offs, pos_id = s["offs"].long(), s["ids"].long()
    p1, lk, rm, mb, k = PIPE["p1_lists"], PIPE["limit_k"], case["rerank_m"], PIPE["mini_batch"], case["k"]
    base, out, col = s["base"].double(), [], torch.arange(int(sizes.max()), device=DEV)[None]
    for b in range(0, case["nq"], max(1, (1 << 26) // case["n"])):
        q = s["q"][b:b + max(1, (1 << 26) // case["n"])].double()
        nq = q.shape[0]
        pd, pi = _sq(q, s["cent"].double()).topk(case["nprobe"], dim=1, largest=False)
        use = pd <= 100.0 * pd[:, :1]
        d = _sq(q, x)
        cand = torch.full_like(d, math.inf)
        low = torch.full((nq,), math.inf, device=DEV, dtype=torch.float64)
        for p in range(min(p1, case["nprobe"])):
            size = sizes[pi[:, p]]
            ok = (col < size[:, None]) & use[:, p:p + 1]
            at = (offs[pi[:, p]][:, None] + col).clamp(max=x.shape[0] - 1)
            v, i = torch.where(ok, torch.gather(d, 1, at), math.inf).sort(dim=1)
            w = size.clamp(max=lk)
            cut = torch.where(use[:, p] & (size > 0), torch.gather(v, 1, (w - 1).clamp(min=0)[:, None])[:, 0], 0.0)
            low = torch.where(cut > 0, torch.minimum(low, cut), low)
            v, i = v[:, :lk], torch.gather(at, 1, i[:, :lk])
            cand.scatter_reduce_(1, i, v, "amin")
        late = torch.zeros((nq, case["nlist"]), dtype=torch.bool, device=DEV).scatter_(1, pi[:, p1:], use[:, p1:])
        reach = late[:, lists] & (d <= (low * PIPE["threshold_coeff"])[:, None])
        cand = torch.where(reach, d, cand)
        v, i = cand.topk(min(rm, x.shape[0]), dim=1, largest=False)
        total = (v < math.inf).sum(1)
        ids = pos_id[i]
        top = torch.full((nq, k), math.inf, device=DEV, dtype=torch.float64)
        stable, live = torch.zeros(nq, dtype=torch.int64, device=DEV), total > 0
        for off in range(0, rm, mb):
            live = live & (off < total) & (stable < PIPE["beta"])
            if not bool(live.any()):
                break
            rows = ids[:, off:off + mb]
            e = (base[rows] - q[:, None]).square_().sum(2)
            e[torch.arange(off, off + rows.shape[1], device=DEV)[None] >= total[:, None]] = math.inf
            both, src = torch.cat([top, e], 1).sort(dim=1, stable=True)
            new = both[:, :k]
            chg = ((src[:, :k] >= k) & (new < math.inf)).sum(1)
            calm = (chg.float() / k) <= PIPE["eps"]
            top = torch.where(live[:, None], new, top)
            stable = torch.where(live, torch.where(calm, stable + 1, 0), stable)
        out.append(torch.where(top < math.inf, top, torch.finfo(torch.float32).max))
    return None, torch.cat(out)


def _exact_assign(x, c):
    step = max(1, (1 << 27) // c.shape[0])
    v = [_sq(x[b:b + step].double(), c).min(1) for b in range(0, x.shape[0], step)]
    return torch.cat([t.indices for t in v]), torch.cat([t.values for t in v])


def _exact_update(x, a, k):
    s = torch.zeros((k, x.shape[1]), dtype=torch.float64, device=DEV).index_add_(0, a, x.double())
    cnt = torch.bincount(a, minlength=k)[:, None]
    return torch.where(cnt > 0, s / cnt.clamp(min=1), 0.0)


def _exact_build(case, s):
    if case["init_mode"] != 0:
        return None  # each k-means++ pick depends on all rounded distances before it
    n, k, x = case["n"], case["nlist"], s["base"]
    mt = np.random.MT19937()
    mt._legacy_seeding(42)
    stride = max(1, n // k)
    c = x[torch.tensor([(i * stride + int(mt.random_raw()) % stride) % n for i in range(k)], device=DEV)].double()
    for _ in range(case["iters"]):
        c = _exact_update(x, _exact_assign(x, c)[0], k)
    return None, None, None, c, None


def _mix64(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _exact_graph(case, s):
    n, k, itopk = case["n"], case["k"], case["itopk"]
    out = []
    for b in range(0, case["nq"], 2048):
        q = s["q"][b:b + 2048].double()
        nq = q.shape[0]
        i = np.arange(b, b + nq, dtype=np.uint64)[:, None] << np.uint64(20) | np.arange(64, dtype=np.uint64)[None]
        cand = torch.from_numpy((_mix64(np.uint64(1) ^ _mix64(i)) % np.uint64(n)).astype(np.int64)).to(DEV)
        seen = torch.zeros((nq, (1 << 16) + 1), dtype=torch.bool, device=DEV)  # the last column takes the dropped ones
        dist = torch.full((nq, itopk), math.inf, dtype=torch.float64, device=DEV)
        node = torch.full((nq, itopk), n, device=DEV)
        done = torch.ones((nq, itopk), dtype=torch.bool, device=DEV)
        for step in range(case["max_iter"] + 1):
            cand = cand.sort(dim=1).values
            bit = ((cand * 2654435761) & 0xFFFFFFFF) >> 16
            keep = (cand < n) & ~torch.gather(seen, 1, bit)
            keep[:, 1:] &= cand[:, 1:] != cand[:, :-1]
            seen.scatter_(1, torch.where(keep, bit, 1 << 16), True)
            d = (s["base"][cand.clamp(max=n - 1)].double() - q[:, None]).square_().sum(2).masked_fill_(~keep, math.inf)
            d, order = torch.cat([dist, d], 1).sort(dim=1, stable=True)
            dist, order = d[:, :itopk], order[:, :itopk]
            node = torch.gather(torch.cat([node, cand], 1), 1, order)
            done = torch.gather(torch.cat([done, ~keep], 1), 1, order) | (dist == math.inf)
            if step == case["max_iter"] or bool(done.all()):
                break
            take = ~done & ((~done).cumsum(1) <= case["width"])
            done |= take
            at = torch.where(take, torch.arange(itopk, device=DEV)[None], itopk).sort(dim=1).values[:, :case["width"]]
            from_ = torch.where(at < itopk, torch.gather(node, 1, at.clamp(max=itopk - 1)), n)
            nb = s["graph"][from_.clamp(max=n - 1)].long()
            cand = torch.where((from_ < n)[:, :, None], nb, n).view(nq, -1)
        out.append(dist[:, :k])
    return None, torch.cat(out), None


def exact(case, seed):
    op = case["op"]
    if op == "pipeline" and case["n"] * case["nq"] > 3e9:
        return None  # the full distance matrix, several times over
    s = _inputs(case, seed)
    if op == "search":
        return _exact_search(case, s)
    if op == "pipeline":
        return _exact_pipeline(case, s)
    if op == "lloyd":
        a, d = _exact_assign(s["base"], s["cent"].double())
        return None, d[:, None], _exact_update(s["base"], a, case["nlist"]), None
    if op == "build":
        return _exact_build(case, s)
    if op == "graph":
        return _exact_graph(case, s)
    out, base = [], s["base"].double()
    for b in range(0, case["nq"], max(1, (1 << 28) // case["n"])):
        q = s["q"][b:b + max(1, (1 << 28) // case["n"])].double()
        out.append(_sq(q, base).topk(case["k"], dim=1, largest=False).values)
    return None, torch.cat(out)
