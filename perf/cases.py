"""Performance cases of the IVF-Flat framework: the calls its users make.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` builds what a user's program holds before the call (the
index, the queries, the bound model), ``run`` is one pass through the public
entry points, ``work`` the bytes and operations a pass cannot do without, and
``exact`` the same outputs in 64-bit arithmetic from plain torch.

Data follow the repository's workload recipes (integer mixtures of sigma 20
in [0, 255], the same with Zipf popularity, heavy-tailed reals, unit-norm
reals); the quantizer is a few Lloyd rounds over a sample, computed here.
"""
import numpy as np
import torch

from harmonyclient_amd import index as hx

_ALGO = {"plain": hx.ALGO_PLAIN, "pruned": hx.ALGO_PRUNED, "batched": hx.ALGO_BATCHED}
_F32MAX = float(np.finfo(np.float32).max)


def _search(name, data, rows, d, nlist, n, nprobe, k, algo="plain", metric="l2", bound="warmup",
            buffers="host", graph=False, per_query=False):
    c = dict(op="search", data=data, rows=rows, d=d, nlist=nlist, n=n, nprobe=nprobe, k=k, algo=algo, metric=metric,
             bound=bound, buffers=buffers, graph=graph, per_query=per_query)
    return dict(c, name=name) if name else c


def _op(name, op, **kw):
    c = dict(op=op, **kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # an interactive lookup: one query with every default, host buffers
        _search("one_query", "int", 200_000, 128, 512, 1, 16, 10),
        # a handful of concurrent requests served as one batched call, ragged count and dimension
        _search("batched_37", "real", 100_000, 96, 300, 37, 24, 20, "batched"),
        # an evaluation batch with the default algorithm (exact recall runs, ground truth)
        _search("plain_1k", "int", 500_000, 128, 1024, 1000, 32, 100),
        # the reference's dimension-block pruning under its warm-up bound
        _search("pruned_2k", "int", 500_000, 128, 1024, 2000, 48, 100, "pruned", buffers="device"),
        # maximum inner product over unit-norm embeddings, odd dimension
        _search("ip_500", "unit", 200_000, 201, 400, 500, 20, 50, metric="ip", buffers="device"),
        # the headline: 10k queries on 1M x 128 under the learned bound, replayed as a captured graph
        _search("learned_10k_graph", "int", 1_000_000, 128, 1024, 10_000, 64, 100, "batched", bound="learned",
                buffers="device", graph=True),
        # skewed lists with a probe count per query, the serve front-end's batch size
        _search("zipf_4k", "zipf", 500_000, 128, 1024, 4096, 64, 100, "batched", buffers="device", per_query=True),
        # heavy-tailed real vectors, the widest ordinary dimension
        _search("real_d420", "real", 250_000, 420, 500, 2000, 50, 100, "batched", buffers="device"),
        # lists rebuilt from new rows, then the first batch searched on them
        _op("add_500k", "add", data="int", rows=500_000, d=128, nlist=1024, n=4096, nprobe=16, k=100),
        # quantizer training: 256 rows per centroid
        _op("train_131k", "train", data="real", rows=131_072, d=96, nlist=512, niter=10),
        # the bound model's backward over a trace batch
        _op("bound_grad_8k", "grad", n=8192, hidden=128),
        # merge of eight partitions' rows (list-sharded search)
        _op("merge_8x10k", "merge", parts=8, n=10_000, k_in=100, k=100, metric="l2"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    u = rng.random()
    if u < 0.08:
        return _op(None, "add", data=rng.choice(["int", "real"]), rows=_log_int(rng, 20_000, 400_000),
                   d=rng.randint(16, 128), nlist=_log_int(rng, 64, 1024), n=_log_int(rng, 64, 4096),
                   nprobe=rng.randint(4, 24), k=rng.randint(5, 100))
    if u < 0.16:
        nlist = _log_int(rng, 32, 500)
        return _op(None, "train", data=rng.choice(["int", "real"]), rows=nlist * rng.randint(64, 256),
                   d=rng.randint(16, 100), nlist=nlist, niter=rng.randint(2, 10))
    if u < 0.22:
        return _op(None, "grad", n=_log_int(rng, 200, 8192), hidden=rng.choice([32, 64, 72, 128]))
    if u < 0.30:
        return _op(None, "merge", parts=rng.randint(2, 8), n=_log_int(rng, 10, 10_000), k_in=rng.randint(10, 100),
                   k=rng.randint(10, 100), metric=rng.choice(["l2", "ip"]))
    nlist = _log_int(rng, 64, 1024)
    rows = max(nlist * 50, _log_int(rng, 20_000, 500_000))
    k = _log_int(rng, 1, 200)
    nprobe = min(nlist, rng.randint(4, 64))
    if u < 0.52:  # per-query algorithms
        metric = rng.choice(["l2", "l2", "ip"])
        data = rng.choice(["int", "real"]) if metric == "l2" else "unit"
        algo = rng.choice(["plain", "pruned"]) if metric == "l2" else "plain"
        return _search(None, data, rows, rng.randint(16, 128) if metric == "l2" else rng.randint(50, 200), nlist,
                       _log_int(rng, 1, 1000), min(nprobe, 32), k, algo, metric,
                       buffers=rng.choice(["host", "device"]))
    data = rng.choice(["int", "int", "zipf", "real"])
    device = rng.random() < 0.7
    learned = data != "real" and rng.random() < 0.4
    d = rng.randint(16, 128) if data != "real" else rng.randint(32, 420)
    return _search(None, data, min(rows, 200_000) if d > 200 else rows, d, nlist,
                   _log_int(rng, 2, 1500 if d > 200 else 8000), max(nprobe, 32) if learned else nprobe,
                   k, "batched", bound="learned" if learned else "warmup", buffers="device" if device else "host",
                   graph=device and rng.random() < 0.4, per_query=device and rng.random() < 0.3)


# -- data -----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _mixture(case, g):
    """The workload's centres, component weights and per-dimension scale."""
    d, ncomp = case["d"], case["nlist"]
    kind = case["data"]
    w = torch.ones(ncomp, device="cuda")
    scale = torch.ones(d, device="cuda")
    if kind in ("int", "zipf"):
        centres = torch.rand(ncomp, d, device="cuda", generator=g) * 255.0
        if kind == "zipf":
            w = 1.0 / torch.arange(1, ncomp + 1, device="cuda", dtype=torch.float32) ** 1.1
    elif kind == "real":
        centres = torch.randn(ncomp, d, device="cuda", generator=g) * 3.0
        scale = torch.exp(torch.randn(d, device="cuda", generator=g) * 0.5)
    else:
        centres = torch.randn(ncomp, d, device="cuda", generator=g)
    return centres, w, scale


def _points(kind, mix, n, g):
    centres, w, scale = mix
    comp = torch.multinomial(w, n, replacement=True, generator=g)
    x = torch.randn(n, centres.shape[1], device="cuda", generator=g)
    if kind in ("int", "zipf"):
        return torch.clamp(torch.round(centres[comp] + 20.0 * x), 0.0, 255.0)
    if kind == "real":  # Student-t, 3 degrees of freedom, per dimension
        chi = torch.zeros_like(x)
        for _ in range(3):
            chi += torch.randn(x.shape, device="cuda", generator=g) ** 2
        return centres[comp] + x / torch.sqrt(chi / 3.0) * scale
    x = centres[comp] + 0.7 * x
    return x / x.norm(dim=1, keepdim=True)


def _lloyd(x, cent, rounds, ip=False):
    """Lloyd rounds in FP64, a centroid without rows keeping its value."""
    x, cent = x.double(), cent.double()
    for _ in range(rounds):
        label = _nearest(x, cent, 1, ip)[1][:, 0]
        order = torch.sort(label, stable=True)[1]
        cnt = torch.bincount(label, minlength=cent.shape[0])
        run = torch.cumsum(x[order], 0)
        end = torch.cumsum(cnt, 0)
        run = torch.cat([torch.zeros(1, x.shape[1], dtype=x.dtype, device=x.device), run])
        mean = (run[end] - run[end - cnt]) / cnt.clamp(min=1)[:, None]
        cent = torch.where(cnt[:, None] > 0, mean, cent).float().double()
    return cent


def _nearest(x, c, p, ip=False, chunk=65536):
    """(distances, ids) of the p best of c for every row of x, in x's type."""
    D, I = [], []
    cn = (c * c).sum(1)
    for s in range(0, x.shape[0], chunk):
        xs = x[s:s + chunk]
        dots = xs @ c.T
        r = -dots if ip else (xs * xs).sum(1)[:, None] + cn[None] - 2.0 * dots
        v, i = torch.topk(r, p, dim=1, largest=False, sorted=True)
        D.append(v)
        I.append(i)
    return torch.cat(D), torch.cat(I)


def _inputs(case, seed):
    """(rows, centroids, queries, training queries) on the GPU, from the seed alone."""
    g = _gen(seed)
    mix = _mixture(case, g)
    xb = _points(case["data"], mix, case["rows"], g)
    xq = _points(case["data"], mix, case["n"], g)
    nt = 16384 if case.get("bound") == "learned" else 0
    xt = _points(case["data"], mix, nt, g) if nt else None
    m = min(case["rows"], 32 * case["nlist"])
    sample = xb[torch.randperm(case["rows"], device="cuda", generator=g)[:m]]
    cent = _lloyd(sample, sample[:case["nlist"]].clone(), 2, case.get("metric") == "ip").float()
    return xb, cent, xq, xt


def _per_query(case, seed):
    if not case.get("per_query"):
        return None
    g = _gen(seed + 77)
    return torch.randint(1 + case["nprobe"] // 8, case["nprobe"] + 1, (case["n"],), device="cuda", generator=g,
                         dtype=torch.int32)


def _metric(case):
    return hx.METRIC_IP if case.get("metric") == "ip" else hx.METRIC_L2


def _grad_inputs(case, seed):
    r = np.random.default_rng(seed)
    h, n = case["hidden"], case["n"]
    x = np.sort(r.gamma(4.0, 2.0, (n, hx.N_FEATURES)).astype(np.float32), axis=1)
    dy = (np.where(r.random(n) < 0.9, -0.9, 0.1) / n).astype(np.float32)
    mu, sd = x.mean(0), x.std(0) + 1e-3
    lim = [np.sqrt(6.0 / f) for f in (hx.N_FEATURES, h, h)]
    p = np.concatenate([r.uniform(-lim[0], lim[0], hx.N_FEATURES * h), r.normal(0, 0.1, h),
                        r.uniform(-lim[1], lim[1], h * h), r.normal(0, 0.1, h), r.uniform(-lim[2], lim[2], h),
                        [8.0], mu, sd, [1.0, 0.0]]).astype(np.float32)
    return x, dy, p


def _merge_inputs(case, seed):
    g = _gen(seed)
    parts, n, k_in = case["parts"], case["n"], case["k_in"]
    D = torch.sort(torch.randint(20_000, 200_000, (parts, n, k_in), device="cuda", generator=g).float(), dim=2,
                   descending=case["metric"] == "ip")[0]
    part = torch.arange(parts, device="cuda").view(parts, 1, 1)
    I = torch.rand(parts, n, k_in, device="cuda", generator=g).argsort(dim=2) * parts + part
    return D.contiguous(), I.to(torch.int64).contiguous()


# -- the cases ------------------------------------------------------------
def prepare(case, seed):
    op = case["op"]
    if op == "grad":
        x, dy, p = _grad_inputs(case, seed)
        m = hx.TauModel(hidden=case["hidden"])
        m.set_params(p)
        return dict(op=op, model=m, x=x, dy=dy)
    if op == "merge":
        D, I = _merge_inputs(case, seed)
        n, k = case["n"], case["k"]
        return dict(op=op, case=case, D=D, I=I, oD=torch.empty(n, k, device="cuda"),
                    oI=torch.empty(n, k, dtype=torch.int64, device="cuda"))
    if op == "train":
        g = _gen(seed)
        x = _points(case["data"], _mixture(case, g), case["rows"], g)
        init = x[torch.randperm(case["rows"], device="cuda", generator=g)[:case["nlist"]]]
        return dict(op=op, idx=hx.Index(case["d"], case["nlist"]), x=x.cpu().numpy(), init=init.cpu().numpy(),
                    niter=case["niter"])
    xb, cent, xq, xt = _inputs(case, seed)
    idx = hx.Index(case["d"], case["nlist"], case["nprobe"], _metric(case))
    idx.set_centroids(cent.cpu().numpy())
    if op == "add":
        return dict(op=op, idx=idx, xb=xb.cpu().numpy(), xq=xq.cpu().numpy(), k=case["k"],
                    params=hx.make_params(algo=hx.ALGO_BATCHED))
    idx.add(case["rows"], xb.cpu().numpy())
    del xb
    if xt is not None:  # the benchmark's recipe for the bound: a high quantile, hardly any misses
        idx.train_tau_model(xt.cpu().numpy(), case["k"], case["nprobe"], epochs=40, quantile=0.999, miss_rate=0.0005)
    npq = _per_query(case, seed)
    tau = {"warmup": hx.TAU_WARMUP, "learned": hx.TAU_LEARNED}[case["bound"]]
    state = dict(op=op, idx=idx, n=case["n"], k=case["k"], npq=npq, buffers=case["buffers"])
    state["params"] = hx.make_params(nprobe=case["nprobe"], algo=_ALGO[case["algo"]], tau=tau, use_graph=case["graph"],
                                     nprobe_per_query_dev=npq.data_ptr() if npq is not None else None)
    if case["buffers"] == "host":
        state["xq"] = xq.cpu().numpy()
    else:
        state["xq"] = xq.contiguous()
        state["D"] = torch.empty(case["n"], case["k"], device="cuda")
        state["I"] = torch.empty(case["n"], case["k"], dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    op = state["op"]
    if op == "grad":
        return {"grad": state["model"].grad(state["x"], state["dy"])}
    if op == "merge":
        c = state["case"]
        hx.merge_topk_device(hx.METRIC_IP if c["metric"] == "ip" else hx.METRIC_L2, c["n"], c["parts"], c["k_in"],
                             state["D"].data_ptr(), state["I"].data_ptr(), c["k"], state["oD"].data_ptr(),
                             state["oI"].data_ptr())
        return {"D": state["oD"], "I": state["oI"]}
    idx = state["idx"]
    if op == "train":
        idx.train(state["x"].shape[0], state["x"], init_centroids=state["init"], niter=state["niter"])
        return {"centroids": idx.centroids}
    if op == "add":
        idx.add(state["xb"].shape[0], state["xb"])
        D, I, _ = idx.search(state["xq"].shape[0], state["xq"], state["k"], params=state["params"])
        return {"D": D, "I": I}
    if state["buffers"] == "host":
        D, I, _ = idx.search(state["n"], state["xq"], state["k"], params=state["params"])
        return {"D": D, "I": I}
    idx.search_device(state["n"], state["xq"].data_ptr(), state["k"], state["D"].data_ptr(), state["I"].data_ptr(),
                      state["params"], stats=False)
    return {"D": state["D"], "I": state["I"]}


def work(case):
    op = case["op"]
    if op == "grad":
        n, h, f = case["n"], case["hidden"], hx.N_FEATURES
        # forward, then the products for the inputs' and the weights' gradients
        return {"bytes": 4.0 * (n * (f + 1) + 2 * (f * h + h * h)), "flops": 2.0 * n * (2 * f * h + 3 * h * h + 3 * h)}
    if op == "merge":
        return {"bytes": 12.0 * case["n"] * (case["parts"] * case["k_in"] + case["k"]), "flops": 0.0}
    rows, d, nlist = case["rows"], case["d"], case["nlist"]
    if op == "train":
        return {"bytes": 4.0 * rows * d + 8.0 * nlist * d, "flops": 2.0 * rows * nlist * d * case["niter"]}
    n, k, P = case["n"], case["k"], min(case["nprobe"], nlist)
    if case.get("per_query"):
        P *= 0.56
    pairs = n * P * rows / nlist  # (query, row) pairs at the mean list size
    flops = 2.0 * d * (n * nlist + pairs)
    io = 4.0 * n * d + 12.0 * n * k + 4.0 * nlist * d
    if op == "add":
        return {"bytes": io + 8.0 * rows * d, "flops": flops + 2.0 * rows * nlist * d}
    return {"bytes": io + 4.0 * d * min(rows, pairs), "flops": flops}


def exact(case, seed):
    op = case["op"]
    if op == "grad":
        x, dy, p = (torch.from_numpy(v).double() for v in _grad_inputs(case, seed))
        h, f = case["hidden"], hx.N_FEATURES
        parts = torch.split(p, [f * h, h, h * h, h, h, 1, f, f, 2])
        W1, b1, W2, b2, w3, _, mu, sd, _ = parts
        W1, W2 = W1.view(f, h), W2.view(h, h)
        # the library's inputs of the layers are standardised in FP32
        xs = (x - mu) / sd
        h1 = torch.relu(xs @ W1 + b1)
        h2 = torch.relu(h1 @ W2 + b2)
        dz2 = dy[:, None] * w3[None] * (h2 > 0)
        dz1 = (dz2 @ W2.T) * (h1 > 0)
        zero = torch.zeros(2 * f + 2, dtype=torch.float64)
        return {"grad": torch.cat([(xs.T @ dz1).reshape(-1), dz1.sum(0), (h1.T @ dz2).reshape(-1), dz2.sum(0),
                                   h2.T @ dy, dy.sum().view(1), zero])}
    if op == "merge":
        D, I = _merge_inputs(case, seed)
        n = case["n"]
        flat = D.permute(1, 0, 2).reshape(n, -1).double()
        top = torch.topk(flat, min(case["k"], flat.shape[1]), dim=1, largest=case["metric"] == "ip")[0]
        pad = case["k"] - top.shape[1]
        fill = -_F32MAX if case["metric"] == "ip" else _F32MAX
        return {"D": torch.nn.functional.pad(top, (0, pad), value=fill), "I": None}
    if op == "train":
        g = _gen(seed)
        x = _points(case["data"], _mixture(case, g), case["rows"], g)
        init = x[torch.randperm(case["rows"], device="cuda", generator=g)[:case["nlist"]]]
        return {"centroids": _lloyd(x, init, case["niter"])}
    xb, cent, xq, _ = _inputs(case, seed)
    ip = case.get("metric") == "ip"
    n, k, P = case["n"], case["k"], min(case["nprobe"], case["nlist"])
    xb, cent, xq = xb.double(), cent.double(), xq.double()
    label = _nearest(xb, cent, 1, ip)[1][:, 0]
    probes = _nearest(xq, cent, P, ip)[1]
    probed = torch.zeros(n, case["nlist"], dtype=torch.bool, device="cuda")
    npq = _per_query(case, seed)
    on = torch.ones_like(probes, dtype=torch.bool)
    if npq is not None:
        on = torch.arange(P, device="cuda")[None] < npq[:, None]
    probed.scatter_(1, probes, on)
    bn = (xb * xb).sum(1)
    fill = -_F32MAX if ip else _F32MAX
    # the rows grouped by list, so that only probed lists' columns count
    out = torch.full((n, k), fill, dtype=torch.float64, device="cuda")
    step = max(1, 40_000_000 // xb.shape[0])
    for s in range(0, n, step):
        q = xq[s:s + step]
        r = q @ xb.T
        r = -r if ip else ((q * q).sum(1)[:, None] + bn[None] - 2.0 * r).clamp_(min=0.0)
        r.masked_fill_(~probed[s:s + step][:, label], float("inf"))
        v = torch.topk(r, min(k, r.shape[1]), dim=1, largest=False, sorted=True)[0]
        v = torch.where(torch.isinf(v), torch.full_like(v, _F32MAX), v)
        out[s:s + step, :v.shape[1]] = -v if ip else v
    return {"D": out, "I": None}
