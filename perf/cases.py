"""Timed cases of the sparse CPD library: what a program linked against it
has it do, through its public entry points.

Kinds of case:
  mttkrp      one MTTKRP of every mode with factors in GPU memory
              (splatt_amd_mttkrp_dev), the loop body of a caller's own ALS
  mttkrp_host the drop-in splatt_mttkrp with host factors and output, every
              mode in turn
  csf         splatt_csf_convert of a coordinate tensor in host memory: the
              CSF arrays
  cpd         splatt_cpd from given start factors, unconstrained or with
              every mode non-negative (row-chunked ADMM, default chunks)
  stream      splatt_amd_cpd_stream_coo over a short stream of time slices
  serve       the multi-stream server: open, submit, drain, read factors

Tensors are drawn on the GPU from the seed (distinct coordinates, Zipf or
uniform per mode, no empty index), then handed over in host arrays as a
caller would.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "splatt-stream_amd"))
import pysplatt as ps  # noqa: E402

ALLOC = {"one": ps.CSF_ONEMODE, "two": ps.CSF_TWOMODE, "all": ps.CSF_ALLMODE}
FORGET, FROB, OUTER = 0.95, 1e-2, 5          # the streaming workloads' settings
UNEVEN = (1.0, 0.5, 1.6, 0.8, 2.0, 0.3)      # slices' nonzeros, relative


def listed():
    return [
        # a small tensor as in the unit-sized fixtures: rank 10 (the CLI's
        # default), default two-CSF allocation; launches and latency count
        dict(name="mttkrp_small_f64_r10", kind="mttkrp", d0=300, d1=200, d2=100, d3=0,
             nnz=8000, zipf=0.0, rank=10, dtype="f64", alloc="two"),
        # the benchmark's tensor: 50M nonzeros, Zipf(1.2), FP32, all-mode CSF
        dict(name="mttkrp_zipf50m_f32_r32", kind="mttkrp", d0=200000, d1=150000, d2=50000,
             d3=0, nnz=50000000, zipf=1.2, rank=32, dtype="f32", alloc="all"),
        # the reference's value type and its smallest allocation: one CSF
        # serves root, internal and leaf outputs
        dict(name="mttkrp_zipf10m_f64_r32_one", kind="mttkrp", d0=120000, d1=80000, d2=30000,
             d3=0, nnz=10000000, zipf=1.2, rank=32, dtype="f64", alloc="one"),
        # four modes at rank 64 (the 4-mode CPD workload at a tenth of its
        # nonzeros), default allocation
        dict(name="mttkrp_4mode10m_f32_r64", kind="mttkrp", d0=100000, d1=60000, d2=20000,
             d3=500, nnz=10000000, zipf=1.1, rank=64, dtype="f32", alloc="two"),
        # a rank that is no multiple of anything
        dict(name="mttkrp_odd5m_f32_r35", kind="mttkrp", d0=50021, d1=39983, d2=29989, d3=0,
             nnz=4999999, zipf=1.1, rank=35, dtype="f32", alloc="all"),
        # the drop-in call: host arrays in and out
        dict(name="mttkrp_host2m_f64_r16", kind="mttkrp_host", d0=40000, d1=25000, d2=8000,
             d3=0, nnz=2000000, zipf=1.1, rank=16, dtype="f64", alloc="two"),
        # CSF construction from host coordinates
        dict(name="csf_convert4m_all", kind="csf", d0=60000, d1=45000, d2=15000, d3=0,
             nnz=4000000, zipf=1.2, rank=0, dtype="f64", alloc="all"),
        # plain CPD-ALS of the small benchmark workload
        dict(name="cpd_1m_f64_r16", kind="cpd", d0=1000, d1=800, d2=600, d3=0, nnz=1000000,
             zipf=0.0, rank=16, dtype="f64", alloc="two", its=20, nonneg=False),
        # 4-mode CPD-ALS at rank 64 with FP32 MTTKRP
        dict(name="cpd_4mode5m_f32_r64", kind="cpd", d0=50000, d1=30000, d2=10000, d3=400,
             nnz=5000000, zipf=1.1, rank=64, dtype="f32", alloc="two", its=10, nonneg=False),
        # non-negative CPD, the constraint in commonest use
        dict(name="cpd_nonneg2m_f64_r32", kind="cpd", d0=40000, d1=25000, d2=8000, d3=0,
             nnz=2000000, zipf=1.1, rank=32, dtype="f64", alloc="two", its=5, nonneg=True),
        # one stream: slices of uneven size, rank 32
        dict(name="stream6_f64_r32", kind="stream", d0=100000, d1=50000, slices=6, nnz=150000,
             rank=32),
        # many streams at once
        dict(name="serve8x2_f64", kind="serve", d0=60000, d1=30000, slices=2, nnz=60000,
             streams=8, rank=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tensor(rng, lo, hi, modes, dmax):
    """Sizes of a drawn tensor: dims spread over the range with room for the
    nonzeros to be distinct."""
    nnz = _log(rng, lo, hi)
    zipf = rng.choice([0.0, 1.1, 1.2])
    while True:
        d = [_log(rng, 60, dmax) for _ in range(min(modes, 3))]
        if modes == 4:
            d.append(_log(rng, 20, 1000))
        cells = math.prod(d)
        if nnz * (40 if zipf == 0.0 else 3000) <= cells < 1 << 61 and 2 * max(d) <= nnz:
            break
    d += [0] * (4 - len(d))
    return dict(d0=d[0], d1=d[1], d2=d[2], d3=d[3], nnz=nnz, zipf=zipf)


def draw(rng):
    kind = rng.choices(["mttkrp", "mttkrp_host", "csf", "cpd", "stream", "serve"],
                       [50, 5, 8, 24, 10, 3])[0]
    if kind in ("mttkrp", "mttkrp_host"):
        modes = rng.choice([3, 3, 4])
        rank = rng.choice([8, 16, 32, 64]) if rng.random() < 0.5 else rng.randint(5, 80)
        hi = 3e6 if kind == "mttkrp_host" else min(2e7, 8e8 / rank)
        return dict(kind=kind, **_tensor(rng, 4e3, hi, modes, 1.5e5), rank=rank,
                    dtype="f64" if kind == "mttkrp_host" else rng.choice(["f32", "f64"]),
                    alloc=rng.choice(["one", "two", "all"]))
    if kind == "csf":
        return dict(kind=kind, **_tensor(rng, 2e4, 4e6, rng.choice([3, 4]), 1e5), rank=0,
                    dtype="f64", alloc=rng.choice(["one", "two", "all"]))
    if kind == "cpd":
        rank = rng.choice([16, 32, 64]) if rng.random() < 0.5 else rng.randint(5, 64)
        nonneg = rng.random() < 0.4
        return dict(kind=kind, **_tensor(rng, 1e4, 2e6 if nonneg else 4e6, rng.choice([3, 3, 4]),
                                         5e4), rank=rank,
                    dtype=rng.choice(["f32", "f64"]), alloc="two",
                    its=rng.randint(3, 5) if nonneg else rng.randint(5, 15), nonneg=nonneg)
    if kind == "stream":
        return dict(kind=kind, d0=_log(rng, 5e3, 1e5), d1=_log(rng, 5e3, 5e4),
                    slices=rng.randint(2, 6), nnz=_log(rng, 5e3, 1.5e5),
                    rank=rng.choice([8, 16, 32, rng.randint(5, 48)]))
    return dict(kind=kind, d0=_log(rng, 1e4, 6e4), d1=_log(rng, 1e4, 3e4), slices=2,
                nnz=_log(rng, 5e3, 6e4), streams=rng.randint(3, 8), rank=0)


# ---- inputs -----------------------------------------------------------------

def _dims(case):
    return [case["d%d" % m] for m in range(4) if case.get("d%d" % m)]


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + what) % (1 << 62))


def _indices(dim, zipf, n, g):
    """n draws from [0, dim): uniform, or Zipf ranks under a random relabelling."""
    if zipf == 0.0:
        return torch.randint(dim, (n,), generator=g, device="cuda")
    cdf = torch.arange(1, dim + 1, device="cuda", dtype=torch.float64).pow_(-zipf).cumsum_(0)
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * cdf[-1]
    return torch.searchsorted(cdf, u).clamp_(max=dim - 1)


def _coords(dims, zipf, nnz, g, cover=True):
    """nnz distinct coordinates in random order; with cover, every index of
    every mode occurs at least once."""
    relabel = [torch.randperm(d, generator=g, device="cuda") for d in dims]
    # position p of the longest mode with p modulo the others' sizes
    must = torch.zeros(max(dims) if cover else 0, dtype=torch.int64, device="cuda")
    p = torch.arange(must.numel(), device="cuda")
    for d in dims:
        must.mul_(d).add_(p % d)
    must = must[:nnz]
    keys = torch.empty(0, dtype=torch.int64, device="cuda")
    while keys.numel() < nnz - must.numel():
        need = nnz - must.numel() - keys.numel()
        k = torch.zeros(int(need * 1.15) + 64, dtype=torch.int64, device="cuda")
        for d in dims:
            k.mul_(d).add_(_indices(d, zipf, k.numel(), g))
        keys = torch.unique(torch.cat([keys, k]))
        keys = keys[~torch.isin(keys, must)]
    keep = torch.randperm(keys.numel(), generator=g, device="cuda")[:nnz - must.numel()]
    keys = torch.cat([must, keys[keep]])
    keys = keys[torch.randperm(nnz, generator=g, device="cuda")]
    inds = [None] * len(dims)
    for m in reversed(range(len(dims))):
        inds[m] = relabel[m][keys % dims[m]]
        keys = keys // dims[m]
    return inds


def _host(t):
    return t.cpu().numpy().view(np.uint64) if t.dtype == torch.int64 else t.cpu().numpy()


def _coo(case, seed):
    """The tensor on the GPU: indices, FP64 values, dims."""
    g = _gen(seed, 1)
    dims, n = _dims(case), case["nnz"]
    inds = _coords(dims, case["zipf"], n, g)
    if case["kind"] == "cpd":
        vals = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
        if not case["nonneg"] and len(dims) == 4:
            vals = 2 * vals - 1
    else:
        vals = torch.randn(n, generator=g, device="cuda", dtype=torch.float64).exp_()
    return inds, vals, dims


def _factors(case, dims, seed):
    """Start or input factors, FP64 on the GPU."""
    g = _gen(seed, 2)
    u = [torch.rand(d, case["rank"], generator=g, device="cuda", dtype=torch.float64)
         for d in dims]
    if case["kind"] == "cpd" and not case["nonneg"]:
        u = [3 * (2 * x - 1) for x in u]
    if case["dtype"] == "f32" and case["kind"] == "mttkrp":
        u = [x.float() for x in u]
    return u


def _slices(case, seed):
    """Streams of time slices: per stream its dims, rank and slices (i, j, values)."""
    g = _gen(seed, 3)
    streams = []
    for k in range(case.get("streams", 1)):
        shrink = 1.0 - 0.4 * k / max(1, case.get("streams", 1))
        dims = [int(case["d0"] * shrink), int(case["d1"] * shrink)]
        sl = []
        for t in range(case["slices"]):
            n = int(case["nnz"] * UNEVEN[(t + k) % len(UNEVEN)])
            ij = _coords(dims, 1.2, n, g, cover=False)
            v = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
            sl.append((_host(ij[0]), _host(ij[1]), _host(v)))
        streams.append(dict(dims=dims, rank=case["rank"] or (8, 16, 32, 64)[k % 4], slices=sl))
    return streams


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, kind=kind)
    if kind == "serve":
        s["streams"] = _slices(case, seed)
        return s
    if kind == "stream":
        one = _slices(case, seed)[0]
        s["inds"] = [np.concatenate([x[m] for x in one["slices"]]) for m in range(2)]
        s["inds"].append(np.concatenate([np.full(len(x[2]), t, dtype=np.uint64)
                                         for t, x in enumerate(one["slices"])]))
        s["vals"] = np.concatenate([x[2] for x in one["slices"]])
        s["dims"] = one["dims"] + [case["slices"]]
        return s
    inds, vals, dims = _coo(case, seed)
    s["dims"] = dims
    hi, hv = [_host(i) for i in inds], _host(vals)
    s["opts"] = ps.Opts(csf_alloc=ALLOC[case["alloc"]])
    if kind == "csf":
        s["inds"], s["vals"] = hi, hv
        # the arrays whose length depends on the pattern are handed on in
        # buffers of the longest they can be
        count = {"one": 1, "two": 2, "all": len(dims)}[case["alloc"]]
        s["bufs"] = [{} for _ in range(count)]
        for b in s["bufs"]:
            for l in range(1, len(dims) - 1):
                b["fptr%d" % l] = torch.full((case["nnz"] + 1,), -1, dtype=torch.int64)
                b["fids%d" % l] = torch.full((case["nnz"],), -1, dtype=torch.int64)
        return s
    del inds, vals
    s["csf"] = ps.CsfSet.convert(hi, hv, s["opts"])
    u = _factors(case, dims, seed)
    if kind == "mttkrp":
        s["mats"] = u
        s["outs"] = [torch.empty_like(x) for x in u]
        s["ptrs"] = (C.c_void_p * len(u))(*[x.data_ptr() for x in u])
        s["prec"] = ps.F32 if case["dtype"] == "f32" else ps.F64
    elif kind == "mttkrp_host":
        s["mats"] = [x.cpu().numpy() for x in u]
    else:
        s["start"] = [x.cpu().numpy() for x in u]
        L = ps.lib()
        s["copts"] = L.splatt_alloc_cpd_opts()
        s["copts"][0].max_iterations = case["its"]
        s["copts"][0].tolerance = 0.0
        if case["nonneg"]:
            modes = np.arange(len(dims), dtype=np.uint64)
            L.splatt_register_nonneg(s["copts"], modes.ctypes.data_as(ps.u64p), len(dims))
        s["gopts"] = L.splatt_alloc_global_opts()
        s["gopts"][0].verbosity = 0
        # the Kruskal tensor a caller owns, its factor arrays overwritten by each call
        k = ps.SplattKruskal()
        s["factors"] = [np.empty_like(x) for x in s["start"]]
        s["lambda"] = np.ones(case["rank"])
        k.rank, k.nmodes = case["rank"], len(dims)
        k.lambda_ = s["lambda"].ctypes.data_as(ps.f64p)
        for m, f in enumerate(s["factors"]):
            k.factors[m] = f.ctypes.data_as(ps.f64p)
            k.dims[m] = dims[m]
        s["kruskal"] = k
    return s


# ---- one pass ---------------------------------------------------------------

def _check(rc, what):
    if rc != ps.SUCCESS:
        raise RuntimeError("%s failed: %s" % (what, ps.last_error()))


def run(s):
    kind, case = s["kind"], s["case"]
    L = ps.lib()
    if kind == "mttkrp":
        for m, o in enumerate(s["outs"]):
            _check(L.splatt_amd_mttkrp_dev(m, case["rank"], s["csf"].ptr, s["ptrs"], o.data_ptr(),
                                           s["prec"], s["opts"].ptr, None), "mttkrp")
        return s["outs"]
    if kind == "mttkrp_host":
        return [s["csf"].mttkrp(m, s["mats"]) for m in range(len(s["dims"]))]
    if kind == "csf":
        csf = ps.CsfSet.convert(s["inds"], s["vals"], s["opts"])
        return [_arrays(csf, i, b) for i, b in enumerate(s["bufs"])]
    if kind == "cpd":
        for f, x in zip(s["factors"], s["start"]):
            np.copyto(f, x)
        s["lambda"][:] = 1.0
        L.splatt_amd_set_mttkrp_precision(ps.F32 if case["dtype"] == "f32" else ps.F64)
        rc = L.splatt_cpd(s["csf"].ptr, case["rank"], s["copts"], s["gopts"],
                          C.byref(s["kruskal"]))
        L.splatt_amd_set_mttkrp_precision(ps.F64)
        _check(rc, "cpd")
        return dict(factors=s["factors"], lam=s["lambda"], fit=float(s["kruskal"].fit))
    if kind == "stream":
        r = ps.run_stream(s["inds"], s["vals"], s["dims"], case["rank"], 2, forget=FORGET,
                          max_its=OUTER, seed=4, frob=FROB)
        f = [_placed(r["factors"][m], s["dims"][m], r["iperm"][m].view(np.int64))
             for m in range(2)]
        return dict(factors=f + [r["factors"][2]], local_err=r["local_err"],
                    final_err=r["final_err"])
    sv = ps.Server(budget=4 << 30, max_inflight=8)
    try:
        ids = [sv.open(x["dims"] + [1], x["rank"], 2, forget=FORGET, max_its=OUTER, frob=FROB,
                       seed=1 + k) for k, x in enumerate(s["streams"])]
        tickets = []
        for t in range(case["slices"]):
            for k, x in enumerate(s["streams"]):
                i, j, v = x["slices"][t]
                tickets.append(sv.submit(ids[k], [i, j, np.full(len(v), t, dtype=np.uint64)], v))
        sv.drain()
        f = [[_placed(sv.factors(sid, m), x["dims"][m]) for m in range(2)] + [sv.factors(sid, 2)]
             for sid, x in zip(ids, s["streams"])]
        return dict(factors=f,
                    local_err=[sv.slice(x)["local_err"] for x in tickets])
    finally:
        sv.free()


def _owned(csf, ptr, n, ctype, dtype):
    """An array of csf in place, which keeps csf."""
    a = (ctype * n).from_address(C.addressof(ptr.contents))
    a.owner = csf
    return np.frombuffer(a, dtype=dtype)


def _arrays(csf, i, bufs):
    """Arrays of one CSF's single tile: in place, or copied into bufs."""
    ct = csf.ptr[i]
    n, pt = int(ct.nmodes), ct.pt[0]
    nf = [int(pt.nfibs[l]) for l in range(n)]
    d = dict(perm=[int(ct.dim_perm[l]) for l in range(n)],
             vals=_owned(csf, pt.vals, nf[-1], C.c_double, np.float64))
    for l in range(n):
        if l < n - 1:
            d["fptr%d" % l] = _owned(csf, pt.fptr[l], nf[l] + 1, C.c_int64, np.int64)
        if l > 0:
            d["fids%d" % l] = _owned(csf, pt.fids[l], nf[l], C.c_int64, np.int64)
    for k, b in bufs.items():
        b[:len(d[k])].copy_(torch.from_numpy(d[k]))
        d[k] = b
    return d


def _placed(rows, n, at=None):
    """Factor rows in an n-row matrix: at their original indices, or first."""
    out = np.zeros((n, rows.shape[1]))
    out[slice(len(rows)) if at is None else at[:len(rows)]] = rows
    return out


# ---- cost and accuracy ------------------------------------------------------

def work(case):
    """Bytes and operations of one pass: 4-byte indices, every array once a
    use (an MTTKRP reads the leaf ids, the values and the other modes'
    factors and writes its output; a CPD iteration is one MTTKRP and one
    solve a mode)."""
    kind, nnz, R = case["kind"], case["nnz"], case["rank"]
    if kind in ("stream", "serve"):
        R = R or 30
        rows = min(case["d0"], nnz) + min(case["d1"], nnz)
        its = OUTER * case["slices"] * case.get("streams", 1)
        return dict(bytes=its * (3 * nnz * 16 + 5 * rows * R * 8.0),
                    flops=its * (3 * 4 * nnz * R + 8.0 * rows * R * R))
    dims, sv = _dims(case), 4 if case["dtype"] == "f32" else 8
    n = len(dims)
    if kind == "csf":
        count = {"one": 1, "two": 2, "all": n}[case["alloc"]]
        return dict(bytes=float(nnz * (8 * n + 8) + count * nnz * 24), flops=0.0)
    sweep = n * (nnz * (sv + 4.0) + sum(dims) * R * sv)
    flops = n * 2.0 * R * nnz * (1 if n == 3 else 1.5)
    if kind != "cpd":
        return dict(bytes=sweep, flops=flops)
    return dict(bytes=case["its"] * (sweep + 3 * sum(dims) * R * 8.0),
                flops=case["its"] * (flops + 4.0 * sum(dims) * R * R))


def tolerance(case):
    """About four times what the library was seen to differ from exact()."""
    kind = case["kind"]
    if kind == "csf":
        return "exact"
    if kind == "mttkrp_host" or (kind == "mttkrp" and case["dtype"] == "f64"):
        return {"rel": 3e-15}
    if kind == "mttkrp":
        return {"rel": 1e-6}
    if kind == "cpd":
        return {"rel": 1.5e-5 if case["dtype"] == "f32" else 1e-10}
    return {"rel": 2e-9}


def _mttkrp64(inds, vals, u, mode):
    """Plain FP64 MTTKRP on the GPU, by pieces; heavy rows are spread over
    copies of the output that are added up at the end."""
    rows, R = u[mode].shape
    k = max(1, min(256, (1 << 29) // (rows * R)))
    out = torch.zeros(rows * k, R, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // R)
    for a in range(0, vals.numel(), step):
        x = vals[a:a + step, None].expand(-1, R)
        for m, f in enumerate(u):
            if m != mode:
                x = x * f[inds[m][a:a + step]]
        at = inds[mode][a:a + step] * k
        out.index_add_(0, at + torch.arange(at.numel(), device="cuda") % k, x)
    return out.view(rows, k, R).sum(1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "csf":
        return None                      # whole numbers and copies of the input
    if kind == "stream":
        one = _slices(case, seed)[0]
        f, le, fe, lab = _stream64(one["slices"], case["rank"], 4)
        for m in range(2):
            f[m] = _placed(f[m], one["dims"][m], np.array(list(lab[m])))
        return dict(factors=f, local_err=le, final_err=fe)
    if kind == "serve":
        got = [_stream64(x["slices"], x["rank"], 1 + k)
               for k, x in enumerate(_slices(case, seed))]
        le = [float(g[1][t]) for t in range(case["slices"]) for g in got]
        f = [[_placed(g[0][m], x["dims"][m]) for m in range(2)] + [g[0][2]]
             for g, x in zip(got, _slices(case, seed))]
        return dict(factors=f, local_err=le)
    inds, vals, dims = _coo(case, seed)
    u = [x.double() for x in _factors(case, dims, seed)]
    if kind != "cpd":
        return [_mttkrp64(inds, vals, u, m) for m in range(len(dims))]
    xnorm = float(vals.square().sum())
    R = case["rank"]
    dev = dict(dtype=torch.float64, device="cuda")
    for m in range(len(u)):
        u[m] = u[m] / u[m].norm(dim=0)
    gram = [x.T @ x for x in u]
    dual = [torch.zeros_like(x) for x in u]
    lam = torch.ones(R, **dev)
    for _ in range(case["its"]):
        for m in range(len(u)):
            M = _mttkrp64(inds, vals, u, m)
            G = torch.ones(R, R, **dev)
            for k in range(len(u)):
                if k != m:
                    G = G * gram[k]
            if case["nonneg"]:
                u[m], dual[m] = _admm_nonneg64(M, G, u[m], dual[m])
            else:
                u[m] = torch.linalg.solve(G, M.T).T.contiguous()
                lam = u[m].norm(dim=0)
                u[m] = u[m] / lam
            gram[m] = u[m].T @ u[m]
    G = torch.ones(R, R, **dev)
    for g in gram:
        G = G * g
    znorm = float((lam @ G @ lam).abs())
    inner = float(((u[-1] * M).sum(0) * lam).sum())
    fit = 1.0 - (xnorm + znorm - 2 * inner) / xnorm
    if not case["nonneg"]:
        for m in range(len(u)):
            c = u[m].norm(dim=0)
            u[m] = u[m] / c
            lam = lam * c
    return dict(factors=[x.cpu() for x in u], lam=lam.cpu(), fit=fit)


def _admm_nonneg64(M, G, P, D, chunk=50, its=50, tol=1e-2):
    """Non-negative least squares by ADMM, every chunk of rows to its own convergence."""
    n, R = M.shape
    rho = float(G.trace()) / R
    inv = torch.linalg.inv(G + rho * torch.eye(R, dtype=G.dtype, device=G.device))
    inv = (inv + inv.T) / 2
    nc = -(-n // chunk)

    def split(x):
        return torch.cat([x, x.new_zeros(nc * chunk - n, R)]).view(nc, chunk, R)

    M, P, D = split(M), split(P), split(D)
    live = torch.arange(nc, device=M.device)
    for _ in range(its):
        p0, d0 = P[live], D[live]
        aux = (M[live] + rho * (p0 + d0)) @ inv
        p = (aux - d0).clamp_(min=0)
        d = d0 + (p - aux)
        P[live], D[live] = p, d
        pn, pr, dr, dn = ((x * x).sum((1, 2)) for x in (p, p - aux, p - p0, d))
        live = live[~((pr <= tol * pn) & (dr <= tol * dn))]
        if live.numel() == 0:
            break
    return P.view(-1, R)[:n].contiguous(), D.view(-1, R)[:n].contiguous()


def _rand_fill(libc, rows, R):
    """Factor entries as the library draws them: magnitude from one rand(), sign from the next."""
    r = libc.rand
    x = np.array([r() for _ in range(2 * rows * R)], dtype=np.int64).reshape(rows, R, 2)
    v = 3.0 * (x[:, :, 0] / 2147483647.0)
    return np.where(x[:, :, 1] % 2 == 0, -v, v)


def _stream64(slices, R, seed):
    """The streaming CPD of 3-mode slices (time last): factors (modes
    relabelled by first appearance), per-slice errors, the final error and
    the labels."""
    # labels and new rows first: library calls in between may draw from rand() too
    libc = C.CDLL(None)
    libc.rand.restype = C.c_int
    libc.srand(C.c_uint(seed))
    lab = [{}, {}]
    parsed = []
    for i, j, v in slices:
        order = np.lexsort((j, i))
        ind, rows = [], []
        for t, x in zip(lab, (i, j)):
            before = len(t)
            ind.append(np.array([t.setdefault(k, len(t)) for k in x[order].tolist()]))
            rows.append(_rand_fill(libc, len(t) - before, R))
        parsed.append((ind, v[order], rows))
    dev = dict(dtype=torch.float64, device="cuda")
    new = [torch.zeros(0, R, **dev) for _ in range(2)]
    old = [torch.zeros(0, R, **dev) for _ in range(2)]
    gram = [None, None]
    tg = torch.zeros(R, R, **dev)
    eye = torch.eye(R, **dev)
    times, local, seen = [], [], []
    for s, (ind, v, rows) in enumerate(parsed):
        ind = [torch.from_numpy(x).cuda() for x in ind]
        v = torch.from_numpy(v).cuda()
        seen.append((ind, v))
        for m in range(2):
            new[m] = torch.cat([new[m], torch.from_numpy(rows[m]).cuda()])
            old[m] = torch.cat([old[m], torch.zeros(len(rows[m]), R, **dev)])
            gram[m] = new[m].T @ new[m]
        if s == 0:
            new = [x / x.norm(dim=0) for x in new]
        prev = 0.0
        for it in range(OUTER):
            mt = (v[:, None] * new[0][ind[0]] * new[1][ind[1]]).sum(0)
            row = torch.linalg.solve(gram[0] * gram[1] + FROB * eye, mt)
            before = tg
            tg = before + row[:, None] * row[None, :]
            delta = 0.0
            for m in range(2):
                o = 1 - m
                M = torch.zeros_like(new[m])
                M.index_add_(0, ind[m], v[:, None] * new[o][ind[o]] * row)
                M += old[m] @ (before * (old[o].T @ new[o]))
                new[m] = _admm_colnorm64(M, gram[o] * tg, new[m])
                gram[m] = new[m].T @ new[m]
                delta += float((old[m] - new[m]).norm() / new[m].norm())
            if it > 0 and abs(delta - prev) < 5e-2:
                break
            prev = delta
        tg = tg * FORGET
        old = [x.clone() for x in new]
        times.append(row)
        xn = float(v.square().sum())
        inner = float((v[:, None] * new[0][ind[0]] * new[1][ind[1]] * row).sum())
        zn = float((gram[0] * gram[1] * (row[:, None] * row)).sum())
        local.append((xn + zn - 2 * inner) / xn)
    T = torch.stack(times)
    xn = sum(float(v.square().sum()) for _, v in seen)
    inner = sum(float((v[:, None] * new[0][ind[0]] * new[1][ind[1]] * T[k]).sum())
                for k, (ind, v) in enumerate(seen))
    zn = float((gram[0] * gram[1] * (T.T @ T)).sum())
    return ([x.cpu().numpy() for x in (*new, T)], np.array(local),
            (xn + zn - 2 * inner) / xn, lab)


def _admm_colnorm64(M, G, P, its=25, tol=7e-2):
    """ADMM for columns of norm at most one, from a zero dual."""
    R = M.shape[1]
    rho = float(G.trace()) / R
    inv = torch.linalg.inv(G + rho * torch.eye(R, dtype=G.dtype, device=G.device))
    inv = (inv + inv.T) / 2
    D = torch.zeros_like(P)
    for _ in range(its):
        aux = (M + rho * (P + D)) @ inv
        p = aux - D
        n = p.norm(dim=0)
        p = torch.where(n > 1, p / n, p)
        D = D + (p - aux)
        pn, pr, dr, dn = (float(x.square().sum()) for x in (p, p - aux, p - P, D))
        P = p
        if pr <= tol * pn and dr <= tol * dn:
            break
    return P
