"""What the speed of this framework is measured on.

A case is one call of a program that uses the engine on data resident in HBM:
association tests of a chunk of genes (eqtlbma_bf), their permutations, Bayes
factors from given summary statistics, the EM of eqtlbma_hm, the averages and
posteriors of eqtlbma_avg_bfs, and one step of the permutation allocator.
Sizes are those of the tests and of bench.py, a chunk at a time, and odd ones
around them; `draw` covers the same ranges.

`exact` restates every model in 64 bits with torch alone.
"""
import ctypes as C
import math

import numpy as np
import torch

from eqtlbma_amd import _abi, synth
from eqtlbma_amd import engine as eng

F64 = torch.float64


def listed():
    return [
        # one gene of the plain-method workload: what an interactive call costs
        dict(name="uvlr_one_gene", kind="uvlr", genes=1, snps=201, subgroups=3, samples=100, covars=0, bfs="all",
             grid=25, dosage=False, stats=True, missing=0.0),
        # the plain-method workload: 200 genes, every output that the files need
        dict(name="uvlr_plain", kind="uvlr", genes=200, snps=201, subgroups=3, samples=100, covars=0, bfs="all",
             grid=25, dosage=False, stats=True, missing=0.0),
        # many tissues of uneven size, dosages, covariates, singleton configurations: Bayes factors only
        dict(name="uvlr_tissues", kind="uvlr", genes=160, snps=1500, subgroups=44, samples=500, covars=3, bfs="sin",
             grid=50, dosage=True, stats=False, missing=0.0),
        # separate analysis: summary statistics only, ragged sizes, missing levels
        dict(name="sep_ragged", kind="sep", genes=120, snps=613, subgroups=11, samples=337, covars=5, bfs="gen",
             grid=25, dosage=True, stats=True, missing=0.03),
        # Bayes factors from summary statistics that were computed elsewhere
        dict(name="inss", kind="inss", pairs=60001, subgroups=5, bfs="all", grid=25),
        # multivariate error model, consistent configuration
        dict(name="mvlr", kind="mvlr", genes=120, snps=800, subgroups=9, samples=150, covars=0, bfs="gen", grid=50),
        # hybrid error model: levels missing per subgroup, covariates of each subgroup
        dict(name="hybrid", kind="hybrid", genes=60, snps=800, subgroups=9, samples=150, covars=3, bfs="gen",
             grid=50, missing=0.15),
        # gene-level p-values: a file chunk of genes, 10,000 permutations each
        dict(name="perm_max", kind="perm", genes=24, snps=1000, subgroups=5, samples=300, nperm=10000, covars=0,
             dosage=False, use_max=True, missing=0.0),
        # the same where covariates, dosages and missing levels rule the closed forms out
        dict(name="perm_covariates", kind="perm", genes=3, snps=300, subgroups=3, samples=200, nperm=400, covars=2,
             dosage=True, use_max=False, missing=0.05),
        # EM on the raw Bayes factors of every configuration of five subgroups
        dict(name="hm_configs", kind="hm", model="configs", genes=1000, snps=1500, dim=31, subgroups=5, grid=10,
             iters=6),
        # averages and every posterior on the same shape
        dict(name="avg_configs", kind="avg", model="configs", genes=600, snps=1500, dim=31, subgroups=5, grid=10),
        # one step of the permutation allocator: LD spectra of new genes, a training step, a prediction
        dict(name="allocator", kind="alloc", genes=48, snps=1000, samples=300, rows=2000),
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["uvlr", "uvlr", "sep", "inss", "mvlr", "hybrid", "perm", "perm", "hm", "avg", "alloc"])
    if kind in ("uvlr", "sep"):
        S = rng.choice([1, 2, 3, 4, 5, 6, 9, 17, 31, 44])
        c = dict(kind=kind, genes=_log_between(rng, 1, 150), snps=_log_between(rng, 20, 1500), subgroups=S,
                 samples=rng.randint(60, 500), covars=rng.choice([0, 1, 3, 5]),
                 bfs=rng.choice(["gen", "sin", "all"] if S <= 6 else ["gen", "sin"]), grid=rng.choice([25, 50]),
                 dosage=rng.random() < 0.5, stats=rng.random() < 0.5, missing=rng.choice([0.0, 0.05]))
        if kind == "sep":
            c.update(bfs="gen", stats=True)
        return c
    if kind == "inss":
        return dict(kind=kind, pairs=_log_between(rng, 100, 100000), subgroups=rng.choice([1, 2, 3, 5, 6]),
                    bfs=rng.choice(["gen", "sin", "all"]), grid=rng.choice([25, 50]))
    if kind in ("mvlr", "hybrid"):
        c = dict(kind=kind, genes=_log_between(rng, 1, 50), snps=_log_between(rng, 30, 900),
                 subgroups=rng.choice([2, 3, 5, 7, 9]), samples=rng.randint(70, 300), covars=rng.choice([0, 2, 3, 5]),
                 bfs=rng.choice(["gen", "sin"]), grid=rng.choice([25, 50]))
        if kind == "hybrid":
            c["missing"] = rng.choice([0.05, 0.15, 0.25])
        return c
    if kind == "perm":
        if rng.random() < 0.6:
            return dict(kind=kind, genes=_log_between(rng, 1, 24), snps=rng.randint(100, 1500),
                        subgroups=rng.choice([1, 2, 3, 5]), samples=rng.randint(80, 400),
                        nperm=_log_between(rng, 500, 10000), covars=0, dosage=False, use_max=rng.random() < 0.7,
                        missing=0.0)
        return dict(kind=kind, genes=rng.randint(1, 3), snps=rng.randint(50, 400), subgroups=rng.choice([2, 3, 4]),
                    samples=rng.randint(80, 300), nperm=rng.randint(50, 400), covars=rng.choice([0, 2]), dosage=True,
                    use_max=rng.random() < 0.5, missing=0.05)
    if kind in ("hm", "avg"):
        model = rng.choice(["configs", "configs", "types"])
        S = rng.choice([3, 4, 5])
        c = dict(kind=kind, model=model, genes=_log_between(rng, 3, 600), snps=_log_between(rng, 20, 1500),
                 dim=(1 << S) - 1 if model == "configs" else rng.choice([2, 3]), subgroups=S,
                 grid=rng.choice([5, 10, 25]))
        if c["grid"] * c["dim"] > 310:
            c["grid"] = 10
        if kind == "hm":
            c["iters"] = rng.randint(3, 8)
        return c
    return dict(kind="alloc", genes=_log_between(rng, 1, 48), snps=_log_between(rng, 50, 1500),
                samples=rng.randint(80, 400), rows=_log_between(rng, 64, 2000))


# ---- sizes that do not depend on the seed --------------------------------

def _sizes(case):
    """Cis SNPs per gene: Poisson about the mean, the same for every seed."""
    r = np.random.default_rng(case["genes"] * 7919 + case["snps"])
    return np.maximum(r.poisson(case["snps"], case["genes"]), 4).astype(np.int64) if case["genes"] > 1 else \
        np.array([case["snps"]], np.int64)


def _grids(case):
    large = synth.make_grid("general", 10 if case["grid"] == 50 else 5)
    return large, (large if case["grid"] == 50 else synth.make_grid("small"))


_engines = {}


def _engine(case):
    """One context per pair of grids, as a program keeps it."""
    key = case.get("grid") if case["kind"] in ("uvlr", "sep", "inss", "mvlr", "hybrid") else None
    if key not in _engines:
        e = eng.Engine(0)
        e.set_grids(*(_grids(case) if key else (synth.make_grid("general"), synth.make_grid("small"))))
        _engines[key] = e
    return _engines[key]


# ---- inputs ---------------------------------------------------------------

def _genes(case, seed):
    """Genotypes, levels, membership and covariates of a chunk of genes."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = np.random.default_rng(seed)
    S, N, Q, G = case.get("subgroups", 1), case["samples"], case.get("covars", 0), case["genes"]
    P = _sizes(case)
    off = np.concatenate([[0], np.cumsum(P)]).astype(np.int64)
    n = int(off[-1])
    maf = torch.rand(n, device="cuda", generator=g) * 0.45 + 0.05
    x = (torch.rand((N, n), device="cuda", generator=g) < maf).float()
    x += (torch.rand((N, n), device="cuda", generator=g) < maf).float()
    x[0], x[1], x[2] = 0, 1, 2  # no SNP without variation
    if case.get("dosage"):
        x += 0.05 * torch.randn((N, n), device="cuda", generator=g)
        x.clamp_(0, 2)
    member = torch.ones((S, N), dtype=torch.bool, device="cuda")
    if case["kind"] in ("uvlr", "sep") and (S > 6 or case["missing"]):
        member = torch.rand((S, N), device="cuda", generator=g) < 0.2 + 0.6 * torch.rand((S, 1), device="cuda", generator=g)
        member[:, :min(N, 24)] = True
    cov = torch.randn((S, max(Q, 1), N), device="cuda", generator=g, dtype=F64)
    if case["kind"] == "mvlr":
        cov[:] = cov[:1].clone()
    y = torch.randn((G, S, N), device="cuda", generator=g, dtype=F64)
    if case["kind"] in ("mvlr", "hybrid") and S > 1:
        low = np.linalg.cholesky(np.full((S, S), 0.5) + 0.5 * np.eye(S))
        y = torch.matmul(torch.from_numpy(low).cuda(), y)
    if Q:
        y += 0.3 * cov[:, :Q].sum(1)
    for k in rnd.choice(G, size=max(1, int(round(0.12 * G))), replace=False):
        on = torch.from_numpy((rnd.random(S) < 0.6).astype(np.float64)).cuda()
        y[k] += rnd.normal(0, 0.5) * on[:, None] * x[:, int(off[k] + rnd.integers(P[k]))].double()
    y[:, ~member] = float("nan")
    if case.get("missing"):
        lost = torch.rand(y.shape, device="cuda", generator=g) < case["missing"]
        lost[:, :, :24] = False
        y[lost] = float("nan")
    return dict(G=G, S=S, N=N, Q=Q, P=P, off=off, x=x.contiguous(), y=y.contiguous(), member=member, cov=cov)


def _chunk(d):
    """The engine's description of the chunk; the tensors live in `d`."""
    S, N, n = d["S"], d["N"], int(d["off"][-1])
    ones = lambda *shape: torch.ones(shape, dtype=torch.uint8, device="cuda")  # noqa: E731
    d["t"] = t = dict(gene_in=ones(d["G"], S), geno_in=d["member"].to(torch.uint8).contiguous(),
                      count=torch.full((S,), d["Q"], dtype=torch.int32, device="cuda"), cov_in=ones(S, N),
                      gset=torch.zeros(S, dtype=torch.int32, device="cuda"), snp_in=ones(n, S),
                      off=torch.from_numpy(d["off"]).cuda(), snp=torch.arange(n, dtype=torch.int32, device="cuda"))
    c = _abi.Chunk()
    c.n_genes, c.n_subgroups, c.n_samples, c.n_covars_max = d["G"], S, N, d["cov"].shape[1]
    c.n_pairs = c.n_snps = c.geno_ld = n
    c.explevels, c.genotypes, c.covars = d["y"].data_ptr(), d["x"].data_ptr(), d["cov"].data_ptr()
    c.gene_in_sbgrp, c.geno_in_sbgrp = t["gene_in"].data_ptr(), t["geno_in"].data_ptr()
    c.covar_count, c.covar_in_sbgrp = t["count"].data_ptr(), t["cov_in"].data_ptr()
    c.n_geno_sets, c.geno_dtype, c.geno_set_stride = 1, _abi.F32, N * n
    c.geno_set_of_sbgrp, c.snp_in_sbgrp = t["gset"].data_ptr(), t["snp_in"].data_ptr()
    c.pair_offset, c.pair_snp = t["off"].data_ptr(), t["snp"].data_ptr()
    return c


def _outputs(case, S, n, stats, std, raw_dtype):
    gl, gs = (len(g) for g in _grids(case))
    nc = _abi.n_configs(case["bfs"], S)
    o = dict(n=torch.zeros((S, n), dtype=torch.int32, device="cuda"))
    if stats:
        o["sstats"] = torch.zeros((5, S, n), dtype=F64, device="cuda")
    if std:
        o["std"] = torch.zeros((3, S, n), dtype=F64, device="cuda")
    if raw_dtype is not None:
        o["raw"] = torch.zeros((3 * gl + nc * gs, n), dtype=raw_dtype, device="cuda")
        o["w"] = torch.zeros((5 + nc, n), dtype=F64, device="cuda")
    a = _abi.AssocOut()
    a.n = o["n"].data_ptr()
    a.sstats = o["sstats"].data_ptr() if "sstats" in o else None
    a.stdsstats = o["std"].data_ptr() if "std" in o else None
    a.raw_abf = o["raw"].data_ptr() if "raw" in o else None
    a.w_abf = o["w"].data_ptr() if "w" in o else None
    return o, a


def _inss_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    S, n = case["subgroups"], case["pairs"]
    u = lambda lo, hi: torch.rand((S, n), device="cuda", generator=g, dtype=F64) * (hi - lo) + lo  # noqa: E731
    size = torch.randint(60, 500, (S, n), device="cuda", generator=g)
    sig, se = u(0.7, 1.4), u(0.04, 0.2)
    beta = se * torch.randn((S, n), device="cuda", generator=g, dtype=F64)
    beta += 0.5 * (torch.rand((S, n), device="cuda", generator=g) < 0.02)
    return size, sig, beta, se


def _raw_inputs(case, seed):
    """Raw log10 ABFs as eqtlbma_bf writes them, and the models' weights."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = np.random.default_rng(seed)
    P = _sizes(case)
    off = np.concatenate([[0], np.cumsum(P)]).astype(np.int64)
    types = case["model"] == "types"
    G, L, K, S = case["genes"], case["grid"], case["dim"], case["subgroups"]
    D = S if types else K
    raw = torch.empty((int(off[-1]), D, L), dtype=F64, device="cuda").normal_(-0.6, 0.4, generator=g)
    hot = np.nonzero(r.random(G) < 0.3)[0]
    if hot.size:
        at = torch.from_numpy(off[hot] + r.integers(0, P[hot])).cuda()
        b = torch.empty((hot.size, D, L), dtype=F64, device="cuda").uniform_(1.0, 3.0, generator=g)
        raw[at] += b * (torch.rand((hot.size, D, L), device="cuda", generator=g) < 0.6)
    w = dict(grid=r.dirichlet(np.full(L, 5.0)), dim=r.dirichlet(np.full(K, 5.0)),
             sub=r.uniform(0.2, 0.9, (K, S)) if types else None)
    return dict(raw=raw, off=off, types=types, G=G, L=L, K=K, S=S, w=w)


def prepare(case, seed):
    kind = case["kind"]
    e = _engine(case)
    s = dict(kind=kind, eng=e)
    if kind in ("uvlr", "sep", "mvlr", "hybrid", "perm", "alloc"):
        d = _genes(case, seed)
        s["data"], s["chunk"] = d, _chunk(d)
        n = int(d["off"][-1])
    if kind in ("uvlr", "sep"):
        sep = kind == "sep"
        tiled = not sep and not case["stats"]
        s["out"], s["a"] = _outputs(case, d["S"], n, case["stats"], case["stats"] and not sep,
                                    None if sep else torch.float32 if tiled else F64)
        s["opts"] = _abi.AssocOpts(_abi.ANALYSIS["sep" if sep else "join"], _abi.BFS[case["bfs"]], _abi.PREC["mixed"],
                                   _abi.F32_TILED if tiled else _abi.F64)
    elif kind in ("mvlr", "hybrid"):
        s["out"], s["a"] = _outputs(case, d["S"], n, kind == "hybrid", False, F64)
        s["opts"] = (eng.MvlrOpts if kind == "mvlr" else eng.HybridOpts)(_abi.BFS[case["bfs"]], 0.5)
    elif kind == "inss":
        s["in"] = _inss_inputs(case, seed)
        s["bfs"] = case["bfs"]
        s["si"] = eng.SstatsIn(case["pairs"], case["subgroups"], *[t.data_ptr() for t in s["in"]])
        s["out"], s["a"] = _outputs(case, case["subgroups"], case["pairs"], False, True, F64)
    elif kind == "perm":
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        G, N, nperm = d["G"], d["N"], case["nperm"]
        s["tables"] = torch.empty((G, nperm, N), dtype=torch.int32, device="cuda")
        for k in range(G):
            s["tables"][k] = torch.rand((nperm, N), device="cuda", generator=g).argsort(1).to(torch.int32)
        s["which"] = np.arange(G, dtype=np.int32)
        s["stats"] = torch.zeros((G, nperm), dtype=F64, device="cuda")
        # the true statistics that such a program has from its association pass
        o, a = _outputs(dict(kind="perm", bfs="all", grid=25), d["S"], n, False, False, F64)
        torch.cuda.synchronize()  # the engine's stream does not wait for torch's
        e.assoc_uvlr_device(s["chunk"], _abi.AssocOpts(1, _abi.BFS["all"], _abi.PREC["mixed"], _abi.F64), a)
        e.sync()
        s["true"] = torch.stack([w.max() if case["use_max"] else _lmean(w, 0)
                                 for w in torch.split(o["w"][-1], [int(p) for p in d["P"]])])
        s["opts"] = eng.PermOpts(_abi.ANALYSIS["join"], _abi.PBF["all"], int(case["use_max"]), -1, _abi.PREC["mixed"])
        s["nperm"] = nperm
    elif kind in ("hm", "avg"):
        d = _raw_inputs(case, seed)
        s["data"] = d
        s["off"] = torch.from_numpy(d["off"]).cuda()
        if kind == "hm":
            o = eng.HmOpts()
            o.model, o.dim, o.n_subgroups, o.n_grid = int(d["types"]), d["K"], d["S"], d["L"]
            o.thresh, o.max_iters, o.stepmax = 1e-300, case["iters"], 1.0
            s["opts"] = o
        else:
            n, K, S, G = int(d["off"][-1]), d["K"], d["S"], d["G"]
            z = lambda *shape: torch.zeros(shape, dtype=F64, device="cuda")  # noqa: E731
            s["out"] = dict(gene_bf=z(G), gene_post=z(G), snp_bf=z(n), dim_bf=z(n, K), post_the=z(n), post_an=z(n),
                            post_dim=z(n, K), post_sub=z(n, S),
                            best_dim=torch.zeros(n, dtype=torch.int32, device="cuda"))
            s["a"] = eng.AvgOut(*[s["out"][f[0]].data_ptr() for f in eng.AvgOut._fields_])
            w = d["w"]
            s["keep"] = np.arange(d["L"], dtype=np.int32)
            s["masks"] = np.array(list(_abi.config_masks("all", S)), np.uint64) if not d["types"] else None
            ptr = lambda a: None if a is None else a.ctypes.data  # noqa: E731
            s["opts"] = eng.AvgOpts(int(d["types"]), K, S, d["L"], d["L"], ptr(s["keep"]), ptr(w["grid"]),
                                    ptr(w["dim"]), ptr(s["masks"]), ptr(w["sub"]), 0.6, 31)
    elif kind == "alloc":
        r = np.random.default_rng(seed)
        if "net" not in _engines:
            _engines["net"] = eng.Mlp(e, 24, 256, 3, 3, 1)
        s["net"] = _engines["net"]
        s["x"] = r.normal(0, 1, (case["rows"], 24)).astype(np.float32)
        s["t"] = (np.tanh(s["x"][:, :3]) + r.normal(0, 0.3, (case["rows"], 3))).astype(np.float32)
    torch.cuda.synchronize()
    return s


def run(s):
    kind, e = s["kind"], s["eng"]
    if kind in ("uvlr", "sep"):
        e.assoc_uvlr_device(s["chunk"], s["opts"], s["a"])
        return s["out"]
    if kind == "mvlr":
        e.assoc_mvlr_device(s["chunk"], s["opts"], s["a"])
        return s["out"]
    if kind == "hybrid":
        e.assoc_hybrid_device(s["chunk"], s["opts"], s["a"])
        return s["out"]
    if kind == "inss":
        e.abf_from_sstats_device(s["si"], s["bfs"], _abi.F64, s["a"])
        return s["out"]
    if kind == "perm":
        e.perm_stats_fp64_ties_device(s["chunk"], s["opts"], s["tables"].data_ptr(), s["tables"].shape[0], s["which"],
                                      s["nperm"], 5e-5, s["stats"].data_ptr(), s["true"].data_ptr())
        return [s["stats"], s["true"]]
    if kind == "hm":
        d, w = s["data"], s["data"]["w"]
        grid, dim = w["grid"].copy(), w["dim"].copy()
        sub = w["sub"].copy() if d["types"] else None
        p = eng.HmParamsC()
        p.pi0, p.grid = 0.5, grid.ctypes.data
        if d["types"]:
            p.type, p.subgroup = dim.ctypes.data, sub.ctypes.data
        else:
            p.config = dim.ctypes.data
        lik, iters = e.hm_em_device(d["raw"].data_ptr(), int(d["off"][-1]), s["off"].data_ptr(), d["G"], s["opts"], p)
        return [p.pi0, grid, dim, sub, lik, int(iters)]
    if kind == "avg":
        d = s["data"]
        e.avg_bfs_device(d["raw"].data_ptr(), int(d["off"][-1]), s["off"].data_ptr(), d["G"], s["opts"], s["a"])
        return s["out"]
    eig = e.ld_eigenvalues_device(s["chunk"], s["data"]["G"], 20)
    loss, grad = s["net"].loss_grad(s["x"], s["t"], np.ones(3, np.float32))
    return [eig, loss, grad, s["net"].forward(s["x"])]


# ---- what one pass cannot do without -------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("hm", "avg"):
        n, L, K, S = int(_sizes(case).sum()), case["grid"], case["dim"], case["subgroups"]
        rows = K if case["model"] == "configs" else S
        out = 8 * (3 + 2 * K + S) * n if kind == "avg" else 8 * (K + L)
        return {"bytes": 8 * n * rows * L + out, "flops": 2 * n * rows * L}
    if kind == "alloc":
        n, N, G = int(_sizes(case).sum()), case["samples"], case["genes"]
        return {"bytes": 4 * N * n + 80 * G, "flops": N * N * n + G * N ** 3 + 2 * 4 * case["rows"] * 138000}
    S = case["subgroups"]
    if kind == "perm":
        n, N, G = int(_sizes(case).sum()), case["samples"], case["genes"]
        return {"bytes": 4 * N * n + 8 * G * S * N + G * case["nperm"] * (4 * N + 8),
                "flops": 2 * n * case["nperm"] * N * S}
    gl, nc = case["grid"], _abi.n_configs(case["bfs"], S)
    rows = 0 if kind == "sep" else 3 * gl + nc * (50 if gl == 50 else 10)
    if kind == "inss":
        n = case["pairs"]
        return {"bytes": n * (S * (32 + 4 + 24) + 8 * (rows + 5 + nc)), "flops": 10 * n * rows}
    n, N, Q, G = int(_sizes(case).sum()), case["samples"], case["covars"], case["genes"]
    read = 4 * N * n + 8 * G * S * N
    raw = 4 if kind == "uvlr" and not case["stats"] else 8
    out = 4 * S + (40 * S if kind in ("sep", "hybrid") or case.get("stats") else 0)
    if kind != "sep":
        out += (24 * S if case.get("stats") else 0) + raw * rows + 8 * (5 + nc)
    sums = 2 * n * N * S * (2 + 1 + Q)
    if kind == "mvlr":
        sums += n * rows * 6 * S * S
    if kind == "hybrid":
        sums += n * N * S * (S - 1) * (6 + 2 * Q) + n * rows * 6 * S * S
    return {"bytes": read + n * out, "flops": sums + 10 * n * rows * (1 if kind == "mvlr" else min(S, 6))}


# ---- the same outputs in 64 bits, with torch alone -----------------------

LN10 = math.log(10.0)


def _lws(v, w, dim):
    """log10 of the sum of w 10^v along dim; w has one weight per entry."""
    shape = [1] * v.dim()
    shape[dim] = -1
    m = v.amax(dim, keepdim=True)
    return (m + torch.log10((w.reshape(shape) * torch.exp((v - m) * LN10)).sum(dim, keepdim=True))).squeeze(dim)


def _lmean(v, dim):
    return _lws(v, torch.full((v.shape[dim],), 1.0 / v.shape[dim], dtype=F64, device=v.device), dim)


def _beta_fraction(a, b, x):
    """Continued fraction of the incomplete beta function (modified Lentz)."""
    c = torch.ones_like(x)
    d = 1 / (1 - (a + b) * x / (a + 1))
    h = d.clone()
    for m in range(1, 400):
        k = m * (b - m) * x / ((a - 1 + 2 * m) * (a + 2 * m))
        d, c = 1 / (1 + k * d), 1 + k / c
        h *= d * c
        k = -(a + m) * (a + b + m) * x / ((a + 2 * m) * (a + 1 + 2 * m))
        d, c = 1 / (1 + k * d), 1 + k / c
        h *= d * c
        if m % 16 == 0 and bool(((d * c - 1).abs() < 4e-16).all()):
            break
    return h


def _t_tail(t, nu):
    """P(T <= -|t|) of Student's t with nu degrees of freedom."""
    t, nu = torch.broadcast_tensors(t, nu)
    out = torch.empty(t.shape, dtype=F64, device=t.device)
    o, tt, nn = out.view(-1), t.reshape(-1), nu.reshape(-1)
    for i in range(0, tt.numel(), 1 << 22):
        t2, v = tt[i:i + (1 << 22)] ** 2, nn[i:i + (1 << 22)]
        a, b = v / 2, torch.full_like(v, 0.5)
        x, y = v / (v + t2), t2 / (v + t2)
        left = x < (a + 1) / (a + b + 2)
        front = torch.lgamma(a + b) - torch.lgamma(a) - torch.lgamma(b) + a * torch.log(x) + b * torch.log(y)
        p, q = torch.where(left, a, b), torch.where(left, b, a)
        part = torch.exp(front) * _beta_fraction(p, q, torch.where(left, x, y)) / p
        o[i:i + (1 << 22)] = 0.5 * torch.where(left, part, 1 - part)
    return out


def _z_of_t(t, nu, table=None):
    """|z| with the normal tail of |t|'s Student tail; `table`: knots for one nu."""
    if table is None:
        return -torch.special.ndtri(_t_tail(t, nu))
    u = t.abs() / table[0]
    i = u.floor().clamp(1, table[1].numel() - 3).long()
    f = u - i
    a, b, c, d = (table[1][i + k] for k in (-1, 0, 1, 2))
    return (-f * (f - 1) * (f - 2) / 6 * a + (f + 1) * (f - 1) * (f - 2) / 2 * b - (f + 1) * f * (f - 2) / 2 * c
            + (f + 1) * f * (f - 1) / 6 * d)


def _z_table(nu, largest):
    h = 2.0 ** -11
    knots = torch.arange(int(largest / h) + 4, dtype=F64, device="cuda") * h
    return h, _z_of_t(knots, torch.full_like(knots, nu))


def _ols(x, y, member, cov, Q):
    """n [S] and x'x, x'y, residual squares, total squares [S][P] of one gene."""
    S, N = y.shape
    on = (member & ~torch.isnan(y)).double()
    n = on.sum(1)
    design = torch.cat([torch.ones((S, 1, N), dtype=F64, device="cuda"), cov[:, :Q]], 1) * on[:, None]
    low = torch.linalg.cholesky(torch.matmul(design, design.transpose(1, 2)))
    u = torch.linalg.solve_triangular(low, design, upper=False)
    y0 = torch.nan_to_num(y) * on
    yc = y0 - torch.matmul(torch.matmul(y0[:, None], u.transpose(1, 2).contiguous()), u)[:, 0]
    xm = on[:, :, None] * x[None]
    xc = xm - torch.matmul(u.transpose(1, 2).contiguous(), torch.matmul(u, xm))
    xx = (xc * xc).sum(1)
    beta = (xc * yc[:, :, None]).sum(1) / xx
    rss = ((yc[:, :, None] - beta[:, None] * xc) ** 2).sum(1)
    tss = (((y0 - (y0.sum(1) / n)[:, None]) * on) ** 2).sum(1)
    return n, xx, beta, rss, tss[:, None]


def _sstats(n, xx, beta, rss, tss, Q):
    nu = (n - 2 - Q)[:, None].expand_as(beta)
    sig = torch.sqrt(rss / nu)
    se = sig / torch.sqrt(xx)
    return sig, se, nu, 1 - rss / tss


def _standard(beta, sig, se, z):
    return torch.sign(beta) * z * se / sig, se / sig, -z


def _abf(b, se, t, phi, oma):
    """log10 ABF of the active subgroups given as rows (Wen and Stephens)."""
    v, keep = se * se, t.abs() >= 1e-8
    k = torch.where(keep, 1 / (v + phi), 0.0)
    one = torch.where(keep, 0.5 * torch.log10(v / (v + phi)) + 0.5 * t * t * phi * k / LN10, 0.0).sum(0)
    den = k.sum(0)
    bbar, var = (torch.where(keep, b, 0.0) * k).sum(0) / den, 1 / den
    q = bbar * bbar / var
    all_ = 0.5 * torch.log10(var / (var + oma)) + 0.5 * q * oma / (var + oma) / LN10
    return torch.where((den > 0) & (bbar != 0), all_ + one, 0.0)


def _weights(masks, S):
    return torch.tensor([1.0 / S / math.comb(S, bin(m).count("1")) for m in masks], dtype=F64, device="cuda")


def _bma(w, gen, bfs, S, n):
    nan = torch.full((n,), float("nan"), dtype=F64, device="cuda")
    if bfs == "gen":
        return [nan, nan]
    lite = _lws(torch.cat([w[:S], gen[None]]), torch.tensor([0.5 / S] * S + [0.5], dtype=F64, device="cuda"), 0)
    return [lite, _lws(w, _weights(_abi.config_masks(bfs, S), S), 0) if bfs == "all" else nan]


def _abfs(case, b, se, t, has=None):
    """raw [rows][n] and averaged [5 + configurations][n] Bayes factors."""
    S, n = b.shape
    large, small = _grids(case)
    masks = _abi.config_masks(case["bfs"], S)
    raw = torch.zeros((3 * len(large) + len(masks) * len(small), n), dtype=F64, device="cuda")
    if has is not None:  # a subgroup without results takes no part: |t| below 1e-8 drops it
        b, se, t = (torch.where(has, a, k) for a, k in ((b, 0.0), (se, 1.0), (t, 0.0)))
    L = len(large)
    for i, (phi, oma) in enumerate(large):
        raw[i] = _abf(b, se, t, phi, oma)
        raw[L + i] = _abf(b, se, t, 0.0, phi + oma)
        raw[2 * L + i] = _abf(b, se, t, phi + oma, 0.0)
    for c, m in enumerate(masks):
        on = [s for s in range(S) if (m >> s) & 1]
        for i, (phi, oma) in enumerate(small):
            raw[3 * L + c * len(small) + i] = _abf(b[on], se[on], t[on], phi, oma)
    return raw, _averaged(case, raw, S)


def _averaged(case, raw, S):
    (large, small), n = _grids(case), raw.shape[1]
    L, nc = len(large), _abi.n_configs(case["bfs"], S)
    w = [_lmean(raw[k * L:(k + 1) * L], 0) for k in range(3)]
    cfg = _lmean(raw[3 * L:].reshape(nc, len(small), n), 1) if nc else raw[:0]
    return torch.cat([torch.stack(w), cfg, torch.stack(_bma(cfg, w[0], case["bfs"], S, n))])


def _tiled(raw):
    """Rows laid out in tiles of 64 pairs."""
    rows, n = raw.shape
    full = n // 64 * 64
    a = raw[:, :full].reshape(rows, -1, 64).permute(1, 0, 2).reshape(-1)
    return torch.cat([a, raw[:, full:].reshape(-1)]).reshape(rows, n)


def _exact_uvlr(case, d):
    S, n, Q = d["S"], int(d["off"][-1]), d["Q"]
    num = torch.zeros((S, n), dtype=torch.int32, device="cuda")
    st = torch.zeros((5, S, n), dtype=F64, device="cuda")
    std = torch.zeros((3, S, n), dtype=F64, device="cuda")
    for g in range(d["G"]):
        at = slice(int(d["off"][g]), int(d["off"][g + 1]))
        got = _ols(d["x"][:, at].double(), d["y"][g], d["member"], d["cov"], Q)
        sig, se, nu, pve = _sstats(*got, Q)
        num[:, at] = got[0].to(torch.int32)[:, None]
        tail = _t_tail(got[2] / se, nu)
        for k, v in enumerate((pve, sig, got[2], se, 2 * tail)):
            st[k, :, at] = v
        for k, v in enumerate(_standard(got[2], sig, se, -torch.special.ndtri(tail))):
            std[k, :, at] = v
    out = dict(n=num)
    if case["stats"]:
        out["sstats"] = st
    if case["kind"] == "uvlr":
        if case["stats"]:
            out["std"] = std
        raw, out["w"] = _abfs(case, *std)
        out["raw"] = raw if case["stats"] else _tiled(raw)
    return out


def _exact_inss(case, seed):
    n, sig, beta, se = _inss_inputs(case, seed)
    std = _standard(beta, sig, se, _z_of_t(beta / se, (n - 2).double()))
    raw, w = _abfs(case, *std)
    return dict(n=n.to(torch.int32), std=torch.stack(std), raw=raw, w=w)


def _solve(m, rhs):
    """x of m x = rhs and log |det m| for a batch [...][k][k], by elimination with row exchanges."""
    a, k = torch.cat([m, rhs], -1), m.shape[-1]
    log = 0.0
    for j in range(k):
        p = a[..., j:, j].abs().argmax(-1, keepdim=True) + j
        i = p[..., None].expand(*p.shape, a.shape[-1])
        row, old = a.gather(-2, i), a[..., j:j + 1, :].clone()
        a.scatter_(-2, i, old)
        a[..., j:j + 1, :] = row
        log = log + torch.log(row[..., 0, j].abs())
        a = a - (a[..., :, j:j + 1] / row[..., :, j:j + 1]) * row * (torch.arange(k, device=a.device) != j)[:, None]
    x = a[..., k:] / torch.diagonal(a[..., :k], dim1=-2, dim2=-1)[..., None]
    return x, log


def _mvn_abfs(case, sigma, vinv, b, S):
    """Rows of configurations from effect covariance and error covariance per configuration [n][S][S]."""
    large, small = _grids(case)
    rows = []
    masks = [(1 << S) - 1] + _abi.config_masks(case["bfs"], S)
    for c, mask in enumerate(masks):
        on = torch.tensor([(mask >> s) & 1 for s in range(S)], dtype=F64, device="cuda")
        sg, vi, bv = sigma(on), *vinv(on)
        t = on * torch.sqrt(torch.diagonal(sg, dim1=-2, dim2=-1))
        grid = [(p, o) for p, o in small] if c else \
            [(p, o) for p, o in large] + [(0.0, p + o) for p, o in large] + [(p + o, 0.0) for p, o in large]
        for phi, oma in grid:
            w = oma * t[:, :, None] * t[:, None, :] + torch.diag_embed(phi * t * t)
            m = torch.matmul(vi, w) + torch.eye(S, dtype=F64, device="cuda")
            x, log = _solve(m, bv[..., None])
            quad = torch.matmul(torch.matmul(bv[:, None, :], w), x)[:, 0, 0]
            rows.append((0.5 * quad - 0.5 * log) / LN10)
    raw = torch.stack(rows)
    return raw, _averaged(case, raw, S)


def _exact_mvlr(case, d):
    S, N, Q, n = d["S"], d["N"], d["Q"], int(d["off"][-1])
    f, m = 0.5, Q + 1 + S + 1
    raws, ws = [], []
    design = torch.cat([torch.ones((1, N), dtype=F64, device="cuda"), d["cov"][0, :Q]])
    u = torch.linalg.solve_triangular(torch.linalg.cholesky(design @ design.T), design, upper=False)
    for g in range(d["G"]):
        x = d["x"][:, int(d["off"][g]):int(d["off"][g + 1])].double()
        x = x - u.T @ (u @ x)
        y = d["y"][g] - (d["y"][g] @ u.T) @ u
        null, k, b0 = y @ y.T, (x * x).sum(0), (y @ x).T.contiguous()
        sigma0 = null / N
        res = y[None] - (b0 / k[:, None])[:, :, None] * x.T[:, None, :]
        ss = (res * res).sum(-1) / (N - Q - 2)
        F = b0 * b0 / k[:, None] / ss ** 2
        z = _z_of_t(torch.sqrt(F), torch.full_like(F, N - Q - 2.0))
        fac = torch.where(F < 1e-8, 1.0, torch.sqrt(F) / z)

        def sigma(on):
            either = torch.maximum(on[:, None].expand(S, S), on[None, :].expand(S, S))
            e = null[None] - either * b0[:, :, None] * b0[:, None, :] / k[:, None, None]
            e = (e + 1e-4 * m * torch.eye(S, dtype=F64, device="cuda")) / (m + N)
            return f * e * torch.where(on > 0, fac, 1.0)[:, None, :] + (1 - f) * sigma0[None]

        def vinv(on):
            eye = torch.eye(S, dtype=F64, device="cuda").expand(len(k), S, S)
            inv = _solve(sigma(on), eye)[0]
            return k[:, None, None] * inv, torch.matmul(inv, b0[..., None])[..., 0]

        raw, w = _mvn_abfs(case, sigma, vinv, None, S)
        raws.append(raw)
        ws.append(w)
    return dict(n=torch.full((S, n), N, dtype=torch.int32, device="cuda"), raw=torch.cat(raws, 1), w=torch.cat(ws, 1))


def _exact_hybrid(case, d):
    S, N, Q = d["S"], d["N"], d["Q"]
    f = 0.5
    got = _exact_uvlr(dict(case, kind="sep", stats=True), d)
    raws, ws = [], []
    pairs = [(a, b) for a in range(S) for b in range(a + 1, S)]
    one = torch.tensor([a for a, _ in pairs], device="cuda")
    two = torch.tensor([b for _, b in pairs], device="cuda")

    def gram(mask, cov, x, extra=()):
        """[1, covariates, genotype] cross-products over the masked individuals, per row of mask and SNP."""
        c = torch.cat([torch.ones_like(mask)[:, None], cov], 1) * mask[:, None]
        cc, cx, xx = torch.matmul(c, c.transpose(1, 2).contiguous()), torch.matmul(c, x), mask @ (x * x)
        out = torch.empty((mask.shape[0], x.shape[1], Q + 2, Q + 2), dtype=F64, device="cuda")
        out[..., :Q + 1, :Q + 1] = cc[:, None]
        out[..., :Q + 1, Q + 1] = out[..., Q + 1, :Q + 1] = cx.transpose(1, 2)
        out[..., Q + 1, Q + 1] = xx
        return out, c

    def unit(k, like):
        e = torch.zeros(k, 1, dtype=F64, device="cuda")
        e[-1] = 1
        return e.expand(*like.shape[:-2], k, 1)

    for g in range(d["G"]):
        x = d["x"][:, int(d["off"][g]):int(d["off"][g + 1])].double()
        y = d["y"][g]
        on = (d["member"] & ~torch.isnan(y)).double()
        y = torch.nan_to_num(y)
        cov = d["cov"][:, :Q]

        def cross(mask, c, u, v, full):
            """u'v over the masked individuals after a fit on [1, covariates(, genotype)]."""
            a, cc = gram(mask, c, x)
            cu, cv = (torch.matmul(cc, t[..., None])[..., 0] for t in (u, v))
            if not full:
                s = _solve(a[:, :1, :Q + 1, :Q + 1], cv[:, None, :, None])[0][..., 0]
                return ((u * v * mask).sum(1)[:, None] - (s * cu[:, None]).sum(-1)).expand(-1, x.shape[1])
            r = lambda t, ct: torch.cat([ct[:, None].expand(-1, x.shape[1], -1), ((t * mask) @ x)[..., None]], -1)  # noqa: E731
            s = _solve(a, r(v, cv)[..., None])[0][..., 0]
            return (u * v * mask).sum(1)[:, None] - (s * r(u, cu)).sum(-1)

        n = on.sum(1)[:, None]
        a, _ = gram(on, cov, x)
        sd = (f * cross(on, cov, y, y, True) + (1 - f) * cross(on, cov, y, y, False)) / n
        vd = sd * _solve(a, unit(Q + 2, a))[0][..., -1, 0]
        both, c1 = on[one] * on[two], cov[one]
        s12 = (f * cross(both, c1, y[one], y[two], True) + (1 - f) * cross(both, c1, y[one], y[two], False))
        s12 = s12 / both.sum(1)[:, None]
        g12 = gram(both, c1, x)[0]
        l1 = _solve(gram(on[one], c1, x)[0], unit(Q + 2, g12))[0]
        l2 = _solve(gram(on[two], c1, x)[0], unit(Q + 2, g12))[0]
        v12 = s12 * (l1 * torch.matmul(g12, l2)).sum((-2, -1))
        P = x.shape[1]
        sig, vg = torch.zeros((P, S, S), dtype=F64, device="cuda"), torch.zeros((P, S, S), dtype=F64, device="cuda")
        i = torch.arange(S, device="cuda")
        sig[:, i, i], vg[:, i, i] = sd.T, vd.T
        sig[:, one, two], sig[:, two, one] = s12.T, s12.T
        vg[:, one, two], vg[:, two, one] = v12.T, v12.T
        beta = got["sstats"][2][:, int(d["off"][g]):int(d["off"][g + 1])].T.contiguous()
        inv = _solve(vg, torch.eye(S, dtype=F64, device="cuda").expand(P, S, S))[0]
        bv = torch.matmul(inv, beta[..., None])[..., 0]
        raw, w = _mvn_abfs(case, lambda on_: sig, lambda on_: (inv, bv), None, S)
        raws.append(raw)
        ws.append(w)
    return dict(n=got["n"], sstats=got["sstats"], raw=torch.cat(raws, 1), w=torch.cat(ws, 1))


def _exact_perm(case, seed):
    s = prepare(case, seed)
    d, S, Q = s["data"], s["data"]["S"], s["data"]["Q"]
    c = dict(case, bfs="all", grid=25)
    nu = d["N"] - 2.0
    table = _z_table(nu, 64.0) if not Q and not case["missing"] else None
    small, masks = _grids(c)[1], _abi.config_masks("all", S)
    wt = _weights(masks, S)

    def stat(b, se, t):
        cfg = torch.stack([_lmean(torch.stack([_abf(b[on], se[on], t[on], p, o) for p, o in small]), 0)
                           for on in ([k for k in range(S) if (m >> k) & 1] for m in masks)])
        return _lws(cfg, wt, 0)

    def reduce(v, dim):
        return v.amax(dim) if case["use_max"] else _lmean(v, dim)

    def gene(g, y):
        """[S][...][P] standardised statistics of the levels y [S][N]."""
        x = d["x"][:, int(d["off"][g]):int(d["off"][g + 1])].double()
        o = _ols(x, y, d["member"], d["cov"], Q)
        sig, se, nu_, _ = _sstats(*o, Q)
        return _standard(o[2], sig, se, _z_of_t(o[2] / se, nu_))

    out, true = torch.zeros_like(s["stats"]), torch.zeros_like(s["true"])
    for g in range(d["G"]):
        true[g] = reduce(stat(*gene(g, d["y"][g])), 0)
        idx = s["tables"][g].long()
        if table is None:
            for p0 in range(0, idx.shape[0], 64):
                rows = [gene(g, d["y"][g][:, i]) for i in idx[p0:p0 + 64]]
                b, se, t = (torch.stack([r[k] for r in rows], 1) for k in range(3))
                out[g, p0:p0 + len(rows)] = reduce(stat(b, se, t), -1)
            continue
        x = d["x"][:, int(d["off"][g]):int(d["off"][g + 1])].double()
        x = x - x.mean(0)
        y = d["y"][g] - d["y"][g].mean(1, keepdim=True)
        xx, yy = (x * x).sum(0), (y * y).sum(1)[:, None, None]
        for p0 in range(0, idx.shape[0], 1000):
            xy = torch.matmul(y[:, idx[p0:p0 + 1000]], x)
            beta = xy / xx
            sig = torch.sqrt((yy - beta * xy) / nu)
            se = sig / torch.sqrt(xx)
            z = _z_of_t(beta / se, None, table)
            out[g, p0:p0 + 1000] = reduce(stat(*_standard(beta, sig, se, z)), -1)
    return [out, true]


def _types_point(raw, sub):
    """[n][K][L] log10 products over the subgroups of the types model."""
    q = sub[None, :, :, None]
    return torch.log10(q * torch.exp(raw[:, None] * LN10) + 1 - q).sum(2)


def _exact_hm(case, seed):
    d = _raw_inputs(case, seed)
    raw, G, K, L, S, types = d["raw"], d["G"], d["K"], d["L"], d["S"], d["types"]
    P = torch.from_numpy(np.diff(d["off"])).cuda()
    gene = torch.repeat_interleave(torch.arange(G, device="cuda"), P)
    cuda = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731

    def over_snps(v):
        """log10 of the mean over each gene's SNPs of 10^v, columns of v."""
        i = gene[:, None].expand_as(v)
        m = torch.full((G, v.shape[1]), -math.inf, dtype=F64, device="cuda").scatter_reduce(0, i, v, "amax")
        s = torch.zeros((G, v.shape[1]), dtype=F64, device="cuda")
        for g in range(G):
            a, b = int(d["off"][g]), int(d["off"][g + 1])
            s[g] = torch.exp((v[a:b] - m[g]) * LN10).sum(0)
        return m + torch.log10(s / P[:, None])

    def step(pi0, grid, dim, sub):
        t = _types_point(raw, sub) if types else raw
        cfg = _lws(t, grid, 2)
        snp = over_snps(_lws(cfg, dim, 1)[:, None])[:, 0]
        lik = torch.log10(pi0 + (1 - pi0) * torch.exp(snp * LN10))
        new = lambda v, old: torch.log10(torch.exp((over_snps(v) - lik[:, None]) * LN10).sum(0)) + torch.log10(old)  # noqa: E731
        share = lambda l: torch.exp((l - l.amax()) * LN10) / torch.exp((l - l.amax()) * LN10).sum()  # noqa: E731
        nsub = None
        if types:
            part = torch.log10(sub[None, :, :, None] * torch.exp(raw[:, None] * LN10) + 1 - sub[None, :, :, None])
            num = _lws((raw[:, None] + part.sum(2, keepdim=True) - part).reshape(-1, K * S, L), grid, 2)
            top, low = new(num, torch.ones(K * S, dtype=F64, device="cuda")).reshape(K, S), new(cfg, torch.ones_like(dim))
            nsub = torch.exp((top - low[:, None]) * LN10) * sub
        return float(lik.sum()), float((pi0 / torch.exp(lik * LN10)).mean()), share(new(_lws(t, dim, 1), grid)), \
            share(new(cfg, dim)), nsub

    p = [0.5, cuda(d["w"]["grid"]), cuda(d["w"]["dim"]), cuda(d["w"]["sub"]) if types else None]
    lik, *nxt = step(*p)
    it = 0
    while True:
        it += 1
        old, p = lik, nxt
        lik, *nxt = step(*p)
        if abs(lik - old) < 1e-300 or it == case["iters"] - 1:
            break
    p = nxt
    lik = step(*p)[0]
    return [p[0], p[1], p[2], p[3], lik, None]


def _exact_avg(case, seed):
    d = _raw_inputs(case, seed)
    raw, G, K, L, S, types = d["raw"], d["G"], d["K"], d["L"], d["S"], d["types"]
    cuda = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    ten = lambda v: torch.exp(v * LN10)  # noqa: E731
    grid, dim = cuda(d["w"]["grid"]), cuda(d["w"]["dim"])
    sub = cuda(d["w"]["sub"]) if types else None
    dims = _lws(_types_point(raw, sub) if types else raw, grid, 2)
    snp = _lws(dims, dim, 1)
    gene_bf, gene_post, the, an = [], [], [], []
    for g in range(G):
        v = snp[int(d["off"][g]):int(d["off"][g + 1])]
        m = len(v)
        bf = _lmean(v, 0)
        gene_bf.append(bf)
        gene_post.append(1 / (1 + 0.6 / 0.4 * ten(-bf)))
        e = ten(v - v.max())
        the.append(e / e.sum())
        an.append(1 / (1 + (m - 1) * ten(-v)))
    post = dim * ten(dims - snp[:, None])
    if types:
        part = torch.log10(sub[None, :, :, None] * ten(raw[:, None]) + 1 - sub[None, :, :, None])
        num = _lws((raw[:, None] + part.sum(2, keepdim=True) - part).reshape(-1, K * S, L), grid, 2).reshape(-1, K, S)
        psub = (dim[:, None] * sub * ten(num - snp[:, None, None])).sum(1)
    else:
        bits = torch.tensor([[float((m >> s) & 1) for s in range(S)] for m in _abi.config_masks("all", S)],
                            dtype=F64, device="cuda")
        psub = post @ bits
    return dict(gene_bf=torch.stack(gene_bf), gene_post=torch.stack(gene_post), snp_bf=snp, dim_bf=dims,
                post_the=torch.cat(the), post_an=torch.cat(an), post_dim=post, post_sub=psub.clamp(max=1.0),
                best_dim=None)


def _exact_alloc(case, seed):
    s = prepare(case, seed)
    d = s["data"]
    eig = []
    for g in range(d["G"]):
        x = d["x"][:, int(d["off"][g]):int(d["off"][g + 1])].double()
        x = x - x.mean(0)
        x = x / torch.sqrt((x * x).sum(0))
        eig.append(torch.linalg.eigvalsh((x @ x.T).cpu()).flip(0)[:20].clamp(min=0))
    p = torch.from_numpy(s["net"].get_params())
    sizes, at, pars = [(256, 24), (256, 256), (256, 256), (3, 256)], 0, []
    for o, i in sizes:  # the weights are used as bfloat16, the biases as they are
        w = p[at:at + o * i].reshape(o, i).bfloat16().double()
        pars += [w.requires_grad_(), p[at + o * i:at + o * i + o].double().requires_grad_()]
        at += o * i + o
    h = torch.from_numpy(s["x"]).double()
    for k in range(4):
        h = torch.nn.functional.linear(h, pars[2 * k], pars[2 * k + 1])
        h = torch.nn.functional.gelu(h) if k < 3 else h
    loss = ((h - torch.from_numpy(s["t"]).double()) ** 2).sum() / h.shape[0]
    loss.backward()
    k = d["N"] - 1
    eig = torch.stack(eig)
    rank = torch.from_numpy(np.minimum(d["P"], k))[:, None] > torch.arange(20)[None]
    return [torch.where(rank, eig, 0.0), float(loss.detach()), torch.cat([q.grad.reshape(-1) for q in pars]),
            h.detach()]


def exact(case, seed):
    kind = case["kind"]
    if kind == "inss":
        return _exact_inss(case, seed)
    if kind == "perm":
        return _exact_perm(case, seed)
    if kind == "hm":
        return _exact_hm(case, seed)
    if kind == "avg":
        return _exact_avg(case, seed)
    if kind == "alloc":
        return _exact_alloc(case, seed)
    d = _genes(case, seed)
    return {"uvlr": _exact_uvlr, "sep": _exact_uvlr, "mvlr": _exact_mvlr, "hybrid": _exact_hybrid}[kind](case, d)


def tolerance(case):
    """About four times what the paths are off `exact`, or off themselves with sums in another order."""
    kind = case["kind"]
    if kind == "uvlr":  # Bayes-factor terms in 32 bits over sums that are exact or in 64
        return {"rel": 4e-6, "max": 1e-3}
    if kind == "perm":
        return {"rel": 3e-6, "max": 1e-4}
    if kind == "sep":  # 64 bits; the tabulated Student tail behind the p-values
        return {"rel": 1e-10}
    if kind in ("mvlr", "hybrid"):
        return {"rel": 3e-10, "max": 1e-7}
    if kind == "inss":
        return {"rel": 1e-12}
    if kind in ("hm", "avg"):  # 64 bits throughout; ties of the best configuration
        return {"rel": 1e-12, "differ": 1e-5}
    return {"rel": 4e-3}  # eigenvalues by iteration to a thousandth; the network's weights are bfloat16
