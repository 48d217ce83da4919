"""GPU contraction path for permutations (every sample in every subgroup,
hard-call genotypes, no covariates) against the CPU oracle.

The index tables come from the library's GSL-semantics generator; both sides
evaluate the same tables.  Tolerances (mixed precision): 1e-4 absolute on
each permutation's log10 BF statistic, 1e-6 relative on the sep p-value
statistics.  With the FP64 true statistics and the FP64 re-check of every
permutation statistic within 5e-5 of them (eqbf_perm_stats_fp64_ties) the
reference's counting loop gives the oracle's counts exactly.  Each test also checks from the live
kernel timing which path ran: the contraction kernels (pf_*) or the general
per-permutation path (perm_gather_kernel).
"""
import sys

import numpy as np
import pytest

from eqtlbma_amd import engine, synth

pytestmark = pytest.mark.gpu

GL25 = synth.make_grid("general")
GS10 = synth.make_grid("small")


@pytest.fixture(scope="module")
def eng():
    e = engine.Engine(0)
    e.set_grids(GL25, GS10)
    yield e
    e.close()


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _run(eng, hc, tables, gene_table, analysis, pbf, use_max, sbgrp=-1):
    """Statistics and the kernels launched by this call (the context's
    timing totals are cumulative)."""
    eng.profile(True)
    before = eng.profile_read()
    gpu = eng.perm_stats(hc, tables, gene_table, analysis, pbf, use_max, sep_sbgrp=sbgrp, precision="mixed")
    after = eng.profile_read()
    eng.profile(False)
    ran = {k for k, v in after.items() if v[1] > before.get(k, (0.0, 0))[1]}
    return gpu, ran


def _oracle(orc, hc, tables, gene_table, analysis, pbf, use_max, sbgrp=-1):
    out = np.full((hc.G, tables.shape[1]), np.nan)
    for g in range(hc.G):
        if gene_table[g] < 0:
            continue
        t = tables[gene_table[g]]
        if analysis == "join":
            out[g] = orc.perm_join_stats(hc, g, pbf, use_max, GL25, GS10, t)
        else:
            out[g] = orc.perm_sep_stats(hc, g, sbgrp, t)
    return out


def _check(gpu, ref, analysis):
    assert np.array_equal(np.isnan(gpu), np.isnan(ref))
    fin = np.isfinite(ref)
    if analysis == "join":
        err = np.max(np.abs(gpu[fin] - ref[fin]), initial=0)
        _say("[gpu]   max |stat - oracle| = %.3g" % err)
        assert err <= 1e-4
    else:
        assert np.allclose(gpu[fin], ref[fin], rtol=1e-6, atol=1e-300)


def _true_w_row(pbf, S):
    n_cfg = {"all": 2 ** S - 1, "gen-sin": S, "gen": 0}[pbf]
    return {"all": 3 + n_cfg + 1, "gen-sin": 3 + n_cfg, "gen": 0}[pbf], {"all": "all", "gen-sin": "sin",
                                                                           "gen": "gen"}[pbf]


@pytest.mark.parametrize("pbf", ["all", "gen", "gen-sin"])
@pytest.mark.parametrize("use_max", [True, False])
def test_join_contraction_matches_oracle(eng, orc, pbf, use_max):
    # the permutation workload's shape at small size: 5 subgroups sharing
    # N = 300 individuals, hard calls, 101 permutations (partial blocks)
    hc = synth.plain(seed=1002, S=5, N=300, n_genes=3, snps_per_gene=40, frac_egenes=0.34)
    nperm = 101
    tables = engine.Rng(7).tables(hc.N, 3, nperm)
    gene_table = np.array([0, 1, 2], np.int32)
    _say("[gpu] contraction join pbf=%s max=%s" % (pbf, use_max))
    gpu, prof = _run(eng, hc, tables, gene_table, "join", pbf, use_max)
    assert "pf_gemm_kernel" in prof and "pf_bma_kernel" in prof
    assert "perm_gather_kernel" not in prof
    ref = _oracle(orc, hc, tables, gene_table, "join", pbf, use_max)
    _check(gpu, ref, "join")
    row, bfs = _true_w_row(pbf, hc.S)
    true = orc.assoc_uvlr(hc, "join", bfs, GL25, GS10)
    a_gpu = eng.assoc_uvlr(hc, "join", bfs, precision="mixed")
    t_in = np.array([orc.true_stat(a_gpu.w[row, hc.pair_offset[g]:hc.pair_offset[g + 1]], use_max)
                     for g in range(hc.G)])
    chk, true_gpu, n_re = eng.perm_stats_fp64_ties(hc, tables, gene_table, t_in, "join", pbf, use_max,
                                                   precision="mixed")
    _check(chk, ref, "join")
    near_total = 0
    for g in range(hc.G):
        w = true.w[row, hc.pair_offset[g]:hc.pair_offset[g + 1]]
        t = orc.true_stat(w, use_max)
        near = int(np.sum(np.abs(gpu[g] - t_in[g]) <= 5e-5))
        near_total += near
        assert abs(true_gpu[g] - t) <= (1e-9 if near else 1e-4), (g, true_gpu[g], t)
        a = engine.perm_pvalue(chk[g], true_gpu[g], nperm)
        b = orc.perm_count(ref[g], t, nperm)
        assert a[0] == b[0] and a[1] == b[1], (g, a, b)
    assert n_re == near_total
    _say("[gpu]   near-ties re-checked in FP64: %d" % n_re)


def test_mixed_eligibility_splits_the_genes(eng, orc):
    hc = synth.plain(seed=31, S=3, N=60, n_genes=4, snps_per_gene=15, frac_egenes=0.5)
    hc.explevels[1, 2, 5] = np.nan              # gene 1: a missing value, membership moves
    j = hc.pair_snp[hc.pair_offset[3]]
    hc.genotypes[0, 7, j] += 0.25                # gene 3: a dosage, not a hard call
    nperm = 40
    tables = engine.Rng(11).tables(hc.N, 4, nperm)
    gene_table = np.array([0, 1, 2, 3], np.int32)
    _say("[gpu] contraction + general path in one chunk")
    gpu, prof = _run(eng, hc, tables, gene_table, "join", "all", True)
    assert "pf_gemm_kernel" in prof and "perm_gather_kernel" in prof
    ref = _oracle(orc, hc, tables, gene_table, "join", "all", True)
    _check(gpu, ref, "join")


def _edge_case_chunk():
    hc = synth.plain(seed=5, S=3, N=50, n_genes=2, snps_per_gene=10, frac_egenes=0.0)
    hc.genotypes[0, :, 0] = 1.0                  # first SNP of gene 0: monomorphic
    x = hc.genotypes[0, :, 1].astype(np.float64)
    xc = x - x.mean()
    y = hc.explevels[0, 1].copy()
    y -= (xc @ (y - y.mean())) / (xc @ xc) * xc  # gene 0, subgroup 1: y orthogonal to SNP 1
    hc.explevels[0, 1] = y
    tables = engine.Rng(3).tables(hc.N, 2, 40)
    tables[0, 0] = np.arange(hc.N)               # identity permutations: t = 0 for that pair
    tables[0, 9] = np.arange(hc.N)
    return hc, tables


@pytest.mark.parametrize("pbf", ["all", "gen", "gen-sin"])
def test_join_zero_z_and_monomorphic_snp(eng, orc, pbf):
    hc, tables = _edge_case_chunk()
    gene_table = np.array([0, 1], np.int32)
    _say("[gpu] contraction join edge cases pbf=%s" % pbf)
    gpu, prof = _run(eng, hc, tables, gene_table, "join", pbf, True)
    assert "pf_gemm_kernel" in prof and "perm_gather_kernel" not in prof
    ref = _oracle(orc, hc, tables, gene_table, "join", pbf, True)
    _check(gpu, ref, "join")


@pytest.mark.parametrize("sbgrp", [-1, 0, 2])
def test_sep_contraction_matches_oracle(eng, orc, sbgrp):
    hc = synth.plain(seed=77, S=5, N=120, n_genes=3, snps_per_gene=30, frac_egenes=0.34)
    nperm = 70
    tables = engine.Rng(5).tables(hc.N, 3, nperm)
    gene_table = np.array([0, -1, 1], np.int32)
    _say("[gpu] contraction sep sbgrp=%d" % sbgrp)
    gpu, prof = _run(eng, hc, tables, gene_table, "sep", "gen", True, sbgrp)
    assert "pf_gemm_kernel" in prof and "perm_gather_kernel" not in prof
    ref = _oracle(orc, hc, tables, gene_table, "sep", "gen", True, sbgrp)
    _check(gpu, ref, "sep")
    assert np.all(np.isnan(gpu[1]))


@pytest.mark.parametrize("sbgrp", [-1, 0])
def test_sep_monomorphic_first_snp(eng, orc, sbgrp):
    # std::min_element: with --permsep 2 a NaN first p-value makes the
    # statistic NaN; with --permsep 1 the minimum starts at 1
    hc, tables = _edge_case_chunk()
    gene_table = np.array([0, 1], np.int32)
    _say("[gpu] contraction sep monomorphic first SNP sbgrp=%d" % sbgrp)
    gpu, prof = _run(eng, hc, tables, gene_table, "sep", "gen", True, sbgrp)
    ref = _oracle(orc, hc, tables, gene_table, "sep", "gen", True, sbgrp)
    _check(gpu, ref, "sep")
    assert np.all(np.isnan(gpu[0])) == (sbgrp >= 0)


def test_perfect_fit_falls_back_to_general_path(eng, orc):
    hc = synth.plain(seed=9, S=2, N=40, n_genes=2, snps_per_gene=8, frac_egenes=0.0)
    x = hc.genotypes[0, :, 3].astype(np.float64)
    hc.explevels[0, 0] = 2.0 + 0.5 * x           # gene 0, subgroup 0: y on SNP 3 exactly
    tables = engine.Rng(13).tables(hc.N, 2, 30)
    tables[0, 4] = np.arange(hc.N)
    gene_table = np.array([0, 1], np.int32)
    _say("[gpu] contraction fallback on a perfect fit")
    gpu, prof = _run(eng, hc, tables, gene_table, "join", "all", True)
    assert "pf_gemm_kernel" in prof and "perm_gather_kernel" in prof
    ref = _oracle(orc, hc, tables, gene_table, "join", "all", True)
    # the perfect fit itself (permutation 4 of gene 0) has a residual sum of
    # squares that is rounding noise in the reference's SVD as in any FP64
    # restatement, so its statistic is not compared (parity unpinned)
    keep = np.ones_like(ref, dtype=bool)
    keep[0, 4] = False
    _check(gpu[keep], ref[keep], "join")


@pytest.mark.parametrize("S,N,P,nperm,wide", [
    (1, 5, 1, 1, False),       # one wave with a tile, seven without; one permutation
    (2, 63, 31, 15, False),    # one sample short of a step; a partial tile pair
    (3, 64, 33, 16, False),    # whole steps; a second pair of one SNP
    (4, 65, 300, 17, False),   # a second step of one sample; more tiles than waves
    (5, 512, 70, 33, False),
    (6, 300, 40, 20, False),
    (1, 100, 223, 17, False),  # the last size of the two kernels and the first of the one
    (1, 100, 224, 17, False),
    (3, 64, 255, 33, False),   # eight tile pairs, one SNP less, one more
    (2, 63, 256, 16, False),
    (3, 64, 257, 17, False),
    (5, 320, 127, 20, False),  # the line at four subgroups and more
    (5, 320, 128, 20, False),  # the most samples that fit at each number of subgroups
    (6, 256, 161, 15, False),
    (6, 256, 159, 15, False),
    (4, 448, 130, 18, False),
    (3, 512, 230, 20, False),
    (3, 513, 230, 20, False),  # one step more than the fused kernel holds
    (4, 449, 130, 18, False),  # fragments that do not fit
    (3, 513, 40, 20, False),
    (3, 64, 40, 20, True),     # a genotype too large for its 32-bit digit pairs
    (3, 64, 230, 20, True),
])
def test_max_over_all_configurations_at_tile_edges(eng, orc, S, N, P, nperm, wide):
    # the statistic is the exact one of the SNP with the maximum whichever
    # kernel takes it, so the tolerance is that of the z and FP32 sums
    hc = synth.plain(seed=41 + S, S=S, N=N, n_genes=2, snps_per_gene=P, frac_egenes=0.5)
    if P > 31:
        hc.genotypes[0, :, hc.pair_snp[hc.pair_offset[1] + 30]] = 2.0  # not estimable
    if wide:
        hc.genotypes[0, :, hc.pair_snp[hc.pair_offset[1] + 3]] *= 20.0
    tables = engine.Rng(5).tables(hc.N, 2, nperm)
    gene_table = np.array([0, 1], np.int32)
    _say("[gpu] fused maximum S=%d N=%d P=%d nperm=%d wide=%d" % (S, N, P, nperm, wide))
    gpu, prof = _run(eng, hc, tables, gene_table, "join", "all", True)
    if N > 5:  # with few samples a perfect fit may move a gene to the general path
        fits = N <= {4: 448, 5: 320, 6: 256}.get(S, 512)
        one = not wide and fits and P >= (224 if S <= 3 else 128 if S <= 5 else 160)
        assert ("pf_max_kernel" if one else "pf_gemm_kernel") in prof and "perm_gather_kernel" not in prof
    _check(gpu, _oracle(orc, hc, tables, gene_table, "join", "all", True), "join")


def _linked_chunk(S, block, changed, n_genes=2, N=100, P=300):
    """Genes of P SNPs in linkage blocks: the SNPs of a block are one SNP with a
    share of its calls drawn anew."""
    hc = synth.plain(seed=90 + S, S=S, N=N, n_genes=n_genes, snps_per_gene=P, frac_egenes=0.0)
    rng = np.random.default_rng(17)
    for g in range(n_genes):
        o = hc.pair_offset[g]
        for b in range(0, P, block):
            for j in range(b + 1, min(b + block, P)):
                x = hc.genotypes[0, :, o + b].copy()
                new = rng.random(N) < changed
                x[new] = rng.integers(0, 3, int(new.sum()))
                hc.genotypes[0, :, o + j] = x
    return hc


@pytest.mark.parametrize("S", [1, 3, 5])
@pytest.mark.parametrize("block", [32, 300])
@pytest.mark.parametrize("changed", [0.0, 0.02, 0.1])
def test_max_over_linked_snps(eng, orc, S, block, changed):
    # where SNPs are linked most of them pass the bounds, so that the queues of
    # candidates fill as fast as they can; identical ones are one SNP, whose maxima
    # may lie below its statistic of z = 0
    hc = _linked_chunk(S, block, changed)
    nperm = 100
    tables = engine.Rng(5).tables(hc.N, 2, nperm)
    gene_table = np.array([0, 1], np.int32)
    _say("[gpu] maximum over linked SNPs S=%d block=%d changed=%g" % (S, block, changed))
    gpu, prof = _run(eng, hc, tables, gene_table, "join", "all", True)
    assert "pf_max_kernel" in prof and "perm_gather_kernel" not in prof
    _check(gpu, _oracle(orc, hc, tables, gene_table, "join", "all", True), "join")


@pytest.mark.parametrize("S", [1, 2, 5])
@pytest.mark.parametrize("P", [1, 2, 3, 5])
def test_max_over_few_snps(eng, orc, S, P):
    # a gene of few SNPs has maxima around and below the statistic of z = 0
    hc = synth.plain(seed=60 + 7 * S + P, S=S, N=100, n_genes=4, snps_per_gene=P, frac_egenes=0.0)
    nperm = 200
    tables = engine.Rng(5).tables(hc.N, 4, nperm)
    gene_table = np.arange(4, dtype=np.int32)
    _say("[gpu] maximum over few SNPs S=%d P=%d" % (S, P))
    gpu, prof = _run(eng, hc, tables, gene_table, "join", "all", True)
    assert "pf_gemm_kernel" in prof and "perm_gather_kernel" not in prof
    _check(gpu, _oracle(orc, hc, tables, gene_table, "join", "all", True), "join")


@pytest.mark.parametrize("pbf,use_max", [("all", True), ("all", False), ("gen", True), ("gen-sin", True)])
@pytest.mark.parametrize("P", [12, 240])  # with the maximum of "all": two kernels, one kernel
def test_constant_subgroup_takes_the_general_path(eng, orc, pbf, use_max, P):
    # a subgroup where the gene is not expressed, all zeros: its residual sum of
    # squares is 0 and no statistic of it has a closed form
    hc = synth.plain(seed=23, S=3, N=60, n_genes=3, snps_per_gene=P, frac_egenes=0.34)
    hc.explevels[1, 2] = 0.0
    nperm = 24
    tables = engine.Rng(5).tables(hc.N, 3, nperm)
    gene_table = np.arange(3, dtype=np.int32)
    _say("[gpu] constant subgroup pbf=%s max=%s P=%d" % (pbf, use_max, P))
    gpu, prof = _run(eng, hc, tables, gene_table, "join", pbf, use_max)
    one = pbf == "all" and use_max and P >= 224
    assert ("pf_max_kernel" if one else "pf_gemm_kernel") in prof and "perm_gather_kernel" in prof
    _check(gpu, _oracle(orc, hc, tables, gene_table, "join", pbf, use_max), "join")


@pytest.mark.parametrize("n_small,nperm", [(3, 50), (42, 800)])  # with the large genes, apart from them
def test_genes_of_few_and_of_many_snps_in_one_chunk(eng, orc, n_small, nperm):
    # apart, the genes are taken in another order than the chunk's, in two batches
    sizes = [(3, 1, 4)[k % 3] for k in range(n_small)] + [40]
    sizes[1:1], sizes[3:3] = [230], [224]
    hc = synth.plain(seed=71, S=2, N=60, n_genes=len(sizes), snps_per_gene=230, frac_egenes=0.34)
    hc.pair_snp = np.concatenate([np.arange(g * 230, g * 230 + n) for g, n in enumerate(sizes)]).astype(np.int32)
    hc.pair_offset = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    tables = engine.Rng(5).tables(hc.N, len(sizes) - 1, nperm)
    gene_table = np.arange(len(sizes), dtype=np.int32) - 1
    gene_table[0], gene_table[2] = 1, -1
    _say("[gpu] %d genes of few SNPs, 2 of many" % n_small)
    gpu, prof = _run(eng, hc, tables, gene_table, "join", "all", True)
    assert "pf_max_kernel" in prof and "perm_gather_kernel" not in prof
    assert ("pf_gemm_kernel" in prof) == (n_small == 42)
    assert np.all(np.isnan(gpu[2]))
    _check(gpu, _oracle(orc, hc, tables, gene_table, "join", "all", True), "join")


@pytest.mark.parametrize("pbf,use_max", [("all", True), ("all", False), ("gen", True)])
def test_statistics_against_64_bits(eng, pbf, use_max):
    # z in FP32 with a relative error of 5e-8 rms (rounding of R, of R^2 and of the
    # polynomial) moves a log10 BF by z^2 / ln 10 times that: with sum z^2 of 15 to
    # 25 at the maximum and five subgroups' errors apart, 1.5e-7 to 2.2e-7 rms, and
    # 1e-7 more in quadrature from the sums of FP32 terms.  An error common to every
    # z of the gene, as of a rounded leading coefficient (5e-8 at this N), would add
    # up over the subgroups: 3.8e-7.
    hc = synth.plain(seed=335, S=5, N=300, n_genes=4, snps_per_gene=200, frac_egenes=0.0)
    tables = engine.Rng(3).tables(hc.N, 4, 400)
    gene_table = np.arange(4, dtype=np.int32)
    _say("[gpu] statistics against 64 bits pbf=%s max=%s" % (pbf, use_max))
    gpu, prof = _run(eng, hc, tables, gene_table, "join", pbf, use_max)
    assert "perm_gather_kernel" not in prof
    ref = eng.perm_stats(hc, tables, gene_table, "join", pbf, use_max, precision="fp64_batched")
    rms = float(np.sqrt(np.mean((gpu - ref) ** 2)))
    _say("[gpu]   rms %.3g" % rms)
    assert rms <= 2.6e-7
