/*
 * Multivariate (MVLR) Bayes factors, --error mvlr, in FP64.
 *
 * Reference: GeneSnpPair::CalcAbfsMvlr and CalcAbfsMvlrFor*
 * (gene_snp_pair.cpp:624-758) over class MVLR (MVLR.cpp:26-764) with one
 * SNP per pair.  With T the projection off [1, covariates of the first
 * subgroup], x~ = T x, y~_s = T y_s, k = x~'x~ and b_s = y~_s'x~:
 *   Sigma0 = Y~'Y~ / n                      (compute_Sigma_null :176-195, m = q+s+1)
 *   residual of y_s on [Xc, x] (gamma_s = 1) or on Xc (gamma_s = 0):
 *     (E'E)_ij = (Y~'Y~)_ij - [gamma_i or gamma_j] b_i b_j / k
 *   F -> chi-square factor for gamma_s = 1 (compute_residual :366-410):
 *     T2 = (b_s^2/k) / sigma1^2 with sigma1 = rss_s/(n-q-1) (the reference
 *     divides by the square of a variance), F = T2,
 *     factor = F / chisq_Qinv(fdist_Q(F; 1, n-q-1); 1)
 *            = T2 / Phi^-1(P(T_{n-q-1} <= -sqrt T2))^2  (1 when F < 1e-8,
 *              0 when the F tail probability underflows in FP64)
 *   Sigma = fiterr [ (H m/(m+n) + E'E/(m+n)) C ] + (1 - fiterr) Sigma0,
 *     C = diag(sqrt(factor)), H = 1e-4 I (Sigma C, not C Sigma C: :268-273)
 *   eVb = Sigma^-1 b, t = gamma o sqrt(diag Sigma), W = oma2 t t' + phi2 diag(t^2),
 *   M = I + k Sigma^-1 W,  log10 ABF = (eVb' W M^-1 eVb - ln|det M|) / (2 ln 10)
 *                                                    (:497-512, :559-605)
 * so no n x n matrix is ever formed.  M is factorised with partial pivoting
 * (as gsl_linalg_LU_decomp); ln|det M| is summed from the pivots and
 * M^-1 eVb comes from one solve instead of an explicit inverse.
 *
 * Kernels (one chunk):
 *   mvlr_prep_kernel   one workgroup per gene: common members, basis of
 *                      [1, covariates], y~_s, Y~'Y~, Sigma0 and Sigma0^-1
 *   mvlr_sums_kernel   one wave per 16 pairs: k and b (FP64 sums over members)
 *   mvlr_cfg_kernel    one thread per (pair, configuration): Sigma, Sigma^-1,
 *                      Sigma^-1 t, t, eVb (structure-of-arrays, coalesced)
 *   mvlr_hess_kernel, mvlr_rows_kernel  2 to 10 subgroups: a Hessenberg form per
 *                      (pair, configuration), then log10 ABFs by elimination
 *   mvlr_grid_kernel   the others, one thread per (pair, raw row): M, LU, log10 ABF
 *   mvlr_wavg_kernel   one thread per (pair, weighted row): grid average
 *                      (utils::log10_weighted_sum)
 * followed by the BMA kernel of the univariate path (gen-sin, all).
 */
#include <algorithm>
#include <type_traits>
#include <cstring>
#include <vector>

#include "eqbf_internal.h"

namespace {

enum { MV_OK = 0, MV_SKIP = 1, MV_MISMATCH = 2, MV_FEW = 3 };
struct MvRec {
  int32_t n, flags, qcov, rank;
};

__device__ inline double wsum64(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

/* LU factorisation with partial pivoting of an SM x SM register matrix
 * (largest |a| of the column, first one on ties).  piv[j] = row swapped
 * with j at step j.  Returns ln|det A|. */
template <int SM>
__device__ inline double lu_factor(double (&A)[SM][SM], int (&piv)[SM]) {
  double lnd = 0.0;
#pragma unroll
  for (int j = 0; j < SM; ++j) {
    int p = j;
    double best = fabs(A[j][j]);
#pragma unroll
    for (int i = j + 1; i < SM; ++i)
      if (fabs(A[i][j]) > best) {
        best = fabs(A[i][j]);
        p = i;
      }
    piv[j] = p;
#pragma unroll
    for (int i = j + 1; i < SM; ++i) {
      const bool sw = p == i;
#pragma unroll
      for (int c = 0; c < SM; ++c) {
        const double a = A[j][c], b = A[i][c];
        A[j][c] = sw ? b : a;
        A[i][c] = sw ? a : b;
      }
    }
    const double d = A[j][j];
    lnd += log(fabs(d));
#pragma unroll
    for (int i = j + 1; i < SM; ++i) {
      const double f = A[i][j] / d;
      A[i][j] = f;
#pragma unroll
      for (int c = j + 1; c < SM; ++c) A[i][c] -= f * A[j][c];
    }
  }
  return lnd;
}

/* Solves A x = rhs in place from the factorisation of lu_factor. */
template <int SM>
__device__ inline void lu_apply(const double (&A)[SM][SM], const int (&piv)[SM], double (&x)[SM]) {
#pragma unroll
  for (int j = 0; j < SM; ++j) {
#pragma unroll
    for (int i = j + 1; i < SM; ++i) {
      const bool sw = piv[j] == i;
      const double a = x[j], b = x[i];
      x[j] = sw ? b : a;
      x[i] = sw ? a : b;
    }
  }
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int c = 0; c < i; ++c) x[i] -= A[i][c] * x[c];
#pragma unroll
  for (int i = SM - 1; i >= 0; --i) {
    double s = x[i];
#pragma unroll
    for (int c = i + 1; c < SM; ++c) s -= A[i][c] * x[c];
    x[i] = s / A[i][i];
  }
}

__global__ void mv_zero_kernel(int* p) { *p = 0; }

/* ---- per-gene preparation ------------------------------------------ */
struct MvPrep {
  MvRec* mrec;
  int32_t* midx; /* [G][N] member sample indices            */
  double* Ut;    /* [G][KU][N] orthonormal basis columns     */
  double* Yt;    /* [G][S][N] y~_s over the members          */
  double* YtY;   /* [G][S][S]                                */
  double* S0;    /* [G][S][S] Sigma0                         */
  double* S0inv; /* [G][S][S]                                */
  int* flag;
  int KU;
};

/* Up to eight waves a gene: the first finds the members and the basis, then they
 * share the subgroups and the entries of Y~'Y~.  Bound by the chain of wave sums; 120
 * genes, 9 subgroups of 150, no covariates: 77 us (119 us with one wave).  The
 * registers allow 2,048 waves at a time on the chip, and a wave that waits for the
 * first one's part holds its own, so many genes take fewer waves each: 2,000 genes
 * took 0.59 ms with eight, 0.20 ms with one. */
constexpr int MV_PREP_WAVES = 8;

inline int mv_prep_waves(int G) { return std::max(1, std::min(MV_PREP_WAVES, 2048 / std::max(G, 1))); }

template <int SM>
__global__ void __launch_bounds__(64 * MV_PREP_WAVES) mvlr_prep_kernel(const eqbf_chunk c, const MvPrep pp) {
  __shared__ uint32_t s_kept;
  const int nwv = blockDim.x >> 6;
  const int S = c.n_subgroups, N = c.n_samples, g = blockIdx.x;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KU = pp.KU;
  MvRec r;
  r.n = 0;
  r.flags = MV_OK;
  r.qcov = min(max(c.covar_count[0], 0), c.n_covars_max);
  r.rank = 0;
  for (int s = 0; s < S; ++s)
    if (!c.gene_in_sbgrp[(int64_t)g * S + s]) r.flags = MV_SKIP;
  if (r.flags != MV_OK) {
    if (threadIdx.x == 0) pp.mrec[g] = r;
    return;
  }
  /* members of subgroup 0 (expression level not NaN, genotyped); every other
   * subgroup must have the same ones */
  int32_t* idx = pp.midx + (int64_t)g * N;
  int n = 0;
  bool mismatch = false;
  for (int base = 0; base < N; base += 64) {
    const int i = base + lane;
    bool m0 = false, diff = false;
    if (i < N) {
      m0 = !isnan(c.explevels[((int64_t)g * S) * N + i]) && c.geno_in_sbgrp[i];
      for (int s = 1; s < S; ++s) {
        const bool ms = !isnan(c.explevels[((int64_t)g * S + s) * N + i]) && c.geno_in_sbgrp[(int64_t)s * N + i];
        diff |= ms != m0;
      }
    }
    mismatch |= __ballot(diff) != 0ull;
    const uint64_t bal = __ballot(m0);
    if (m0 && wv == 0) idx[n + __popcll(bal & ((1ull << lane) - 1ull))] = i;
    n += __popcll(bal);
  }
  __syncthreads();
  r.n = n;
  const int Q = r.qcov;
  if (mismatch)
    r.flags = MV_MISMATCH;
  else if (n < Q + 3) /* no residual degree of freedom for the F statistic */
    r.flags = MV_FEW;
  if (r.flags != MV_OK) {
    if (threadIdx.x == 0) pp.mrec[g] = r;
    return;
  }
  if (Q > 0) { /* a member without covariates is a data error (gene_snp_pair.cpp:137-144) */
    int miss = 0;
    for (int k = lane; k < n; k += 64) miss |= !c.covar_in_sbgrp[idx[k]];
    if (__ballot(miss) != 0ull) {
      r.flags = MV_SKIP;
      if (threadIdx.x == 0) {
        atomicOr(pp.flag, FLAG_MISSING_COVAR);
        pp.mrec[g] = r;
      }
      return;
    }
  }
  double* U = pp.Ut + (int64_t)g * KU * N;
  double* Y = pp.Yt + (int64_t)g * S * N;
  /* orthonormal basis of [1, covariates] by two-pass modified Gram-Schmidt;
   * each lane only touches its own rows k = lane + 64 m */
  uint32_t kept = 0;
  for (int j = 0; j <= Q && wv == 0; ++j) {
    double* cj = U + (int64_t)j * N;
    for (int k = lane; k < n; k += 64)
      cj[k] = (j == 0) ? 1.0 : c.covars[((int64_t)(j - 1)) * N + idx[k]];
    double nn = 0;
    for (int k = lane; k < n; k += 64) nn += cj[k] * cj[k];
    const double n0 = sqrt(wsum64(nn));
    for (int pass = 0; pass < 2; ++pass)
      for (int l = 0; l < j; ++l) {
        if (!((kept >> l) & 1u)) continue;
        const double* cl = U + (int64_t)l * N;
        double d = 0;
        for (int k = lane; k < n; k += 64) d += cl[k] * cj[k];
        d = wsum64(d);
        for (int k = lane; k < n; k += 64) cj[k] -= d * cl[k];
      }
    double nv = 0;
    for (int k = lane; k < n; k += 64) nv += cj[k] * cj[k];
    nv = sqrt(wsum64(nv));
    const bool keep = nv > 1e-9 * n0 && nv > 0.0;
    const double sc = keep ? 1.0 / nv : 0.0;
    for (int k = lane; k < n; k += 64) cj[k] *= sc;
    if (keep) {
      kept |= 1u << j;
      ++r.rank;
    }
  }
  if (threadIdx.x == 0) s_kept = kept;
  __syncthreads();
  kept = s_kept;
  for (int j = Q + 1 + wv; j < KU; j += nwv)
    for (int k = lane; k < n; k += 64) U[(int64_t)j * N + k] = 0.0;
  for (int s = wv; s < S; s += nwv) {
    double* ys = Y + (int64_t)s * N;
    for (int k = lane; k < n; k += 64) ys[k] = c.explevels[((int64_t)g * S + s) * N + idx[k]];
    for (int pass = 0; pass < 2; ++pass)
      for (int l = 0; l <= Q; ++l) {
        if (!((kept >> l) & 1u)) continue;
        const double* cl = U + (int64_t)l * N;
        double d = 0;
        for (int k = lane; k < n; k += 64) d += cl[k] * ys[k];
        d = wsum64(d);
        for (int k = lane; k < n; k += 64) ys[k] -= d * cl[k];
      }
  }
  __syncthreads();
  double* yty = pp.YtY + (int64_t)g * S * S;
  int turn = 0;
  for (int a = 0; a < S; ++a)
    for (int b = a; b < S; ++b) {
      if (turn++ % nwv != wv) continue;
      const double* ya = Y + (int64_t)a * N;
      const double* yb = Y + (int64_t)b * N;
      double d = 0;
      for (int k = lane; k < n; k += 64) d += ya[k] * yb[k];
      d = wsum64(d);
      if (lane == 0) {
        yty[a * S + b] = d;
        yty[b * S + a] = d;
      }
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    /* Sigma0 = Y'TY / (n + m - q - s - 1) = Y'TY / n, m = q + s + 1 */
    double A[SM][SM];
    int piv[SM];
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SM; ++j) A[i][j] = (i < S && j < S) ? yty[i * S + j] / (double)n : (i == j ? 1.0 : 0.0);
    for (int i = 0; i < S; ++i)
      for (int j = 0; j < S; ++j) pp.S0[((int64_t)g * S + i) * S + j] = yty[i * S + j] / (double)n;
    (void)lu_factor<SM>(A, piv);
    for (int col = 0; col < S; ++col) {
      double e[SM];
#pragma unroll
      for (int i = 0; i < SM; ++i) e[i] = (i == col) ? 1.0 : 0.0;
      lu_apply<SM>(A, piv, e);
#pragma unroll
      for (int i = 0; i < SM; ++i)
        if (i < S) pp.S0inv[((int64_t)g * S + i) * S + col] = e[i];
    }
    pp.mrec[g] = r;
  }
}

/* ---- per pair: k and b over the members ------------------------------------------ */
struct MvSums {
  const MvRec* mrec;
  const int32_t* midx;
  const double* Ut;
  const double* Yt;
  double* kb;         /* [S + 1][NP]: k, b_0 .. b_{S-1}          */
  int32_t* pgene;     /* [NP]: gene of the pair, -1 = no result    */
  int32_t* n_out;
  double* sstats;
  double* stdsstats;
  int* flag;
  int KU;
};

__device__ inline int gene_of_pair(const int64_t* __restrict__ off, int G, int64_t p) {
  int lo = 0, hi = G - 1; /* largest g with off[g] <= p */
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= p)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

typedef double v4d __attribute__((ext_vector_type(4)));

/* One wave per 16 pairs: the sums over the members are FP64 matrix products of
 * their genotypes with the gene's levels and covariate basis (NG groups of 16
 * columns, rows of A), both read as the operands want them, the genotypes once.
 * Lane l holds pair l % 16, columns l / 16 + 4 r.  The pairs of a wave may belong to
 * several genes: one product each, for its own pairs.
 *
 * Bound by the latency of its reads, four steps in flight.  96,000 pairs, 9
 * subgroups of 150, no covariates: 44 us.  (A thread per pair, 1,500 waves, read the
 * genotypes once per basis column: 437 us.) */
template <int NG>
__global__ void __launch_bounds__(256) mvlr_sums_kernel(const eqbf_chunk c, const MvSums ms) {
  const int64_t NP = c.n_pairs;
  const int lane = threadIdx.x & 63, kl = lane >> 4, pl = lane & 15;
  const int64_t p0 = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / 64 * 16;
  if (p0 >= NP) return;
  const int64_t p = min(p0 + pl, NP - 1);
  const bool act = p0 + pl < NP;
  const int S = c.n_subgroups, N = c.n_samples, KU = ms.KU;
  const int g = gene_of_pair(c.pair_offset, c.n_genes, p);
  const int64_t snp = c.pair_snp[p];
  const MvRec r = ms.mrec[g];
  bool all_geno = true;
  for (int s = 0; s < S; ++s) all_geno &= c.snp_in_sbgrp[snp * S + s] != 0;
  if (act && r.flags == MV_MISMATCH && all_geno) atomicOr(ms.flag, FLAG_MVLR_SAMPLES);
  const bool has = r.flags != MV_SKIP && r.flags != MV_MISMATCH && all_geno;
  const bool fit = act && has && r.flags != MV_FEW;
  /* the reference records the sample size of each subgroup and NaN summary
   * statistics for --error mvlr (gene_snp_pair.cpp:154-158) */
  if (act)
    for (int s = kl; s < S; s += 4) {
      ms.n_out[(int64_t)s * NP + p] = has ? r.n : 0;
      if (ms.sstats)
        for (int k = 0; k < 5; ++k) ms.sstats[((int64_t)k * S + s) * NP + p] = NAN;
      if (ms.stdsstats)
        for (int k = 0; k < 3; ++k) ms.stdsstats[((int64_t)k * S + s) * NP + p] = NAN;
    }
  if (act && kl == 0) ms.pgene[p] = fit ? g : -1;
  const int64_t gbase = (int64_t)c.geno_set_of_sbgrp[0] * c.geno_set_stride + snp;
  const bool f32 = c.geno_dtype == EQBF_F32;
  uint64_t left = __ballot(fit);
  while (left) {
    const int gw = __builtin_amdgcn_readlane(g, __builtin_ctzll(left));
    const bool mine = fit && g == gw;
    left &= ~__ballot(mine);
    const int n = ms.mrec[gw].n;
    const int32_t* idx = ms.midx + (int64_t)gw * N;
    /* this lane's column of each group: levels, then the basis */
    const double* col[NG];
    bool on[NG];
    v4d acc[NG];
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int m = 16 * j + pl;
      on[j] = m < S + KU;
      col[j] = m < S ? ms.Yt + ((int64_t)gw * S + m) * N : ms.Ut + ((int64_t)gw * KU + min(m - S, KU - 1)) * N;
      acc[j] = v4d{0.0, 0.0, 0.0, 0.0};
    }
    double xx = 0.0;
    for (int k0 = 0; k0 < n; k0 += 16) {
      int64_t at[4];
      double x[4], v[4][NG];
#pragma unroll
      for (int u = 0; u < 4; ++u) at[u] = gbase + (int64_t)idx[min(k0 + 4 * u + kl, n - 1)] * c.geno_ld;
      if (f32) {
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = (double)((const float*)c.genotypes)[at[u]];
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = ((const double*)c.genotypes)[at[u]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int j = 0; j < NG; ++j) v[u][j] = col[j][min(k0 + 4 * u + kl, n - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = k0 + 4 * u + kl < n; /* past n the last member once more, with zeros */
        xx += in ? x[u] * x[u] : 0.0;
#pragma unroll
        for (int j = 0; j < NG; ++j)
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(in && on[j] ? v[u][j] : 0.0, x[u], acc[j], 0, 0, 0);
      }
    }
    double proj = 0.0;
#pragma unroll
    for (int j = 0; j < NG; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = 16 * j + kl + 4 * q;
        if (m < S) {
          if (mine) ms.kb[(int64_t)(1 + m) * NP + p] = acc[j][q];
        } else if (m < S + KU) {
          proj += acc[j][q] * acc[j][q];
        }
      }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      xx += __shfl_xor(xx, o, 64);
      proj += __shfl_xor(proj, o, 64);
    }
    if (mine && kl == 0) ms.kb[p] = xx - proj;
  }
}

/* ---- per (pair, configuration): Sigma, Sigma^-1, Sigma^-1 t, t, eVb -------------- */
struct MvCfg {
  const MvRec* mrec;
  const double* YtY;
  const double* S0;
  const double* S0inv;
  const double* kb;
  const int32_t* pgene;
  const double* tz;
  const uint64_t* masks; /* [1 + n_cfg]: the consistent configuration first */
  double* par;           /* [cfg in batch][PSZ][NP]                          */
  double fiterr;
  int cfg0, PSZ;
};

/* Calls launch(std::integral_constant<int, E>) with E the exact subgroup
 * count where SM pads it (5..7 in 8, 9..11 in 12), else E = SM: the
 * per-(pair, configuration) kernels then hold E x E matrices, fewer
 * registers and no identity-padded LU. */
template <int SM, class Launch>
void with_exact_sm(int S, Launch&& launch) {
  if constexpr (SM == 8) {
    if (S == 5) return launch(std::integral_constant<int, 5>{});
    if (S == 6) return launch(std::integral_constant<int, 6>{});
    if (S == 7) return launch(std::integral_constant<int, 7>{});
  } else if constexpr (SM == 12) {
    if (S == 9) return launch(std::integral_constant<int, 9>{});
    if (S == 10) return launch(std::integral_constant<int, 10>{});
    if (S == 11) return launch(std::integral_constant<int, 11>{});
  }
  launch(std::integral_constant<int, SM>{});
}

template <int SM>
__global__ void __launch_bounds__(64) mvlr_cfg_kernel(const eqbf_chunk c, const MvCfg mc) {
  const int64_t NP = c.n_pairs;
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= NP) return;
  const int ci = blockIdx.y;
  const int S = c.n_subgroups;
  const int PSZ = mc.PSZ;
  double* out = mc.par + (int64_t)ci * PSZ * NP + p;
  const int g = mc.pgene[p];
  if (g < 0) {
    out[(int64_t)(PSZ - 1) * NP] = 1.0;
    return;
  }
  const MvRec r = mc.mrec[g];
  const uint64_t gm = mc.masks[mc.cfg0 + ci];
  const double kk = mc.kb[p];
  double b[SM];
#pragma unroll
  for (int s = 0; s < SM; ++s) b[s] = (s < S) ? mc.kb[(int64_t)(1 + s) * NP + p] : 0.0;
  const double* YY = mc.YtY + (int64_t)g * S * S;
  const double* S0 = mc.S0 + (int64_t)g * S * S;
  double Sg[SM][SM];
  const bool fit = !(mc.fiterr < 1e-6);
  if (!fit) {
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SM; ++j) Sg[i][j] = (i < S && j < S) ? S0[i * S + j] : (i == j ? 1.0 : 0.0);
  } else {
    const double nn = (double)r.n;
    const double m = (double)(r.qcov + 1 + S + 1);
    const int nu = r.n - (r.qcov + 1) - 1;
    double cf[SM];
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      cf[i] = 1.0;
      if (i < S && ((gm >> i) & 1ull)) {
        const double b2k = b[i] * b[i] / kk;
        const double s1 = (YY[i * S + i] - b2k) / (double)nu;
        const double T2 = b2k / (s1 * s1);
        if (!(T2 < 1e-8)) {
          const double w = dm::tz_eval(mc.tz, nu, sqrt(T2)); /* -ln P(T_nu <= -sqrt T2) */
          if (2.0 * exp(-w) == 0.0) {
            cf[i] = 0.0; /* the F tail underflows: chi-square quantile +inf */
          } else {
            const double z = dm::gauss_pinv_from_w(w);
            cf[i] = sqrt(T2 / (z * z));
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SM; ++j) {
        if (i < S && j < S) {
          const bool any = ((gm >> i) & 1ull) || ((gm >> j) & 1ull);
          const double ee = YY[i * S + j] - (any ? b[i] * b[j] / kk : 0.0);
          const double h = (i == j) ? 1e-4 : 0.0;
          const double sm = (h * m / (m + nn) + ee / (m + nn)) * cf[j];
          Sg[i][j] = mc.fiterr * sm + (1.0 - mc.fiterr) * S0[i * S + j];
        } else {
          Sg[i][j] = (i == j) ? 1.0 : 0.0;
        }
      }
  }
  double tv[SM];
#pragma unroll
  for (int j = 0; j < SM; ++j) tv[j] = (j < S && ((gm >> j) & 1ull)) ? sqrt(Sg[j][j]) : 0.0;
  double u[SM], eVb[SM];
#pragma unroll
  for (int i = 0; i < SM; ++i) u[i] = eVb[i] = 0.0;
  if (!fit) {
    const double* Si = mc.S0inv + (int64_t)g * S * S;
#pragma unroll
    for (int i = 0; i < SM; ++i)
      if (i < S) {
#pragma unroll
        for (int j = 0; j < SM; ++j)
          if (j < S) {
            const double v = Si[i * S + j];
            out[(int64_t)(i * S + j) * NP] = v;
            u[i] += v * tv[j];
            eVb[i] += v * b[j];
          }
      }
  } else {
    int piv[SM];
    (void)lu_factor<SM>(Sg, piv);
    for (int col = 0; col < S; ++col) {
      double e[SM];
#pragma unroll
      for (int i = 0; i < SM; ++i) e[i] = (i == col) ? 1.0 : 0.0;
      lu_apply<SM>(Sg, piv, e);
      double tc = 0, bc = 0;
#pragma unroll
      for (int j = 0; j < SM; ++j)
        if (j == col) {
          tc = tv[j];
          bc = b[j];
        }
#pragma unroll
      for (int i = 0; i < SM; ++i)
        if (i < S) {
          out[(int64_t)(i * S + col) * NP] = e[i];
          u[i] += e[i] * tc;
          eVb[i] += e[i] * bc;
        }
    }
  }
#pragma unroll
  for (int i = 0; i < SM; ++i)
    if (i < S) {
      out[(int64_t)(S * S + i) * NP] = u[i];
      out[(int64_t)(S * S + S + i) * NP] = tv[i];
      out[(int64_t)(S * S + 2 * S + i) * NP] = eVb[i];
    }
  out[(int64_t)(S * S + 3 * S) * NP] = kk;
  out[(int64_t)(PSZ - 1) * NP] = 0.0;
}

/* ---- per (pair, raw row): one log10 ABF ------------------------------------------ */
struct MvGrid {
  const double* par;
  const double* grid; /* phiL, omaL, phiS, omaS */
  double* raw;        /* [n_raw][NP]            */
  int GL, GS, cfg0, PSZ;
  int64_t row0, nrows, pair_blocks;
};

template <int SM>
__global__ void __launch_bounds__(64) mvlr_grid_kernel(const eqbf_chunk c, const MvGrid mg) {
  const int64_t NP = c.n_pairs;
  /* rows fastest: the blocks in flight share one tile of 64 pairs, whose
   * parameters stay in L2 across the rows */
  const int64_t pb = blockIdx.x / mg.nrows;
  const int64_t rr = blockIdx.x - pb * mg.nrows;
  const int64_t p = pb * 64 + threadIdx.x;
  if (p >= NP || rr >= mg.nrows) return;
  const int64_t row = mg.row0 + rr;
  const int S = c.n_subgroups;
  int cfg, gi, type = 0;
  double p2, o2;
  if (row < 3 * (int64_t)mg.GL) {
    cfg = 0;
    type = (int)(row / mg.GL);
    gi = (int)(row - (int64_t)type * mg.GL);
    p2 = mg.grid[gi];
    o2 = mg.grid[mg.GL + gi];
    if (type == 1) { /* gen-fix: phi2 = 0, oma2 = phi2 + oma2 */
      o2 = p2 + o2;
      p2 = 0.0;
    } else if (type == 2) { /* gen-maxh: phi2 = phi2 + oma2, oma2 = 0 */
      p2 = p2 + o2;
      o2 = 0.0;
    }
  } else {
    const int64_t rs = row - 3 * (int64_t)mg.GL;
    cfg = 1 + (int)(rs / mg.GS);
    gi = (int)(rs - (int64_t)(cfg - 1) * mg.GS);
    p2 = mg.grid[2 * mg.GL + gi];
    o2 = mg.grid[2 * mg.GL + mg.GS + gi];
  }
  const int PSZ = mg.PSZ;
  const double* pr = mg.par + (int64_t)(cfg - mg.cfg0) * PSZ * NP + p;
  double l = NAN;
  if (pr[(int64_t)(PSZ - 1) * NP] == 0.0) {
    const double kk = pr[(int64_t)(S * S + 3 * S) * NP];
    double t[SM], z[SM], u[SM];
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      t[i] = (i < S) ? pr[(int64_t)(S * S + S + i) * NP] : 0.0;
      u[i] = (i < S) ? pr[(int64_t)(S * S + i) * NP] : 0.0;
      z[i] = (i < S) ? pr[(int64_t)(S * S + 2 * S + i) * NP] : 0.0;
    }
    /* M = I + k Sigma^-1 (oma2 t t' + phi2 diag(t^2)) */
    double M[SM][SM];
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SM; ++j) {
        double v = (i == j) ? 1.0 : 0.0;
        if (i < S && j < S) v += kk * (o2 * u[i] * t[j] + p2 * pr[(int64_t)(i * S + j) * NP] * t[j] * t[j]);
        M[i][j] = v;
      }
    double e[SM];
#pragma unroll
    for (int i = 0; i < SM; ++i) e[i] = z[i];
    int piv[SM];
    const double lnd = lu_factor<SM>(M, piv);
    lu_apply<SM>(M, piv, z); /* z = M^-1 eVb */
    /* eVb' W z with W = oma2 t t' + phi2 diag(t^2) */
    double et = 0, tz = 0, q2 = 0;
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      et += e[i] * t[i];
      tz += t[i] * z[i];
      q2 += e[i] * t[i] * t[i] * z[i];
    }
    const double quad = o2 * et * tz + p2 * q2;
    l = (0.5 * quad - 0.5 * lnd) / 2.302585092994045684;
  }
  mg.raw[row * NP + p] = l;
}

/* ---- per (pair, group of rows): Hessenberg form, every grid point ----------------
 * With B = k Sigma^-1 T^2 (T = diag t) and the rank-one term o2 k u t'
 * (u = Sigma^-1 t), the matrix of every row is M = I + p2 B + o2 (k u) t'.
 * An orthogonal similarity Q'BQ = H (Householder reflections, upper
 * Hessenberg) is computed once per (pair, configuration); then for each grid
 * point A = I + p2 H is factorised with partial pivoting in O(S^2) (only
 * adjacent rows can swap), the rank-one term is added by the matrix
 * determinant lemma and Sherman-Morrison, and
 *   ln|det M| = ln|det A| + ln|1 + o2 t~'A^-1 u~|,
 *   M^-1 eVb  = Q (A^-1 z~ - o2 A^-1 u~ (t~'A^-1 z~) / (1 + o2 t~'A^-1 u~)),
 * with u~ = k Q'u, z~ = Q'eVb, t~ = Q't; the quadratic form eVb'W M^-1 eVb
 * = o2 (eVb't)(t~'x~) + p2 (Q'T^2 eVb)'x~.  Rows of the gen-fix type
 * (p2 = 0) reduce to scalars.  The row kernel above builds and factorises
 * each M from scratch (O(S^3) per row); this one gives the same values to
 * rounding.  Groups: for the consistent configuration gen, gen-fix and
 * gen-maxh (GL rows each), for the others their GS rows. */
template <int SM>
struct HessIdx {
  /* position of entry (i, j), j >= i - 1, of an upper Hessenberg SM x SM matrix */
  static constexpr int at(int i, int j) { return i == 0 ? j : SM + (i - 1) * SM - (i - 1) * (i - 2) / 2 + (j - (i - 1)); }
  static constexpr int size = SM == 1 ? 1 : SM + (SM - 1) * SM - (SM - 1) * (SM - 2) / 2;
};

/* per (pair, configuration of the batch): the Hessenberg form and the
 * carried vectors, [cfg][E][NP] with E = HessIdx::size + 4 SM + 1:
 * H's entries, u~ = k Q'u, z~ = Q'eVb, t~ = Q't, v~ = Q'T^2 eVb, eVb't */
template <int SM>
__global__ void __launch_bounds__(64) mvlr_hess_kernel(const eqbf_chunk c, const MvGrid mg, double* __restrict__ hess) {
  const int64_t NP = c.n_pairs;
  const int64_t p = blockIdx.x * (int64_t)64 + threadIdx.x;
  if (p >= NP) return;
  const int cfg = blockIdx.y;
  const int PSZ = mg.PSZ, S = SM;
  constexpr int HS = HessIdx<SM>::size, E = HS + 4 * SM + 1;
  const double* pr = mg.par + (int64_t)cfg * PSZ * NP + p;
  double* out = hess + (int64_t)cfg * E * NP + p;
  if (pr[(int64_t)(PSZ - 1) * NP] != 0.0) return; /* no result: the row kernel writes NaN */
  const double kk = pr[(int64_t)(S * S + 3 * S) * NP];
  double t[SM], ut[SM], zt[SM], tt[SM], vt[SM], B[SM][SM];
  double et = 0.0;
#pragma unroll
  for (int i = 0; i < SM; ++i) t[i] = pr[(int64_t)(S * S + S + i) * NP];
#pragma unroll
  for (int i = 0; i < SM; ++i) {
    const double u = pr[(int64_t)(S * S + i) * NP], z = pr[(int64_t)(S * S + 2 * S + i) * NP];
#pragma unroll
    for (int j = 0; j < SM; ++j) B[i][j] = kk * pr[(int64_t)(i * S + j) * NP] * t[j] * t[j];
    ut[i] = kk * u;
    zt[i] = z;
    tt[i] = t[i];
    vt[i] = t[i] * t[i] * z;
    et += z * t[i];
  }
#pragma unroll
  for (int k = 0; k + 2 < SM; ++k) {
    double nrm2 = 0.0;
#pragma unroll
    for (int i = k + 1; i < SM; ++i) nrm2 += B[i][k] * B[i][k];
    const double x0 = B[k + 1][k];
    double alpha = sqrt(nrm2);
    if (x0 > 0) alpha = -alpha;
    double v[SM];
    double vv = 0.0;
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      v[i] = i == k + 1 ? x0 - alpha : (i > k + 1 ? B[i][k] : 0.0);
      vv += v[i] * v[i];
    }
    const double beta = vv > 0.0 ? 2.0 / vv : 0.0;
#pragma unroll
    for (int j = k; j < SM; ++j) {
      double s = 0.0;
#pragma unroll
      for (int i = k + 1; i < SM; ++i) s += v[i] * B[i][j];
      s *= beta;
#pragma unroll
      for (int i = k + 1; i < SM; ++i) B[i][j] -= v[i] * s;
    }
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      double s = 0.0;
#pragma unroll
      for (int j = k + 1; j < SM; ++j) s += B[i][j] * v[j];
      s *= beta;
#pragma unroll
      for (int j = k + 1; j < SM; ++j) B[i][j] -= s * v[j];
    }
    double s1 = 0.0, s2 = 0.0, s3 = 0.0, s4 = 0.0;
#pragma unroll
    for (int i = k + 1; i < SM; ++i) {
      s1 += v[i] * ut[i];
      s2 += v[i] * zt[i];
      s3 += v[i] * tt[i];
      s4 += v[i] * vt[i];
    }
#pragma unroll
    for (int i = k + 1; i < SM; ++i) {
      ut[i] -= beta * v[i] * s1;
      zt[i] -= beta * v[i] * s2;
      tt[i] -= beta * v[i] * s3;
      vt[i] -= beta * v[i] * s4;
    }
  }
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = (i == 0 ? 0 : i - 1); j < SM; ++j) out[(int64_t)HessIdx<SM>::at(i, j) * NP] = B[i][j];
#pragma unroll
  for (int i = 0; i < SM; ++i) {
    out[(int64_t)(HS + i) * NP] = ut[i];
    out[(int64_t)(HS + SM + i) * NP] = zt[i];
    out[(int64_t)(HS + 2 * SM + i) * NP] = tt[i];
    out[(int64_t)(HS + 3 * SM + i) * NP] = vt[i];
  }
  out[(int64_t)(HS + 4 * SM) * NP] = et;
}

/* a / x with r = rcp_nr(x): the quotient and its remainder's correction */
__device__ __forceinline__ double div_by(double a, double x, double r) {
  const double q = a * r;
  return fma(fma(-q, x, a), r, q);
}

/* per (64 pairs, group of rows): every grid point of the group from the
 * Hessenberg form, the points shared out among four waves.
 *
 * What is needed of M^-1 are the four products of (tt, vt) with M^-1 (ut, zt).  With
 * M = L U, L^-1 (ut, zt) and (tt, vt) U^-1 both follow the elimination row by row,
 * so that a lane holds two rows of the matrix and nothing is solved backwards; H and
 * the carried vectors stay in LDS for the four waves.
 *
 * Bound by the vector unit, about 750 instructions a point (9 subgroups).  96,000
 * pairs, 9 subgroups, 100 points: 0.28 ms.  (With U kept for the solves a wave took
 * 344 registers, one to a SIMD, and an IEEE division for each quotient: 0.40 ms.) */
constexpr int MV_ROW_WAVES = 4;

template <int SM>
__global__ void __launch_bounds__(64 * MV_ROW_WAVES, 3) mvlr_rows_kernel(const eqbf_chunk c, const MvGrid mg,
                                                                      const double* __restrict__ hess) {
  const int64_t NP = c.n_pairs;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool act = blockIdx.x * (int64_t)64 + lane < NP;
  const int64_t p = act ? blockIdx.x * (int64_t)64 + lane : NP - 1;
  const int g = blockIdx.y;
  /* group g -> configuration (relative to the batch) and row type */
  int cfg, type;
  if (mg.cfg0 == 0) {
    cfg = g < 3 ? 0 : g - 2;
    type = g < 3 ? g : 3;
  } else {
    cfg = g;
    type = 3;
  }
  constexpr int HS = HessIdx<SM>::size, E = HS + 4 * SM + 1;
  __shared__ double Hs[HS + 4 * SM][64]; /* H, ut, zt, tt, vt */
  const int PSZ = mg.PSZ, S = SM;
  const double* pr = mg.par + (int64_t)cfg * PSZ * NP + p;
  const bool ok = pr[(int64_t)(PSZ - 1) * NP] == 0.0;
  const int n_rows = type == 3 ? mg.GS : mg.GL;
  const int64_t row_base = type < 3 ? (int64_t)type * mg.GL : 3 * (int64_t)mg.GL + (int64_t)(mg.cfg0 + cfg - 1) * mg.GS;
  const double* gp = type == 3 ? mg.grid + 2 * mg.GL : mg.grid;
  const double* go = type == 3 ? mg.grid + 2 * mg.GL + mg.GS : mg.grid + mg.GL;
  const double ln10 = 2.302585092994045684;
  double* raw = mg.raw + row_base * NP + p;
  if (type == 1) { /* gen-fix: M = I + o2 k u t' */
    const double kk = pr[(int64_t)(S * S + 3 * S) * NP];
    double tu = 0.0, tz = 0.0, et = 0.0;
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      const double t = pr[(int64_t)(S * S + S + i) * NP];
      const double u = pr[(int64_t)(S * S + i) * NP], z = pr[(int64_t)(S * S + 2 * S + i) * NP];
      tu += t * u;
      tz += t * z;
      et += z * t;
    }
    for (int gi = wv; gi < n_rows; gi += MV_ROW_WAVES) {
      const double o2 = gp[gi] + go[gi];
      const double sig = 1.0 + o2 * kk * tu;
      const double quad = o2 * et * (tz / sig);
      if (act) raw[(int64_t)gi * NP] = ok ? (0.5 * quad - 0.5 * log(fabs(sig))) / ln10 : NAN;
    }
    return;
  }
  const double* hv = hess + (int64_t)cfg * E * NP + p;
#pragma unroll 8
  for (int e = wv; e < HS + 4 * SM; e += MV_ROW_WAVES) Hs[e][lane] = hv[(int64_t)e * NP];
  const double et = hv[(int64_t)(HS + 4 * SM) * NP];
  __syncthreads();
  for (int gi = wv; gi < n_rows; gi += MV_ROW_WAVES) {
    double p2, o2;
    if (type == 2) { /* gen-maxh */
      p2 = gp[gi] + go[gi];
      o2 = 0.0;
    } else {
      p2 = gp[gi];
      o2 = go[gi];
    }
    auto entry = [&](int i, int j) { return (i == j ? 1.0 : 0.0) + p2 * Hs[HessIdx<SM>::at(i, j)][lane]; };
    asm volatile("" ::: "memory"); /* H is read again for each point, not kept in registers */
    double cur[SM], nxt[SM], a[SM], b[SM];
#pragma unroll
    for (int i = 0; i < SM; ++i) {
      cur[i] = entry(0, i);
      a[i] = Hs[HS + 2 * SM + i][lane];
      b[i] = Hs[HS + 3 * SM + i][lane];
    }
    double u = Hs[HS][lane], z = Hs[HS + SM][lane]; /* this row of L^-1 (ut, zt) */
    double tu = 0.0, tz = 0.0, vu = 0.0, vz = 0.0;   /* t' M^-1 ut, ... */
    double mant = 1.0;
    int ex = 0;
    /* LU of the Hessenberg matrix, partial pivoting between rows j and j+1 */
#pragma unroll
    for (int j = 0; j < SM; ++j) {
      double un = 0.0, zn = 0.0;
      if (j + 1 < SM) {
#pragma unroll
        for (int col = j; col < SM; ++col) nxt[col] = entry(j + 1, col);
        un = Hs[HS + j + 1][lane];
        zn = Hs[HS + SM + j + 1][lane];
        const bool sw = fabs(nxt[j]) > fabs(cur[j]);
        auto order = [&](double& x, double& y) {
          const double xs = sw ? y : x;
          y = sw ? x : y;
          x = xs;
        };
#pragma unroll
        for (int col = j; col < SM; ++col) order(cur[col], nxt[col]);
        order(u, un);
        order(z, zn);
      }
      const double piv = cur[j], rp = dm::rcp_nr(piv);
      const double ya = div_by(a[j], piv, rp), yb = div_by(b[j], piv, rp);
      tu += ya * u;
      tz += ya * z;
      vu += yb * u;
      vz += yb * z;
      int e;
      mant = frexp(mant * piv, &e);
      ex += e;
      if (j + 1 < SM) {
        const double f = div_by(nxt[j], piv, rp);
#pragma unroll
        for (int col = j + 1; col < SM; ++col) {
          a[col] -= ya * cur[col];
          b[col] -= yb * cur[col];
          cur[col] = nxt[col] - f * cur[col];
        }
        u = un - f * u;
        z = zn - f * z;
      }
    }
    double lnd = log(fabs(mant)) + (double)ex * 0.69314718055994530942;
    if (o2 != 0.0) {
      const double sig = 1.0 + o2 * tu;
      const double coef = o2 * tz / sig;
      tz -= coef * tu;
      vz -= coef * vu;
      lnd += log(fabs(sig));
    }
    const double quad = o2 * et * tz + p2 * vz;
    if (act) raw[(int64_t)gi * NP] = ok ? (0.5 * quad - 0.5 * lnd) / ln10 : NAN;
  }
}

/* ---- per (pair, weighted row): utils::log10_weighted_sum over the grid ------------ */
__global__ void __launch_bounds__(256) mvlr_wavg_kernel(const double* __restrict__ raw, double* __restrict__ w,
                                                         int64_t NP, int GL, int GS, int64_t wrow0, int64_t nw) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= nw * NP) return;
  const int64_t wr = wrow0 + i / NP, p = i % NP;
  const int G = wr < 3 ? GL : GS;
  const int64_t r0 = wr < 3 ? wr * GL : 3 * (int64_t)GL + (wr - 3) * GS;
  const double* v = raw + r0 * NP + p;
  double mx = v[0];
  for (int k = 1; k < G; ++k) {
    const double x = v[(int64_t)k * NP];
    if (x > mx) mx = x;
  }
  const double wt = 1.0 / (double)G;
  double sum = 0;
  for (int k = 0; k < G; ++k) {
    const double x = v[(int64_t)k * NP];
    if (!isnan(x)) sum += wt * exp10(x - mx);
  }
  double res = mx + log10(sum);
  if (fabs(res) <= 2.220446049250313e-16) res = 0.0;
  w[wr * NP + p] = res;
}

/* Raw and grid-averaged rows of every configuration (the consistent one
 * first), then the BMA rows.  fill(c0, nb, par, PSZ, pair_blocks) enqueues
 * the kernel writing the parameters of configurations [c0, c0 + nb) in the
 * layout mvlr_grid_kernel reads: [cfg - c0][PSZ][NP] with Sigma^-1 [S][S],
 * Sigma^-1 t, t, eVb, k and a flag (0 = computed).  Configurations go in
 * batches bounded by the parameter buffer and by the 65535 limit of the
 * grid's y dimension. */
/* the row kernel at the exact subgroup count (no padded rows in the LU) */
void launch_grid_kernel(int S, unsigned blocks, hipStream_t st, const eqbf_chunk& c, const MvGrid& mg) {
#define EQBF_GRID_CASE(n) \
  case n:                 \
    hipLaunchKernelGGL(mvlr_grid_kernel<n>, dim3(blocks), dim3(64), 0, st, c, mg); \
    break;
  switch (S) {
    EQBF_GRID_CASE(1)
    EQBF_GRID_CASE(2)
    EQBF_GRID_CASE(3)
    EQBF_GRID_CASE(4)
    EQBF_GRID_CASE(5)
    EQBF_GRID_CASE(6)
    EQBF_GRID_CASE(7)
    EQBF_GRID_CASE(8)
    EQBF_GRID_CASE(9)
    EQBF_GRID_CASE(10)
    EQBF_GRID_CASE(11)
    EQBF_GRID_CASE(12)
    EQBF_GRID_CASE(13)
    EQBF_GRID_CASE(14)
    EQBF_GRID_CASE(15)
    default:
      hipLaunchKernelGGL(mvlr_grid_kernel<16>, dim3(blocks), dim3(64), 0, st, c, mg);
      break;
  }
#undef EQBF_GRID_CASE
}

/* the Hessenberg kernels at the exact subgroup count, 2 <= S <= 10 */
template <int n>
void launch_hess_rows(unsigned pair_blocks, unsigned nb, unsigned groups, hipStream_t st, const eqbf_chunk& c,
                      const MvGrid& mg, double* hess, eqbf_ctx* ctx) {
  {
    ProfScope ps(ctx, "mvlr_hess_kernel", st);
    hipLaunchKernelGGL(mvlr_hess_kernel<n>, dim3(pair_blocks, nb), dim3(64), 0, st, c, mg, hess);
  }
  ProfScope ps(ctx, "mvlr_rows_kernel", st);
  hipLaunchKernelGGL(mvlr_rows_kernel<n>, dim3(pair_blocks, groups), dim3(64 * MV_ROW_WAVES), 0, st, c, mg,
                     (const double*)hess);
}

constexpr bool hess_ok(int S) { return S >= 2 && S <= 10; }
constexpr int hess_entries(int S) { return (S == 1 ? 1 : S + (S - 1) * S - (S - 1) * (S - 2) / 2) + 4 * S + 1; }

void launch_rows_kernel(int S, unsigned pair_blocks, unsigned nb, unsigned groups, hipStream_t st,
                        const eqbf_chunk& c, const MvGrid& mg, double* hess, eqbf_ctx* ctx) {
  switch (S) {
    case 2: launch_hess_rows<2>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 3: launch_hess_rows<3>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 4: launch_hess_rows<4>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 5: launch_hess_rows<5>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 6: launch_hess_rows<6>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 7: launch_hess_rows<7>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 8: launch_hess_rows<8>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    case 9: launch_hess_rows<9>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
    default: launch_hess_rows<10>(pair_blocks, nb, groups, st, c, mg, hess, ctx); break;
  }
}

template <int SM, class Fill>
int mv_rows_run(eqbf_ctx* ctx, const eqbf_chunk& c, int bfs, eqbf_assoc_out* out, hipStream_t st, Fill fill) {
  const int S = c.n_subgroups;
  const int64_t NP = c.n_pairs;
  const int GL = (int)ctx->phiL.size(), GS = (int)ctx->phiS.size();
  const int64_t n_cfg = eqbf_n_configs(bfs, S);
  const int PSZ = S * S + 3 * S + 2;
  const int64_t total = 1 + n_cfg;
  int64_t per = std::max<int64_t>(1, ((int64_t)1 << 30) / std::max<int64_t>(1, NP * PSZ * 8));
  /* 2 to 10 subgroups: one thread per (pair, group of rows), the grid
   * points of a group from one Hessenberg reduction (mvlr_rows_kernel);
   * otherwise one thread per (pair, row) */
  per = std::min<int64_t>(std::min<int64_t>(per, hess_ok(S) ? 65533 : 65535), total);
  double* par = (double*)ctx_buf(ctx, "mv_par", (size_t)per * NP * PSZ * sizeof(double));
  double* hess = hess_ok(S) ? (double*)ctx_buf(ctx, "mv_hess", (size_t)per * NP * hess_entries(S) * sizeof(double))
                            : nullptr;
  if (!par || (hess_ok(S) && !hess)) return ctx_fail(ctx, EQBF_ERR_HIP, "allocating mvlr buffers failed");
  const int64_t pair_blocks = (NP + 63) / 64;
  for (int64_t c0 = 0; c0 < total; c0 += per) {
    const int nb = (int)std::min<int64_t>(per, total - c0);
    fill(c0, nb, par, PSZ, pair_blocks);
    /* raw rows of configurations [c0, c0 + nb) and their weighted rows */
    const int64_t c1 = c0 + nb;
    const int64_t row0 = c0 == 0 ? 0 : 3 * (int64_t)GL + (c0 - 1) * GS;
    const int64_t row1 = 3 * (int64_t)GL + (c1 - 1) * GS;
    const int64_t wrow0 = c0 == 0 ? 0 : 3 + (c0 - 1);
    const int64_t wrow1 = 3 + (c1 - 1);
    if (hess_ok(S)) {
      MvGrid mg;
      mg.par = par;
      mg.grid = (const double*)ctx->d_grid.ptr;
      mg.raw = (double*)out->raw_abf;
      mg.GL = GL;
      mg.GS = GS;
      mg.cfg0 = (int)c0;
      mg.PSZ = PSZ;
      mg.row0 = row0;
      mg.nrows = row1 - row0;
      mg.pair_blocks = pair_blocks;
      const unsigned groups = (unsigned)(nb + (c0 == 0 ? 2 : 0));
      launch_rows_kernel(S, (unsigned)pair_blocks, (unsigned)nb, groups, st, c, mg, hess, ctx);
    }
    for (int64_t r0 = row0; !hess_ok(S) && r0 < row1;) {
      const int64_t nr = std::min<int64_t>(row1 - r0, std::max<int64_t>(1, ((int64_t)1 << 30) / pair_blocks));
      MvGrid mg;
      mg.par = par;
      mg.grid = (const double*)ctx->d_grid.ptr;
      mg.raw = (double*)out->raw_abf;
      mg.GL = GL;
      mg.GS = GS;
      mg.cfg0 = (int)c0;
      mg.PSZ = PSZ;
      mg.row0 = r0;
      mg.nrows = nr;
      mg.pair_blocks = pair_blocks;
      {
        ProfScope ps(ctx, "mvlr_grid_kernel", st);
        launch_grid_kernel(S, (unsigned)(nr * pair_blocks), st, c, mg);
      }
      r0 += nr;
    }
    const int64_t nw = wrow1 - wrow0;
    hipLaunchKernelGGL(mvlr_wavg_kernel, dim3((unsigned)((nw * NP + 255) / 256)), dim3(256), 0, st,
                       (const double*)out->raw_abf, out->w_abf, NP, GL, GS, wrow0, nw);
    EQBF_HIP(ctx, hipGetLastError());
  }
  return launch_bma(ctx, out->w_abf, NP, S, bfs, st);
}

template <int SM>
int mvlr_run_sm(eqbf_ctx* ctx, const eqbf_chunk& c, const eqbf_mvlr_opts* o, eqbf_assoc_out* out, hipStream_t st) {
  const int S = c.n_subgroups, N = c.n_samples, G = c.n_genes;
  const int64_t NP = c.n_pairs;
  const int64_t n_cfg = eqbf_n_configs(o->bfs, S);
  const int KU = 1 + c.n_covars_max;
  MvPrep pp;
  pp.mrec = (MvRec*)ctx_buf(ctx, "mv_rec", (size_t)G * sizeof(MvRec));
  pp.midx = (int32_t*)ctx_buf(ctx, "mv_idx", (size_t)G * N * sizeof(int32_t));
  pp.Ut = (double*)ctx_buf(ctx, "mv_U", (size_t)G * KU * N * sizeof(double));
  pp.Yt = (double*)ctx_buf(ctx, "mv_Y", (size_t)G * S * N * sizeof(double));
  pp.YtY = (double*)ctx_buf(ctx, "mv_YtY", (size_t)G * S * S * sizeof(double));
  pp.S0 = (double*)ctx_buf(ctx, "mv_S0", (size_t)G * S * S * sizeof(double));
  pp.S0inv = (double*)ctx_buf(ctx, "mv_S0i", (size_t)G * S * S * sizeof(double));
  pp.KU = KU;
  pp.flag = (int*)ctx->d_flag.ptr;
  double* kb = (double*)ctx_buf(ctx, "mv_kb", (size_t)(S + 1) * NP * sizeof(double));
  int32_t* pgene = (int32_t*)ctx_buf(ctx, "mv_pgene", (size_t)NP * sizeof(int32_t));
  /* configuration masks: the consistent one (all subgroups) first */
  std::vector<uint64_t> hm(1 + n_cfg);
  hm[0] = (S >= 64) ? ~0ull : ((1ull << S) - 1ull);
  if (n_cfg > 0) eqbf_config_masks(o->bfs, S, hm.data() + 1);
  uint64_t* dmask = (uint64_t*)ctx_buf(ctx, "mv_masks", hm.size() * sizeof(uint64_t));
  if (!pp.mrec || !pp.midx || !pp.Ut || !pp.Yt || !pp.YtY || !pp.S0 || !pp.S0inv || !kb || !pgene || !dmask)
    return ctx_fail(ctx, EQBF_ERR_HIP, "allocating mvlr buffers failed");
  EQBF_HIP(ctx, hipMemcpyAsync(dmask, hm.data(), hm.size() * sizeof(uint64_t), hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipStreamSynchronize(st)); /* the host vector goes out of scope */
  int rc = ctx_ensure_tz(ctx, N, st);
  if (rc) return rc;
  hipLaunchKernelGGL(mv_zero_kernel, dim3(1), dim3(1), 0, st, (int*)ctx->d_flag.ptr);
  {
    ProfScope ps(ctx, "mvlr_prep_kernel", st);
    with_exact_sm<SM>(c.n_subgroups, [&](auto e) {
      hipLaunchKernelGGL(mvlr_prep_kernel<decltype(e)::value>, dim3(G), dim3(64 * mv_prep_waves(G)), 0, st, c, pp);
    });
  }
  MvSums ms;
  ms.mrec = pp.mrec;
  ms.midx = pp.midx;
  ms.Ut = pp.Ut;
  ms.Yt = pp.Yt;
  ms.kb = kb;
  ms.pgene = pgene;
  ms.n_out = out->n;
  ms.sstats = out->sstats;
  ms.stdsstats = out->stdsstats;
  ms.flag = (int*)ctx->d_flag.ptr;
  ms.KU = KU;
  {
    ProfScope ps(ctx, "mvlr_sums_kernel", st);
    const dim3 grid((unsigned)((NP + 63) / 64));
    const int groups = (S + ms.KU + 15) / 16; /* S <= 16, KU <= 17 */
    if (groups == 1)
      hipLaunchKernelGGL(mvlr_sums_kernel<1>, grid, dim3(256), 0, st, c, ms);
    else if (groups == 2)
      hipLaunchKernelGGL(mvlr_sums_kernel<2>, grid, dim3(256), 0, st, c, ms);
    else
      hipLaunchKernelGGL(mvlr_sums_kernel<3>, grid, dim3(256), 0, st, c, ms);
  }
  EQBF_HIP(ctx, hipGetLastError());
  return mv_rows_run<SM>(ctx, c, o->bfs, out, st, [&](int64_t c0, int nb, double* par, int PSZ, int64_t pair_blocks) {
    MvCfg mc;
    mc.mrec = pp.mrec;
    mc.YtY = pp.YtY;
    mc.S0 = pp.S0;
    mc.S0inv = pp.S0inv;
    mc.kb = kb;
    mc.pgene = pgene;
    mc.tz = ctx_tz_table(ctx);
    mc.masks = dmask;
    mc.par = par;
    mc.fiterr = o->fiterr;
    mc.cfg0 = (int)c0;
    mc.PSZ = PSZ;
    ProfScope ps(ctx, "mvlr_cfg_kernel", st);
    with_exact_sm<SM>(c.n_subgroups, [&](auto e) {
      hipLaunchKernelGGL(mvlr_cfg_kernel<decltype(e)::value>, dim3((unsigned)pair_blocks, (unsigned)nb), dim3(64), 0,
                         st, c, mc);
    });
  });
}

/* ==== --error hybrid ================================================================
 * GeneSnpPair::CalcAbfsHybrid (gene_snp_pair.cpp:1384-1423) and what it
 * calls (:760-1163), with the Bayes factor of CalcLog10AbfMvlr
 * (:1165-1256).  Per pair of a gene expressed in every subgroup and a SNP
 * genotyped in every subgroup:
 *   b_s, Sigma_ss, Vg_ss from the subgroup's own regression over its members
 *     (present: genotyped, expression level not NaN) on [1, x, covariates],
 *     sigma2 = rss / n, Sigma_ss = f s2_full + (1 - f) s2_null and
 *     Vg_ss = Sigma_ss [(X'X)^-1]_xx;
 *   for s1 < s2, over the individuals present in both (rows [1, x, covariates
 *     of s1 read at the individual's index]): Sigma_12 = f full_01 + (1 - f)
 *     null_01 from the ML error covariances Y'(I - H)Y / n12, and
 *     Vg_12 = Sigma_12 [M1^-1 G12 M2^-1]_xx with G12 = X12'X12 and M_s the
 *     same sums over every individual present in s (the reference's
 *     pinv(G12 + Xs'Xs) X12' products, :977-1131);
 *   log10 ABF = (b'Vg^-1 W (I + Vg^-1 W)^-1 Vg^-1 b - ln|det(I + Vg^-1 W)|)
 *     / (2 ln 10), W = (oma2 1 1' + phi2 I) o gamma gamma' o sd sd',
 *     sd_s = sqrt(Sigma_ss): the MVLR row kernel with k = 1 and Vg in place
 *     of Sigma.
 * Every sum over individuals splits into a covariate block that does not
 * depend on the SNP (per gene: A = sum c c', its inverse, the null
 * regression coefficients psi = A^-1 sum c y and the null residual
 * cross-product, hyb_gene_kernel) and SNP terms (u = sum c x, sum x^2,
 * sum x y, hyb_pair_kernel).  With w = A^-1 u and k = sum x^2 - u'w (the
 * Schur complement, x~'x~ of Frisch-Waugh), the genotype column of M^-1 is
 * (-w, 1) / k, so
 *   [(X'X)^-1]_xx = 1 / k,  x~'y~ = sum x y - u'psi,
 *   rss_full = rss_null - (x~'y~)^2 / k,
 *   [M1^-1 G12 M2^-1]_xx = (w1'A12 w2 - w1'u12 - u12'w2 + sum_12 x^2) / (k1 k2)
 * and no (Q+2) x (Q+2) system is solved per pair.  The reference's
 * pseudo-inverses invert every singular value, so on full-rank designs they
 * are these inverses; the covariate blocks are inverted by Gauss-Jordan
 * elimination with partial pivoting. */
struct HybGene {
  const double* cp;  /* pairwise covariates [S][Qmax][N] (by index in the samples) */
  const double* yp;  /* pairwise expression levels [G][S][N]                       */
  double* rec;       /* [G][NSET][RSZ]                                             */
  int NSET, RSZ, Q1M;
};

/* set j of a gene: 0 <= j < S: members of s with its own covariates and
 * levels; S + s1: members of s1 with the pairwise covariates of s1;
 * 2S + pi: present in s1 and s2 (pair pi = (s1, s2), s1 < s2 in
 * lexicographic order) with the pairwise covariates and levels;
 * 2S + npr + pi: present in s2 with the pairwise covariates of s1. */
__device__ inline void hyb_pair_of(int pi, int S, int& s1, int& s2) {
  s1 = 0;
  while (pi >= S - 1 - s1) {
    pi -= S - 1 - s1;
    ++s1;
  }
  s2 = s1 + 1 + pi;
}

/* present in subgroup s: genotyped there and a level (not NaN) in lev
 * [G][S][N]; the per-subgroup sets read the chunk's levels, the pairwise
 * sets the pairwise levels, which permutations leave as loaded
 * (samples.cpp:148-192) */
__device__ inline bool hyb_present(const eqbf_chunk& c, const double* lev, int g, int s, int i) {
  const int S = c.n_subgroups, N = c.n_samples;
  return c.geno_in_sbgrp[(int64_t)s * N + i] && !isnan(lev[((int64_t)g * S + s) * N + i]);
}

/* record of a set: A^-1 [Q1M][Q1M], A [Q1M][Q1M], psi1 [Q1M], psi2 [Q1M],
 * r (null residual cross-product y1'(I - Hc)y2), n */
__global__ void __launch_bounds__(256) hyb_gene_kernel(const eqbf_chunk c, const HybGene hg) {
  const int g = blockIdx.x, j = blockIdx.y, t = threadIdx.x;
  const int S = c.n_subgroups, N = c.n_samples, QM = c.n_covars_max;
  for (int s = 0; s < S; ++s)
    if (!c.gene_in_sbgrp[(int64_t)g * S + s]) return;
  const int npr = S * (S - 1) / 2;
  int type, sa, sb = -1;
  if (j < S) {
    type = 0;
    sa = j;
  } else if (j < 2 * S) {
    type = 1;
    sa = j - S;
  } else if (j < 2 * S + npr) {
    type = 2;
    hyb_pair_of(j - 2 * S, S, sa, sb);
  } else {
    type = 3;
    hyb_pair_of(j - 2 * S - npr, S, sa, sb);
  }
  const int Q1 = min(max(c.covar_count[sa], 0), QM) + 1, Q1M = hg.Q1M;
  const double* cov = (type == 0) ? c.covars + (int64_t)sa * QM * N : hg.cp + (int64_t)sa * QM * N;
  const bool has_y = type == 0 || type == 2;
  const double* y1 = (type == 0) ? c.explevels + ((int64_t)g * S + sa) * N : hg.yp + ((int64_t)g * S + sa) * N;
  const double* y2 = (type == 0) ? y1 : (type == 2 ? hg.yp + ((int64_t)g * S + sb) * N : nullptr);
  /* entries: the upper triangle of A, then sum c y1, sum c y2, sum y1 y2, n */
  const int nA = Q1 * (Q1 + 1) / 2;
  const int nE = nA + (has_y ? 2 * Q1 + 1 : 0) + 1;
  __shared__ double ent[17 * 18 / 2 + 2 * 17 + 2];
  __shared__ double M[17][34];
  __shared__ double fac[17];
  __shared__ int pivrow;
  /* one wave per entry, lanes striding the individuals */
  const int lane = t & 63, nwv = blockDim.x >> 6;
  const double* lev = (type == 0) ? c.explevels : hg.yp;
  for (int e = t >> 6; e < nE; e += nwv) {
    int kind, a = 0, b = 0;
    if (e < nA) {
      kind = 0;
      int r = e;
      while (r >= Q1 - a) {
        r -= Q1 - a;
        ++a;
      }
      b = a + r;
    } else if (has_y && e < nA + Q1) {
      kind = 1;
      a = e - nA;
    } else if (has_y && e < nA + 2 * Q1) {
      kind = 2;
      a = e - nA - Q1;
    } else if (has_y && e == nA + 2 * Q1) {
      kind = 3;
    } else {
      kind = 4;
    }
    double acc = 0.0;
    for (int i = lane; i < N; i += 64) {
      bool in;
      if (type == 0 || type == 1)
        in = hyb_present(c, lev, g, sa, i);
      else if (type == 2)
        in = hyb_present(c, lev, g, sa, i) && hyb_present(c, lev, g, sb, i);
      else
        in = hyb_present(c, lev, g, sb, i);
      if (!in) continue;
      const double va = a == 0 ? 1.0 : cov[(int64_t)(a - 1) * N + i];
      switch (kind) {
        case 0: acc += va * (b == 0 ? 1.0 : cov[(int64_t)(b - 1) * N + i]); break;
        case 1: acc += va * y1[i]; break;
        case 2: acc += va * y2[i]; break;
        case 3: acc += y1[i] * y2[i]; break;
        default: acc += 1.0; break;
      }
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (lane == 0) ent[e] = acc;
  }
  __syncthreads();
  /* [A | I] */
  for (int e = t; e < Q1 * 2 * Q1; e += blockDim.x) {
    const int r = e / (2 * Q1), col = e - r * 2 * Q1;
    double v;
    if (col < Q1) {
      const int a = min(r, col), b = max(r, col);
      v = ent[a * Q1 - a * (a - 1) / 2 + (b - a)];
    } else {
      v = (col - Q1 == r) ? 1.0 : 0.0;
    }
    M[r][col] = v;
  }
  __syncthreads();
  for (int jc = 0; jc < Q1; ++jc) {
    if (t == 0) {
      int p = jc;
      double best = fabs(M[jc][jc]);
      for (int r = jc + 1; r < Q1; ++r)
        if (fabs(M[r][jc]) > best) {
          best = fabs(M[r][jc]);
          p = r;
        }
      pivrow = p;
    }
    __syncthreads();
    const int p = pivrow;
    if (p != jc && t < 2 * Q1) {
      const double tmp = M[jc][t];
      M[jc][t] = M[p][t];
      M[p][t] = tmp;
    }
    __syncthreads();
    if (t < Q1) fac[t] = (t == jc) ? M[jc][jc] : M[t][jc];
    __syncthreads();
    if (t < 2 * Q1) M[jc][t] /= fac[jc];
    __syncthreads();
    for (int e = t; e < Q1 * 2 * Q1; e += blockDim.x) {
      const int r = e / (2 * Q1), col = e - r * 2 * Q1;
      if (r != jc) M[r][col] -= fac[r] * M[jc][col];
    }
    __syncthreads();
  }
  const int RSZ = hg.RSZ;
  double* out = hg.rec + ((int64_t)g * hg.NSET + j) * RSZ;
  for (int e = t; e < Q1M * Q1M; e += blockDim.x) {
    const int r = e / Q1M, col = e - r * Q1M;
    const bool in = r < Q1 && col < Q1;
    out[e] = in ? M[r][Q1 + col] : 0.0;
    if (in) {
      const int a = min(r, col), b = max(r, col);
      out[Q1M * Q1M + e] = ent[a * Q1 - a * (a - 1) / 2 + (b - a)];
    } else {
      out[Q1M * Q1M + e] = 0.0;
    }
  }
  if (t < Q1M) {
    double p1 = 0.0, p2 = 0.0;
    if (has_y && t < Q1)
      for (int k = 0; k < Q1; ++k) {
        p1 += M[t][Q1 + k] * ent[nA + k];
        p2 += M[t][Q1 + k] * ent[nA + Q1 + k];
      }
    out[2 * Q1M * Q1M + t] = p1;
    out[2 * Q1M * Q1M + Q1M + t] = p2;
  }
  if (t == 0) {
    double r = 0.0;
    if (has_y) {
      r = ent[nA + 2 * Q1];
      for (int k = 0; k < Q1; ++k) {
        double p2 = 0.0;
        for (int l = 0; l < Q1; ++l) p2 += M[k][Q1 + l] * ent[nA + Q1 + l];
        r -= ent[nA + k] * p2;
      }
    }
    out[2 * Q1M * Q1M + 2 * Q1M] = r;
    out[2 * Q1M * Q1M + 2 * Q1M + 1] = ent[nE - 1];
  }
}

struct HybTile {
  int64_t p0;
  int32_t g, n;
};

/* A batch: second subgroups s2 .. s2 + nb - 1 of s1 (nb = 0: none), its groups of
 * columns (ngm against the genotypes, then those against their squares) and base
 * rows.  A column: its base row and the two presence words that it is masked with. */
struct HybBatch {
  int32_t s1, s2, nb, Q1, ngm, ng, nrow, pad;
};
struct HybColumn {
  uint8_t row, wa, wb, pad;
};

struct HybPair {
  const HybTile* tiles;
  const HybBatch* batches;
  const HybColumn* columns; /* [batch][16 HYB_NG] */
  const uint64_t* pres;  /* [G][S][W] presence bits from the chunk's levels  */
  const uint64_t* presp; /* the same from the pairwise levels (may be pres) */
  const double* cp;
  const double* yp;
  const double* rec;
  double* b;      /* [S][NP]    */
  double* Sig;    /* [S*S][NP]  */
  double* Vg;     /* [S*S][NP]  */
  int32_t* pgene; /* [NP]       */
  int32_t* n_out;
  double* sstats;
  int* flag;
  double fiterr;
  int NSET, RSZ, n_tiles, n_batch;
};

template <int Q1M>
__device__ inline double hyb_quad(const double* __restrict__ Ai, const double (&u)[Q1M], const double (&v)[Q1M]) {
  double s = 0.0;
#pragma unroll
  for (int a = 0; a < Q1M; ++a) {
    double r = 0.0;
#pragma unroll
    for (int b = 0; b < Q1M; ++b) r += Ai[a * Q1M + b] * v[b];
    s += u[a] * r;
  }
  return s;
}

/* presence bits: bit i of word w of (gene, subgroup) = individual 64 w + i
 * is genotyped in the subgroup and has a level (not NaN) in lev [G][S][N] */
__global__ void __launch_bounds__(64) hyb_pres_kernel(const eqbf_chunk c, const double* __restrict__ lev,
                                                      uint64_t* __restrict__ pres, int W) {
  const int g = blockIdx.x, s = blockIdx.y, lane = threadIdx.x;
  const int S = c.n_subgroups, N = c.n_samples;
  for (int w = 0; w < W; ++w) {
    const int i = w * 64 + lane;
    const bool in = i < N && c.geno_in_sbgrp[(int64_t)s * N + i] && !isnan(lev[((int64_t)g * S + s) * N + i]);
    const uint64_t m = __ballot(in);
    if (lane == 0) pres[((int64_t)g * S + s) * W + w] = m;
  }
}

/* The sums of the pairs of a tile (64 pairs of one gene) for a first subgroup s1
 * and nb second subgroups, as one FP64 matrix product of the tile's genotypes
 * with columns over the individuals: covariates and levels with zeros where the
 * sum's set has no member.  Columns: u1; u0 and x'y (with the first batch of
 * s1); per second subgroup u12, x'y1, x'y2, u2; then, against the squared
 * genotypes, the columns of ones of every set.
 *
 * Four waves: wave w takes the pairs 32 (w & 1) to + 31 and every second group of
 * 16 columns, so that a genotype operand serves up to three groups and a column
 * operand two tiles of 16 pairs.  The columns are not stored anywhere: a lane
 * reads its base row (covariate, level or ones) from LDS and masks it with its
 * set's presence word.  Rows are padded (HX_LD, HB_LD) so that the 16 rows x 2
 * steps of a half wave fall into different banks.  The sums pass through LDS
 * to the layout of one lane per pair for the closed forms.
 *
 * 48,000 pairs, 9 subgroups of 150, 3 covariates: 0.38 ms, of which the products
 * at the FP64 matrix rate are 0.14; the rest is staging and the closed forms, which
 * three workgroups per CU overlap only in part.  (One lane per pair with the sums
 * of two second subgroups in registers had 750 waves for 1,024 SIMDs, read the
 * genotypes S (S + 1) / 4 times and an LDS word per product: 2.35 ms.)  Past 8
 * covariates the closed forms' registers allow two workgroups. */
constexpr int HX_LD = 80, HB_LD = 66, HO_LD = 65;
constexpr int HYB_NG = 6; /* groups of 16 columns a workgroup has at most */

/* groups of a batch of nb second subgroups */
int hyb_main_groups(int Q1, bool first, int nb) { return (Q1 + (first ? Q1 + 1 : 0) + nb * (2 * Q1 + 2) + 15) / 16; }
int hyb_sq_groups(int nb) { return (2 + 2 * nb + 15) / 16; }

/* Base rows: ones, covariates of s1 (own, pairwise), levels of s1 (own, pairwise),
 * pairwise levels of the second subgroups.  Presence words: s1 by its own levels,
 * s1, the second subgroups (by the pairwise levels), none, all. */
HybColumn hyb_column(const HybBatch& t, int col) {
  const int Q1 = t.Q1, Q = Q1 - 1, none = 2 + t.nb, all = 3 + t.nb;
  const bool first = t.s2 == t.s1 + 1;
  auto make = [](int row, int wa, int wb) { return HybColumn{(uint8_t)row, (uint8_t)wa, (uint8_t)wb, 0}; };
  if (col >= 16 * t.ngm) {
    const int k = col - 16 * t.ngm, b = (k - 2) / 2;
    if (k < 2) return make(0, k, all);
    if (b >= t.nb) return make(0, none, all);
    return (k & 1) ? make(0, 2 + b, all) : make(0, 1, 2 + b);
  }
  int k = col;
  if (k < Q1) return make(k ? Q + k : 0, 1, all);
  k -= Q1;
  if (first) {
    if (k <= Q1) return make(k == Q1 ? 2 * Q + 1 : k, 0, all);
    k -= Q1 + 1;
  }
  const int b = k / (2 * Q1 + 2), r = k % (2 * Q1 + 2);
  if (b >= t.nb) return make(0, none, all);
  if (r < Q1) return make(r ? Q + r : 0, 1, 2 + b);
  if (r < Q1 + 2) return make(r == Q1 ? 2 * Q + 2 : 2 * Q + 3 + b, 1, 2 + b);
  return make(r > Q1 + 2 ? Q + r - Q1 - 2 : 0, 2 + b, all);
}

/* gene of each pair, -1 where the gene or the SNP is missing from a subgroup:
 * gene.cpp:314-321 skips such a pair, which has no sample size and no statistics */
__global__ void __launch_bounds__(64) hyb_skip_kernel(const eqbf_chunk c, const HybPair hp) {
  const HybTile tl = hp.tiles[blockIdx.x];
  const int lane = threadIdx.x, S = c.n_subgroups;
  if (lane >= tl.n) return;
  const int64_t p = tl.p0 + lane, NP = c.n_pairs, snp = c.pair_snp[p];
  bool ok = true;
  for (int s = 0; s < S; ++s)
    ok &= c.gene_in_sbgrp[(int64_t)tl.g * S + s] != 0 && c.snp_in_sbgrp[snp * S + s] != 0;
  hp.pgene[p] = ok ? tl.g : -1;
  if (ok) return;
  for (int s = 0; s < S; ++s) {
    hp.n_out[(int64_t)s * NP + p] = 0;
    if (hp.sstats)
      for (int k = 0; k < 5; ++k) hp.sstats[((int64_t)k * S + s) * NP + p] = NAN;
  }
}

template <int Q1M, class GT>
__global__ void __launch_bounds__(256, Q1M > 8 ? 2 : 3) hyb_pair_kernel(const eqbf_chunk c, const HybPair hp) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint64_t words[2 + 15 + 2];
  __shared__ unsigned long long badm;
  GT* const Xs = (GT*)smem;                                       /* [64][HX_LD] */
  double* const base = (double*)(smem + 64 * HX_LD * sizeof(GT)); /* [rows][HB_LD] */
  double* const sums = (double*)smem;                             /* [columns][HO_LD], after them */
  const int n_items = hp.n_tiles * hp.n_batch, per = (n_items + 7) / 8;
  /* the batches of a tile follow one another on one XCD */
  const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || item >= n_items) return;
  const HybBatch bt = hp.batches[item % hp.n_batch];
  const HybTile tl = hp.tiles[item / hp.n_batch];
  const int g = tl.g, s1 = bt.s1, nb = bt.nb;
  const bool first = bt.s2 == s1 + 1;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool act = lane < tl.n;
  const int64_t p = tl.p0 + (act ? lane : 0);
  const int64_t NP = c.n_pairs;
  const int S = c.n_subgroups, N = c.n_samples, QM = c.n_covars_max;
  const int W = (N + 63) >> 6;
  const bool ok = hp.pgene[p] >= 0 && act;
  const int64_t snp = c.pair_snp[p];
  const int Q1 = bt.Q1, Q = Q1 - 1, ngm = bt.ngm, ng = bt.ng, nrow = bt.nrow;
  const double* cov0 = c.covars + (int64_t)s1 * QM * N;
  const double* covp = hp.cp + (int64_t)s1 * QM * N;
  const double* y0 = c.explevels + ((int64_t)g * S + s1) * N;
  const double* yp1 = hp.yp + ((int64_t)g * S + s1) * N;
  const double* yp2 = hp.yp + ((int64_t)g * S + bt.s2) * N;
  const GT* xb = (const GT*)c.genotypes + (int64_t)c.geno_set_of_sbgrp[s1] * c.geno_set_stride + snp;
  const int64_t ld = c.geno_ld;
  auto base_row = [&](int row) {
    const double* r = cov0 + (int64_t)max(row - 1, 0) * N;
    r = row > Q ? covp + (int64_t)(row - Q - 1) * N : r;
    r = row == 2 * Q + 1 ? y0 : r;
    r = row == 2 * Q + 2 ? yp1 : r;
    r = row > 2 * Q + 2 ? yp2 + (int64_t)(row - 2 * Q - 3) * N : r;
    return row == 0 ? y0 : r; /* read, not used */
  };
  auto word_at = [&](int k, int w) -> uint64_t {
    if (k >= 2 + nb) return k == 2 + nb ? 0ull : ~0ull;
    if (k == 0) return hp.pres[((int64_t)g * S + s1) * W + w];
    return hp.presp[((int64_t)g * S + (k == 1 ? s1 : bt.s2 + k - 2)) * W + w];
  };
  const int half = wv & 1, kl = lane >> 4, pl = lane & 15;
  v4d acc[HYB_NG / 2][2];
  const HybColumn* const cols = hp.columns + (int64_t)(item % hp.n_batch) * (16 * HYB_NG);
  int row[HYB_NG / 2], wa[HYB_NG / 2], wb[HYB_NG / 2];
#pragma unroll
  for (int j = 0; j < HYB_NG / 2; ++j) {
    acc[j][0] = acc[j][1] = v4d{0.0, 0.0, 0.0, 0.0};
    const HybColumn cl = cols[min((wv >> 1) + 2 * j, ng - 1) * 16 + pl];
    row[j] = cl.row * HB_LD;
    wa[j] = cl.wa;
    wb[j] = cl.wb;
  }
  if (tid == 0) badm = 0ull;
  /* a chunk of 64 individuals, read while the one before is worked on: 16 of
   * them of the lane's pair, the lane's of every fourth base row, and a presence
   * word (past N the last individual once more: no set has it) */
  constexpr int BR = (2 * Q1M + 1 + 15 + 3) / 4;
  GT xv[16];
  double bv[BR];
  uint64_t wd = 0ull;
  auto load = [&](int c0) {
#pragma unroll
    for (int k = 0; k < 16; ++k) xv[k] = xb[(int64_t)min(c0 + 16 * wv + k, N - 1) * ld];
#pragma unroll
    for (int k = 0; k < BR; ++k)
      if (wv + 4 * k < nrow) bv[k] = base_row(wv + 4 * k)[min(c0 + lane, N - 1)];
    if (tid < 4 + nb) wd = word_at(tid, c0 >> 6);
  };
  bool bad = false; /* a genotype that is not finite: masked columns don't keep it out */
  load(0);
  for (int c0 = 0; c0 < N; c0 += 64) {
    const int n = min(64, N - c0);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      Xs[(16 * wv + k) * HX_LD + lane] = xv[k];
      bad |= !__builtin_isfinite(xv[k]);
    }
#pragma unroll
    for (int k = 0; k < BR; ++k)
      if (wv + 4 * k < nrow)
        base[(wv + 4 * k) * HB_LD + lane] = wv + 4 * k == 0 ? 1.0 : bv[k];
    if (tid < 4 + nb) words[tid] = wd;
    __syncthreads();
    if (c0 + 64 < N) load(c0 + 64);
    uint64_t m[HYB_NG / 2];
#pragma unroll
    for (int j = 0; j < HYB_NG / 2; ++j) m[j] = (words[wa[j]] & words[wb[j]]) >> kl;
    const GT* xr = Xs + kl * HX_LD + half * 32 + pl;
    const double* br = base + kl;
    /* four steps of J groups at a time, without a branch between their reads; SQ:
     * the last group's columns meet the squares (a wave has one at most) */
    auto steps = [&](auto J, auto SQ) {
      for (int k0 = 0; k0 < n; k0 += 16) {
        GT x0[4], x1[4];
        double v[4][J.value];
        int w[J.value];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          x0[k] = xr[(k0 + 4 * k) * HX_LD];
          x1[k] = xr[(k0 + 4 * k) * HX_LD + 16];
#pragma unroll
          for (int j = 0; j < J.value; ++j) v[k][j] = br[row[j] + k0 + 4 * k];
        }
#pragma unroll
        for (int j = 0; j < J.value; ++j) {
          w[j] = (int)m[j];
          m[j] >>= 16;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double b0 = (double)x0[k], b1 = (double)x1[k];
#pragma unroll
          for (int j = 0; j < J.value; ++j) {
            const int keep = __builtin_amdgcn_sbfe(w[j], 4 * k, 1);
            const double av = __hiloint2double(__double2hiint(v[k][j]) & keep, __double2loint(v[k][j]) & keep);
            const bool sq = SQ.value && j == J.value - 1;
            acc[j][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, sq ? b0 * b0 : b0, acc[j][0], 0, 0, 0);
            acc[j][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, sq ? b1 * b1 : b1, acc[j][1], 0, 0, 0);
          }
        }
      }
    };
    const int nj = (ng - (wv >> 1) + 1) >> 1; /* groups of this wave */
    using std::integral_constant;
    if ((wv >> 1) + 2 * (nj - 1) >= ngm) {
      if (nj == 1) steps(integral_constant<int, 1>(), std::true_type());
      if (nj == 2) steps(integral_constant<int, 2>(), std::true_type());
      if (nj == 3) steps(integral_constant<int, 3>(), std::true_type());
    } else {
      if (nj == 1) steps(integral_constant<int, 1>(), std::false_type());
      if (nj == 2) steps(integral_constant<int, 2>(), std::false_type());
      if (nj == 3) steps(integral_constant<int, 3>(), std::false_type());
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < HYB_NG / 2; ++j) {
    const int gr = (wv >> 1) + 2 * j;
    if (gr < ng) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sums[(gr * 16 + kl + 4 * r) * HO_LD + half * 32 + 16 * u + pl] = acc[j][u][r];
    }
  }
  if (__any(bad)) {
    const uint64_t bal = __ballot(bad);
    if (lane == 0) atomicOr(&badm, (unsigned long long)bal);
  }
  __syncthreads();
  if (badm != 0ull) { /* such pairs: the members of each set only, one by one */
    if ((badm >> lane) & 1ull)
      for (int col = wv; col < ng * 16; col += 4) {
        const HybColumn cl = cols[col];
        double a = 0.0;
        for (int i = 0; i < N; ++i)
          if (((word_at(cl.wa, i >> 6) & word_at(cl.wb, i >> 6)) >> (i & 63)) & 1ull) {
            const double x = (double)xb[(int64_t)i * ld];
            a += (cl.row == 0 ? 1.0 : base_row(cl.row)[i]) * (col >= 16 * ngm ? x * x : x);
          }
        sums[col * HO_LD + lane] = a;
      }
    __syncthreads();
  }
  /* closed forms, one lane per pair; wave w takes every fourth second subgroup */
  const int npr = S * (S - 1) / 2, RSZ = hp.RSZ;
  const double* R = hp.rec + (int64_t)g * hp.NSET * RSZ;
  const double f = hp.fiterr;
  auto col_at = [&](int col) { return sums[col * HO_LD + lane]; };
  /* records are zero past Q1, and so is what goes with them: no branches */
  auto take = [&](int col, double (&u)[Q1M]) {
#pragma unroll
    for (int a = 0; a < Q1M; ++a) {
      const double v = col_at(col + min(a, Q1 - 1));
      u[a] = a < Q1 ? v : 0.0;
    }
  };
  auto mul = [&](const double* __restrict__ Ai, const double (&u)[Q1M], double (&w)[Q1M]) {
#pragma unroll
    for (int a = 0; a < Q1M; ++a) {
      double r = 0.0;
#pragma unroll
      for (int b = 0; b < Q1M; ++b) r += Ai[a * Q1M + b] * u[b];
      w[a] = r;
    }
  };
  const int sq = 16 * ngm;
  /* w1 = A1^-1 u1, k1: the genotype column of M1^-1 is (-w1, 1) / k1 */
  double w1[Q1M], k1 = col_at(sq + 1);
  {
    double u1[Q1M];
    take(0, u1);
    mul(R + (int64_t)(S + s1) * RSZ, u1, w1);
#pragma unroll
    for (int a = 0; a < Q1M; ++a)
      k1 -= u1[a] * w1[a];
  }
  if (first && wv == 3) {
    const double* R0 = R + (int64_t)s1 * RSZ;
    double u0[Q1M];
    take(Q1, u0);
    const double k0 = col_at(sq) - hyb_quad<Q1M>(R0, u0, u0);
    double xty = col_at(2 * Q1);
#pragma unroll
    for (int a = 0; a < Q1M; ++a)
      xty -= u0[a] * R0[2 * Q1M * Q1M + a];
    const double rss0 = R0[2 * Q1M * Q1M + 2 * Q1M], n0 = R0[2 * Q1M * Q1M + 2 * Q1M + 1];
    const double rss1 = rss0 - xty * xty / k0;
    const double sg = f * rss1 / n0 + (1.0 - f) * rss0 / n0;
    if (ok) {
      hp.b[(int64_t)s1 * NP + p] = xty / k0;
      hp.Sig[(int64_t)(s1 * S + s1) * NP + p] = sg;
      hp.Vg[(int64_t)(s1 * S + s1) * NP + p] = sg / k0;
    }
  }
  const int col0 = Q1 + (first ? Q1 + 1 : 0);
  for (int b = wv; b < nb; b += 4) {
    const int s2 = bt.s2 + b, pi = s1 * S - s1 * (s1 + 1) / 2 + s2 - s1 - 1;
    const double* R2 = R + (int64_t)(2 * S + pi) * RSZ;
    const double* R3 = R + (int64_t)(2 * S + npr + pi) * RSZ;
    const double n12 = R2[2 * Q1M * Q1M + 2 * Q1M + 1];
    if (ok && !(n12 > 0.0)) atomicOr(hp.flag, FLAG_HYB_NO_COMMON);
    const int cb = col0 + b * (2 * Q1 + 2);
    double u12[Q1M];
    take(cb, u12);
    const double sxx12 = col_at(sq + 2 + 2 * b);
    const double k12 = sxx12 - hyb_quad<Q1M>(R2, u12, u12);
    double xty1 = col_at(cb + Q1), xty2 = col_at(cb + Q1 + 1);
#pragma unroll
    for (int a = 0; a < Q1M; ++a) {
      xty1 -= u12[a] * R2[2 * Q1M * Q1M + a];
      xty2 -= u12[a] * R2[2 * Q1M * Q1M + Q1M + a];
    }
    const double s12 = R2[2 * Q1M * Q1M + 2 * Q1M] / n12 - f * xty1 * xty2 / (k12 * n12);
    double u2[Q1M], w2[Q1M];
    take(cb + Q1 + 2, u2);
    mul(R3, u2, w2);
    double k2 = col_at(sq + 3 + 2 * b), wu = 0.0;
#pragma unroll
    for (int a = 0; a < Q1M; ++a) {
      k2 -= u2[a] * w2[a];
      wu += w1[a] * u12[a] + u12[a] * w2[a];
    }
    const double aw = hyb_quad<Q1M>(R2 + Q1M * Q1M, w1, w2);
    const double a11 = (aw - wu + sxx12) / (k1 * k2);
    if (ok) {
      hp.Sig[(int64_t)(s1 * S + s2) * NP + p] = s12;
      hp.Sig[(int64_t)(s2 * S + s1) * NP + p] = s12;
      hp.Vg[(int64_t)(s1 * S + s2) * NP + p] = s12 * a11;
      hp.Vg[(int64_t)(s2 * S + s1) * NP + p] = s12 * a11;
    }
  }
}

/* per (pair, configuration): Vg^-1, Vg^-1 t, t = gamma o sqrt(diag Sigma),
 * Vg^-1 b and k = 1, in the layout of mvlr_grid_kernel */
struct HybCfg {
  const double* b;
  const double* Sig;
  const double* Vg;
  const int32_t* pgene;
  const uint64_t* masks;
  double* par;
  int cfg0, PSZ;
};

template <int SM>
__global__ void __launch_bounds__(64) hyb_cfg_kernel(const eqbf_chunk c, const HybCfg hc) {
  const int64_t NP = c.n_pairs;
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= NP) return;
  const int ci = blockIdx.y;
  const int S = c.n_subgroups, PSZ = hc.PSZ;
  double* out = hc.par + (int64_t)ci * PSZ * NP + p;
  if (hc.pgene[p] < 0) {
    out[(int64_t)(PSZ - 1) * NP] = 1.0;
    return;
  }
  const uint64_t gm = hc.masks[hc.cfg0 + ci];
  double A[SM][SM], b[SM], tv[SM];
#pragma unroll
  for (int i = 0; i < SM; ++i) {
    b[i] = (i < S) ? hc.b[(int64_t)i * NP + p] : 0.0;
    tv[i] = (i < S && ((gm >> i) & 1ull)) ? sqrt(hc.Sig[(int64_t)(i * S + i) * NP + p]) : 0.0;
#pragma unroll
    for (int j = 0; j < SM; ++j) A[i][j] = (i < S && j < S) ? hc.Vg[(int64_t)(i * S + j) * NP + p] : (i == j ? 1.0 : 0.0);
  }
  int piv[SM];
  (void)lu_factor<SM>(A, piv);
  double u[SM], eVb[SM];
#pragma unroll
  for (int i = 0; i < SM; ++i) u[i] = eVb[i] = 0.0;
  for (int col = 0; col < S; ++col) {
    double e[SM];
#pragma unroll
    for (int i = 0; i < SM; ++i) e[i] = (i == col) ? 1.0 : 0.0;
    lu_apply<SM>(A, piv, e);
    double tc = 0, bc = 0;
#pragma unroll
    for (int j = 0; j < SM; ++j)
      if (j == col) {
        tc = tv[j];
        bc = b[j];
      }
#pragma unroll
    for (int i = 0; i < SM; ++i)
      if (i < S) {
        out[(int64_t)(i * S + col) * NP] = e[i];
        u[i] += e[i] * tc;
        eVb[i] += e[i] * bc;
      }
  }
#pragma unroll
  for (int i = 0; i < SM; ++i)
    if (i < S) {
      out[(int64_t)(S * S + i) * NP] = u[i];
      out[(int64_t)(S * S + S + i) * NP] = tv[i];
      out[(int64_t)(S * S + 2 * S + i) * NP] = eVb[i];
    }
  out[(int64_t)(S * S + 3 * S) * NP] = 1.0;
  out[(int64_t)(PSZ - 1) * NP] = 0.0;
}

template <int SM, int Q1M>
int hybrid_run_sm(eqbf_ctx* ctx, const eqbf_chunk& c, const eqbf_hybrid_opts* o, eqbf_assoc_out* out,
                  hipStream_t st) {
  const int S = c.n_subgroups, N = c.n_samples, G = c.n_genes;
  const int64_t NP = c.n_pairs;
  const int64_t n_cfg = eqbf_n_configs(o->bfs, S);
  /* sample sizes and summary statistics: the separate analysis; the batched
   * path (FP64 sums when summary statistics are asked for) where it applies,
   * else the FP64 plain path */
  int KU = 1;
  while (KU < c.n_covars_max + 1) KU = (KU == 1) ? 4 : KU * 2;
  const int prec = uvlr_fast_eligible(c, KU) ? EQBF_PREC_MIXED : EQBF_PREC_FP64_BATCHED;
  eqbf_assoc_opts so{EQBF_ANALYSIS_SEP, EQBF_BFS_GEN, prec, EQBF_F64};
  eqbf_assoc_out sout;
  memset(&sout, 0, sizeof sout);
  sout.n = out->n;
  sout.sstats = out->sstats;
  int rc = assoc_uvlr_run(ctx, &c, &so, &sout, st);
  if (rc) return rc;
  const int npr = S * (S - 1) / 2;
  const int NSET = 2 * S + 2 * npr;
  const int RSZ = 2 * Q1M * Q1M + 2 * Q1M + 2;
  /* tiles of at most 64 pairs of one gene */
  std::vector<int64_t> off(G + 1);
  std::vector<int32_t> q1(S);
  EQBF_HIP(ctx, hipMemcpyAsync(off.data(), c.pair_offset, (G + 1) * sizeof(int64_t), hipMemcpyDeviceToHost, st));
  EQBF_HIP(ctx, hipMemcpyAsync(q1.data(), c.covar_count, S * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  EQBF_HIP(ctx, hipStreamSynchronize(st));
  std::vector<HybTile> tiles;
  for (int g = 0; g < G; ++g)
    for (int64_t p0 = off[g]; p0 < off[g + 1]; p0 += 64)
      tiles.push_back(HybTile{p0, g, (int32_t)std::min<int64_t>(64, off[g + 1] - p0)});
  if (tiles.empty()) return EQBF_OK;
  /* batches of second subgroups: as many as a workgroup's groups of columns
   * hold, of even size */
  std::vector<HybBatch> batches;
  std::vector<HybColumn> columns;
  size_t lds = 0;
  for (int s1 = 0; s1 < S; ++s1) {
    const int Q1 = std::min(std::max(q1[s1], 0), c.n_covars_max) + 1, n2 = S - 1 - s1;
    int nb_max = 15;
    while (hyb_main_groups(Q1, true, nb_max) + hyb_sq_groups(nb_max) > HYB_NG) --nb_max;
    const int k = std::max(1, (n2 + nb_max - 1) / nb_max);
    for (int b = 0; b < k; ++b) {
      const int lo = s1 + 1 + n2 * b / k, nb = s1 + 1 + n2 * (b + 1) / k - lo;
      const int ngm = hyb_main_groups(Q1, b == 0, nb);
      batches.push_back(HybBatch{s1, lo, nb, Q1, ngm, ngm + hyb_sq_groups(nb), 2 * Q1 + 1 + nb, 0});
      const HybBatch& t = batches.back();
      for (int col = 0; col < 16 * HYB_NG; ++col)
        columns.push_back(col < 16 * t.ng ? hyb_column(t, col) : HybColumn{});
      const size_t in = 64 * HX_LD * (c.geno_dtype == EQBF_F32 ? 4 : 8) + (size_t)t.nrow * HB_LD * 8;
      lds = std::max(lds, std::max(in, (size_t)16 * t.ng * HO_LD * 8));
    }
  }
  const size_t tb = tiles.size() * sizeof(HybTile), btb = batches.size() * sizeof(HybBatch);
  std::vector<unsigned char> lists(tb + btb + columns.size() * sizeof(HybColumn));
  memcpy(lists.data(), tiles.data(), tb);
  memcpy(lists.data() + tb, batches.data(), btb);
  memcpy(lists.data() + tb + btb, columns.data(), lists.size() - tb - btb);
  if (tiles.size() * batches.size() > (size_t)INT32_MAX - 8)
    return ctx_fail(ctx, EQBF_ERR_UNSUPPORTED, "too many pairs in a chunk for --error hybrid");
  HybTile* dtiles = (HybTile*)ctx_buf(ctx, "hyb_tiles", lists.size());
  double* rec = (double*)ctx_buf(ctx, "hyb_rec", (size_t)G * NSET * RSZ * sizeof(double));
  double* bb = (double*)ctx_buf(ctx, "hyb_b", (size_t)S * NP * sizeof(double));
  double* sig = (double*)ctx_buf(ctx, "hyb_sig", (size_t)S * S * NP * sizeof(double));
  double* vg = (double*)ctx_buf(ctx, "hyb_vg", (size_t)S * S * NP * sizeof(double));
  int32_t* pgene = (int32_t*)ctx_buf(ctx, "mv_pgene", (size_t)NP * sizeof(int32_t));
  std::vector<uint64_t> hm(1 + n_cfg);
  hm[0] = (S >= 64) ? ~0ull : ((1ull << S) - 1ull);
  if (n_cfg > 0) eqbf_config_masks(o->bfs, S, hm.data() + 1);
  uint64_t* dmask = (uint64_t*)ctx_buf(ctx, "mv_masks", hm.size() * sizeof(uint64_t));
  if (!dtiles || !rec || !bb || !sig || !vg || !pgene || !dmask)
    return ctx_fail(ctx, EQBF_ERR_HIP, "allocating hybrid buffers failed");
  EQBF_HIP(ctx, hipMemcpyAsync(dtiles, lists.data(), lists.size(), hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipMemcpyAsync(dmask, hm.data(), hm.size() * sizeof(uint64_t), hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipStreamSynchronize(st)); /* the host vectors go out of scope */
  HybGene hg;
  hg.cp = o->covars_by_position ? o->covars_by_position : c.covars;
  hg.yp = o->explevels_pairs ? o->explevels_pairs : c.explevels;
  hg.rec = rec;
  hg.NSET = NSET;
  hg.RSZ = RSZ;
  hg.Q1M = Q1M;
  {
    ProfScope ps(ctx, "hyb_gene_kernel", st);
    hipLaunchKernelGGL(hyb_gene_kernel, dim3(G, NSET), dim3(256), 0, st, c, hg);
  }
  const int W = (N + 63) / 64;
  const bool split = hg.yp != c.explevels;
  uint64_t* pres = (uint64_t*)ctx_buf(ctx, "hyb_pres", (size_t)(split ? 2 : 1) * G * S * W * sizeof(uint64_t));
  if (!pres) return ctx_fail(ctx, EQBF_ERR_HIP, "allocating hybrid buffers failed");
  uint64_t* presp = split ? pres + (size_t)G * S * W : pres;
  hipLaunchKernelGGL(hyb_pres_kernel, dim3(G, S), dim3(64), 0, st, c, c.explevels, pres, W);
  if (split) hipLaunchKernelGGL(hyb_pres_kernel, dim3(G, S), dim3(64), 0, st, c, hg.yp, presp, W);
  HybPair hp;
  hp.tiles = dtiles;
  hp.batches = (const HybBatch*)(dtiles + tiles.size());
  hp.columns = (const HybColumn*)(hp.batches + batches.size());
  hp.n_tiles = (int)tiles.size();
  hp.n_batch = (int)batches.size();
  hp.pres = pres;
  hp.presp = presp;
  hp.cp = hg.cp;
  hp.yp = hg.yp;
  hp.rec = rec;
  hp.b = bb;
  hp.Sig = sig;
  hp.Vg = vg;
  hp.pgene = pgene;
  hp.n_out = out->n;
  hp.sstats = out->sstats;
  hp.flag = (int*)ctx->d_flag.ptr;
  hp.fiterr = o->fiterr;
  hp.NSET = NSET;
  hp.RSZ = RSZ;
  hipLaunchKernelGGL(hyb_skip_kernel, dim3((unsigned)tiles.size()), dim3(64), 0, st, c, hp);
  {
    ProfScope ps(ctx, "hyb_pair_kernel", st);
    const dim3 grid((unsigned)((tiles.size() * batches.size() + 7) / 8 * 8));
    if (c.geno_dtype == EQBF_F32)
      hipLaunchKernelGGL((hyb_pair_kernel<Q1M, float>), grid, dim3(256), lds, st, c, hp);
    else
      hipLaunchKernelGGL((hyb_pair_kernel<Q1M, double>), grid, dim3(256), lds, st, c, hp);
  }
  EQBF_HIP(ctx, hipGetLastError());
  return mv_rows_run<SM>(ctx, c, o->bfs, out, st, [&](int64_t c0, int nb, double* par, int PSZ, int64_t pair_blocks) {
    HybCfg hc;
    hc.b = bb;
    hc.Sig = sig;
    hc.Vg = vg;
    hc.pgene = pgene;
    hc.masks = dmask;
    hc.par = par;
    hc.cfg0 = (int)c0;
    hc.PSZ = PSZ;
    ProfScope ps(ctx, "hyb_cfg_kernel", st);
    with_exact_sm<SM>(c.n_subgroups, [&](auto e) {
      hipLaunchKernelGGL(hyb_cfg_kernel<decltype(e)::value>, dim3((unsigned)pair_blocks, (unsigned)nb), dim3(64), 0,
                         st, c, hc);
    });
  });
}

template <int SM>
int hybrid_run_q(eqbf_ctx* ctx, const eqbf_chunk& c, const eqbf_hybrid_opts* o, eqbf_assoc_out* out,
                 hipStream_t st) {
  const int Q1 = c.n_covars_max + 1;
  if (Q1 <= 4) return hybrid_run_sm<SM, 4>(ctx, c, o, out, st);
  if (Q1 <= 8) return hybrid_run_sm<SM, 8>(ctx, c, o, out, st);
  return hybrid_run_sm<SM, 17>(ctx, c, o, out, st);
}

}  // namespace

int mvlr_run(eqbf_ctx* ctx, const eqbf_chunk* cp, const eqbf_mvlr_opts* o, eqbf_assoc_out* out, hipStream_t st) {
  const eqbf_chunk& c = *cp;
  const int S = c.n_subgroups, N = c.n_samples, G = c.n_genes;
  const int GL = (int)ctx->phiL.size(), GS = (int)ctx->phiS.size();
  if (S < 1 || S > 16) return ctx_fail(ctx, EQBF_ERR_UNSUPPORTED, "--error mvlr supports 1 to 16 subgroups (S=%d)", S);
  if (N < 1 || G < 0 || c.n_pairs < 0 || c.n_covars_max < 0 || c.n_covars_max > 16)
    return ctx_fail(ctx, EQBF_ERR_ARG, "chunk sizes out of range (N=%d G=%d Q=%d)", N, G, c.n_covars_max);
  if (o->bfs != EQBF_BFS_GEN && o->bfs != EQBF_BFS_SIN && o->bfs != EQBF_BFS_ALL)
    return ctx_fail(ctx, EQBF_ERR_ARG, "unknown --bfs value %d", o->bfs);
  if (!(o->fiterr >= 0.0 && o->fiterr <= 1.0)) return ctx_fail(ctx, EQBF_ERR_ARG, "--fiterr must be in [0, 1]");
  if (GL < 1 || (o->bfs != EQBF_BFS_GEN && GS < 1))
    return ctx_fail(ctx, EQBF_ERR_ARG, "--error mvlr needs the grids (eqbf_set_grids)");
  if (!out || !out->n || !out->w_abf || !out->raw_abf) return ctx_fail(ctx, EQBF_ERR_ARG, "missing output buffers");
  if (G == 0 || c.n_pairs == 0) return EQBF_OK;
  if (S <= 4) return mvlr_run_sm<4>(ctx, c, o, out, st);
  if (S <= 8) return mvlr_run_sm<8>(ctx, c, o, out, st);
  if (S <= 12) return mvlr_run_sm<12>(ctx, c, o, out, st);
  return mvlr_run_sm<16>(ctx, c, o, out, st);
}

int hybrid_run(eqbf_ctx* ctx, const eqbf_chunk* cp, const eqbf_hybrid_opts* o, eqbf_assoc_out* out, hipStream_t st) {
  const eqbf_chunk& c = *cp;
  const int S = c.n_subgroups, N = c.n_samples, G = c.n_genes;
  const int GL = (int)ctx->phiL.size(), GS = (int)ctx->phiS.size();
  if (S < 1 || S > 16) return ctx_fail(ctx, EQBF_ERR_UNSUPPORTED, "--error hybrid supports 1 to 16 subgroups (S=%d)", S);
  if (N < 1 || G < 0 || c.n_pairs < 0 || c.n_covars_max < 0 || c.n_covars_max > 16)
    return ctx_fail(ctx, EQBF_ERR_ARG, "chunk sizes out of range (N=%d G=%d Q=%d)", N, G, c.n_covars_max);
  if (o->bfs != EQBF_BFS_GEN && o->bfs != EQBF_BFS_SIN && o->bfs != EQBF_BFS_ALL)
    return ctx_fail(ctx, EQBF_ERR_ARG, "unknown --bfs value %d", o->bfs);
  if (!(o->fiterr >= 0.0 && o->fiterr <= 1.0)) return ctx_fail(ctx, EQBF_ERR_ARG, "--fiterr must be in [0, 1]");
  if (GL < 1 || (o->bfs != EQBF_BFS_GEN && GS < 1))
    return ctx_fail(ctx, EQBF_ERR_ARG, "--error hybrid needs the grids (eqbf_set_grids)");
  if (!out || !out->n || !out->w_abf || !out->raw_abf) return ctx_fail(ctx, EQBF_ERR_ARG, "missing output buffers");
  if (G == 0 || c.n_pairs == 0) return EQBF_OK;
  if (S <= 4) return hybrid_run_q<4>(ctx, c, o, out, st);
  if (S <= 8) return hybrid_run_q<8>(ctx, c, o, out, st);
  if (S <= 12) return hybrid_run_q<12>(ctx, c, o, out, st);
  return hybrid_run_q<16>(ctx, c, o, out, st);
}
