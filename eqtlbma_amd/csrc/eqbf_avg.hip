/*
 * eqtlbma_avg_bfs on the device: raw log10 ABFs averaged over the grid and
 * over the configurations or types, gene and SNP Bayes factors and the
 * posteriors (src/eqtlbma_avg_bfs.cpp:371-796).
 *
 * Layout: raw [n_pairs][R][L] in FP64, R = dim rows (configs model: the
 * j-th configuration row of the SNP) or n_subgroups rows (types model:
 * subgroup-specific rows); a gene's pairs are contiguous (gene_offset).
 * Every sum is utils::log10_weighted_sum (utils_math.cpp:100-159): the
 * maximum starts from the first value (a NaN first value makes the result
 * NaN), NaN terms are skipped, |result| <= DBL_EPSILON gives 0.
 *
 * Kernels:
 *   avg_grid_kernel  one thread per raw row: the row averaged over the kept
 *                    grid points (BayesFactor::avg_raw_bfs, :371-382)
 *   avg_pair_kernel  one wave per pair (four waves a block striding over
 *                    the pairs), lanes over the dimensions: the
 *                    per-dimension BFs (Snp::avg_raw_bfs, :418-475), the
 *                    SNP BF over them and the first strict maximum; then,
 *                    when asked, post_dim and its argmax (:683-718) and the
 *                    configs model's subgroup posteriors (:722-745)
 *   avg_rows_kernel  the same for the configs model where every grid point is
 *                    kept and a row fits a lane's registers (at most 16
 *                    points, 64 configurations)
 *   avg_gene_kernel  one wave per gene, lanes over its SNPs: the gene BF
 *                    (Gene::avg_raw_bfs, :598-622), gene_post (:634-643),
 *                    post_the (:647-662), post_an (:664-680)
 *   avg_post_kernel  the types model's subgroup posteriors (:749-796)
 * The roofline is HBM: each raw value is read once by avg_pair_kernel (and
 * again by avg_post_kernel for the types model's subgroup posteriors).
 */
#include <algorithm>
#include <cstring>
#include <vector>

#include "eqbf_internal.h"

namespace {

constexpr double kEps = 2.220446049250313e-16;

__device__ inline double wmax(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ inline double wsum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ inline double l10_round(double r) { return fabs(r) <= kEps ? 0.0 : r; }

struct AvgArgs {
  const double* raw;
  const int64_t* off;
  const int32_t* keep;
  const double* gw;   /* [L] grid weights                          */
  const double* dw;   /* [D] configuration or type weights         */
  const uint64_t* cs; /* [D] subgroups of each configuration        */
  const double* sw;   /* [D][S] subgroup weights per type           */
  double* gene_bf;
  double* gene_post;
  double* snp_bf;
  double* dim_bf;
  double* post_the;
  double* post_an;
  double* post_dim;
  double* post_sub;
  int32_t* best_dim;
  double pi0;
  int64_t NP, G;
  int D, S, L, nk, types, want;
  double gw_row[16]; /* the grid weights as kernel arguments, where L fits and every point is kept */
};

/* sum over the subgroups of log10(q 10^x + 1 - q) at kept grid point i,
 * skipping subgroup `skip` (types model, :464-466, :778-782) */
__device__ inline double types_point(const AvgArgs& a, int64_t p, int k, int i, int skip) {
  const double* r = a.raw + (size_t)p * a.S * a.L + a.keep[i];
  double v = 0.0;
  for (int s = 0; s < a.S; ++s) {
    if (s == skip) continue;
    const double q = a.sw[(size_t)k * a.S + s];
    v += log10(q * exp10(r[(size_t)s * a.L]) + 1 - q);
  }
  return v;
}

/* log10 sum_i w_i 10^v_i over the kept grid points, values from f(i) */
template <class F>
__device__ inline double grid_lws(const AvgArgs& a, F f) {
  double mx = f(0);
  for (int i = 1; i < a.nk; ++i) {
    const double v = f(i);
    if (v > mx) mx = v;
  }
  double sum = 0.0;
  for (int i = 0; i < a.nk; ++i) {
    const double v = f(i);
    if (!isnan(v)) sum += a.gw[a.keep[i]] * exp10(v - mx);
  }
  return l10_round(mx + log10(sum));
}

__global__ void __launch_bounds__(256) avg_grid_kernel(const double* __restrict__ raw, int64_t n_rows, int L,
                                                       const double* __restrict__ gw, const int32_t* __restrict__ keep,
                                                       int nk, double* __restrict__ out) {
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= n_rows) return;
  const double* v = raw + r * L;
  double mx = v[keep[0]];
  for (int i = 1; i < nk; ++i)
    if (v[keep[i]] > mx) mx = v[keep[i]];
  double sum = 0.0;
  for (int i = 0; i < nk; ++i) {
    const double x = v[keep[i]];
    if (!isnan(x)) sum += gw[keep[i]] * exp10(x - mx);
  }
  out[r] = l10_round(mx + log10(sum));
}

/* Value of the lane that a step of a butterfly over aligned groups pairs this
 * one with: within 16 lanes by data-parallel moves (quads by permutation, the
 * halves mirrored, which pairs equal partial results), 16 and 32 apart through
 * LDS. */
template <int STEP>
__device__ __forceinline__ int partner(int v) {
  if (STEP == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);  /* quad [1,0,3,2] */
  if (STEP == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);  /* quad [2,3,0,1] */
  if (STEP == 4) return __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true); /* 8 lanes mirrored */
  if (STEP == 8) return __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true); /* 16 lanes mirrored */
  return __shfl_xor(v, STEP, 64);
}
template <int STEP>
__device__ __forceinline__ double partner(double v) {
  return __hiloint2double(partner<STEP>(__double2hiint(v)), partner<STEP>(__double2loint(v)));
}
/* reduction over the aligned group of w lanes (w a power of two <= 64), the
 * result in every lane */
template <class T, class F>
__device__ __forceinline__ T greduce(T v, int w, F f) {
  if (w > 1) v = f(v, partner<1>(v));
  if (w > 2) v = f(v, partner<2>(v));
  if (w > 4) v = f(v, partner<4>(v));
  if (w > 8) v = f(v, partner<8>(v));
  if (w > 16) v = f(v, partner<16>(v));
  if (w > 32) v = f(v, partner<32>(v));
  return v;
}
__device__ __forceinline__ double gmax(double v, int w) {
  return greduce(v, w, [](double a, double b) { return fmax(a, b); });
}
__device__ __forceinline__ double gsum(double v, int w) {
  return greduce(v, w, [](double a, double b) { return a + b; });
}

/* first index of the strict maximum scanning from index 0 (the reference's
 * "j == 0 || v[j] > v[best]"): v0 is the first value, mx the group's largest,
 * (lmax, larg) the lane's largest value and its first index (larg = n when it
 * has none) */
__device__ __forceinline__ int first_max(double v0, double mx, double lmax, int larg, int n, int w) {
  const int cand = greduce((larg < n && lmax == mx) ? larg : n, w, [](int a, int b) { return min(a, b); });
  if (isnan(v0) || !(mx > v0)) return 0;
  return cand >= n ? 0 : cand;
}

/* Posterior of a dimension of weight w and log10 BF d: its term t of the SNP's
 * sum over that sum, against mx; where the sum leaves the normal numbers (the
 * largest d has weight 0, or a weight is negative), the reference's expression. */
__device__ __noinline__ double post_apart(double w, double d, double mx, double sum) {
  return exp10(log10(w) + d - l10_round(mx + log10(sum)));
}
__device__ __forceinline__ double post_of(double w, double t, double sum, double d, double mx) {
  if (__builtin_expect(!(sum > 1e-290) || !(w >= 0.0), 0)) return post_apart(w, d, mx, sum);
  return t / sum;
}

constexpr int kAvgWaves = 4;
constexpr int kAvgRow = 16; /* longest row that a lane holds in registers (AvgArgs::gw_row) */

/* log10 sum_i w_i 10^r_i over a row of LV values that all are kept: the row in
 * registers, 16-byte loads where VEC; a row with a value that is not finite
 * goes through the general form */
template <int LV, bool VEC>
__device__ __forceinline__ double row_lws(const AvgArgs& a, const double* __restrict__ r) {
  double x[LV];
  if (VEC) {
#pragma unroll
    for (int i = 0; i + 1 < LV; i += 2) {
      const double2 t = *reinterpret_cast<const double2*>(r + i);
      x[i] = t.x;
      x[i + 1] = t.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < LV; ++i) x[i] = r[i];
  }
  double mx = x[0], z = 0.0;
#pragma unroll
  for (int i = 0; i < LV; ++i) {
    mx = fmax(mx, x[i]);
    z = fma(0.0, x[i], z);
  }
  if (__builtin_expect(isnan(z), 0)) return grid_lws(a, [&](int i) { return r[i]; });
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < LV; ++i) sum = fma(a.gw_row[i], dm::exp10_core(fmax(x[i] - mx, -400.0)), sum);
  return l10_round(mx + log10(sum));
}

/* A group of w lanes per pair (w = the power of two >= dim, at most 64:
 * 64 / w pairs a wave), four waves a block striding over the pairs; lanes
 * over the dimensions.  Also writes post_dim, its best dimension and the
 * configs model's subgroup posteriors when asked: they need only the pair's
 * own values, and the posterior of a dimension is its term of the SNP's sum
 * over that sum.  The general form: any number of dimensions, kept points and
 * row lengths, both models. */
__global__ void __launch_bounds__(64 * kAvgWaves) avg_pair_kernel(const AvgArgs a, int w) {
  const int lane = threadIdx.x & 63;
  const int gl = lane & (w - 1), g0 = lane - gl; /* lane in the group, group's first lane */
  const int per_wave = 64 / w;
  const int D = a.D;
  const bool dims_post = (a.want & 16) || (!a.types && (a.want & 8));
  const bool sub_post = !a.types && (a.want & 8);
  /* the lane's first dimension: its weight and subgroups stay in registers */
  const double dw0 = gl < D ? a.dw[gl] : 0.0;
  const uint64_t cs0 = sub_post && gl < D ? a.cs[gl] : 0;
  const int64_t step = (int64_t)gridDim.x * kAvgWaves * per_wave;
  for (int64_t pb = ((int64_t)blockIdx.x * kAvgWaves + (threadIdx.x >> 6)) * per_wave; pb < a.NP; pb += step) {
    const int64_t p = pb + lane / w;
    const bool on = p < a.NP; /* every lane still takes part in the shuffles */
    double* dims = a.dim_bf + (size_t)p * D;
    /* per-dimension BFs; the lane's largest value and its first index */
    double lmax = -INFINITY, dk = NAN;
    int larg = D;
    for (int k = gl; on && k < D; k += w) {
      double d;
      if (!a.types) {
        const double* r = a.raw + ((size_t)p * D + k) * a.L;
        d = grid_lws(a, [&](int i) { return r[a.keep[i]]; });
      } else {
        d = grid_lws(a, [&](int i) { return types_point(a, p, k, i, -1); });
      }
      dims[k] = d;
      if (k == gl) dk = d;
      if (d > lmax) {
        lmax = d;
        larg = k;
      }
    }
    const double d0 = __shfl(dk, g0, 64); /* the group's first lane holds dims[0] */
    /* maximum as the reference scans it: from the first value, strict > */
    const double top = gmax(lmax, w);
    double mx = top;
    if (isnan(d0)) mx = NAN;
    if (!(mx > d0)) mx = d0;
    int best = a.types ? -1 : first_max(d0, top, lmax, larg, D, w);
    /* the terms w_k 10^(d_k - mx) of the SNP's sum, the first one kept */
    double sum = 0.0, tk = 0.0;
    for (int k = gl; on && k < D; k += w) {
      const double d = (k == gl) ? dk : dims[k];
      const double t = ((k == gl) ? dw0 : a.dw[k]) * dm::exp10_sum(d - mx);
      if (k == gl) tk = t;
      if (!isnan(d)) sum += t;
    }
    sum = gsum(sum, w);
    const double sbp = l10_round(mx + log10(sum));
    if (dims_post) {
      double* pd = a.post_dim + (size_t)p * D;
      double pmax = -INFINITY, pk = NAN;
      int parg = D;
      for (int k = gl; on && k < D; k += w) {
        const double wk = (k == gl) ? dw0 : a.dw[k];
        const double t = (k == gl) ? tk : wk * dm::exp10_sum(dims[k] - mx);
        double v = post_of(wk, t, sum, (k == gl) ? dk : dims[k], mx);
        if (v > 1.0) v = 1.0;
        pd[k] = v;
        if (k == gl) pk = v;
        if (v > pmax) {
          pmax = v;
          parg = k;
        }
      }
      best = first_max(__shfl(pk, g0, 64), gmax(pmax, w), pmax, parg, D, w);
      if (sub_post) {
        for (int s = 0; s < a.S; ++s) {
          double acc = 0.0;
          for (int k = gl; on && k < D; k += w)
            if ((((k == gl) ? cs0 : a.cs[k]) >> s) & 1ull) acc += (k == gl) ? pk : pd[k];
          acc = gsum(acc, w);
          if (on && gl == 0) a.post_sub[(size_t)p * a.S + s] = acc > 1.0 ? 1.0 : acc;
        }
      }
    }
    if (on && gl == 0) {
      a.snp_bf[p] = sbp;
      a.best_dim[p] = best;
    }
  }
}

/* Configs model with at most 64 dimensions and rows of LV values that are all
 * kept: a wave takes n_it passes of 64 / w pairs, one lane per row.
 *
 * Bound by the FP64 instructions (11 exponentials and a logarithm per row and
 * six reductions over the lanes of a pair) next to the one read of the raw
 * values.  So a row is held in registers (16-byte loads where VEC), the SNP's
 * logarithms wait in LDS until the wave has one for each of its lanes, and a
 * posterior is its term over the sum instead of a logarithm and an exponential
 * of its own.  On 9.0e5 pairs of 31 x 10 values with every posterior 0.67 ms
 * (4.1 TB/s); the general form took 2.0 ms. */
template <int LV, bool VEC>
__global__ void __launch_bounds__(64 * kAvgWaves) __attribute__((amdgpu_waves_per_eu(4, 8)))
avg_rows_kernel(const AvgArgs a, int w, int n_it) {
  __shared__ double2 held[kAvgWaves][64]; /* maximum and sum of each pair of the wave */
  __shared__ int hbest[kAvgWaves][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int gl = lane & (w - 1), grp = lane / w, g0 = lane - gl;
  const int per_wave = 64 / w, D = a.D;
  const bool dims_post = a.want & (16 | 8), sub_post = a.want & 8;
  const bool in = gl < D;
  const double dw0 = in ? a.dw[gl] : 0.0;
  const uint64_t cs0 = sub_post && in ? a.cs[gl] : 0;
  const int64_t base = ((int64_t)blockIdx.x * kAvgWaves + wv) * (n_it * per_wave);
  const int n_pairs = (int)min((int64_t)n_it * per_wave, max(a.NP - base, (int64_t)0));
  for (int q = grp; q - grp < n_pairs; q += per_wave) {
    const int64_t p = base + q;
    const bool on = q < n_pairs && in; /* every lane takes part in the reductions */
    double d = NAN;
    if (on) {
      d = row_lws<LV, VEC>(a, a.raw + ((size_t)p * D + gl) * LV);
      a.dim_bf[(size_t)p * D + gl] = d;
    }
    const double d0 = __shfl(d, g0, 64);
    /* maximum as the reference scans it: from the first value, strict > */
    const double lmax = d > -INFINITY ? d : -INFINITY, top = gmax(lmax, w);
    double mx = top;
    if (isnan(d0)) mx = NAN;
    if (!(mx > d0)) mx = d0;
    const double t = dw0 * dm::exp10_sum(d - mx);
    const double sum = gsum(isnan(d) ? 0.0 : t, w);
    int best;
    if (dims_post) {
      double v = post_of(dw0, t, sum, d, mx);
      if (v > 1.0) v = 1.0;
      if (on) a.post_dim[(size_t)p * D + gl] = v;
      const double pmax = v > -INFINITY && on ? v : -INFINITY;
      best = first_max(__shfl(v, g0, 64), gmax(pmax, w), pmax, v > -INFINITY && on ? gl : D, D, w);
      if (sub_post) {
        /* lane s of the group keeps subgroup s */
        double mine = 0.0;
        for (int s = 0; s < a.S; ++s) {
          const double acc = gsum(((cs0 >> s) & 1ull) ? v : 0.0, w);
          if (w >= a.S) {
            if (gl == s) mine = acc;
          } else if (gl == 0 && q < n_pairs) {
            a.post_sub[(size_t)p * a.S + s] = acc > 1.0 ? 1.0 : acc;
          }
        }
        if (w >= a.S && gl < a.S && q < n_pairs) a.post_sub[(size_t)p * a.S + gl] = mine > 1.0 ? 1.0 : mine;
      }
    } else {
      best = first_max(d0, top, lmax, d > -INFINITY ? gl : D, D, w);
    }
    if (gl == 0 && q < n_pairs) {
      held[wv][q] = make_double2(mx, sum);
      hbest[wv][q] = best;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (lane < n_pairs) {
    const double2 h = held[wv][lane];
    a.snp_bf[base + lane] = l10_round(h.x + log10(h.y));
    a.best_dim[base + lane] = hbest[wv][lane];
  }
}

/* launch of the instance for rows of L values, LV counted down to it */
template <int LV>
void launch_avg_rows(const AvgArgs& a, int w, int n_it, hipStream_t st) {
  if constexpr (LV > 1)
    if (a.L != LV) return launch_avg_rows<LV - 1>(a, w, n_it, st);
  const int64_t per_block = (int64_t)kAvgWaves * n_it * (64 / w);
  const dim3 grid((unsigned)((a.NP + per_block - 1) / per_block)), block(64 * kAvgWaves);
  if (LV % 2 == 0 && ((uintptr_t)a.raw & 15) == 0)
    hipLaunchKernelGGL((avg_rows_kernel<LV, LV % 2 == 0>), grid, block, 0, st, a, w, n_it);
  else
    hipLaunchKernelGGL((avg_rows_kernel<LV, false>), grid, block, 0, st, a, w, n_it);
}

__global__ void __launch_bounds__(64) avg_gene_kernel(const AvgArgs a) {
  const int64_t g = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t p0 = a.off[g], m = a.off[g + 1] - p0;
  if (m <= 0) {
    if (lane == 0) a.gene_bf[g] = NAN;
    return;
  }
  const double* sb = a.snp_bf + p0;
  const double x0 = sb[0];
  double lm = -INFINITY;
  for (int64_t q = lane; q < m; q += 64) lm = fmax(lm, sb[q]);
  double mx = wmax(lm);
  if (isnan(x0)) mx = NAN;
  if (!(mx > x0)) mx = x0;
  const double w = 1 / ((double)m);
  double s1 = 0.0, s2 = 0.0;
  for (int64_t q = lane; q < m; q += 64) {
    const double x = sb[q];
    if (!isnan(x)) {
      const double e = exp10(x - mx);
      s1 += w * e;
      s2 += e;
    }
  }
  s1 = wsum(s1);
  s2 = wsum(s2);
  const double gbf = l10_round(mx + log10(s1));
  if (lane == 0) {
    a.gene_bf[g] = gbf;
    if (a.want & 1) {
      /* lws of (0, gbf) with weights (pi0, 1 - pi0) */
      double om = 0.0;
      if (gbf > om) om = gbf;
      double s = a.pi0 * exp10(0.0 - om);
      if (!isnan(gbf)) s += (1 - a.pi0) * exp10(gbf - om);
      const double ol = l10_round(om + log10(s));
      const double pp = exp10(log10(1.0 - a.pi0) + gbf - ol);
      a.gene_post[g] = pp > 1.0 ? 1.0 : pp;
    }
  }
  if (a.want & 2) {
    const double tot = l10_round(mx + log10(s2));
    for (int64_t q = lane; q < m; q += 64) {
      const double pt = exp10(sb[q] - tot);
      a.post_the[p0 + q] = pt > 1.0 ? 1.0 : pt;
    }
  }
  if (a.want & 4) {
    const double w0 = 1.0 - 1 / (double)m, w1 = 1 / (double)m;
    for (int64_t q = lane; q < m; q += 64) {
      const double x = sb[q];
      double om = 0.0;
      if (x > om) om = x;
      double s = w0 * exp10(0.0 - om);
      if (!isnan(x)) s += w1 * exp10(x - om);
      a.post_an[p0 + q] = exp10(-log10((double)m) + x - l10_round(om + log10(s)));
    }
  }
}

/* types model's subgroup posteriors (:749-796): one wave per pair
 * (grid-stride), lanes over the subgroups */
__global__ void __launch_bounds__(64 * kAvgWaves) avg_post_kernel(const AvgArgs a) {
  const int lane = threadIdx.x & 63;
  const int D = a.D, S = a.S;
  for (int64_t p = (int64_t)blockIdx.x * kAvgWaves + (threadIdx.x >> 6); p < a.NP;
       p += (int64_t)gridDim.x * kAvgWaves) {
    const double sbp = a.snp_bf[p];
    for (int s = lane; s < S; s += 64) {
      double acc = 0.0;
      for (int k = 0; k < D; ++k) {
        double t = log10(a.dw[k]) + log10(a.sw[(size_t)k * S + s]) - sbp;
        const double* rs = a.raw + ((size_t)p * S + s) * a.L;
        t += grid_lws(a, [&](int i) { return rs[a.keep[i]] + types_point(a, p, k, i, s); });
        acc += exp10(t);
      }
      a.post_sub[(size_t)p * S + s] = acc > 1.0 ? 1.0 : acc;
    }
  }
}

}  // namespace

int avg_bfs_run(eqbf_ctx* ctx, const double* raw, int64_t NP, const int64_t* off, int64_t G, const eqbf_avg_opts* o,
                const double* d_gw, const int32_t* d_keep, const double* d_dw, const uint64_t* d_cs,
                const double* d_sw, eqbf_avg_out* out, hipStream_t st) {
  AvgArgs a;
  memset(&a, 0, sizeof a);
  a.raw = raw;
  a.off = off;
  a.keep = d_keep;
  a.gw = d_gw;
  a.dw = d_dw;
  a.cs = d_cs;
  a.sw = d_sw;
  a.gene_bf = out->gene_bf;
  a.gene_post = out->gene_post;
  a.snp_bf = out->snp_bf;
  a.dim_bf = out->dim_bf;
  a.post_the = out->post_the;
  a.post_an = out->post_an;
  a.post_dim = out->post_dim;
  a.post_sub = out->post_sub;
  a.best_dim = out->best_dim;
  a.pi0 = o->pi0;
  a.NP = NP;
  a.G = G;
  a.D = o->dim;
  a.S = o->n_subgroups;
  a.L = o->n_grid;
  a.nk = o->n_keep;
  a.types = o->model == EQBF_AVG_TYPES;
  a.want = o->want;
  /* rows that are kept whole and fit a lane's registers */
  bool rows = !a.types && a.D <= 64 && a.L <= kAvgRow && a.nk == a.L;
  for (int i = 0; i < a.nk && rows; ++i) rows = o->keep[i] == i;
  for (int i = 0; i < a.L && rows; ++i) a.gw_row[i] = o->grid_weights[i];
  /* lanes per pair: the power of two >= dim, at most 64; enough blocks to
   * fill every CU several times over, each wave then strides over the pairs */
  int w = 1;
  while (w < a.D && w < 64) w <<= 1;
  const int64_t per_block = (int64_t)kAvgWaves * (64 / w);
  const unsigned pblocks = (unsigned)std::min<int64_t>((NP + per_block - 1) / per_block, (int64_t)256 * 64);
  if (NP > 0) {
    ProfScope ps(ctx, "avg_pair_kernel", st);
    if (rows) {
      /* passes per wave: as many as give every lane a pair, fewer while that
       * leaves compute units without a workgroup */
      const int64_t passes = (NP + 64 / w - 1) / (64 / w);
      const int n_it = (int)std::max<int64_t>(
          1, std::min<int64_t>(w, passes / ((int64_t)kAvgWaves * 4 * std::max(ctx->n_cu, 1))));
      launch_avg_rows<kAvgRow>(a, w, n_it, st);
    } else {
      hipLaunchKernelGGL(avg_pair_kernel, dim3(pblocks), dim3(64 * kAvgWaves), 0, st, a, w);
    }
  }
  if (G > 0) {
    ProfScope ps(ctx, "avg_gene_kernel", st);
    hipLaunchKernelGGL(avg_gene_kernel, dim3((unsigned)G), dim3(64), 0, st, a);
  }
  if (NP > 0 && a.types && (a.want & 8)) {
    ProfScope ps(ctx, "avg_post_kernel", st);
    const unsigned qblocks = (unsigned)std::min<int64_t>((NP + kAvgWaves - 1) / kAvgWaves, (int64_t)256 * 64);
    hipLaunchKernelGGL(avg_post_kernel, dim3(qblocks), dim3(64 * kAvgWaves), 0, st, a);
  }
  EQBF_HIP(ctx, hipGetLastError());
  return EQBF_OK;
}

int avg_grid_run(eqbf_ctx* ctx, const double* raw, int64_t n_rows, int L, const double* gw, const int32_t* keep,
                 int nk, double* out, hipStream_t st) {
  if (n_rows <= 0) return EQBF_OK;
  {
    ProfScope ps(ctx, "avg_grid_kernel", st);
    hipLaunchKernelGGL(avg_grid_kernel, dim3((unsigned)((n_rows + 255) / 256)), dim3(256), 0, st, raw, n_rows, L,
                       gw, keep, nk, out);
  }
  EQBF_HIP(ctx, hipGetLastError());
  return EQBF_OK;
}

namespace {

int avg_check(eqbf_ctx* ctx, int64_t NP, int64_t G, const eqbf_avg_opts* o) {
  if (!o) return ctx_fail(ctx, EQBF_ERR_ARG, "null options");
  if (o->model != EQBF_AVG_CONFIGS && o->model != EQBF_AVG_TYPES)
    return ctx_fail(ctx, EQBF_ERR_ARG, "unknown model %d", o->model);
  if (o->dim < 1 || o->n_grid < 1 || o->n_keep < 1 || o->n_keep > o->n_grid || NP < 0 || G < 0 ||
      (o->model == EQBF_AVG_TYPES && (o->n_subgroups < 1 || o->n_subgroups > 64)) || o->n_subgroups < 0 ||
      o->n_subgroups > 64)
    return ctx_fail(ctx, EQBF_ERR_ARG, "sizes out of range (dim=%d grid=%d keep=%d S=%d)", o->dim, o->n_grid,
                    o->n_keep, o->n_subgroups);
  if (!o->keep || !o->grid_weights || !o->dim_weights ||
      (o->model == EQBF_AVG_TYPES && !o->sub_weights) ||
      (o->model == EQBF_AVG_CONFIGS && (o->want & EQBF_AVG_POST_D) && !o->cfg_subgroups))
    return ctx_fail(ctx, EQBF_ERR_ARG, "missing weights");
  for (int i = 0; i < o->n_keep; ++i)
    if (o->keep[i] < 0 || o->keep[i] >= o->n_grid) return ctx_fail(ctx, EQBF_ERR_ARG, "grid index %d out of range", o->keep[i]);
  return EQBF_OK;
}

/* the option tables on the device */
struct AvgTables {
  double *gw = nullptr, *dw = nullptr, *sw = nullptr;
  int32_t* keep = nullptr;
  uint64_t* cs = nullptr;
};

/* in one buffer and one copy (each small copy costs a few microseconds); `host`
 * has to live until the stream has made it */
int avg_tables(eqbf_ctx* ctx, const eqbf_avg_opts* o, AvgTables& t, std::vector<uint64_t>& host, hipStream_t st) {
  const size_t D = o->dim, S = std::max(o->n_subgroups, 0), L = o->n_grid, nk = o->n_keep;
  const size_t sw = o->sub_weights ? D * S : 0, cs = o->cfg_subgroups ? D : 0;
  host.resize(L + D + cs + sw + (nk + 1) / 2);
  uint64_t* h = host.data();
  memcpy(h, o->grid_weights, L * sizeof(double));
  memcpy(h + L, o->dim_weights, D * sizeof(double));
  if (cs) memcpy(h + L + D, o->cfg_subgroups, D * sizeof(uint64_t));
  if (sw) memcpy(h + L + D + cs, o->sub_weights, sw * sizeof(double));
  memcpy(h + L + D + cs + sw, o->keep, nk * sizeof(int32_t));
  uint64_t* d = (uint64_t*)ctx_buf(ctx, "avg_tables", host.size() * sizeof(uint64_t));
  if (!d) return ctx_fail(ctx, EQBF_ERR_HIP, "allocating tables failed");
  t.gw = (double*)d;
  t.dw = (double*)(d + L);
  t.cs = d + L + D;
  t.sw = (double*)(d + L + D + cs);
  t.keep = (int32_t*)(d + L + D + cs + sw);
  EQBF_HIP(ctx, hipMemcpyAsync(d, h, host.size() * sizeof(uint64_t), hipMemcpyHostToDevice, st));
  return EQBF_OK;
}

}  // namespace

extern "C" int eqbf_avg_bfs_device(eqbf_ctx* ctx, const double* raw, int64_t NP, const int64_t* off, int64_t G,
                                   const eqbf_avg_opts* o, eqbf_avg_out* out, void* stream) {
  if (!ctx || !out) return EQBF_ERR_ARG;
  int rc = avg_check(ctx, NP, G, o);
  if (rc) return rc;
  if ((NP > 0 && (!raw || !out->snp_bf || !out->dim_bf || !out->best_dim)) || (G > 0 && (!off || !out->gene_bf)))
    return ctx_fail(ctx, EQBF_ERR_ARG, "missing input or output");
  const bool types = o->model == EQBF_AVG_TYPES;
  const bool dims_post = (o->want & EQBF_AVG_POST_DIMS) || (!types && (o->want & EQBF_AVG_POST_D));
  if (((o->want & EQBF_AVG_POST_A) && !out->gene_post) || ((o->want & EQBF_AVG_POST_B) && !out->post_the) ||
      ((o->want & EQBF_AVG_POST_C) && !out->post_an) || ((o->want & EQBF_AVG_POST_D) && !out->post_sub) ||
      (dims_post && !out->post_dim))
    return ctx_fail(ctx, EQBF_ERR_ARG, "missing output for a requested posterior");
  EQBF_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t st = stream ? (hipStream_t)stream : ctx->stream;
  AvgTables t;
  std::vector<uint64_t> tables;
  if ((rc = avg_tables(ctx, o, t, tables, st))) return rc;
  rc = avg_bfs_run(ctx, raw, NP, off, G, o, t.gw, t.keep, t.dw, t.cs, t.sw, out, st);
  if (rc) return rc;
  /* the host tables must outlive the copies */
  EQBF_HIP(ctx, hipStreamSynchronize(st));
  return EQBF_OK;
}

extern "C" int eqbf_avg_bfs(eqbf_ctx* ctx, const double* raw, int64_t NP, const int64_t* off, int64_t G,
                            const eqbf_avg_opts* o, eqbf_avg_out* out) {
  if (!ctx || !out) return EQBF_ERR_ARG;
  int rc = avg_check(ctx, NP, G, o);
  if (rc) return rc;
  if ((NP > 0 && !raw) || !off) return ctx_fail(ctx, EQBF_ERR_ARG, "missing input");
  EQBF_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int D = o->dim, S = o->n_subgroups, R = o->model == EQBF_AVG_TYPES ? S : D;
  const size_t np = (size_t)std::max<int64_t>(NP, 1), ng = (size_t)std::max<int64_t>(G, 1);
  auto buf = [&](const char* name, size_t bytes) { return ctx_buf(ctx, name, bytes); };
  double* d_raw = (double*)buf("avg_raw", np * R * o->n_grid * sizeof(double));
  int64_t* d_off = (int64_t*)buf("avg_off", (ng + 1) * sizeof(int64_t));
  eqbf_avg_out d;
  d.gene_bf = (double*)buf("avg_gbf", ng * sizeof(double));
  d.gene_post = (double*)buf("avg_gpost", ng * sizeof(double));
  d.snp_bf = (double*)buf("avg_sbf", np * sizeof(double));
  d.dim_bf = (double*)buf("avg_dbf", np * D * sizeof(double));
  d.post_the = (double*)buf("avg_pthe", np * sizeof(double));
  d.post_an = (double*)buf("avg_pan", np * sizeof(double));
  d.post_dim = (double*)buf("avg_pdim", np * D * sizeof(double));
  d.post_sub = (double*)buf("avg_psub", np * std::max(S, 1) * sizeof(double));
  d.best_dim = (int32_t*)buf("avg_best", np * sizeof(int32_t));
  if (!d_raw || !d_off || !d.gene_bf || !d.gene_post || !d.snp_bf || !d.dim_bf || !d.post_the || !d.post_an ||
      !d.post_dim || !d.post_sub || !d.best_dim)
    return ctx_fail(ctx, EQBF_ERR_HIP, "allocating eqtlbma_avg_bfs buffers failed");
  if (NP > 0)
    EQBF_HIP(ctx, hipMemcpyAsync(d_raw, raw, (size_t)NP * R * o->n_grid * sizeof(double), hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipMemcpyAsync(d_off, off, (size_t)(G + 1) * sizeof(int64_t), hipMemcpyHostToDevice, st));
  AvgTables t;
  std::vector<uint64_t> tables;
  if ((rc = avg_tables(ctx, o, t, tables, st))) return rc;
  rc = avg_bfs_run(ctx, d_raw, NP, d_off, G, o, t.gw, t.keep, t.dw, t.cs, t.sw, &d, st);
  if (rc) return rc;
  auto back = [&](void* h, const void* dv, size_t bytes) -> int {
    if (h && bytes) EQBF_HIP(ctx, hipMemcpyAsync(h, dv, bytes, hipMemcpyDeviceToHost, st));
    return EQBF_OK;
  };
  const bool types = o->model == EQBF_AVG_TYPES;
  const bool dims_post = (o->want & EQBF_AVG_POST_DIMS) || (!types && (o->want & EQBF_AVG_POST_D));
  if ((rc = back(out->gene_bf, d.gene_bf, (size_t)G * sizeof(double))) ||
      (rc = back(out->snp_bf, d.snp_bf, (size_t)NP * sizeof(double))) ||
      (rc = back(out->dim_bf, d.dim_bf, (size_t)NP * D * sizeof(double))) ||
      (rc = back(out->best_dim, d.best_dim, (size_t)NP * sizeof(int32_t))) ||
      ((o->want & EQBF_AVG_POST_A) && (rc = back(out->gene_post, d.gene_post, (size_t)G * sizeof(double)))) ||
      ((o->want & EQBF_AVG_POST_B) && (rc = back(out->post_the, d.post_the, (size_t)NP * sizeof(double)))) ||
      ((o->want & EQBF_AVG_POST_C) && (rc = back(out->post_an, d.post_an, (size_t)NP * sizeof(double)))) ||
      (dims_post && (rc = back(out->post_dim, d.post_dim, (size_t)NP * D * sizeof(double)))) ||
      ((o->want & EQBF_AVG_POST_D) && (rc = back(out->post_sub, d.post_sub, (size_t)NP * S * sizeof(double)))))
    return rc;
  EQBF_HIP(ctx, hipStreamSynchronize(st));
  return EQBF_OK;
}

extern "C" int eqbf_avg_grid(eqbf_ctx* ctx, const double* raw, int64_t n_rows, int32_t L, const double* gw,
                             const int32_t* keep, int32_t nk, double* out) {
  if (!ctx) return EQBF_ERR_ARG;
  if (n_rows < 0 || L < 1 || nk < 1 || nk > L || !gw || !keep || (n_rows > 0 && (!raw || !out)))
    return ctx_fail(ctx, EQBF_ERR_ARG, "invalid arguments");
  for (int i = 0; i < nk; ++i)
    if (keep[i] < 0 || keep[i] >= L) return ctx_fail(ctx, EQBF_ERR_ARG, "grid index %d out of range", keep[i]);
  if (n_rows == 0) return EQBF_OK;
  EQBF_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  double* d_raw = (double*)ctx_buf(ctx, "avg_raw", (size_t)n_rows * L * sizeof(double));
  double* d_out = (double*)ctx_buf(ctx, "avg_gout", (size_t)n_rows * sizeof(double));
  double* d_gw = (double*)ctx_buf(ctx, "avg_gw", (size_t)L * sizeof(double));
  int32_t* d_keep = (int32_t*)ctx_buf(ctx, "avg_keep", (size_t)nk * sizeof(int32_t));
  if (!d_raw || !d_out || !d_gw || !d_keep) return ctx_fail(ctx, EQBF_ERR_HIP, "allocating buffers failed");
  EQBF_HIP(ctx, hipMemcpyAsync(d_raw, raw, (size_t)n_rows * L * sizeof(double), hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipMemcpyAsync(d_gw, gw, (size_t)L * sizeof(double), hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipMemcpyAsync(d_keep, keep, (size_t)nk * sizeof(int32_t), hipMemcpyHostToDevice, st));
  int rc = avg_grid_run(ctx, d_raw, n_rows, L, d_gw, d_keep, nk, d_out, st);
  if (rc) return rc;
  EQBF_HIP(ctx, hipMemcpyAsync(out, d_out, (size_t)n_rows * sizeof(double), hipMemcpyDeviceToHost, st));
  EQBF_HIP(ctx, hipStreamSynchronize(st));
  return EQBF_OK;
}
