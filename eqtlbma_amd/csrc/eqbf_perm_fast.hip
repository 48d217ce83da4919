/*
 * Permutation statistics, contraction path.
 *
 * Applies to the genes of a chunk whose every sample is a member of every
 * subgroup (expression present everywhere, one genotype file, hard-call
 * genotypes, no covariates).  Then the members of a subgroup do not change
 * under a permutation, x'x and sum(x) are fixed per SNP, y'y is fixed per
 * subgroup, and the only quantity that moves is x'y_perm:
 *
 *   XY[snp][s][p] = sum_i x[i][snp] * yc_s[perm_p(i)]        (yc = y - ybar)
 *
 * for all SNPs of the gene, all subgroups and all permutations: a dense
 * contraction G^T . Y_perm on the matrix cores (MakePermutationsJoin /
 * MakePermutationsSep*, gene.cpp:380-717, recompute this one fit at a time
 * through GeneSnpPair::CalcSstatsOneSbgrp).
 *
 * Exactness: genotypes are small integers and are held exactly in int8.
 * yc is held in 32-bit fixed point (scaled by 2^E per gene and subgroup so
 * that max|yc| maps to ~2^30) and split into four signed 8-bit digits;
 * v_mfma_i32_16x16x64_i8 gives each digit's dot product exactly in int32,
 * and the digits are recombined exactly in FP64.  x'yc is therefore exact up
 * to the fixed-point rounding of yc (2^-31 of its range), far below FP64's
 * own rounding of the reference's SVD fit.
 *
 * From XY the fit (FitSingleGeneWithSingleSnp, utils_math.cpp:166-209) is
 * closed form in FP64 (the residual sum of squares y'y - (x'y)^2/x'x included);
 * the standardised z (gene_snp_pair.cpp:256-290) comes from a table of
 * z(asinh(|t|/sqrt(nu))) = z(atanh(R)) in FP32, R = |x'y| / sqrt(x'x y'y),
 * from a polynomial fitted to that table where R < 1/2, or from the FP64 tail functions for |t| < 1e-5, where the reference's
 * |z| > 1e-8 test is decided.
 *
 * Because every subgroup has the same members, the standardised variance
 * v = 1/x'x is the same in every subgroup, and the log10 ABF of a
 * configuration gamma with m = |gamma| active subgroups at grid point
 * (phi2, omega2) (CalcLog10AbfUvlr, gene_snp_pair.cpp:297-356) reduces to
 *   l = Cabf_m + q * Z2 + D_m * Z1^2,
 *   Z1 = sum_{s in gamma} z_s,  Z2 = sum_{s in gamma} z_s^2,
 *   r = 1/(v+phi2), q = phi2 r/(2 ln10), Cabf_m = m/2 log10(v r) -
 *   1/2 log10(1 + m r omega2), D_m = omega2 v r^2 / (2 ln10 (1 + m r omega2)),
 * with per-SNP coefficients and per-permutation Z1, Z2.  A subgroup with
 * |z| <= 1e-8 drops out of A and B in the reference; here it contributes
 * z = 0 to Z1 and Z2 and m counts only the others.  The statistic
 * (BMA over configurations, BMAlite, or the consistent configuration,
 * gene_snp_pair.cpp:552-602, then max or log10 average over SNPs,
 * gene.cpp:575-596) is a sum of 2^(l log2 10) terms per SNP with the weights
 * folded into the exponents.
 *
 * Anything the closed forms do not cover for a permutation (a residual sum of
 * squares <= 0, |t| past the tail table, an FP32 sum that overflows) marks
 * the gene, and the caller recomputes that gene on the general path, which
 * is exact for every input.
 */
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

#include "eqbf_internal.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int PF_NMAX = 2048;        /* samples (LDS holds the digit fragments) */
constexpr int ZT_STRIDE = 3;                             /* every third t-tail node   */
constexpr int ZT_NODES = (TZ_NODES - 1) / ZT_STRIDE + 1; /* nodes of the z table      */
constexpr int ZP = 8;                                    /* terms of z(R) / R in R^2  */
constexpr float ZP_RMAX = 0.5f;                          /* ... used for R below this */
constexpr int ZT_ROW = 4 + 2 * ZT_NODES + ZP + 1;        /* floats per z-table row    */
constexpr int PF_SB = 64;            /* SNPs per Bayes-factor work item         */
constexpr float kLog2_10f = 3.32192809488736235f;
constexpr double kLog2_10 = 3.32192809488736235;

/* floats per (SNP, grid point) of the coefficients: q, C_1..S, D_1..S, padded
 * so that a lane reads a row of its own SNP in 16-byte pieces */
__host__ __device__ constexpr int pf_ncf(int S) { return (1 + 2 * S + 3) / 4 * 4; }

enum { PF_JOIN_ALL = 0, PF_JOIN_GEN = 1, PF_JOIN_GENSIN = 2, PF_SEP = 3 };

/* ---- which genes qualify ------------------------------------------------------
 * Bit 0 of bad[g]: gene g does not; bit 1: some genotype is past PFX_XMAX, too
 * large for pf_max_kernel.  One workgroup per 64 pairs of a gene (blockIdx
 * = gene, block of pairs; the first block looks at the levels too): lanes over
 * pairs, the four waves over samples.  24 genes of 1,000 pairs and 300 samples
 * took 1.0 ms with one workgroup per gene. */
constexpr int PFX_XMAX = 31;

__global__ void __launch_bounds__(64) pf_clear_kernel(int* __restrict__ p, int n) {
  for (int i = blockIdx.x * 64 + threadIdx.x; i < n; i += gridDim.x * 64) p[i] = 0;
}

template <class T>
__global__ void __launch_bounds__(256) pf_check_kernel(const eqbf_chunk c, int* __restrict__ bad) {
  const int g = blockIdx.x, S = c.n_subgroups, N = c.n_samples;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t p0 = c.pair_offset[g], np = c.pair_offset[g + 1] - p0;
  int b = 0;
  if (blockIdx.y == 0) {
    for (int e = threadIdx.x; e < S * N; e += blockDim.x) {
      if (!c.geno_in_sbgrp[e]) b = 1;
      const double y = c.explevels[(int64_t)g * S * N + e];
      if (!(fabs(y) < INFINITY)) b = 1;
    }
    for (int s = threadIdx.x; s < S; s += blockDim.x)
      if (!c.gene_in_sbgrp[(int64_t)g * S + s]) b = 1;
    if (np <= 0) b = 1;
  }
  for (int64_t q = (int64_t)blockIdx.y * 64 + lane; q < np; q += (int64_t)gridDim.y * 64) {
    const int64_t snp = c.pair_snp[p0 + q];
    const T* x = (const T*)c.genotypes + snp;
#pragma unroll 8
    for (int i = w; i < N; i += 4) {
      const T v = x[(int64_t)i * c.geno_ld];
      b |= !(v == rint(v)) || v < (T)-127 || v > (T)127;
      b |= v < (T)-PFX_XMAX || v > (T)PFX_XMAX ? 2 : 0;
    }
    for (int s = w; s < S; s += 4) b |= !c.snp_in_sbgrp[snp * S + s];
  }
  if (__any(b != 0)) {
    const int bits = (__any(b & 1) ? 1 : 0) | (__any(b & 2) ? 2 : 0);
    if (lane == 0) atomicOr(&bad[g], bits);
  }
}

/* ---- per (gene, subgroup): centred y in four signed 8-bit digits ---------------- */
struct YStat {
  double yy;    /* sum (y - ybar)^2                        */
  double scale; /* 2^-E: value of one fixed-point unit      */
  double tsum;  /* sum of the fixed-point values (integer)  */
};

__device__ inline double block_sum(double v, double* red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (tid < o) red[tid] += red[tid + o];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}
__device__ inline double block_max(double v, double* red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (tid < o) red[tid] = fmax(red[tid], red[tid + o]);
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

/* One workgroup per (batch gene, subgroup).  Levels that are all equal (a gene
 * that a subgroup does not express), or whose sum of squares leaves the normal
 * numbers, have no R: such a gene goes to the general path (fallback, null where
 * the caller looks after y'y = 0 itself). */
__global__ void __launch_bounds__(256) pf_prep_y_kernel(const eqbf_chunk c, const int32_t* __restrict__ bgene,
                                                        int Npad, uint32_t* __restrict__ W, YStat* __restrict__ ys,
                                                        int* __restrict__ fallback) {
  __shared__ double red[256];
  const int S = c.n_subgroups, N = c.n_samples;
  const int bi = blockIdx.x / S, s = blockIdx.x - bi * S;
  const int g = bgene[bi];
  const double* y = c.explevels + ((int64_t)g * S + s) * N;
  double a = 0;
  for (int i = threadIdx.x; i < N; i += blockDim.x) a += y[i];
  const double ybar = block_sum(a, red) / (double)N;
  double q = 0, mx = 0;
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    const double d = y[i] - ybar;
    q += d * d;
    mx = fmax(mx, fabs(d));
  }
  const double yy = block_sum(q, red);
  mx = block_max(mx, red);
  int ex = 0;
  if (mx > 0) {
    int e2;
    (void)frexp(mx, &e2); /* mx < 2^e2 */
    ex = 30 - e2;         /* max |yc| 2^ex < 2^30 */
  }
  const double up = ldexp(1.0, ex);
  double ts = 0;
  uint32_t* Wg = W + ((int64_t)bi * S + s) * Npad;
  for (int i = threadIdx.x; i < Npad; i += blockDim.x) {
    int64_t v = 0;
    if (i < N) v = (int64_t)llrint((y[i] - ybar) * up);
    ts += (double)v;
    uint32_t word = 0;
    for (int j = 0; j < 3; ++j) {
      int d = (int)(v & 0xff);
      if (d >= 128) d -= 256;
      v = (v - d) >> 8;
      word |= (uint32_t)(d & 0xff) << (8 * j);
    }
    word |= (uint32_t)((int)v & 0xff) << 24;
    Wg[i] = word;
  }
  ts = block_sum(ts, red);
  if (threadIdx.x == 0) {
    ys[(int64_t)bi * S + s] = YStat{yy, ldexp(1.0, -ex), ts};
    if (fallback && !(yy >= DBL_MIN && yy < INFINITY)) atomicOr(&fallback[bi], 1);
  }
}

/* Genotypes of the batch pairs, SNP-major int8 [pair][Npad], and per pair
 * x'x - (sum x)^2 / N, 1 / that, sum x and the not-estimable flag
 * (uvlr_stats: x'x - |U'x|^2 <= 1e-12 x'x). */
struct PStat {
  double xx, inv_xx, sx, rs_xx; /* rs_xx = 1/sqrt(xx), NaN when not estimable */
};
/* 64 pairs a workgroup, lane = pair and the waves over groups of four samples;
 * the int8 rows go through LDS so that they are written whole.  The batch's
 * pairs are those of its genes in order: pair b of batch gene bi is pair
 * goff[bi] + b - bpoff[bi] of the chunk. */
template <class T>
__global__ void __launch_bounds__(256) pf_prep_x_kernel(const eqbf_chunk c, const int64_t* __restrict__ bpoff,
                                                        const int64_t* __restrict__ goff, int nb, int Npad,
                                                        int8_t* __restrict__ G8, PStat* __restrict__ ps,
                                                        uint8_t* __restrict__ pflag) {
  extern __shared__ uint32_t rows8[]; /* [64][Npad / 4 + 1] */
  __shared__ int red[2][4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, N = c.n_samples;
  const int nw = Npad / 4, pitch = nw + 1;
  const int64_t nbp = bpoff[nb], b0 = (int64_t)blockIdx.x * 64, b = min(b0 + lane, nbp - 1);
  int lo = 0, hi = nb; /* bpoff[lo] <= b < bpoff[hi] */
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (bpoff[mid] <= b)
      lo = mid;
    else
      hi = mid;
  }
  const T* x = (const T*)c.genotypes + c.pair_snp[goff[lo] + (b - bpoff[lo])];
  int sx = 0, sxx = 0; /* exact: |x| <= 127, at most PF_NMAX samples */
#pragma unroll 2
  for (int k = w; k < nw; k += 4) {
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = 4 * k + j;
      const T v = x[(int64_t)min(i, N - 1) * c.geno_ld];
      const int xi = i < N ? (int)v : 0;
      sx += xi;
      sxx += xi * xi;
      word |= (uint32_t)(xi & 0xff) << (8 * j);
    }
    rows8[lane * pitch + k] = word;
  }
  red[0][w][lane] = sx;
  red[1][w][lane] = sxx;
  __syncthreads();
  const int n = (int)min((int64_t)64, nbp - b0) * nw;
  uint32_t* out = (uint32_t*)(G8 + b0 * Npad);
  for (int e = threadIdx.x; e < n; e += 256) out[e] = rows8[(e / nw) * pitch + e % nw];
  if (w == 0 && b0 + lane < nbp) {
    const double fx = (double)(red[0][0][lane] + red[0][1][lane] + red[0][2][lane] + red[0][3][lane]);
    const double fxx = (double)(red[1][0][lane] + red[1][1][lane] + red[1][2][lane] + red[1][3][lane]);
    const double xx = fxx - fx * fx / (double)N;
    const bool flagged = !(xx > 1e-12 * fxx);
    ps[b] = PStat{xx, 1.0 / xx, fx, flagged ? NAN : 1.0 / sqrt(xx)};
    pflag[b] = flagged;
  }
}

/* ---- z as a function of s = asinh(|t| / sqrt(nu)) for one nu -------------------- */
/* From every third node of the t-tail table row of nu (segment A, s in
 * [0, sA]): value and derivative of |z| = -Phi^-1(exp(-w)), d|z|/dw =
 * exp(-w + z^2/2) sqrt(2 pi).  11 KB, so that it sits in LDS. */
/* After the nodes: |z| / R as a polynomial in R^2 for R <= ZP_RMAX (s = atanh R),
 * the interpolant at ZP Chebyshev nodes in R^2; z(R) / R is smooth in R^2 for
 * every nu (its nearest singularity is R^2 = 1), so that eight terms leave
 * about 1e-10 of it, far below the FP32 result.  The constant term is kept in two
 * parts: its rounding alone would be the same relative error in every z of a nu
 * (5e-8 at nu = 298, of 7e-8 rms).  Rounding against 64 bits (nu 10 to 2000, t
 * from 1 to 7): 4e-8 to 5e-8 rms, 1.7e-7 at most; the table has 1.0e-7 and
 * 4.7e-7. */
__device__ void pf_zeta_poly(const double* __restrict__ tz, int nu, float* __restrict__ out) {
  double x[ZP], d[ZP], c[ZP];
  for (int k = 0; k < ZP; ++k) {
    x[k] = 0.5 * (double)ZP_RMAX * ZP_RMAX * (1.0 + cos(3.14159265358979323846 * (2 * k + 1) / (2 * ZP)));
    const double R = sqrt(x[k]), w = dm::tz_eval(tz, nu, sqrt((double)nu * x[k] / (1.0 - x[k])));
    d[k] = -dm::gauss_pinv_from_w(w) / R;
  }
  for (int j = 1; j < ZP; ++j) /* divided differences */
    for (int k = ZP - 1; k >= j; --k) d[k] = (d[k] - d[k - 1]) / (x[k] - x[k - j]);
  for (int k = 0; k < ZP; ++k) c[k] = 0.0;
  for (int k = ZP - 1; k >= 0; --k) { /* c = c (X - x_k) + d_k */
    for (int m = ZP - 1; m > 0; --m) c[m] = c[m - 1] - x[k] * c[m];
    c[0] = d[k] - x[k] * c[0];
  }
  for (int k = 0; k < ZP; ++k) out[k] = (float)c[k];
  out[ZP] = (float)(c[0] - (double)out[0]);
}

struct PfZeta {
  float c[ZP], lo;
};
__device__ __forceinline__ PfZeta pf_zeta_load(const float* __restrict__ zt) {
  PfZeta p;
#pragma unroll
  for (int k = 0; k < ZP; ++k) p.c[k] = zt[4 + 2 * ZT_NODES + k];
  p.lo = zt[4 + 2 * ZT_NODES + ZP];
  return p;
}
/* |z| / R at x = R^2 */
__device__ __forceinline__ float pf_zeta_ratio(const PfZeta& p, float x) {
  float v = p.c[ZP - 1];
#pragma unroll
  for (int k = ZP - 2; k > 0; --k) v = fmaf(v, x, p.c[k]);
  return p.c[0] + fmaf(v, x, p.lo);
}

__global__ void pf_zeta_table_kernel(const double* __restrict__ tz, int nu, float* __restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k == ZT_NODES) pf_zeta_poly(tz, nu, out + 4 + 2 * ZT_NODES);
  const double* row = tz + (size_t)nu * TZ_ROW;
  const double h = row[0] * ZT_STRIDE, sA = row[1];
  if (k == 0) {
    out[0] = (float)h;
    out[1] = (float)sA;
    out[2] = (float)(1.0 / h);
    out[3] = 0.f;
  }
  if (k >= ZT_NODES) return;
  const double w = row[4 + 2 * ZT_STRIDE * k], dw = row[4 + 2 * ZT_STRIDE * k + 1];
  const double z = -dm::gauss_pinv_from_w(w);
  const double dz = exp(-w + 0.5 * z * z) * 2.5066282746310002 * dw;
  out[4 + 2 * k] = (float)z;
  out[4 + 2 * k + 1] = (float)dz;
}

/* |z| at s (< sA) by cubic Hermite interpolation of the table. */
__device__ inline float pf_zeta_abs(const float* __restrict__ zt, float s) {
  const float h = zt[0], inv_h = zt[2];
  const float u = s * inv_h;
  int k = (int)u;
  if (k > ZT_NODES - 2) k = ZT_NODES - 2;
  const float f = u - (float)k;
  const float2 a = ((const float2*)(zt + 4))[k], b = ((const float2*)(zt + 4))[k + 1];
  const float f2 = f * f, f3 = f2 * f;
  const float h00 = 2.f * f3 - 3.f * f2 + 1.f, h10 = f3 - 2.f * f2 + f, h01 = -2.f * f3 + 3.f * f2, h11 = f3 - f2;
  return h00 * a.x + h10 * (a.y * h) + h01 * b.x + h11 * (b.y * h);
}

/* z where the reference decides |z| > 1e-8: the FP64 tail functions that the
 * association path uses (rarely taken, kept out of line). */
__device__ __noinline__ float pf_zeta_exact(const double* __restrict__ tz, int nu, double tt, double sxy) {
  const double z = fabs(dm::gauss_pinv_from_w(dm::tz_eval(tz, nu, sqrt(tt))));
  return z > 1e-8 ? (float)copysign(z, sxy) : 0.f;
}

/* z (signed) where the polynomial does not serve: R past ZP_RMAX through the
 * table of z(atanh R), |t| below 1e-5 through the FP64 tails; fb is set when the
 * closed forms do not cover the value.  d has the sign of x'y. */
__device__ __forceinline__ float pf_zeta_slow(const float* __restrict__ zt, const double* __restrict__ tz, int nu,
                                              double R, double d, bool& fb) {
  const double omR = 1.0 - R;
  const float Rf = (float)R;
  if (!(omR > 0.0)) { /* rss <= 0 */
    fb = true;
    return 0.f;
  }
  if (Rf * Rf * (float)nu < 1e-10f) return pf_zeta_exact(tz, nu, (double)nu * R * R / (omR * (1.0 + R)), d);
  const float sv = 0.34657359027997264f * __log2f((1.f + Rf) * __builtin_amdgcn_rcpf((float)omR));
  if (!(sv < zt[1])) {
    fb = true;
    return 0.f;
  }
  return copysignf(pf_zeta_abs(zt, sv), (float)d);
}

/* ---- the contraction ---------------------------------------------------------------
 * One workgroup per (batch gene, 16 permutations, subgroup).  Phase 1 gathers
 * yc_s[perm(i)] for its 16 permutations into LDS as the B fragments of every
 * 64-sample step (4 digits x 64 lanes x 16 bytes per step).  Phase 2: each
 * wave takes pairs of 16-SNP tiles; per step two A fragments (16 samples of one
 * SNP per lane) and eight MFMAs (one per digit and tile), so that a B fragment
 * is read from LDS once for two products (with one, LDS was the bound of the
 * products).  Lane l's 16 bytes of A and of B cover the same 16 samples, in the
 * same order, so the product is the sum over samples whatever the hardware's k
 * order within an operand.
 *
 * Bound by the epilogue, about 30 instructions per (SNP, permutation): the
 * digits recombined and R formed in FP64, z = R P(R^2) in FP32.  (A table of
 * z(atanh R) in LDS behind a series for atanh took 170.)  Four waves a SIMD: left
 * to itself the compiler takes 160 registers for the two tiles, and with three
 * waves a call on 300 genes of 5 SNPs and 1,000 permutations, S = 5, N = 300, took
 * 1.07 ms under sep, 0.87 with four; 24 genes of 1,000, 5,000 permutations 1.89 and
 * 1.60, under gen 4.88 and 4.61. */
struct PfGemmArgs {
  const int8_t* G8;
  const uint32_t* W;
  const YStat* ys;
  const PStat* ps;
  const uint8_t* pflag;
  const int64_t* bpoff;
  const int32_t* tables;
  const int32_t* btable;
  const float* zt;
  const double* tz;
  float* zeta;   /* join: [nbp][S][NPP]  */
  double* tmax;  /* sep:  [nb][S][NPP] max t^2 over SNPs (-1: none) */
  int* fallback; /* [nb] */
  int S, N, Npad, nks, nu, n_items, npb16, s_lo, ns; /* item = (gene * npb16 + 16 permutations) * ns + s - s_lo */
  int64_t nperm, NPP;
};

__device__ inline uint32_t perm_b(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }

/* B fragments of 16 permutations of one subgroup: digit words Ws in LDS
 * through the index table rows, into Bf[step][digit][64 lanes]. */
__device__ __forceinline__ void pf_gather(const uint32_t* Ws, const int32_t* __restrict__ tab, int64_t pb, int64_t nperm,
                                          int N, int nks, v4i* Bf, int tid, int nt) {
  for (int e = tid; e < nks * 64; e += nt) {
    const int ks = e >> 6, ln = e & 63;
    const int64_t p = min(pb * 16 + (ln & 15), nperm - 1);
    const int k0 = ks * 64 + (ln >> 4) * 16;
    const int32_t* row = tab + p * N;
    uint32_t wd[16];
    if ((N & 3) == 0 && k0 + 16 <= N) { /* 16-byte aligned rows: four vector loads */
      const int4* r4 = (const int4*)(row + k0);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int4 v = r4[b];
        wd[4 * b] = Ws[min(max(v.x, 0), N - 1)];
        wd[4 * b + 1] = Ws[min(max(v.y, 0), N - 1)];
        wd[4 * b + 2] = Ws[min(max(v.z, 0), N - 1)];
        wd[4 * b + 3] = Ws[min(max(v.w, 0), N - 1)];
      }
    } else {
#pragma unroll
      for (int b = 0; b < 16; ++b) {
        const int k = k0 + b;
        int idx = k < N ? row[k] : 0;
        idx = min(max(idx, 0), N - 1);
        wd[b] = Ws[idx];
      }
    }
    uint32_t o[4][4];
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const uint32_t w0 = wd[4 * gq], w1 = wd[4 * gq + 1], w2 = wd[4 * gq + 2], w3 = wd[4 * gq + 3];
      const uint32_t t0 = perm_b(w1, w0, 0x05010400u), t1 = perm_b(w1, w0, 0x07030602u);
      const uint32_t u0 = perm_b(w3, w2, 0x05010400u), u1 = perm_b(w3, w2, 0x07030602u);
      o[0][gq] = perm_b(u0, t0, 0x05040100u);
      o[1][gq] = perm_b(u0, t0, 0x07060302u);
      o[2][gq] = perm_b(u1, t1, 0x05040100u);
      o[3][gq] = perm_b(u1, t1, 0x07060302u);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      v4i f;
      f.x = (int)o[d][0];
      f.y = (int)o[d][1];
      f.z = (int)o[d][2];
      f.w = (int)o[d][3];
      Bf[(ks * 4 + d) * 64 + ln] = f;
    }
  }
}

/* exact value of the four digit sums */
__device__ __forceinline__ double pf_fold(const v4i (&acc)[4], int r) {
  return fma(16777216.0, (double)acc[3][r], fma(65536.0, (double)acc[2][r], fma(256.0, (double)acc[1][r], (double)acc[0][r])));
}

/* the same where |x| <= PFX_XMAX: pairs of digits fit 32 bits (2048 samples x 31
 * x 128 x 257 < 2^31), two conversions less */
__device__ __forceinline__ double pf_fold_narrow(const v4i (&acc)[4], int r) {
  return fma(65536.0, (double)(acc[2][r] + 256 * acc[3][r]), (double)(acc[0][r] + 256 * acc[1][r]));
}

template <int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8))) pf_gemm_kernel(const PfGemmArgs a) {
  extern __shared__ __align__(16) unsigned char sm[];
  uint32_t* Ws = (uint32_t*)sm;
  v4i* Bf = (v4i*)(sm + (size_t)a.Npad * 4);
  __shared__ double redt[4][16];
  /* XCD-aware order (blockIdx & 7 = XCD): contiguous item ranges per XCD, so
   * that neighbouring permutation blocks write their z rows through one L2 */
  const int nit = a.n_items, per = (nit + 7) / 8;
  const int itx = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (itx >= nit) return;
  const int s = a.s_lo + itx % a.ns, pb = (itx / a.ns) % a.npb16, bi = itx / a.ns / a.npb16;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int N = a.N;
  {
    const uint32_t* Wg = a.W + ((int64_t)bi * a.S + s) * a.Npad;
    for (int i = tid; i < a.Npad; i += 256) Ws[i] = Wg[i];
  }
  __syncthreads();
  pf_gather(Ws, a.tables + (int64_t)a.btable[bi] * a.nperm * N, pb, a.nperm, N, a.nks, Bf, tid, 256);
  __syncthreads();

  const int64_t P0 = a.bpoff[bi], np = a.bpoff[bi + 1] - P0;
  const int npair = (int)((np + 31) / 32); /* pairs of tiles */
  const YStat y = a.ys[(int64_t)bi * a.S + s];
  const double kc = y.tsum / (double)N, nu = (double)a.nu, inv_yy = 1.0 / y.yy;
  const double k_row = MODE == PF_SEP ? y.scale * y.scale * inv_yy : y.scale * sqrt(inv_yy);
  PfZeta zp = {};
  if (MODE != PF_SEP) zp = pf_zeta_load(a.zt);
  const int64_t perm = (int64_t)pb * 16 + (lane & 15);
  const bool pvalid = perm < a.nperm;
  const int64_t row_step = (int64_t)a.S * a.NPP;
  double r2mx = -1.0; /* sep: max R^2 = (x'y)^2 / (x'x y'y) over SNPs; t^2 = nu R^2 / (1 - R^2) */
  bool fb = false;
  for (int t = w; t < npair; t += 4) {
    v4i acc[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[u][d] = v4i{0, 0, 0, 0};
    const v4i* ap[2];
    /* the epilogue's per-SNP inputs of this lane's eight rows, loaded ahead of
     * the products so that their latency overlaps the matrix work: sx tsum / N
     * and rs_xx (join) or inv_xx (sep) with the gene's factors; NaN where the
     * SNP is not estimable, past the last one and past the last permutation */
    double cc[2][4], sc[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ap[u] = (const v4i*)(a.G8 + (P0 + min((int64_t)t * 32 + 16 * u + (lane & 15), np - 1)) * a.Npad) + (lane >> 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t q = (int64_t)t * 32 + 16 * u + 4 * (lane >> 4) + r, pr = P0 + min(q, np - 1);
        const PStat st = a.ps[pr];
        const bool on = q < np && pvalid && !a.pflag[pr];
        cc[u][r] = st.sx * kc;
        sc[u][r] = on ? (MODE == PF_SEP ? st.inv_xx : st.rs_xx) * k_row : NAN;
      }
    }
    /* two 64-sample steps per round; the next round's A loads are issued
     * before this round's products */
    v4i af[2][2], an[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int k = 0; k < 2; ++k) af[u][k] = k < a.nks ? ap[u][k * 4] : v4i{0, 0, 0, 0};
    for (int ks0 = 0; ks0 < a.nks; ks0 += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int k = 0; k < 2; ++k) an[u][k] = ks0 + 2 + k < a.nks ? ap[u][(ks0 + 2 + k) * 4] : v4i{0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (ks0 + k < a.nks) {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const v4i b = Bf[((ks0 + k) * 4 + d) * 64 + lane];
#pragma unroll
            for (int u = 0; u < 2; ++u)
              acc[u][d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[u][k], b, acc[u][d], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int k = 0; k < 2; ++k) af[u][k] = an[u][k];
    }
    float* zrow = MODE == PF_SEP ? nullptr
                                 : a.zeta + ((P0 + (int64_t)t * 32 + 4 * (lane >> 4)) * a.S + s) * a.NPP + perm;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double d = pf_fold(acc[u], r) - cc[u][r];
        if (MODE == PF_SEP) {
          /* R^2 = 1 - rss / y'y; the residual sum of squares stays in FP64 */
          const double r2 = d * d * sc[u][r];
          if (isnan(sc[u][r])) continue;
          if (!(1.0 - r2 >= 0.0)) { /* rss < 0: NaN statistic */
            if (t == 0 && u == 0 && r == 0 && lane < 16) fb = true; /* a NaN first statistic: general path */
            continue;
          }
          r2mx = fmax(r2mx, d != 0.0 ? r2 : 0.0);
        } else {
          /* R = |x'y| / sqrt(x'x y'y); |t| / sqrt(nu) = R / sqrt(1 - R^2) */
          const double R = fabs(d) * sc[u][r];
          const float Rf = (float)R, x = Rf * Rf;
          float z = copysignf(pf_zeta_ratio(zp, x) * Rf, (float)d);
          const bool on = !isnan(R);
          if (__builtin_expect(on && (!(Rf < ZP_RMAX) || x * (float)a.nu < 1e-10f), 0))
            z = pf_zeta_slow(a.zt, a.tz, a.nu, R, d, fb);
          /* SNPs that are not estimable have no z (the statistic's kernels handle them) */
          if (on) zrow[(16 * u + r) * row_step] = z;
        }
      }
    }
  }
  if (fb) a.fallback[bi] = 1;
  if (MODE == PF_SEP) {
    r2mx = fmax(r2mx, __shfl_xor(r2mx, 16, 64));
    r2mx = fmax(r2mx, __shfl_xor(r2mx, 32, 64));
    if (lane < 16) redt[w][lane] = r2mx;
    __syncthreads();
    if (tid < 16) {
      const int64_t p = (int64_t)pb * 16 + tid;
      const double m = fmax(fmax(redt[0][tid], redt[1][tid]), fmax(redt[2][tid], redt[3][tid]));
      if (p < a.nperm) a.tmax[((int64_t)bi * a.S + s) * a.NPP + p] = m < 0.0 ? -1.0 : nu * m / (1.0 - m);
    }
  }
}

/* ---- per-SNP coefficients of the Bayes factors ---------------------------------------
 * coef[pair][j][0..2S]: q, Cabf_1..S, D_1..S at grid point j of the grids
 * the statistic uses (large grid first when used, then small), scaled by
 * log2(10) so that the terms are 2^l. */
__global__ void pf_coef_kernel(const PStat* __restrict__ ps, const uint8_t* __restrict__ pflag, int64_t nbp,
                               const double* __restrict__ phi, const double* __restrict__ oma, int ngrid, int S,
                               float* __restrict__ coef) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nbp * ngrid) return;
  const int64_t b = e / ngrid;
  const int j = (int)(e - b * ngrid);
  const int nc = pf_ncf(S);
  float* out = coef + (b * ngrid + j) * nc;
  for (int k = 1 + 2 * S; k < nc; ++k) out[k] = 0.f;
  if (pflag[b]) {
    for (int k = 0; k < 1 + 2 * S; ++k) out[k] = 0.f;
    return;
  }
  const double v = ps[b].inv_xx, p2 = phi[j], o2 = oma[j];
  const double r = 1.0 / (v + p2);
  const double c2 = 1.0 / (2.0 * 0.69314718055994531); /* log2(10) / (2 ln 10) */
  out[0] = (float)(p2 * r * c2);
  const double lvr = log2(v * r);
  for (int m = 1; m <= S; ++m) {
    const double den = 1.0 + m * r * o2;
    out[m] = (float)(0.5 * m * lvr - 0.5 * log2(den));
    out[S + m] = (float)(o2 * v * r * r * c2 / den);
  }
}

/* ---- Bayes-factor statistic per (SNP, permutation) --------------------------------------
 * Work item = (batch gene, 64 permutations, block of SNPs); one wave, lane =
 * permutation, so the SNP's coefficients are uniform across the wave.  Writes
 * the block's max (or sum) over SNPs of the linear-scale statistic. */
struct PfBmaArgs {
  const float* zeta;
  const float* coef;
  const uint8_t* pflag;
  const int4* items; /* (bi, pb, sb, slot) */
  const int64_t* bpoff;
  float* pmax;  /* [slot][NPP] */
  double* psum; /* [slot][NPP] */
  int* fallback;
  float lw[2][9]; /* log2 weights: [0] large-grid terms by m, [1] small-grid terms by m */
  float lwc[9];   /* log2 C(S, m) (bounds of pf_bma_max_kernel) */
  int GL, GS, use_max, n_items;
  int64_t NPP, nperm;
};

/* One row of coefficients, read in 16-byte pieces.  The loops over a SNP's rows
 * hold the two next ones: where each lane reads a SNP of its own a row takes
 * longer to arrive than to use. */
template <int S>
struct PfRow {
  float v[pf_ncf(S)];
};
template <int S>
__device__ __forceinline__ PfRow<S> pf_row(const float* cf, int j) {
  PfRow<S> r;
  const float4* p = reinterpret_cast<const float4*>(cf + j * pf_ncf(S));
#pragma unroll
  for (int k = 0; k < pf_ncf(S) / 4; ++k) {
    const float4 f = p[k];
    r.v[4 * k] = f.x;
    r.v[4 * k + 1] = f.y;
    r.v[4 * k + 2] = f.z;
    r.v[4 * k + 3] = f.w;
  }
  return r;
}
/* f(row) for the GS rows at cf, in order */
template <int S, class F>
__device__ __forceinline__ void pf_rows(const float* cf, int GS, F f) {
  PfRow<S> r0 = pf_row<S>(cf, 0), r1 = pf_row<S>(cf, min(1, GS - 1));
  for (int j = 0; j < GS; ++j) {
    const PfRow<S> r2 = pf_row<S>(cf, min(j + 2, GS - 1));
    f(r0.v);
    r0 = r1;
    r1 = r2;
  }
}

/* Some |z| <= 1e-8: those subgroups drop out of their configurations
 * (rare; kept out of line). */
template <int S>
struct PfZ {
  float v[S];
};
template <int S>
__device__ __noinline__ float pf_sum_all_zero(const PfZ<S> z, const float* __restrict__ cf, int GS, const PfZ<9> lw,
                                              int nzm) {
  constexpr int NC = (1 << S) - 1;
  constexpr int NCF = pf_ncf(S);
  float sum = 0.f;
  for (int g = 1; g <= NC; ++g) {
    float Z1 = 0.f, Z2 = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s)
      if ((g >> s) & 1) {
        Z1 += z.v[s];
        Z2 = fmaf(z.v[s], z.v[s], Z2);
      }
    Z1 *= Z1;
    const int m = __popc(g), me = __popc(g & nzm);
    for (int j = 0; j < GS; ++j) {
      const float* row = cf + j * NCF;
      float l = lw.v[m];
      if (me > 0) l += fmaf(row[S + me], Z1, fmaf(row[0], Z2, row[me]));
      sum += __builtin_amdgcn_exp2f(l);
    }
  }
  return sum;
}

template <int S>
__device__ inline float pf_sum_all(const float (&z)[S], const float* __restrict__ cf, int GS, const float* lw,
                                   int nzm) {
  constexpr int NC = (1 << S) - 1;
  constexpr int NCF = pf_ncf(S);
  if (nzm != NC) {
    PfZ<S> zz;
    PfZ<9> ww;
#pragma unroll
    for (int s = 0; s < S; ++s) zz.v[s] = z[s];
#pragma unroll
    for (int m = 0; m < 9; ++m) ww.v[m] = lw[m];
    return pf_sum_all_zero<S>(zz, cf, GS, ww, nzm);
  }
  float Z1[NC + 1], Z2[NC + 1];
  Z1[0] = 0.f;
  Z2[0] = 0.f;
#pragma unroll
  for (int g = 1; g <= NC; ++g) {
    const int lo = g & (g - 1), s = __builtin_ctz(g);
    Z1[g] = Z1[lo] + z[s];
    Z2[g] = fmaf(z[s], z[s], Z2[lo]);
  }
#pragma unroll
  for (int g = 1; g <= NC; ++g) Z1[g] = Z1[g] * Z1[g];
  float part[4] = {0.f, 0.f, 0.f, 0.f}; /* four partial sums: independent add chains */
  pf_rows<S>(cf, GS, [&](const float(&row)[NCF]) {
    const float q = row[0];
    float C[S + 1], D[S + 1];
#pragma unroll
    for (int m = 1; m <= S; ++m) {
      C[m] = row[m] + lw[m];
      D[m] = row[S + m];
    }
#pragma unroll
    for (int g = 1; g <= NC; ++g) {
      const int m = __builtin_popcount(g);
      part[g & 3] += __builtin_amdgcn_exp2f(fmaf(D[m], Z1[g], fmaf(q, Z2[g], C[m])));
    }
  });
  return (part[0] + part[1]) + (part[2] + part[3]);
}

template <int S>
__device__ inline float pf_sum_gen(const float (&z)[S], const float* __restrict__ cf, int G, float lw, int nzm) {
  constexpr int NCF = pf_ncf(S);
  float Z1 = 0.f, Z2 = 0.f;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    Z1 += z[s];
    Z2 = fmaf(z[s], z[s], Z2);
  }
  Z1 *= Z1;
  const int me = __popc(nzm);
  float sum = 0.f;
  if (me == 0) return (float)G * __builtin_amdgcn_exp2f(lw);
  for (int j = 0; j < G; ++j) {
    const float* row = cf + j * NCF;
    sum += __builtin_amdgcn_exp2f(fmaf(row[S + me], Z1, fmaf(row[0], Z2, row[me] + lw)));
  }
  return sum;
}

template <int S>
__device__ inline float pf_sum_sin(const float (&z)[S], const float* __restrict__ cf, int G, float lw) {
  constexpr int NCF = pf_ncf(S);
  float sum = 0.f;
  for (int j = 0; j < G; ++j) {
    const float* row = cf + j * NCF;
    const float c1 = row[1] + lw, k1 = row[0] + row[S + 1];
#pragma unroll
    for (int s = 0; s < S; ++s) sum += __builtin_amdgcn_exp2f(z[s] != 0.f ? fmaf(k1, z[s] * z[s], c1) : lw);
  }
  return sum;
}

template <int S, int MODE>
__global__ void __launch_bounds__(256) pf_bma_kernel(const PfBmaArgs a) {
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= a.n_items) return;
  const int lane = threadIdx.x & 63;
  const int4 it = a.items[item];
  const int bi = it.x, pb = it.y, sb = it.z, slot = it.w;
  const int64_t P0 = a.bpoff[bi], np = a.bpoff[bi + 1] - P0;
  const int64_t q0 = (int64_t)sb * PF_SB, q1 = min(np, q0 + PF_SB);
  const int64_t p = (int64_t)pb * 64 + lane;
  const bool valid = p < a.nperm;
  const int64_t pp = valid ? p : 0;
  const int NCF = pf_ncf(S);
  const int ngrid = (MODE == PF_JOIN_ALL) ? a.GS : (MODE == PF_JOIN_GEN ? a.GL : a.GL + a.GS);
  float mx = 0.f;
  double sm = 0.0;
  bool bad = false;
  for (int64_t q = q0; q < q1; ++q) {
    const int64_t pr = P0 + q;
    float val;
    if (a.pflag[pr]) {
      val = 1.f; /* every ABF of a non-estimable SNP is 1 */
    } else {
      float z[S];
      int nzm = 0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        z[s] = a.zeta[(pr * S + s) * a.NPP + pp];
        nzm |= (z[s] != 0.f) << s;
      }
      const float* cf = a.coef + pr * (int64_t)ngrid * NCF;
      if (MODE == PF_JOIN_ALL) {
        val = pf_sum_all<S>(z, cf, a.GS, a.lw[1], nzm);
      } else if (MODE == PF_JOIN_GEN) {
        val = pf_sum_gen<S>(z, cf, a.GL, a.lw[0][S], nzm);
      } else {
        val = pf_sum_gen<S>(z, cf, a.GL, a.lw[0][S], nzm) + pf_sum_sin<S>(z, cf + a.GL * NCF, a.GS, a.lw[1][1]);
      }
    }
    bad |= !(val < INFINITY) || !(val > 1e-30f);
    mx = fmaxf(mx, val);
    sm += (double)val;
  }
  if (valid) {
    a.pmax[(int64_t)slot * a.NPP + p] = mx;
    a.psum[(int64_t)slot * a.NPP + p] = sm;
    if (bad) a.fallback[bi] = 1;
  }
}

/* ---- statistic per (gene, permutation) --------------------------------------------- */
struct PfFinalArgs {
  const float* pmax;
  const double* psum;
  const double* tmax;
  const int32_t* bgene;
  const int64_t* bpoff;
  const int32_t* bslot; /* first slot of each batch gene */
  const uint8_t* pflag;
  const double* tz;
  double* stats; /* [G][nperm] */
  int nb, S, nu, mode, use_max, sep_sbgrp;
  int one_slot; /* the maximum of each (gene, permutation) is in its first slot */
  int64_t nperm, NPP;
};

__global__ void pf_final_kernel(const PfFinalArgs a) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)a.nb * a.nperm) return;
  const int bi = (int)(e / a.nperm);
  const int64_t p = e - (int64_t)bi * a.nperm;
  const int64_t np = a.bpoff[bi + 1] - a.bpoff[bi];
  double res;
  if (a.mode == PF_SEP) {
    double m = -1.0;
    if (a.sep_sbgrp >= 0) {
      m = a.tmax[((int64_t)bi * a.S + a.sep_sbgrp) * a.NPP + p];
    } else {
      for (int s = 0; s < a.S; ++s) m = fmax(m, a.tmax[((int64_t)bi * a.S + s) * a.NPP + p]);
    }
    if (a.sep_sbgrp >= 0 && a.pflag[a.bpoff[bi]]) {
      res = NAN; /* std::min_element: the first SNP's p-value is NaN */
    } else if (m < 0) {
      res = 1.0;
    } else {
      const double pv = 2.0 * exp(-dm::tz_eval(a.tz, a.nu, sqrt(m)));
      res = pv < 1.0 ? pv : 1.0;
    }
  } else {
    const int nsb = a.one_slot ? 1 : (int)((np + PF_SB - 1) / PF_SB);
    const int slot0 = a.bslot[bi];
    if (a.use_max) {
      float m = 0.f;
      for (int k = 0; k < nsb; ++k) m = fmaxf(m, a.pmax[(int64_t)(slot0 + k) * a.NPP + p]);
      res = log10((double)m);
    } else {
      double sm = 0.0;
      for (int k = 0; k < nsb; ++k) sm += a.psum[(int64_t)(slot0 + k) * a.NPP + p];
      res = log10(sm / (double)np);
    }
    if (fabs(res) <= 2.220446049250313e-16) res = 0.0;
  }
  a.stats[(int64_t)a.bgene[bi] * a.nperm + p] = res;
}

/* ---- --pbf all --maxbf: the maximum over SNPs without evaluating every SNP --------------
 * Work item = (batch gene, 4 x 64 permutations), one wave per 64
 * permutations (lane = permutation), the gene's SNPs in blocks of 64 whose
 * Bayes-factor coefficients are staged in LDS.  Every configuration of
 * size m and grid point j has an exponent (log2) of at most
 *   E_mj = lw_m + C_mj + q_j Z2max_m + D_mj Z1max_m^2,
 * Z2max_m = the sum of the m largest z^2, Z1max_m^2 = the larger square of
 * the sums of the m largest and of the m smallest z (q, D >= 0).  Two bounds
 * of log2(statistic) follow: log2(number of terms) + max E_mj (a few
 * operations per grid point, every SNP), and log2 sum_m,j C(S, m) 2^E_mj (one
 * exponential per (m, j), the SNPs that pass the first).  Only a SNP whose
 * bounds reach the lane's running maximum can raise it: those go through two
 * queues in LDS, 64 entries at a time, and are evaluated exactly by
 * pf_sum_all (the arithmetic of pf_bma_kernel), so the running maxima, and the
 * final maximum, are exactly pf_bma_kernel's.  A SNP with some z = 0 (its
 * subgroup drops out of the configurations) skips the bounds. */
constexpr int PFQ = 128;  /* entries per queue and wave      */
constexpr int PF_WG = 4;  /* waves (permutation blocks) per item */

template <int S>
struct PfSorted {
  float Z2[S + 1], Q1[S + 1];
};

template <int S>
__device__ inline PfSorted<S> pf_sorted(const float (&z)[S]) {
  float a[S], b[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    a[s] = z[s];
    b[s] = z[s] * z[s];
  }
#pragma unroll
  for (int i = 1; i < S; ++i)
#pragma unroll
    for (int k = i; k > 0; --k) {
      const float lo = fminf(a[k - 1], a[k]), hi = fmaxf(a[k - 1], a[k]);
      a[k - 1] = lo;
      a[k] = hi;
      const float bl = fmaxf(b[k - 1], b[k]), bs = fminf(b[k - 1], b[k]);
      b[k - 1] = bl;
      b[k] = bs;
    }
  PfSorted<S> r;
  float top = 0.f, bot = 0.f, sq = 0.f;
#pragma unroll
  for (int m = 1; m <= S; ++m) {
    top += a[S - m];
    bot += a[m - 1];
    sq += b[m - 1];
    r.Z2[m] = sq;
    r.Q1[m] = fmaxf(top * top, bot * bot);
  }
  return r;
}

/* first bound: max over (m, j) of E_mj (without the log2 of the term count) */
template <int S>
__device__ inline float pf_bound_max(const PfSorted<S>& t, const float* cf, int GS, const float* lw) {
  constexpr int NCF = pf_ncf(S);
  float u = -INFINITY;
  for (int j = 0; j < GS; ++j) {
    const float* row = cf + j * NCF;
    const float q = row[0];
#pragma unroll
    for (int m = 1; m <= S; ++m) u = fmaxf(u, fmaf(row[S + m], t.Q1[m], fmaf(q, t.Z2[m], row[m] + lw[m])));
  }
  return u;
}

/* second bound: log2 sum over (m, j) of C(S, m) 2^E_mj; lwc_m = lw_m + log2 C(S, m) */
template <int S>
__device__ inline float pf_bound_sum(const PfSorted<S>& t, const float* cf, int GS, const float* lwc) {
  constexpr int NCF = pf_ncf(S);
  float sum = 0.f;
  pf_rows<S>(cf, GS, [&](const float(&row)[NCF]) {
#pragma unroll
    for (int m = 1; m <= S; ++m)
      sum += __builtin_amdgcn_exp2f(fmaf(row[S + m], t.Q1[m], fmaf(row[0], t.Z2[m], row[m] + lwc[m])));
  });
  return __builtin_amdgcn_logf(sum);
}

template <int S>
__global__ void __launch_bounds__(64 * PF_WG) pf_bma_max_kernel(const PfBmaArgs a) {
  extern __shared__ __align__(16) float cfs[]; /* [64 SNPs][GS][NCF] */
  __shared__ uint32_t q1s[PF_WG][PFQ], q2s[PF_WG][PFQ], mbs[PF_WG][64];
  constexpr int NC = (1 << S) - 1;
  constexpr int NCF = pf_ncf(S);
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int4 it = a.items[blockIdx.x];
  const int bi = it.x, slot = it.w;
  const int64_t P0 = a.bpoff[bi], np = a.bpoff[bi + 1] - P0;
  const int64_t pbase = ((int64_t)it.y + wv) * 64;
  const int64_t p = pbase + lane;
  const bool valid = p < a.nperm;
  const int GS = a.GS, rowf = GS * NCF;
  uint32_t* q1 = q1s[wv];
  uint32_t* q2 = q2s[wv];
  uint32_t* mb = mbs[wv];
  float lw[S + 1], lwc[S + 1];
#pragma unroll
  for (int m = 1; m <= S; ++m) {
    lw[m] = a.lw[1][m];
    lwc[m] = a.lw[1][m] + a.lwc[m];
  }
  const float lg_terms = __builtin_amdgcn_logf((float)(NC * GS));
  mb[lane] = 0u; /* +0.0f: statistics are > 0 */
  float lm = -INFINITY; /* log2 of this lane's running maximum */
  int n1 = 0, n2 = 0;
  bool bad = false;
  int64_t b0 = 0; /* first SNP of the staged block */

  auto zload = [&](int64_t pr, int64_t pp, float (&z)[S]) {
#pragma unroll
    for (int s = 0; s < S; ++s) z[s] = a.zeta[(pr * S + s) * a.NPP + pp];
  };
  /* exact statistics of the first k entries of queue 2 */
  auto drain2 = [&](int k) {
    if (lane < k) {
      const uint32_t e = q2[lane];
      const int ql = (int)(e >> 6), le = (int)(e & 63u);
      float z[S];
      zload(P0 + b0 + ql, pbase + le, z);
      int nzm = 0;
#pragma unroll
      for (int s = 0; s < S; ++s) nzm |= (z[s] != 0.f) << s;
      const float val = pf_sum_all<S>(z, cfs + ql * rowf, GS, a.lw[1], nzm);
      bad |= !(val < INFINITY) || !(val > 1e-30f);
      atomicMax(&mb[le], __float_as_uint(val));
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    const int rest = n2 - k;
    if (lane < rest) {
      const uint32_t v = q2[k + lane];
      q2[lane] = v;
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    n2 = rest;
    lm = __builtin_amdgcn_logf(__uint_as_float(mb[lane]));
  };
  /* second bound of the first k entries of queue 1; survivors to queue 2 */
  auto drain1 = [&](int k) {
    bool pass = false;
    const uint32_t e = lane < k ? q1[lane] : 0u;
    const int le = lane < k ? (int)(e & 63u) : lane;
    const float lmq = __shfl(lm, le, 64); /* every lane takes part */
    if (lane < k) {
      const int ql = (int)(e >> 6);
      float z[S];
      zload(P0 + b0 + ql, pbase + le, z);
      bool zero = false;
#pragma unroll
      for (int s = 0; s < S; ++s) zero |= z[s] == 0.f;
      pass = zero || !(pf_bound_sum<S>(pf_sorted<S>(z), cfs + ql * rowf, GS, lwc) + 0.00390625f < lmq);
    }
    const uint64_t bal = __ballot(pass);
    const int pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
    if (pass) q2[n2 + pos] = e;
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    n2 += __popcll(bal);
    if (n2 >= 64) drain2(64);
    const int rest = n1 - k;
    if (lane < rest) {
      const uint32_t v = q1[k + lane];
      q1[lane] = v;
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    n1 = rest;
  };

  for (b0 = 0; b0 < np; b0 += 64) {
    const int nq = (int)min((int64_t)64, np - b0);
    __syncthreads(); /* every wave is done with the previous block */
    {
      const float* src = a.coef + (P0 + b0) * (int64_t)rowf;
      for (int e = threadIdx.x; e < nq * rowf; e += 64 * PF_WG) cfs[e] = src[e];
    }
    __syncthreads();
    if (pbase >= a.nperm) continue; /* a wave past the last permutation only joins the barriers */
    float zn[S];
    zload(P0 + b0, valid ? p : pbase, zn);
    for (int ql = 0; ql < nq; ++ql) {
      float z[S];
#pragma unroll
      for (int s = 0; s < S; ++s) z[s] = zn[s];
      if (ql + 1 < nq) zload(P0 + b0 + ql + 1, valid ? p : pbase, zn);
      if (a.pflag[P0 + b0 + ql]) { /* every ABF of a non-estimable SNP is 1 */
        if (valid) atomicMax(&mb[lane], __float_as_uint(1.f));
        __builtin_amdgcn_s_waitcnt(0);
        lm = __builtin_amdgcn_logf(__uint_as_float(mb[lane]));
        continue;
      }
      bool zero = false;
#pragma unroll
      for (int s = 0; s < S; ++s) zero |= z[s] == 0.f;
      const float u = pf_bound_max<S>(pf_sorted<S>(z), cfs + ql * rowf, GS, lw) + lg_terms;
      /* a margin of 2^-8 for the FP32 rounding of the bound and the maximum */
      const bool cand = valid && (zero || !(u + 0.00390625f < lm));
      const uint64_t bal = __ballot(cand);
      if (bal) {
        const int pos =
            __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
        if (cand) q1[n1 + pos] = ((uint32_t)ql << 6) | (uint32_t)lane;
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
        n1 += __popcll(bal);
        if (n1 >= 64) drain1(64);
      }
    }
    while (n1 > 0) drain1(min(n1, 64));
    while (n2 > 0) drain2(min(n2, 64));
  }
  if (bad) atomicOr(&a.fallback[bi], 1);
  if (valid) a.pmax[(int64_t)slot * a.NPP + p] = __uint_as_float(mb[lane]);
}

/* ---- --pbf all --maxbf in one kernel: contraction, bounds and maximum ----------------
 * The z values of all SNPs and permutations (4.8 GB for 24 genes of 1,000 SNPs,
 * 5 subgroups and 10,000 permutations) were written in 64-byte pieces and read
 * again, which bounded both kernels (4.6 and 3.9 ms).  Here a workgroup takes 16
 * permutations of a gene with the digit fragments of every subgroup in LDS, so
 * that a lane holds all S z values of its (SNP, permutation)s, and nothing but
 * the maxima is written.
 *
 * A SNP is evaluated exactly (pf_sum_all, as in pf_bma_kernel) only if an upper
 * bound of its statistic reaches the running maximum, so the maxima are exactly
 * those of all SNPs.  First bound, one comparison: with T = sum_s z_s^2,
 *   statistic <= sum_m,j [(m/S) 2^(C_mj + (q_j + m D_mj) T) + (1 - m/S) 2^C_mj]
 *                / (S GS) = 2^F(T),
 * since Z1^2 <= m Z2 in a configuration of m subgroups, and the sum over the
 * configurations of size m is then convex in the z_s^2, so largest where one of
 * them is T.  F is convex with a slope of at most 1 / (2 ln 2), so from the T at
 * which F reaches a level L below the running maximum M (pf_thr_kernel), or would
 * reach it at that slope, M asks for at least (M - L) 2 ln 2 more.  Second bound: pf_bound_sum.  Survivors pass
 * through two queues per wave, 64 at a time, and what is left of all queues at the
 * end is shared out in full waves.  A z of 0 (its subgroup drops out of the
 * configurations) skips the bounds.  A wave starts with the exact value of its
 * largest T of each permutation, so that the bounds have a maximum to work against:
 * 3 % of the SNPs then pass the first bound and 0.7 % the second. (With lower
 * bounds from single terms as the start 70 % passed the first.)  Bound by the
 * vector unit: two FP64 conversions, a product and the polynomial per z, at two
 * waves per SIMD.  24 genes of 1,000 SNPs, 5 subgroups of 300 samples, 10,000
 * permutations: 4.8 ms, from 4.6 + 3.9 ms for the two kernels.
 *
 * The digits' 64-sample steps are held in registers, so more than PFX_NKS of them,
 * fragments that don't fit in LDS, or a genotype past PFX_XMAX take the two
 * kernels. */
constexpr int PFX_WG = 8;     /* waves per workgroup               */
constexpr int PFX_NKS = 8;    /* 64-sample steps held in registers  */
constexpr int PFX_PAD = 32;   /* rows past the batch's last pair    */
constexpr int PFX_BINS = 32;  /* levels L = PFX_L0 + bin            */
constexpr float PFX_L0 = -2.f;

/* SNPs from which a gene is worth the one kernel: its eight waves take 32 SNPs at
 * a time, and those without a tile wait for the others.  All kernels of both kinds,
 * one and two, us for 1,000 permutations of (genes x SNPs): S = 1, N = 100: 1,034 /
 * 312 (375 x 64), 408 / 349 (125 x 192), 360 / 411 (93 x 256); S = 3, N = 200:
 * 2,004 / 914, 751 / 791, 654 / 880; S = 5, N = 300: 1,738 / 1,045 (187 x 64),
 * 1,196 / 926 (125 x 96), 914 / 976 (93 x 128); S = 6, N = 150: 1,375 / 1,268 (93 x
 * 128), 1,054 / 1,250 (62 x 192). */
constexpr int64_t pf_max_snps(int S) { return S <= 3 ? 224 : S <= 5 ? 128 : 160; }

/* bytes of LDS: fragments, then the digit words (phase 1) or the queues */
size_t pf_max_lds(int S, int Npad) {
  const size_t frag = (size_t)S * (Npad / 64) * 4 * 64 * 16;
  const size_t words = (size_t)S * Npad * 4, queues = (size_t)PFX_WG * 2 * PFQ * (S + 1) * 4;
  return frag + std::max(words, queues);
}

/* thr[bin][pair]: a lower bound of the T at which F reaches the bin's level, from
 * F at T = 0..63 (lane = T): the chords of a convex function lie above it.  Where
 * F(0) is above the level, the T below 0 at which the steepest slope would reach
 * it, so that a maximum M asks for T >= (M - F(0)) 2 ln 2 of such a SNP.  One wave
 * per pair. */
template <int S>
__global__ void __launch_bounds__(256) pf_thr_kernel(const float* __restrict__ coef, int64_t nbp, int GS,
                                                     float* __restrict__ thr) {
  constexpr int NCF = pf_ncf(S);
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= nbp) return;
  const int lane = threadIdx.x & 63;
  const float T = (float)lane;
  float sum = 0.f;
  for (int j = 0; j < GS; ++j) {
    const float* row = coef + (b * GS + j) * NCF;
#pragma unroll
    for (int m = 1; m <= S; ++m)
      sum += __builtin_amdgcn_exp2f(row[m]) *
             ((float)m / S * __builtin_amdgcn_exp2f((row[0] + m * row[S + m]) * T) + 1.f - (float)m / S);
  }
  const float F = __builtin_amdgcn_logf(sum / (float)(S * GS));
  for (int k = 0; k < PFX_BINS; ++k) {
    const float L = PFX_L0 + k - 0.0078125f; /* margin of the FP32 sums */
    const int n = __popcll(__ballot(F <= L)); /* F grows with T */
    float t;
    if (n >= 64) {
      t = 63.f;
    } else if (n == 0) {
      t = (L - __shfl(F, 0, 64)) * 1.38629436f - 0.001f; /* 2 ln 2 */
    } else {
      const float f0 = __shfl(F, n - 1, 64), f1 = __shfl(F, n, 64);
      t = (float)(n - 1) + (L - f0) / (f1 - f0) - 0.001f;
    }
    if (lane == 0) thr[(int64_t)k * nbp + b] = t;
  }
}

struct PfMaxArgs {
  PfGemmArgs g; /* zeta, tmax, s_lo, ns unused */
  const float* coef;
  const float* thr;
  const int32_t* bslot;
  float* pmax; /* [slot][NPP] */
  float lw[9], lwc[9];
  int GS;
  int64_t nbp;
};

template <int S>
__global__ void __launch_bounds__(64 * PFX_WG) pf_max_kernel(const PfMaxArgs x) {
  extern __shared__ __align__(16) unsigned char sm[];
  const PfGemmArgs& a = x.g;
  constexpr int NCF = pf_ncf(S), QW = PFQ * (S + 1); /* words of a queue */
  __shared__ uint32_t mb[16], lb[16]; /* running maxima, lower bounds of them (positive floats) */
  __shared__ int left1[PFX_WG], left2[PFX_WG];
  __shared__ double kcs[S], krs[S];
  v4i* Bf = (v4i*)sm; /* [S][nks][4][64] */
  unsigned char* rest = sm + (size_t)S * a.nks * 4 * 64 * 16;
  const int nit = a.n_items, per = (nit + 7) / 8;
  const int itx = (blockIdx.x & 7) * per + (blockIdx.x >> 3); /* XCD-aware, as in pf_gemm_kernel */
  if (itx >= nit) return;
  const int pb = itx % a.npb16, bi = itx / a.npb16;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = a.N;
  {
    uint32_t* Ws = (uint32_t*)rest;
    const uint32_t* Wg = a.W + (int64_t)bi * S * a.Npad;
    for (int i = tid; i < S * a.Npad; i += 64 * PFX_WG) Ws[i] = Wg[i];
    if (tid < 16) mb[tid] = lb[tid] = 0u;
    if (tid < S) {
      const YStat y = a.ys[(int64_t)bi * S + tid];
      kcs[tid] = y.tsum / (double)N;
      krs[tid] = y.scale * sqrt(1.0 / y.yy);
    }
    __syncthreads();
    const int32_t* tab = a.tables + (int64_t)a.btable[bi] * a.nperm * N;
#pragma unroll 1
    for (int s = 0; s < S; ++s)
      pf_gather(Ws + s * a.Npad, tab, pb, a.nperm, N, a.nks, Bf + (size_t)s * a.nks * 256, tid, 64 * PFX_WG);
    __syncthreads();
  }
  /* two queues per wave: entry (SNP of the gene << 4 | permutation) and its z */
  uint32_t* const queues = (uint32_t*)rest;
  uint32_t* q1 = queues + wv * 2 * QW;
  uint32_t* q2 = q1 + QW;
  const int64_t P0 = a.bpoff[bi], np = a.bpoff[bi + 1] - P0;
  const int npair = (int)((np + 31) / 32);
  const PfZeta zp = pf_zeta_load(a.zt);
  const int pl = lane & 15;
  const bool pvalid = (int64_t)pb * 16 + pl < a.nperm;
  int n1 = 0, n2 = 0;
  bool fb = false;

  auto sync_wave = [&]() { /* LDS of this wave written by one lane, read by another */
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  auto put = [&](uint32_t* q, int& n, bool on, uint32_t e, const float (&z)[S]) {
    const uint64_t bal = __ballot(on);
    const int pos = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
    if (on) {
      q[pos] = e;
#pragma unroll
      for (int s = 0; s < S; ++s) q[(s + 1) * PFQ + pos] = __float_as_uint(z[s]);
    }
    n += __popcll(bal);
    sync_wave();
  };
  auto get = [&](const uint32_t* q, int at, float (&z)[S]) {
#pragma unroll
    for (int s = 0; s < S; ++s) z[s] = __uint_as_float(q[(s + 1) * PFQ + at]);
    return q[at];
  };
  auto shift = [&](uint32_t* q, int& n, int k) { /* drops the first k entries */
    const int left = n - k;
    uint32_t v[S + 1];
    if (lane < left) {
#pragma unroll
      for (int s = 0; s <= S; ++s) v[s] = q[s * PFQ + k + lane];
    }
    sync_wave();
    if (lane < left) {
#pragma unroll
      for (int s = 0; s <= S; ++s) q[s * PFQ + lane] = v[s];
    }
    n = left;
    sync_wave();
  };
  auto row_of = [&](uint32_t e) { return x.coef + (P0 + (int64_t)(e >> 4)) * (int64_t)(x.GS * NCF); };
  /* log2 of what is known of the maximum of permutation p */
  auto known = [&](uint32_t p) {
    const uint32_t m = __hip_atomic_load(&mb[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const uint32_t l = __hip_atomic_load(&lb[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return __builtin_amdgcn_logf(__uint_as_float(max(m, l)));
  };
  /* exact statistic of a lane's entry */
  auto exact = [&](bool on, uint32_t e, const float (&z)[S]) {
    if (on) {
      int nzm = 0;
#pragma unroll
      for (int s = 0; s < S; ++s) nzm |= (z[s] != 0.f) << s;
      const float val = pf_sum_all<S>(z, row_of(e), x.GS, x.lw, nzm);
      fb |= !(val < INFINITY) || !(val > 1e-30f);
      atomicMax(&mb[e & 15u], __float_as_uint(val));
    }
  };
  /* second bound of a lane's entry; survivors to queue 2 */
  auto second = [&](bool on, uint32_t e, const float (&z)[S]) {
    bool pass = false;
    if (on) {
      bool zero = false;
#pragma unroll
      for (int s = 0; s < S; ++s) zero |= z[s] == 0.f;
      pass = zero ||
             !(pf_bound_sum<S>(pf_sorted<S>(z), row_of(e), x.GS, x.lwc) + 0.00390625f < known(e & 15u));
    }
    put(q2, n2, pass, e, z);
  };
  /* entry i of all waves' queue q (0 or 1) together, `left` of them in each */
  auto joint = [&](int q, const int* left, int i, uint32_t& e, float (&z)[S]) {
    bool on = false;
    e = 0u;
    for (int w = 0; w < PFX_WG; ++w) {
      if (!on && i >= 0 && i < left[w]) {
        on = true;
        e = get(queues + (w * 2 + q) * QW, i, z);
      }
      i -= left[w];
    }
    return on;
  };

  /* After a wave's last tiles (phase 0) the rest of all queues 1 (phase 1) and
   * then of all queues 2 (phase 2) is shared out in full waves.  One loop, so
   * that the code of the bounds and of the sums is there once. */
  int t = wv, phase = 0;
  if (t >= npair) { /* no tiles for this wave */
    phase = 1;
    if (lane == 0) left1[wv] = 0;
    __syncthreads();
  }
  while (phase < 3) {
    const int64_t r0 = (int64_t)t * 32 + 4 * (lane >> 4);
    float z[S][8], T[8], th[2][4];
    uint32_t mask = 0, zero = 0; /* rows of this lane for the first queue; with some z of 0 */
    const bool first = phase == 0 && t == wv;
    /* thresholds of T: the level is the one below the wave's least maximum, and
     * a lane's maximum asks for more; every SNP while a maximum is below the
     * lowest level */
    auto thresholds = [&]() {
      const float lm = known(pl) - 0.00390625f;
      float least = pvalid ? lm : INFINITY;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) least = fminf(least, __shfl_xor(least, o, 64));
      const int bin = (int)fminf(fmaxf(floorf(least - PFX_L0), 0.f), (float)(PFX_BINS - 1));
      const float over = lm < PFX_L0 + bin ? -INFINITY : (lm - (PFX_L0 + bin)) * 1.38629436f; /* 2 ln 2 */
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        __builtin_memcpy(th[u], x.thr + (int64_t)bin * x.nbp + P0 + r0 + 16 * u, 16);
#pragma unroll
        for (int r = 0; r < 4; ++r) th[u][r] += over;
      }
    };
    if (phase == 0) {
      /* the tiles' genotypes (all steps), per-row statistics and thresholds */
      v4i af[2][PFX_NKS];
      double sx[2][4], rs[2][4];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        /* rows past the gene's last SNP are read (the arrays have PFX_PAD more)
         * and masked by their NaN */
        const v4i* ap = (const v4i*)(a.G8 + (P0 + (int64_t)t * 32 + 16 * u + pl) * a.Npad) + (lane >> 4);
#pragma unroll
        for (int k = 0; k < PFX_NKS; ++k)
          if (k < a.nks) af[u][k] = ap[k * 4];
        const PStat* st = a.ps + P0 + r0 + 16 * u;
        const int live = pvalid ? (int)min((int64_t)4, np - (r0 + 16 * u)) : 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sx[u][r] = st[r].sx;
          const double v = st[r].rs_xx;
          rs[u][r] = r < live ? v : NAN;
          if (__builtin_expect(r < live && isnan(v), 0))
            atomicMax(&mb[pl], __float_as_uint(1.f)); /* every ABF of such a SNP is 1 */
        }
      }
      if (!first) thresholds();
#pragma unroll
      for (int k = 0; k < 8; ++k) T[k] = 0.f;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        v4i acc[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int d = 0; d < 4; ++d) acc[u][d] = v4i{0, 0, 0, 0};
        const v4i* bs = Bf + (size_t)s * a.nks * 256 + lane;
#pragma unroll
        for (int k = 0; k < PFX_NKS; ++k)
          if (k < a.nks) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              const v4i b = bs[(k * 4 + d) * 64];
#pragma unroll
              for (int u = 0; u < 2; ++u)
                acc[u][d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[u][k], b, acc[u][d], 0, 0, 0);
            }
          }
        const double kc = kcs[s], kr = krs[s];
        const float tiny = 1e-5f * __builtin_amdgcn_rsqf((float)a.nu);
        double dv[8];
        bool any_slow = false;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          /* as in pf_gemm_kernel */
          const int u = k >> 2, r = k & 3;
          dv[k] = pf_fold_narrow(acc[u], r) - sx[u][r] * kc;
          const float Rf = (float)(fabs(dv[k]) * (rs[u][r] * kr)), x2 = Rf * Rf;
          const float v = pf_zeta_ratio(zp, x2);
          z[s][k] = __uint_as_float((__float_as_uint(v * Rf) & 0x7fffffffu) |
                                    ((uint32_t)__double2hiint(dv[k]) & 0x80000000u));
          any_slow |= Rf >= ZP_RMAX || Rf < tiny; /* NaN: no SNP */
        }
        /* the rare values that the polynomial does not serve, one at a time: one
         * copy of that code per subgroup */
        if (__any(any_slow)) {
#pragma unroll 1
          for (int k = 0; k < 8; ++k) {
            double d = dv[0], rk = rs[0][0];
#pragma unroll
            for (int i = 1; i < 8; ++i) {
              d = k == i ? dv[i] : d;
              rk = k == i ? rs[i >> 2][i & 3] : rk;
            }
            const double R = fabs(d) * (rk * kr);
            const float Rf = (float)R;
            if (Rf >= ZP_RMAX || Rf < tiny) {
              const float v = pf_zeta_slow(a.zt, a.tz, a.nu, R, d, fb);
              zero |= v == 0.f ? 1u << k : 0u;
#pragma unroll
              for (int i = 0; i < 8; ++i) z[s][i] = k == i ? v : z[s][i];
            }
          }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) T[k] = fmaf(z[s][k], z[s][k], T[k]);
      }
      if (first) {
        /* a lower bound to start from: the statistic of the largest T that the
         * wave has for each permutation, four lanes to one (their sums are in
         * another order than pf_sum_all's, so it does not count as the value) */
        float bestT = -1.f, zb[S] = {};
        int best = -1;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const bool up = T[k] > bestT && !((zero >> k) & 1u); /* NaN: no SNP */
          bestT = up ? T[k] : bestT;
          best = up ? (int)(16 * (k >> 2) + (k & 3) + 4 * (lane >> 4)) : best;
#pragma unroll
          for (int s = 0; s < S; ++s) zb[s] = up ? z[s][k] : zb[s];
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) {
          const float oT = __shfl_xor(bestT, o, 64);
          const int ob = __shfl_xor(best, o, 64);
          const bool up = oT > bestT || (oT == bestT && ob > best);
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const float oz = __shfl_xor(zb[s], o, 64);
            zb[s] = up ? oz : zb[s];
          }
          bestT = up ? oT : bestT;
          best = up ? ob : best;
        }
        float sum = 0.f;
        if (best >= 0) {
          const float* cf = row_of((uint32_t)(t * 32 + best) << 4);
          for (int j = lane >> 4; j < x.GS; j += 4) sum += pf_sum_all<S>(zb, cf + j * NCF, 1, x.lw, (1 << S) - 1);
        }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if (pvalid && best >= 0 && sum < 1e30f) atomicMax(&lb[pl], __float_as_uint(sum * 0.99f));
        sync_wave();
        thresholds();
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) mask |= T[k] >= th[k >> 2][k & 3] ? 1u << k : 0u; /* NaN: no SNP */
      mask |= zero;
    }
    for (int c = 0;; ++c) {
      float ze[S] = {};
      uint32_t e = 0u;
      /* Room in the queues: a turn puts at most 64 entries into queue 1, and only
       * where 64 fit, so n1 <= PFQ; then one action, which is due whenever a queue
       * has 64, takes 64 of them.  Queue 2 gets at most 64, and only while it has
       * fewer than 64.  So n1 <= 128 and n2 < 128 whatever passes, and what a
       * shift keeps is at most 64. */
      if (phase == 0 && n1 <= PFQ - 64 && __any(mask != 0)) {
        const int k = __builtin_ctz(mask | 0x100u);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          ze[s] = z[s][0];
#pragma unroll
          for (int i = 1; i < 8; ++i) ze[s] = k == i ? z[s][i] : ze[s];
        }
        put(q1, n1, mask != 0, (uint32_t)((r0 + 16 * (k >> 2) + (k & 3)) << 4 | pl), ze);
        mask &= mask - 1;
      }
      /* what to do next: 1 the second bound, 2 the exact statistic of 64 entries */
      int act = 0;
      bool on = false;
      if (phase == 0) {
        act = n2 >= 64 ? 2 : (n1 >= 64 ? 1 : 0);
        if (act) {
          on = true;
          e = get(act == 2 ? q2 : q1, lane, ze);
        }
      } else {
        const int* left = phase == 1 ? left1 : left2;
        int total = 0;
        for (int w = 0; w < PFX_WG; ++w) total += left[w];
        if ((wv + PFX_WG * c) * 64 < total) {
          act = phase;
          on = joint(phase - 1, left, (wv + PFX_WG * c) * 64 + lane, e, ze);
        }
      }
      if (act == 2) exact(on, e, ze);
      if (act == 1) second(on, e, ze);
      if (phase == 0 && act) shift(act == 2 ? q2 : q1, act == 2 ? n2 : n1, 64);
      if (!act && !__any(mask != 0)) break;
    }
    if (phase == 0) {
      t += PFX_WG;
      if (t < npair) continue;
      phase = 1;
      if (lane == 0) left1[wv] = n1;
      __syncthreads();
    } else {
      if (phase == 1 && lane == 0) left2[wv] = n2;
      ++phase;
      __syncthreads();
    }
  }
  /* a maximum of nothing: the general path (the bounds keep the largest SNP, and
   * the last barrier above is after every update) */
  if (tid < 16 && (int64_t)pb * 16 + tid < a.nperm) fb |= mb[tid] == 0u;
  if (fb) atomicOr(&a.fallback[bi], 1);
  if (tid < 16 && (int64_t)pb * 16 + tid < a.nperm)
    x.pmax[(int64_t)x.bslot[bi] * a.NPP + (int64_t)pb * 16 + tid] = __uint_as_float(mb[tid]);
}

template <int S>
void launch_pf_max_s(eqbf_ctx* ctx, hipStream_t st, const PfMaxArgs& x, float* thr, size_t lds) {
  {
    ProfScope ps(ctx, "pf_thr_kernel", st);
    hipLaunchKernelGGL(pf_thr_kernel<S>, dim3((unsigned)((x.nbp + 3) / 4)), dim3(256), 0, st, x.coef, x.nbp, x.GS, thr);
  }
  ProfScope ps(ctx, "pf_max_kernel", st);
  hipLaunchKernelGGL(pf_max_kernel<S>, dim3((unsigned)((x.g.n_items + 7) / 8 * 8)), dim3(64 * PFX_WG), lds, st, x);
}
void launch_pf_max(eqbf_ctx* ctx, int S, hipStream_t st, const PfMaxArgs& x, float* thr, size_t lds) {
  switch (S) {
    case 1: return launch_pf_max_s<1>(ctx, st, x, thr, lds);
    case 2: return launch_pf_max_s<2>(ctx, st, x, thr, lds);
    case 3: return launch_pf_max_s<3>(ctx, st, x, thr, lds);
    case 4: return launch_pf_max_s<4>(ctx, st, x, thr, lds);
    case 5: return launch_pf_max_s<5>(ctx, st, x, thr, lds);
    case 6: return launch_pf_max_s<6>(ctx, st, x, thr, lds);
    default: return;
  }
}

template <int MODE>
void launch_bma_s(int S, dim3 grid, hipStream_t st, const PfBmaArgs& a) {
  switch (S) {
#define PF_CASE(SS) \
  case SS: hipLaunchKernelGGL((pf_bma_kernel<SS, MODE>), grid, dim3(256), 0, st, a); break;
    PF_CASE(1) PF_CASE(2) PF_CASE(3) PF_CASE(4) PF_CASE(5) PF_CASE(6)
#undef PF_CASE
    default: break;
  }
}
template <>
void launch_bma_s<PF_JOIN_GEN>(int S, dim3 grid, hipStream_t st, const PfBmaArgs& a) {
  switch (S) {
#define PF_CASE(SS) \
  case SS: hipLaunchKernelGGL((pf_bma_kernel<SS, PF_JOIN_GEN>), grid, dim3(256), 0, st, a); break;
    PF_CASE(1) PF_CASE(2) PF_CASE(3) PF_CASE(4) PF_CASE(5) PF_CASE(6) PF_CASE(7) PF_CASE(8)
#undef PF_CASE
    default: break;
  }
}
template <>
void launch_bma_s<PF_JOIN_GENSIN>(int S, dim3 grid, hipStream_t st, const PfBmaArgs& a) {
  switch (S) {
#define PF_CASE(SS) \
  case SS: hipLaunchKernelGGL((pf_bma_kernel<SS, PF_JOIN_GENSIN>), grid, dim3(256), 0, st, a); break;
    PF_CASE(1) PF_CASE(2) PF_CASE(3) PF_CASE(4) PF_CASE(5) PF_CASE(6) PF_CASE(7) PF_CASE(8)
#undef PF_CASE
    default: break;
  }
}

void launch_bma_max(int S, dim3 grid, hipStream_t st, const PfBmaArgs& a) {
  const size_t lds = (size_t)64 * a.GS * pf_ncf(S) * sizeof(float);
  switch (S) {
#define PF_CASE(SS) \
  case SS: hipLaunchKernelGGL((pf_bma_max_kernel<SS>), grid, dim3(64 * PF_WG), lds, st, a); break;
    PF_CASE(1) PF_CASE(2) PF_CASE(3) PF_CASE(4) PF_CASE(5) PF_CASE(6)
#undef PF_CASE
    default: break;
  }
}

double lg2(double x) { return std::log2(x); }

}  // namespace

/* Eligible genes of the chunk go through the contraction path; done[g] = 1
 * for each gene whose statistics it wrote.  The caller runs the rest (and
 * any gene marked for fallback) on the general path. */
int perm_fast_run(eqbf_ctx* ctx, const eqbf_chunk* cp, const eqbf_perm_opts* po, const int32_t* tables_dev,
                  int32_t n_tables, const int32_t* gene_table, int64_t nperm, double* stats_dev, hipStream_t st,
                  std::vector<uint8_t>& done) {
  const eqbf_chunk& c = *cp;
  const int S = c.n_subgroups, N = c.n_samples, G = c.n_genes;
  done.assign(G, 0);
  const bool join = po->analysis == EQBF_ANALYSIS_JOIN;
  if (po->precision != EQBF_PREC_MIXED || c.n_geno_sets != 1 || N > PF_NMAX || N < 4 || nperm <= 0) return EQBF_OK;
  int mode;
  if (!join)
    mode = PF_SEP;
  else
    mode = po->pbf == EQBF_PBF_ALL ? PF_JOIN_ALL : (po->pbf == EQBF_PBF_GEN ? PF_JOIN_GEN : PF_JOIN_GENSIN);
  if (S < 1 || S > (mode == PF_JOIN_ALL ? 6 : 8)) return EQBF_OK;
  if (!join && po->sep_sbgrp >= S) return EQBF_OK;
  const int GL = (int)ctx->phiL.size(), GS = (int)ctx->phiS.size();
  if (join && ((mode != PF_JOIN_ALL && GL < 1) || (mode != PF_JOIN_GEN && GS < 1))) return EQBF_OK;
  {
    std::vector<int32_t> cc(S);
    EQBF_HIP(ctx, hipMemcpyAsync(cc.data(), c.covar_count, S * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    EQBF_HIP(ctx, hipStreamSynchronize(st));
    for (int s = 0; s < S; ++s)
      if (cc[s] != 0) return EQBF_OK;
  }
  /* eligibility per gene */
  int* d_bad = (int*)ctx_buf(ctx, "pf_ok", (size_t)G * sizeof(int) + 64);
  if (!d_bad) return EQBF_ERR_HIP; /* ctx_buf has set the message */
  const bool f32 = c.geno_dtype == EQBF_F32;
  hipLaunchKernelGGL(pf_clear_kernel, dim3((unsigned)std::min(256, (G + 63) / 64)), dim3(64), 0, st, d_bad, G);
  /* enough blocks per gene for its share of the chunk's pairs, 64 at a time */
  const unsigned per_gene = (unsigned)std::min<int64_t>(64, std::max<int64_t>(1, c.n_pairs / G / 64 + 1));
  hipLaunchKernelGGL((f32 ? pf_check_kernel<float> : pf_check_kernel<double>), dim3((unsigned)G, per_gene), dim3(256), 0,
                     st, c, d_bad);
  EQBF_HIP(ctx, hipGetLastError());
  std::vector<int> bad(G);
  std::vector<int64_t> off(G + 1);
  EQBF_HIP(ctx, hipMemcpyAsync(bad.data(), d_bad, G * sizeof(int), hipMemcpyDeviceToHost, st));
  EQBF_HIP(ctx, hipMemcpyAsync(off.data(), c.pair_offset, (G + 1) * sizeof(int64_t), hipMemcpyDeviceToHost, st));
  EQBF_HIP(ctx, hipStreamSynchronize(st));
  std::vector<int> genes;
  bool wide = false;
  for (int g = 0; g < G; ++g)
    if (gene_table[g] >= 0 && gene_table[g] < n_tables && !(bad[g] & 1) && off[g + 1] > off[g]) {
      genes.push_back(g);
      wide |= (bad[g] & 2) != 0;
    }
  if (genes.empty()) return EQBF_OK;

  const int nu = N - 2;
  int rc = ctx_ensure_tz(ctx, N, st);
  if (rc) return rc;
  float* d_zt = nullptr;
  if (join) {
    d_zt = (float*)ctx_buf(ctx, "pf_zt", (size_t)ZT_ROW * sizeof(float));
    if (!d_zt) return EQBF_ERR_HIP; /* ctx_buf has set the message */
    hipLaunchKernelGGL(pf_zeta_table_kernel, dim3(ZT_NODES / 256 + 1), dim3(256), 0, st, ctx_tz_table(ctx), nu,
                       d_zt);
    EQBF_HIP(ctx, hipGetLastError());
  }
  const int Npad = (N + 63) / 64 * 64, nks = Npad / 64;
  const int64_t NPP = (nperm + 63) / 64 * 64;
  const int npb16 = (int)((nperm + 15) / 16), npb64 = (int)((nperm + 63) / 64);
  const int ngrid = mode == PF_JOIN_ALL ? GS : (mode == PF_JOIN_GEN ? GL : GL + GS);
  const int NCF = pf_ncf(S);
  /* batch: z values of at most 16 GB */
  size_t zeta_budget = (size_t)16 << 30;
  {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess) zeta_budget = std::min(zeta_budget, fr / 4);
    zeta_budget = std::max(zeta_budget, (size_t)256 << 20);
  }
  /* --pbf all --maxbf: in one kernel where its fragments fit the LDS and the
   * genotypes of a tile its registers, else with the bounds on stored z values.
   * Genes of few SNPs (pf_max_snps) take the latter too, last and in batches of
   * their own, where no gene has more or where they are enough work: a batch costs
   * 50 to 150 us in launches, which 2,048 workgroups (gene x 16 permutations) of
   * the one kernel cost more than.  24 genes, 10,000 permutations, S = 5: six genes
   * of 20 SNPs among 18 of 1,000, 5,580 us together, 4,755 apart; one among 23,
   * 5,494 and 5,558; ten genes, 1,000 permutations, S = 3, one of 20 SNPs among 500,
   * 325 and 479. */
  const bool prune = join && mode == PF_JOIN_ALL && po->use_max_bf && S <= 6 &&
                     (size_t)64 * GS * NCF * sizeof(float) <= 48 * 1024;
  const bool fits = prune && !wide && nks <= PFX_NKS && pf_max_lds(S, Npad) <= (size_t)158 * 1024;
  auto large = [&](int g) { return off[g + 1] - off[g] >= pf_max_snps(S); };
  const int64_t n_large = std::count_if(genes.begin(), genes.end(), large), n_small = (int64_t)genes.size() - n_large;
  const bool apart = n_large == 0 || n_small * npb16 > 2048;
  auto in_one = [&](int g) { return fits && (!apart || large(g)); };
  if (fits && apart) std::stable_partition(genes.begin(), genes.end(), in_one);
  const int s_lo = (!join && po->sep_sbgrp >= 0) ? po->sep_sbgrp : 0;
  const int s_hi = (!join && po->sep_sbgrp >= 0) ? po->sep_sbgrp + 1 : S;

  /* log2 weights of the terms (gene_snp_pair.cpp:552-602, utils_math.cpp:100-159) */
  PfBmaArgs ba;
  memset(&ba, 0, sizeof ba);
  for (int m = 0; m <= 8; ++m) {
    if (mode == PF_JOIN_ALL && m >= 1 && m <= S) {
      double ch = 1;
      for (int k = 0; k < m; ++k) ch = ch * (S - k) / (k + 1);
      ba.lw[1][m] = (float)lg2(1.0 / ((double)S * ch * GS));
      ba.lwc[m] = (float)lg2(ch);
    }
    if (mode == PF_JOIN_GEN) ba.lw[0][m] = (float)lg2(1.0 / GL);
    if (mode == PF_JOIN_GENSIN) {
      ba.lw[0][m] = (float)lg2(0.5 / GL);
      ba.lw[1][m] = (float)lg2(0.5 / ((double)S * GS));
    }
  }

  std::vector<int> fb_all;
  size_t gi = 0;
  while (gi < genes.size()) {
    const bool fused = in_one(genes[gi]);
    /* gather the batch */
    std::vector<int32_t> bgene, btable, bslot;
    std::vector<int64_t> bpoff(1, 0), goff;
    size_t zbytes = 0;
    int nslots = 0;
    while (gi < genes.size()) {
      const int g = genes[gi];
      if (in_one(g) != fused) break;
      const int64_t np = off[g + 1] - off[g];
      const size_t zb = join && !fused ? (size_t)np * S * NPP * sizeof(float) : 0;
      if (!bgene.empty() && (zbytes + zb > zeta_budget || bgene.size() >= 4096 || bpoff.back() + np > ((int64_t)1 << 23) ||
                             (int64_t)(bgene.size() + 1) * npb16 * (s_hi - s_lo) > ((int64_t)1 << 30)))
        break;
      zbytes += zb;
      bgene.push_back(g);
      btable.push_back(gene_table[g]);
      bslot.push_back(nslots);
      nslots += fused ? 1 : (int)((np + PF_SB - 1) / PF_SB);
      goff.push_back(off[g]);
      bpoff.push_back(bpoff.back() + np);
      ++gi;
    }
    const int nb = (int)bgene.size();
    const int64_t nbp = bpoff.back();
    const int64_t n_gitems = (int64_t)nb * npb16 * (fused ? 1 : s_hi - s_lo);
    std::vector<int4> bitems;
    /* pf_bma_max_kernel: one item per (gene, PF_WG x 64 permutations) over all
     * the gene's SNPs; otherwise blocks of PF_SB SNPs */
    if (join && !fused)
      for (int b = 0; b < nb; ++b) {
        if (prune) {
          for (int pb = 0; pb < npb64; pb += PF_WG) bitems.push_back(make_int4(b, pb, 0, bslot[b]));
          continue;
        }
        const int nsb = (int)((bpoff[b + 1] - bpoff[b] + PF_SB - 1) / PF_SB);
        for (int pb = 0; pb < npb64; ++pb)
          for (int sb = 0; sb < nsb; ++sb) bitems.push_back(make_int4(b, pb, sb, bslot[b] + sb));
      }
    /* device buffers */
    uint8_t* meta = (uint8_t*)ctx_buf(ctx, "pf_meta", (size_t)nb * 3 * sizeof(int32_t) +
                                                          (size_t)(2 * nb + 1) * sizeof(int64_t) +
                                                          bitems.size() * sizeof(int4) + 256);
    int8_t* d_G8 = (int8_t*)ctx_buf(ctx, "pf_g8", (size_t)(nbp + PFX_PAD) * Npad);
    uint32_t* d_W = (uint32_t*)ctx_buf(ctx, "pf_w", (size_t)nb * S * Npad * sizeof(uint32_t));
    YStat* d_ys = (YStat*)ctx_buf(ctx, "pf_ys", (size_t)nb * S * sizeof(YStat));
    PStat* d_ps = (PStat*)ctx_buf(ctx, "pf_ps", (size_t)(nbp + PFX_PAD) * sizeof(PStat));
    uint8_t* d_pf = (uint8_t*)ctx_buf(ctx, "pf_pflag", (size_t)nbp + 64);
    int* d_fb = (int*)ctx_buf(ctx, "pf_fb", (size_t)nb * sizeof(int) + 64);
    if (!meta || !d_G8 || !d_W || !d_ys || !d_ps || !d_pf || !d_fb)
      return EQBF_ERR_HIP; /* ctx_buf has set the message */
    float* d_zeta = nullptr;
    float* d_coef = nullptr;
    float* d_thr = nullptr;
    float* d_pmax = nullptr;
    double* d_psum = nullptr;
    double* d_tmax = nullptr;
    if (join) {
      if (!fused) d_zeta = (float*)ctx_buf(ctx, "pf_zeta", zbytes + 64);
      d_coef = (float*)ctx_buf(ctx, "pf_coef", (size_t)nbp * ngrid * NCF * sizeof(float) + 64);
      d_pmax = (float*)ctx_buf(ctx, "pf_pmax", (size_t)nslots * NPP * sizeof(float) + 64);
      if (!fused) d_psum = (double*)ctx_buf(ctx, "pf_psum", (size_t)nslots * NPP * sizeof(double) + 64);
      if (fused) d_thr = (float*)ctx_buf(ctx, "pf_thr", ((size_t)PFX_BINS * nbp + PFX_PAD) * sizeof(float));
      if (!d_coef || !d_pmax || (fused ? !d_thr : !d_zeta || !d_psum))
        return EQBF_ERR_HIP; /* ctx_buf has set the message */
    } else {
      d_tmax = (double*)ctx_buf(ctx, "pf_tmax", (size_t)nb * S * NPP * sizeof(double) + 64);
      if (!d_tmax) return EQBF_ERR_HIP; /* ctx_buf has set the message */
      /* subgroups that are not computed (--permsep 2) are never read */
    }
    /* the batch's tables, in one copy: offsets, first pairs, work items, genes */
    int64_t* d_bpoff = (int64_t*)meta;
    int64_t* d_goff = d_bpoff + nb + 1;
    int4* d_bitems = (int4*)(((uintptr_t)(d_goff + nb) + 15) & ~(uintptr_t)15);
    int32_t* d_bgene = (int32_t*)(d_bitems + bitems.size());
    int32_t* d_btable = d_bgene + nb;
    int32_t* d_bslot = d_btable + nb;
    std::vector<uint8_t> hmeta((uint8_t*)(d_bslot + nb) - meta);
    auto put = [&](const void* dev, const void* src, size_t bytes) {
      if (bytes) memcpy(hmeta.data() + ((const uint8_t*)dev - meta), src, bytes);
    };
    put(d_bpoff, bpoff.data(), (nb + 1) * sizeof(int64_t));
    put(d_goff, goff.data(), nb * sizeof(int64_t));
    put(d_bitems, bitems.data(), bitems.size() * sizeof(int4));
    put(d_bgene, bgene.data(), nb * sizeof(int32_t));
    put(d_btable, btable.data(), nb * sizeof(int32_t));
    put(d_bslot, bslot.data(), nb * sizeof(int32_t));
    EQBF_HIP(ctx, hipMemcpyAsync(meta, hmeta.data(), hmeta.size(), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(pf_clear_kernel, dim3((unsigned)std::min(256, (nb + 63) / 64)), dim3(64), 0, st, d_fb, nb);
    {
      ProfScope ps(ctx, "pf_prep_kernel", st);
      hipLaunchKernelGGL(pf_prep_y_kernel, dim3(nb * S), dim3(256), 0, st, c, d_bgene, Npad, d_W, d_ys,
                         join ? d_fb : nullptr); /* sep: pf_gemm_kernel's own rule */
      hipLaunchKernelGGL((f32 ? pf_prep_x_kernel<float> : pf_prep_x_kernel<double>), dim3((unsigned)((nbp + 63) / 64)),
                         dim3(256), (size_t)64 * (Npad / 4 + 1) * sizeof(uint32_t), st, c, d_bpoff, d_goff, nb, Npad, d_G8,
                         d_ps, d_pf);
    }
    EQBF_HIP(ctx, hipGetLastError());
    if (join) {
      const int64_t ne = nbp * ngrid;
      std::vector<double> gphi, goma;
      if (mode != PF_JOIN_ALL) {
        gphi.insert(gphi.end(), ctx->phiL.begin(), ctx->phiL.end());
        goma.insert(goma.end(), ctx->omaL.begin(), ctx->omaL.end());
      }
      if (mode != PF_JOIN_GEN) {
        gphi.insert(gphi.end(), ctx->phiS.begin(), ctx->phiS.end());
        goma.insert(goma.end(), ctx->omaS.begin(), ctx->omaS.end());
      }
      double* d_g = (double*)ctx_buf(ctx, "pf_grid", 2 * gphi.size() * sizeof(double) + 64);
      if (!d_g) return EQBF_ERR_HIP; /* ctx_buf has set the message */
      EQBF_HIP(ctx, hipMemcpyAsync(d_g, gphi.data(), gphi.size() * sizeof(double), hipMemcpyHostToDevice, st));
      EQBF_HIP(ctx, hipMemcpyAsync(d_g + gphi.size(), goma.data(), goma.size() * sizeof(double), hipMemcpyHostToDevice,
                                   st));
      ProfScope ps(ctx, "pf_coef_kernel", st);
      hipLaunchKernelGGL(pf_coef_kernel, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, st, d_ps, d_pf, nbp, d_g,
                         d_g + gphi.size(), ngrid, S, d_coef);
      EQBF_HIP(ctx, hipGetLastError());
    }
    PfGemmArgs ga;
    memset(&ga, 0, sizeof ga);
    ga.G8 = d_G8;
    ga.W = d_W;
    ga.ys = d_ys;
    ga.ps = d_ps;
    ga.pflag = d_pf;
    ga.bpoff = d_bpoff;
    ga.tables = tables_dev;
    ga.btable = d_btable;
    ga.zt = d_zt;
    ga.tz = ctx_tz_table(ctx);
    ga.zeta = d_zeta;
    ga.tmax = d_tmax;
    ga.fallback = d_fb;
    ga.S = S;
    ga.N = N;
    ga.Npad = Npad;
    ga.nks = nks;
    ga.nu = nu;
    ga.nperm = nperm;
    ga.NPP = NPP;
    ga.n_items = (int)n_gitems;
    ga.npb16 = npb16;
    ga.s_lo = s_lo;
    ga.ns = s_hi - s_lo;
    const size_t lds = (size_t)Npad * 4 + (size_t)nks * 4 * 64 * 16;
    if (fused) {
      PfMaxArgs xa;
      memset(&xa, 0, sizeof xa);
      xa.g = ga;
      xa.coef = d_coef;
      xa.thr = d_thr;
      xa.bslot = d_bslot;
      xa.pmax = d_pmax;
      memcpy(xa.lw, ba.lw[1], sizeof xa.lw);
      for (int m = 0; m <= 8; ++m) xa.lwc[m] = ba.lw[1][m] + ba.lwc[m];
      xa.GS = GS;
      xa.nbp = nbp;
      launch_pf_max(ctx, S, st, xa, d_thr, pf_max_lds(S, Npad));
    } else {
      ProfScope ps(ctx, "pf_gemm_kernel", st);
      if (join)
        hipLaunchKernelGGL(pf_gemm_kernel<PF_JOIN_ALL>, dim3((unsigned)((n_gitems + 7) / 8 * 8)), dim3(256), lds, st, ga);
      else
        hipLaunchKernelGGL(pf_gemm_kernel<PF_SEP>, dim3((unsigned)((n_gitems + 7) / 8 * 8)), dim3(256), lds, st, ga);
    }
    EQBF_HIP(ctx, hipGetLastError());
    if (join && !fused) {
      ba.zeta = d_zeta;
      ba.coef = d_coef;
      ba.pflag = d_pf;
      ba.items = d_bitems;
      ba.bpoff = d_bpoff;
      ba.pmax = d_pmax;
      ba.psum = d_psum;
      ba.fallback = d_fb;
      ba.GL = GL;
      ba.GS = GS;
      ba.use_max = po->use_max_bf;
      ba.n_items = (int)bitems.size();
      ba.NPP = NPP;
      ba.nperm = nperm;
      const dim3 grid((unsigned)((bitems.size() + 3) / 4));
      ProfScope ps(ctx, "pf_bma_kernel", st);
      if (prune)
        launch_bma_max(S, dim3((unsigned)bitems.size()), st, ba);
      else if (mode == PF_JOIN_ALL)
        launch_bma_s<PF_JOIN_ALL>(S, grid, st, ba);
      else if (mode == PF_JOIN_GEN)
        launch_bma_s<PF_JOIN_GEN>(S, grid, st, ba);
      else
        launch_bma_s<PF_JOIN_GENSIN>(S, grid, st, ba);
      EQBF_HIP(ctx, hipGetLastError());
    }
    {
      PfFinalArgs fa;
      memset(&fa, 0, sizeof fa);
      fa.pmax = d_pmax;
      fa.psum = d_psum;
      fa.tmax = d_tmax;
      fa.bgene = d_bgene;
      fa.bpoff = d_bpoff;
      fa.bslot = d_bslot;
      fa.pflag = d_pf;
      fa.tz = ctx_tz_table(ctx);
      fa.stats = stats_dev;
      fa.nb = nb;
      fa.S = S;
      fa.nu = nu;
      fa.mode = mode;
      fa.use_max = po->use_max_bf;
      fa.sep_sbgrp = po->sep_sbgrp;
      fa.one_slot = prune ? 1 : 0;
      fa.nperm = nperm;
      fa.NPP = NPP;
      const int64_t ne = (int64_t)nb * nperm;
      ProfScope ps(ctx, "pf_final_kernel", st);
      hipLaunchKernelGGL(pf_final_kernel, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, st, fa);
      EQBF_HIP(ctx, hipGetLastError());
    }
    std::vector<int> fb(nb);
    EQBF_HIP(ctx, hipMemcpyAsync(fb.data(), d_fb, nb * sizeof(int), hipMemcpyDeviceToHost, st));
    EQBF_HIP(ctx, hipStreamSynchronize(st));
    for (int b = 0; b < nb; ++b)
      if (!fb[b]) done[bgene[b]] = 1;
  }
  return EQBF_OK;
}
