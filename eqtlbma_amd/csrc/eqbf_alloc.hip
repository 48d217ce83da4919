/*
 * Learned permutation allocator: the per-gene inputs of its network and the
 * targets it is trained on.  No counterpart in the reference.
 *
 *  - LD eigenvalues: the k largest eigenvalues of the correlation matrix of
 *    a gene's cis genotypes (P x P).  They are the k largest eigenvalues of
 *    Z Z^T / N (N x N), Z the N x P standardised genotypes, so the kernels
 *    form that Gram matrix (64 x 64 tiles, FP32) and run a blocked subspace
 *    iteration on it (32 vectors, FP32 products, FP64 Cholesky-QR, then the
 *    Rayleigh-Ritz matrix diagonalised by Jacobi rotations in FP64, p/2
 *    disjoint pairs per round).  A batch's pairs are consecutive, so its
 *    kernels take the first one and the genes' offsets from it.
 *  - GEV fit: location, scale and shape of each gene's permutation
 *    statistics by probability-weighted moments (Hosking, Wallis & Wood
 *    1985, Technometrics 27:251-261): the draws are sorted in LDS (bitonic,
 *    NaN last and not counted) and the moments b0, b1, b2 summed in FP64.
 */
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "eqbf_internal.h"

namespace {

constexpr int EIG_NMAX = 512;  /* samples for the eigenvalue kernel (LDS) */
constexpr int EIG_P = 32;      /* subspace vectors                        */
constexpr int EIG_ITERS = 20;
constexpr int EIG_NT = 512;    /* threads of the eigenvalue kernel, >= EIG_NMAX */
constexpr int GEV_NMAX = 16384; /* permutations per gene for the GEV fit    */

template <class T>
__device__ inline T al_geno(const eqbf_chunk& c, int64_t i, int64_t j) {
  return ((const T*)c.genotypes)[i * c.geno_ld + j];
}

/* mean and 1/sd of each pair's SNP over the chunk's samples (missing values
 * excluded; a constant SNP gets 1/sd = 0, so it adds nothing): 64 pairs a
 * workgroup, the samples over its four waves */
template <class T>
__global__ void __launch_bounds__(256) al_snpstat_kernel(const eqbf_chunk c, int64_t b0, int64_t nbp,
                                                         float2* __restrict__ ms) {
  __shared__ double ps[4][64], ps2[4][64];
  __shared__ int pn[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t b = (int64_t)blockIdx.x * 64 + lane;
  const int64_t snp = b < nbp ? c.pair_snp[b0 + b] : 0;
  double s = 0, s2 = 0;
  int n = 0;
  if (b < nbp) {
#pragma unroll 8
    for (int i = wv; i < c.n_samples; i += 4) {
      const double x = (double)al_geno<T>(c, i, snp);
      if (x == x) {
        s += x;
        s2 += x * x;
        ++n;
      }
    }
  }
  ps[wv][lane] = s;
  ps2[wv][lane] = s2;
  pn[wv][lane] = n;
  __syncthreads();
  if (wv || b >= nbp) return;
  for (int k = 1; k < 4; ++k) {
    s += ps[k][lane];
    s2 += ps2[k][lane];
    n += pn[k][lane];
  }
  const double m = n ? s / n : 0.0;
  const double v = n ? s2 / n - m * m : 0.0;
  ms[b] = make_float2((float)m, v > 1e-12 * (s2 / (n ? n : 1)) ? (float)(1.0 / sqrt(v)) : 0.f);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

/* K[gene][a][b] = sum_j z[a][j] z[b][j] / N over the gene's pairs j: 64 x 64
 * outputs a workgroup for the tiles on and above the diagonal, the others
 * mirrored; 32 pairs a stage, the next stage's genotypes in registers
 * meanwhile, FP32 matrix instructions (each wave 32 x 32).  48 genes of 300
 * samples and 1,000 pairs: 0.13 ms (0.41 ms with 16 pairs a stage, every tile and
 * scalar products). */
template <class T>
__global__ void __launch_bounds__(256) al_gram_kernel(const eqbf_chunk c, int64_t b0,
                                                      const int64_t* __restrict__ bpoff, const float2* __restrict__ ms,
                                                      int nt, float* __restrict__ K) {
  __shared__ float Za[32][65], Zb[32][65];
  const int N = c.n_samples, tri = nt * (nt + 1) / 2;
  const int bi = blockIdx.x / tri;
  int ta = 0, tb = blockIdx.x % tri; /* tile (ta, tb), ta <= tb */
  while (tb >= nt - ta) {
    tb -= nt - ta;
    ++ta;
  }
  tb += ta;
  const int ra0 = ta * 64, rb0 = tb * 64;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int kk = tid & 31, r0 = tid >> 5; /* consecutive threads: consecutive SNPs of one sample */
  const int64_t j0 = bpoff[bi], j1 = bpoff[bi + 1];
  float za[8], zb[8];
  auto fetch = [&](int64_t jj) { /* indexes held inside, so that the loads need no branches */
    const int64_t j = min(jj + kk, j1 - 1);
    const bool on = jj + kk < j1;
    const float2 s = ms[j];
    const T* g = (const T*)c.genotypes + c.pair_snp[b0 + j];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int a = ra0 + r0 + 8 * i, b = rb0 + r0 + 8 * i;
      const float xa = (float)g[(int64_t)min(a, N - 1) * c.geno_ld];
      const float ya = (xa - s.x) * s.y;
      za[i] = on && a < N && xa == xa ? ya : 0.f;
      if (ta != tb) {
        const float xb = (float)g[(int64_t)min(b, N - 1) * c.geno_ld];
        const float yb = (xb - s.x) * s.y;
        zb[i] = on && b < N && xb == xb ? yb : 0.f;
      }
    }
  };
  f32x4 acc[2][2] = {};
  const int wa = (wv >> 1) * 32, wb = (wv & 1) * 32, lr = lane & 15, lk = lane >> 4;
  if (j0 < j1) fetch(j0);
  for (int64_t jj = j0; jj < j1; jj += 32) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      Za[kk][r0 + 8 * i] = za[i];
      Zb[kk][r0 + 8 * i] = ta == tb ? za[i] : zb[i];
    }
    __syncthreads();
    if (jj + 32 < j1) fetch(jj + 32);
#pragma unroll
    for (int k4 = 0; k4 < 32; k4 += 4) {
      float a[2], b[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        a[u] = Za[k4 + lk][wa + 16 * u + lr];
        b[u] = Zb[k4 + lk][wb + 16 * u + lr];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) acc[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[v], acc[u][v], 0, 0, 0);
    }
    __syncthreads();
  }
  const float invN = 1.f / (float)N;
  float* Kg = K + (int64_t)bi * N * N;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int a = ra0 + wa + 16 * u + lk * 4 + i, b = rb0 + wb + 16 * v + lr;
        if (a < N && b < N) {
          Kg[(int64_t)a * N + b] = acc[u][v][i] * invN;
          if (ta != tb) Kg[(int64_t)b * N + a] = acc[u][v][i] * invN;
        }
      }
}

/* value of lane `from` (the same for every lane) */
__device__ __forceinline__ double lane_value(double v, int from) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), from),
                          __builtin_amdgcn_readlane(__double2loint(v), from));
}

/* k largest eigenvalues of one gene's K (one workgroup per gene).
 *
 * Bound by the chain of its 20 iterations on one compute unit.  So the two
 * products of an iteration run on the matrix instructions (W = K V in FP32,
 * K's rows read from L2 straight into the operand; G in FP64), the Cholesky
 * factor is made by one wave with a row per lane, without a barrier, and a
 * round of Jacobi rotations is one barrier: each thread rotates one 2 x 2 block
 * from one copy of the matrix into the other.  LDS rows of EIG_PV values keep
 * the operands' four rows on different banks.  48 genes of 300 samples: 0.85 ms
 * (4.06 ms with scalar products, a barrier per Cholesky update and twelve sweeps
 * of three barriers a round). */
constexpr int EIG_PV = EIG_P + 1;

__host__ __device__ inline int eig_rows(int N) { return (N + 31) / 32 * 32; }

__global__ void __launch_bounds__(EIG_NT) al_eig_kernel(const float* __restrict__ Kall, int N, int k,
                                                     float* __restrict__ eig) {
  constexpr int p = EIG_P, pv = EIG_PV;
  extern __shared__ __align__(16) unsigned char smem[];
  const int Np = eig_rows(N);
  double* G = (double*)smem;                 /* [p][p], two copies for the rotations */
  double* G2 = G + p * p;
  float* V = (float*)(G2 + p * p);           /* [Np][pv], rows past N zero */
  float* W = V + (size_t)Np * pv;            /* [Np][pv] */
  __shared__ double dinv[p];
  __shared__ int ok;
  const float* K = Kall + (int64_t)blockIdx.x * N * N;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lk = lane >> 4;
  /* start: a fixed pseudo-random block */
  for (int e = tid; e < Np * p; e += EIG_NT) {
    uint32_t h = (uint32_t)e * 2654435761u ^ 0x9e3779b9u;
    h ^= h >> 15;
    h *= 2246822519u;
    h ^= h >> 13;
    V[(e / p) * pv + e % p] = e < N * p ? (float)(h & 0xffff) / 65536.f - 0.5f : 0.f;
  }
  __syncthreads();
  for (int it = 0; it <= EIG_ITERS; ++it) {
    /* W = K V, 16 rows a wave at a time, eight operands of K in flight (K is
     * symmetric: A[m][kk] read as K[kk][m]) */
    for (int r0 = wv * 16; r0 < Np; r0 += (EIG_NT / 64) * 16) {
      /* past the last sample K's last row is read: V's rows there are zero, and
       * such rows of W are written as zero */
      const float* Kr = K + min(r0 + lr, N - 1);
      f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
      float cur[8], nxt[8];
      auto fetch = [&](float (&x)[8], int kb) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          x[u] = Kr[(int64_t)min(kb + 4 * u + lk, N - 1) * N];
        }
      };
      fetch(cur, 0);
      for (int kb = 0; kb < Np; kb += 32) {
        if (kb + 32 < Np) fetch(nxt, kb + 32);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const float* v = V + (kb + 4 * u + lk) * pv + lr;
          a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[u], v[0], a0, 0, 0, 0);
          a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[u], v[16], a1, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) cur[u] = nxt[u];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + lk * 4 + i;
        W[r * pv + lr] = r < N ? a0[i] : 0.f;
        W[r * pv + lr + 16] = r < N ? a1[i] : 0.f;
      }
    }
    __syncthreads();
    /* G = V^T W (Rayleigh-Ritz on the last pass) or W^T W (orthonormalise,
     * its lower half): a 16 x 16 tile each for the first four waves */
    if (wv < 4 && (it == EIG_ITERS || wv != 1)) {
      const float* X = it == EIG_ITERS ? V : W;
      const int ma = (wv >> 1) * 16 + lr, nb = (wv & 1) * 16 + lr;
      f64x4 g = {0.0, 0.0, 0.0, 0.0};
      for (int kb = lk; kb < Np; kb += 4)
        g = __builtin_amdgcn_mfma_f64_16x16x4f64((double)X[kb * pv + ma], (double)W[kb * pv + nb], g, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) G[((wv >> 1) * 16 + lk + 4 * i) * p + nb] = g[i];
    }
    __syncthreads();
    if (it == EIG_ITERS) break;
    /* Cholesky G = L L^T in wave 0, lane i holding row i and a step's column
     * passing through LDS; a pivot below 1e-14 of the first (rank-deficient
     * block) is raised.  L's columns over G, the reciprocal pivots in dinv. */
    if (wv == 0) {
      const double first = G[0];
      if (lane == 0) ok = first > 0;
      const double floor_ = 1e-14 * first;
      double r[p];
#pragma unroll
      for (int c2 = 0; c2 < p; ++c2) r[c2] = G[(lane & 31) * p + c2];
#pragma unroll
      for (int j = 0; j < p; ++j) {
        const double inv = 1.0 / sqrt(fmax(lane_value(r[j], j), floor_));
        r[j] *= inv;
        dinv[j] = inv; /* the same in every lane: no branch, which would let the updates sink past it */
        /* two buffers, so that one wait orders a step against the next */
        double* col = G2 + (j & 1) * 64;
        col[lane] = r[j];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
#pragma unroll
        for (int c2 = j + 1; c2 < p; ++c2) r[c2] = fma(-r[j], col[c2], r[c2]);
        __builtin_amdgcn_sched_barrier(0); /* a step's reads stay in it: registers */
      }
      /* L below the diagonal, column after column: the order of the
       * substitution below */
#pragma unroll
      for (int d = 0; d < p; ++d)
        if (lane > d && lane < p) G[d * (2 * p - 1 - d) / 2 + lane - d - 1] = r[d];
    }
    __syncthreads();
    if (!ok) break;
    /* V = W L^-T by forward substitution (an inverse of L would not be stable
     * for the rank-deficient blocks), a row per thread; the next eight values
     * of L are on their way from LDS during eight steps */
    if (tid < N) {
      constexpr int n_l = p * (p - 1) / 2, U = 8;
      double s[p], cur[U], nxt[U];
#pragma unroll
      for (int c2 = 0; c2 < p; ++c2) s[c2] = W[tid * pv + c2];
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = G[u];
      int d = 0, c2 = 1; /* known at compile time throughout */
      double v = 0.0;
#pragma unroll
      for (int e = 0; e < n_l; e += U) {
        if (e + U < n_l) {
#pragma unroll
          for (int u = 0; u < U; ++u) nxt[u] = G[e + U + u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (c2 == d + 1) {
            const float f = (float)(s[d] * dinv[d]);
            V[tid * pv + d] = f;
            v = (double)f;
          }
          s[c2] = fma(-v, cur[u], s[c2]);
          if (++c2 == p) {
            ++d;
            c2 = d + 1;
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) cur[u] = nxt[u];
        __builtin_amdgcn_sched_barrier(0);
      }
      V[tid * pv + p - 1] = (float)(s[p - 1] * dinv[p - 1]);
    }
    __syncthreads();
  }
  /* Jacobi on the symmetrised p x p Rayleigh-Ritz matrix, parallel
   * (tournament) ordering: the p/2 pairs of a round are disjoint, so thread
   * (q1, q2) rotates the 2 x 2 block of pairs q1 and q2 from one copy into the
   * other.  Sweeps until no element off the diagonal was above 1e-13 of the
   * largest on it (their effect on an eigenvalue is of second order), at most
   * 12. */
  if (!ok) {
    if (tid < k) eig[(int64_t)blockIdx.x * k + tid] = NAN;
    return;
  }
  for (int e = tid; e < p * p; e += EIG_NT) {
    const int a = e / p, b = e % p;
    if (b > a) {
      const double m = 0.5 * (G[a * p + b] + G[b * p + a]);
      G[a * p + b] = G[b * p + a] = m;
    }
  }
  __syncthreads();
  double big = 0.0;
  for (int a = 0; a < p; ++a) big = fmax(big, fabs(G[a * p + a]));
  const int q2 = lane & 15, q1 = (tid >> 4) & 15;
  double *src = G, *dst = G2;
  for (int sweep = 0; sweep < 12; ++sweep) {
    bool far = false;
    for (int r = 0; r < p - 1; ++r) {
      /* every wave works out all p/2 rotations, lane q of each 16 the one of
       * pair q, so that the block below needs no other wave */
      int a = r, b = p - 1;
      if (q2) {
        a = (r + q2) % (p - 1);
        b = (r - q2 + (p - 1)) % (p - 1);
      }
      if (a > b) {
        const int t2 = a;
        a = b;
        b = t2;
      }
      const double apq = src[a * p + b];
      far |= __any(fabs(apq) > 1e-13 * big);
      double c2 = 1.0, s2 = 0.0;
      if (fabs(apq) > 1e-300) {
        const double th = (src[b * p + b] - src[a * p + a]) / (2 * apq);
        const double tt = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1));
        c2 = 1 / sqrt(tt * tt + 1);
        s2 = tt * c2;
      }
      if (tid < (p / 2) * (p / 2)) {
        const int a1 = __shfl(a, q1, 64), b1 = __shfl(b, q1, 64);
        const double c1 = __shfl(c2, q1, 64), s1 = __shfl(s2, q1, 64);
        /* rows a1, b1 of columns a, b: the columns first, then the rows */
        const double gaa = src[a1 * p + a], gab = src[a1 * p + b], gba = src[b1 * p + a], gbb = src[b1 * p + b];
        const double taa = c2 * gaa - s2 * gab, tab = s2 * gaa + c2 * gab;
        const double tba = c2 * gba - s2 * gbb, tbb = s2 * gba + c2 * gbb;
        dst[a1 * p + a] = c1 * taa - s1 * tba;
        dst[a1 * p + b] = c1 * tab - s1 * tbb;
        dst[b1 * p + a] = s1 * taa + c1 * tba;
        dst[b1 * p + b] = s1 * tab + c1 * tbb;
      }
      __syncthreads();
      double* t3 = src;
      src = dst;
      dst = t3;
    }
    if (!far) break; /* the same in every wave */
  }
  /* the k largest diagonal entries, descending */
  if (wv == 0) {
    double d = lane < p ? src[lane * p + lane] : -INFINITY;
    if (isnan(d)) d = -INFINITY;
    int rank = 0;
    for (int j = 0; j < p; ++j) {
      const double o = lane_value(d, j);
      rank += o > d || (o == d && j < lane);
    }
    if (lane < p && rank < k) eig[(int64_t)blockIdx.x * k + rank] = (float)d;
  }
}

/* GEV by probability-weighted moments of one gene's statistics. */
__global__ void __launch_bounds__(1024) al_gev_kernel(const double* __restrict__ stats, int64_t nperm, int npow,
                                                      double* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* x = (double*)smem;
  __shared__ double red[3][1024];
  __shared__ int nvalid;
  const int tid = threadIdx.x;
  const double* s = stats + (int64_t)blockIdx.x * nperm;
  if (tid == 0) nvalid = 0;
  __syncthreads();
  int cnt = 0;
  for (int i = tid; i < npow; i += 1024) {
    const double v = i < nperm ? s[i] : NAN;
    const bool valid = v == v;
    cnt += valid;
    x[i] = valid ? v : INFINITY;
  }
  atomicAdd(&nvalid, cnt);
  __syncthreads();
  for (int kk = 2; kk <= npow; kk <<= 1)
    for (int j = kk >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < npow; i += 1024) {
        const int l = i ^ j;
        if (l > i) {
          const double a = x[i], b = x[l];
          const bool up = (i & kk) == 0;
          if ((a > b) == up) {
            x[i] = b;
            x[l] = a;
          }
        }
      }
      __syncthreads();
    }
  const int n = nvalid;
  double b0 = 0, b1 = 0, b2 = 0;
  for (int i = tid; i < n; i += 1024) {
    const double v = x[i], j = (double)i;
    b0 += v;
    b1 += j / (n - 1) * v;
    b2 += j * (j - 1) / ((double)(n - 1) * (n - 2)) * v;
  }
  red[0][tid] = b0;
  red[1][tid] = b1;
  red[2][tid] = b2;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (tid < o)
      for (int q = 0; q < 3; ++q) red[q][tid] += red[q][tid + o];
    __syncthreads();
  }
  if (tid == 0) {
    double* o3 = out + (int64_t)blockIdx.x * 3;
    if (n < 3) {
      o3[0] = o3[1] = o3[2] = NAN;
      return;
    }
    b0 = red[0][0] / n;
    b1 = red[1][0] / n;
    b2 = red[2][0] / n;
    const double cc = (2 * b1 - b0) / (3 * b2 - b0) - 0.63092975357145743710; /* ln 2 / ln 3 */
    const double k = 7.8590 * cc + 2.9554 * cc * cc;
    double mu, sigma;
    if (fabs(k) < 1e-6) {
      sigma = (2 * b1 - b0) / 0.69314718055994531;
      mu = b0 - 0.57721566490153286 * sigma;
    } else {
      const double g = tgamma(1 + k);
      sigma = (2 * b1 - b0) * k / (g * (1 - exp2(-k)));
      mu = b0 + sigma * (g - 1) / k;
    }
    o3[0] = mu;
    o3[1] = sigma;
    o3[2] = fabs(k) < 1e-6 ? 0.0 : -k;
  }
}

}  // namespace

/* k largest LD eigenvalues of every gene of a chunk whose pointers are
 * device addresses (off: host copy of pair_offset). */
static int ld_eig_run(eqbf_ctx* ctx, const eqbf_chunk& d, const std::vector<int64_t>& off, int32_t n_eig,
                      float* eig) {
  const int N = d.n_samples, G = d.n_genes;
  const hipStream_t st = ctx->stream;
  const int nt = (N + 63) / 64;
  const bool f32 = d.geno_dtype == EQBF_F32;
  const size_t lds = (size_t)2 * eig_rows(N) * EIG_PV * sizeof(float) + (size_t)2 * EIG_P * EIG_P * sizeof(double);
  /* batches of genes: Gram matrices of at most ~1 GB */
  const int gb = std::max(1, (int)std::min<int64_t>(G, ((int64_t)1 << 30) / ((int64_t)N * N * 4)));
  float* dK = (float*)ctx_buf(ctx, "al_gram", (size_t)gb * N * N * sizeof(float));
  float* deig = (float*)ctx_buf(ctx, "al_eig", (size_t)gb * n_eig * sizeof(float));
  if (!dK || !deig) return EQBF_ERR_HIP; /* ctx_buf has set the message */
  std::vector<int64_t> boff;
  for (int g0 = 0; g0 < G; g0 += gb) {
    const int g1 = std::min(G, g0 + gb), nb = g1 - g0;
    /* pairs of the batch: off[g0] .. off[g1] - 1 */
    boff.resize(nb + 1);
    for (int g = g0; g <= g1; ++g) boff[g - g0] = off[g] - off[g0];
    const int64_t n_src = boff[nb];
    float2* dms = (float2*)ctx_buf(ctx, "al_ms", (size_t)std::max<int64_t>(n_src, 1) * sizeof(float2));
    int64_t* doff = (int64_t*)ctx_buf(ctx, "al_off", (nb + 1) * sizeof(int64_t));
    if (!dms || !doff) return EQBF_ERR_HIP;
    EQBF_HIP(ctx, hipMemcpyAsync(doff, boff.data(), boff.size() * sizeof(int64_t), hipMemcpyHostToDevice, st));
    if (n_src > 0)
      hipLaunchKernelGGL((f32 ? al_snpstat_kernel<float> : al_snpstat_kernel<double>),
                         dim3((unsigned)((n_src + 63) / 64)), dim3(256), 0, st, d, off[g0], n_src, dms);
    {
      ProfScope ps(ctx, "al_gram_kernel", st);
      hipLaunchKernelGGL((f32 ? al_gram_kernel<float> : al_gram_kernel<double>),
                         dim3((unsigned)(nb * (nt * (nt + 1) / 2))), dim3(256), 0, st, d, off[g0], doff, dms, nt, dK);
    }
    {
      ProfScope ps(ctx, "al_eig_kernel", st);
      hipLaunchKernelGGL(al_eig_kernel, dim3((unsigned)nb), dim3(EIG_NT), lds, st, dK, N, n_eig, deig);
    }
    EQBF_HIP(ctx, hipGetLastError());
    EQBF_HIP(ctx, hipMemcpyAsync(eig + (int64_t)g0 * n_eig, deig, (size_t)nb * n_eig * sizeof(float),
                                 hipMemcpyDeviceToHost, st));
    EQBF_HIP(ctx, hipStreamSynchronize(st)); /* boff is refilled for the next batch */
  }
  return EQBF_OK;
}

static int ld_eig_check(eqbf_ctx* ctx, const eqbf_chunk* c, int32_t n_eig, float* eig) {
  if (!ctx) return EQBF_ERR_ARG;
  if (!c || !eig || n_eig < 1 || n_eig > EIG_P - 4)
    return ctx_fail(ctx, EQBF_ERR_ARG, "n_eig must be in 1..%d", EIG_P - 4);
  if (c->n_genes > 0 && (c->n_samples < 2 || c->n_samples > EIG_NMAX))
    return ctx_fail(ctx, EQBF_ERR_UNSUPPORTED, "LD eigenvalues support 2..%d samples", EIG_NMAX);
  return EQBF_OK;
}

extern "C" int eqbf_ld_eigenvalues_device(eqbf_ctx* ctx, const eqbf_chunk* chunk_dev, int32_t n_eig, float* eig) {
  int rc = ld_eig_check(ctx, chunk_dev, n_eig, eig);
  if (rc || chunk_dev->n_genes == 0) return rc;
  std::vector<int64_t> off(chunk_dev->n_genes + 1);
  EQBF_HIP(ctx, hipMemcpyAsync(off.data(), chunk_dev->pair_offset, off.size() * sizeof(int64_t), hipMemcpyDeviceToHost,
                               ctx->stream));
  EQBF_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return ld_eig_run(ctx, *chunk_dev, off, n_eig, eig);
}

extern "C" int eqbf_ld_eigenvalues(eqbf_ctx* ctx, const eqbf_chunk* chunk, int32_t n_eig, float* eig) {
  int rc = ld_eig_check(ctx, chunk, n_eig, eig);
  if (rc || chunk->n_genes == 0) return rc;
  const eqbf_chunk& c = *chunk;
  const hipStream_t st = ctx->stream;
  eqbf_chunk d = c;
  const size_t gbytes = (size_t)c.n_samples * c.geno_ld * (c.geno_dtype == EQBF_F32 ? 4 : 8);
  void* g = ctx_buf(ctx, "al_geno", gbytes);
  void* ps = ctx_buf(ctx, "al_psnp", (size_t)std::max<int64_t>(c.n_pairs, 1) * sizeof(int32_t));
  if (!g || !ps) return EQBF_ERR_HIP;
  EQBF_HIP(ctx, hipMemcpyAsync(g, c.genotypes, gbytes, hipMemcpyHostToDevice, st));
  EQBF_HIP(ctx, hipMemcpyAsync(ps, c.pair_snp, (size_t)c.n_pairs * sizeof(int32_t), hipMemcpyHostToDevice, st));
  d.genotypes = g;
  d.pair_snp = (const int32_t*)ps;
  std::vector<int64_t> off(c.pair_offset, c.pair_offset + c.n_genes + 1);
  return ld_eig_run(ctx, d, off, n_eig, eig);
}

extern "C" int eqbf_gev_fit(eqbf_ctx* ctx, const double* stats, int64_t n_genes, int64_t nperm, double* params) {
  if (!ctx || !stats || !params || n_genes < 0 || nperm < 3) return ctx ? ctx_fail(ctx, EQBF_ERR_ARG, "gev") : 1;
  if (nperm > GEV_NMAX) return ctx_fail(ctx, EQBF_ERR_UNSUPPORTED, "GEV fit supports at most %d draws", GEV_NMAX);
  if (n_genes == 0) return EQBF_OK;
  const hipStream_t st = ctx->stream;
  int npow = 1;
  while (npow < nperm) npow <<= 1;
  const int64_t gb = std::min<int64_t>(n_genes, 65536);
  double* ds = (double*)ctx_buf(ctx, "gev_in", (size_t)gb * nperm * sizeof(double));
  double* dp = (double*)ctx_buf(ctx, "gev_out", (size_t)gb * 3 * sizeof(double));
  if (!ds || !dp) return EQBF_ERR_HIP;
  for (int64_t g0 = 0; g0 < n_genes; g0 += gb) {
    const int64_t nb = std::min(gb, n_genes - g0);
    EQBF_HIP(ctx, hipMemcpyAsync(ds, stats + g0 * nperm, (size_t)nb * nperm * sizeof(double), hipMemcpyHostToDevice,
                                 st));
    {
      ProfScope ps(ctx, "al_gev_kernel", st);
      hipLaunchKernelGGL(al_gev_kernel, dim3((unsigned)nb), dim3(1024), (size_t)npow * sizeof(double), st, ds, nperm,
                         npow, dp);
    }
    EQBF_HIP(ctx, hipGetLastError());
    EQBF_HIP(ctx, hipMemcpyAsync(params + g0 * 3, dp, (size_t)nb * 3 * sizeof(double), hipMemcpyDeviceToHost, st));
    EQBF_HIP(ctx, hipStreamSynchronize(st));
  }
  return EQBF_OK;
}
