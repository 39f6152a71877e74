// Block-level (one workgroup) FP64 building blocks shared by the single-molecule
// kernels and the persistent ensemble kernel.
#pragma once
#include <math.h>
#include "common.h"

#define EIG_SMALL_CLUSTER 8

__host__ __device__ static size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

struct EigLayout {
  size_t W, d, e, tau, z, scratch, coef, total;
};
__host__ __device__ static EigLayout eig_layout(int l, int nev) {
  EigLayout L;
  size_t off = 0;
  L.W = off; off += al256((size_t)l * l * 8);
  L.d = off; off += al256((size_t)l * 8);
  L.e = off; off += al256((size_t)l * 8);
  L.tau = off; off += al256((size_t)l * 8);
  L.z = off; off += al256((size_t)l * nev * 8);
  L.scratch = off; off += al256((size_t)6 * l * nev * 8);
  L.coef = off; off += al256((size_t)nev * 8);
  L.total = off;
  return L;
}


template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true));
}

// Sum over the wave in every lane: the butterfly v_i + v_{i ^ o}, o = 32, 16, .. 1.  The
// partners come through v_permlane swaps and row rotations (after the step o = 8 a row's
// halves agree, so that a rotation by o reads the same value as lane i ^ o) instead of
// ds_bpermute: 6 steps of ~25 cycles instead of ~120.
__device__ __forceinline__ double wave_sum(double v) {
  {
    const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    v = __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
  }
  {
    const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    v = __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
  }
  v += dpp_f64<0x128>(v);   // row_ror:8
  v += dpp_f64<0x124>(v);   // row_ror:4
  v += dpp_f64<0x122>(v);   // row_ror:2
  v += dpp_f64<0x121>(v);   // row_ror:1
  return v;
}

__device__ double blk_sum(double v, double* sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wv] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += sh[i];
  return s;
}

// maximum over the workgroup (all threads get it)
__device__ double blk_max_any(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wv] = v;
  __syncthreads();
  double m = sh[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = fmax(m, sh[i]);
  return m;
}

// Sturm count: number of eigenvalues of the tridiagonal (d, e) below x.
typedef __attribute__((address_space(3))) double lds_f64;
typedef __attribute__((address_space(3))) int lds_i32;

// d, e in LDS (address-space-3 pointers: ds_read instead of flat loads)
__device__ int sturm_count(const lds_f64* d, const lds_f64* e, int l, double x, double pivmin) {
  int c = 0;
  double q = d[0] - x;
  if (fabs(q) < pivmin) q = -pivmin;
  if (q < 0) ++c;
#pragma unroll 8
  for (int i = 1; i < l; ++i) {
    q = d[i] - x - e[i - 1] * e[i - 1] / q;
    if (fabs(q) < pivmin) q = -pivmin;
    if (q < 0) ++c;
  }
  return c;
}

__device__ __forceinline__ double hash_unit(unsigned int a, unsigned int b) {
  unsigned int h = a * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15; h *= 0x2C1B3C6Du; h ^= h >> 12; h *= 0x297A2D39u; h ^= h >> 15;
  return ((double)(h & 0xFFFFFF) / (double)0xFFFFFF) * 2.0 - 1.0;
}

// LU factorisation of T - lam I with partial pivoting between rows k and k+1
// (u0r: reciprocals of the pivots, u1/u2: the two superdiagonals of U, mlt: the
// multipliers, piv: 1 where rows were interchanged).
__device__ void tri_factor(const double* __restrict__ d, const double* __restrict__ e, int l, double lam,
                           double tiny, double* __restrict__ u0r, double* __restrict__ u1, double* __restrict__ u2,
                           double* __restrict__ mlt, int* __restrict__ piv) {
  double r0 = d[0] - lam, r1 = (l > 1) ? e[0] : 0.0;
  for (int k = 0; k < l - 1; ++k) {
    const double sub = e[k];
    const double a1 = d[k + 1] - lam;
    const double b1 = (k + 1 < l - 1) ? e[k + 1] : 0.0;
    if (fabs(r0) >= fabs(sub)) {
      if (fabs(r0) < tiny) r0 = (r0 >= 0 ? tiny : -tiny);
      const double m = sub / r0;
      u0r[k] = 1.0 / r0; u1[k] = r1; u2[k] = 0.0; mlt[k] = m; piv[k] = 0;
      r0 = a1 - m * r1;
      r1 = b1;
    } else {
      const double m = r0 / sub;
      u0r[k] = 1.0 / sub; u1[k] = a1; u2[k] = b1; mlt[k] = m; piv[k] = 1;
      r0 = r1 - m * a1;
      r1 = -m * b1;
    }
  }
  if (fabs(r0) < tiny) r0 = (r0 >= 0 ? tiny : -tiny);
  u0r[l - 1] = 1.0 / r0;
  u1[l - 1] = 0.0;
  u2[l - 1] = 0.0;
}

// x <- (T - lam I)^{-1} x with the factors of tri_factor.  The entries being
// eliminated are carried in registers; the operands of TRI_B consecutive steps
// are loaded together, without bounds tests (full blocks first, then the
// remainder one step at a time), so one memory latency is paid per block of
// steps instead of per step.
#define TRI_B 8
template <typename D, typename I>
__device__ void tri_apply(int l, const D* __restrict__ u0r, const D* __restrict__ u1, const D* __restrict__ u2,
                          const D* __restrict__ mlt, const I* __restrict__ piv, D* __restrict__ x) {
  double c = x[0];
  int k = 0;
  for (; k + TRI_B <= l - 1; k += TRI_B) {
    double nx[TRI_B], m[TRI_B];
    int pv[TRI_B];
#pragma unroll
    for (int u = 0; u < TRI_B; ++u) {
      nx[u] = x[k + u + 1];
      m[u] = mlt[k + u];
      pv[u] = piv[k + u];
    }
#pragma unroll
    for (int u = 0; u < TRI_B; ++u) {
      const double keep = pv[u] ? nx[u] : c;
      c = pv[u] ? c - m[u] * nx[u] : nx[u] - m[u] * c;
      x[k + u] = keep;
    }
  }
  for (; k < l - 1; ++k) {
    const double nx = x[k + 1], m = mlt[k];
    const double keep = piv[k] ? nx : c;
    c = piv[k] ? c - m * nx : nx - m * c;
    x[k] = keep;
  }
  x[l - 1] = c;
  double x1 = 0.0, x2 = 0.0;
  k = l - 1;
  for (; k - TRI_B + 1 >= 0; k -= TRI_B) {
    double xv[TRI_B], a1[TRI_B], a2[TRI_B], r0[TRI_B];
#pragma unroll
    for (int u = 0; u < TRI_B; ++u) {
      xv[u] = x[k - u];
      a1[u] = u1[k - u];
      a2[u] = u2[k - u];
      r0[u] = u0r[k - u];
    }
#pragma unroll
    for (int u = 0; u < TRI_B; ++u) {
      const double sv = (xv[u] - a1[u] * x1 - a2[u] * x2) * r0[u];
      x[k - u] = sv;
      x2 = x1;
      x1 = sv;
    }
  }
  for (; k >= 0; --k) {
    const double sv = (x[k] - u1[k] * x1 - u2[k] * x2) * u0r[k];
    x[k] = sv;
    x2 = x1;
    x1 = sv;
  }
}


// ---- inverse iteration of one eigenvalue cluster by one wavefront -------------------
// The recurrences (substitution, dot products, norms) are chains over the vector's
// entries: lane 0 runs them on operands in LDS, unrolled so that the reads run ahead of
// the chain.  What is not a chain (updates, scaling, loads, stores) is spread over the
// lanes.  The factors arrive in blocks of 64 steps, one step per lane, the next block's
// loads issued before the current block's steps.  One thread per cluster on global memory
// paid a memory latency per entry and serialised the clusters of a wave: the kernel took
// 17.7 ms for 20 roots at l = 620, this form takes 4.8 ms (same results).
#define EIG_STAGE 320            // LDS doubles per wave: five arrays of 64
#define EIG_STAGE_WAVES 8

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// one forward step: entry x_k leaves as `keep`, the eliminated next entry stays in c
__device__ __forceinline__ double tri_forward(double& c, double nx, double m, int pv) {
  const double keep = pv ? nx : c;
  c = pv ? c - m * nx : nx - m * c;
  return keep;
}

// x <- (T - lam I)^{-1} x with the factors of tri_factor, x (l doubles) and stg in LDS
__device__ void tri_apply_wave(int l, const double* __restrict__ u0r, const double* __restrict__ u1,
                               const double* __restrict__ u2, const double* __restrict__ mlt,
                               const int* __restrict__ piv, lds_f64* x, lds_f64* stg) {
  const int lane = threadIdx.x & 63;
  lds_f64 *sm = stg, *s0 = stg, *s1 = stg + 64, *s2 = stg + 128;
  double c = x[0];
  const int nf = l - 1;                      // forward steps
  double gm = 0.0;
  int gp = 0;
  if (lane < nf) { gm = mlt[lane]; gp = piv[lane]; }
  for (int kb = 0; kb < nf; kb += 64) {
    const int n = nf - kb < 64 ? nf - kb : 64;
    sm[lane] = gm;
    const unsigned long long pm = __ballot(gp != 0);
    wave_lds_fence();
    if (kb + 64 + lane < nf) { gm = mlt[kb + 64 + lane]; gp = piv[kb + 64 + lane]; }
    lds_f64* xb = x + kb;
    if (lane == 0) {
      int h = 0;
      for (; h + 16 <= n; h += 16) {
        double nx[16], m[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) { nx[u] = xb[h + u + 1]; m[u] = sm[h + u]; }
#pragma unroll
        for (int u = 0; u < 16; ++u) xb[h + u] = tri_forward(c, nx[u], m[u], (int)(pm >> (h + u)) & 1);
      }
      for (; h < n; ++h) xb[h] = tri_forward(c, xb[h + 1], sm[h], (int)(pm >> h) & 1);
    }
    wave_lds_fence();
  }
  if (lane == 0) x[l - 1] = c;
  wave_lds_fence();
  // backward: step t handles entry l - 1 - t
  double g0 = 0.0, g1 = 0.0, g2 = 0.0;
  if (lane < l) { g0 = u0r[l - 1 - lane]; g1 = u1[l - 1 - lane]; g2 = u2[l - 1 - lane]; }
  double x1 = 0.0, x2 = 0.0;
  for (int kb = 0; kb < l; kb += 64) {
    const int n = l - kb < 64 ? l - kb : 64;
    s0[lane] = g0;
    s1[lane] = g1;
    s2[lane] = g2;
    wave_lds_fence();
    if (kb + 64 + lane < l) {
      g0 = u0r[l - 65 - kb - lane];
      g1 = u1[l - 65 - kb - lane];
      g2 = u2[l - 65 - kb - lane];
    }
    lds_f64* xb = x + (l - 1 - kb);
    if (lane == 0) {
      int h = 0;
      for (; h + 16 <= n; h += 16) {
        double xv[16], a1[16], a2[16], r0[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          xv[u] = xb[-(h + u)];
          a1[u] = s1[h + u];
          a2[u] = s2[h + u];
          r0[u] = s0[h + u];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const double sv = (xv[u] - a1[u] * x1 - a2[u] * x2) * r0[u];
          xb[-(h + u)] = sv;
          x2 = x1;
          x1 = sv;
        }
      }
      for (; h < n; ++h) {
        const double sv = (xb[-h] - s1[h] * x1 - s2[h] * x2) * s0[h];
        xb[-h] = sv;
        x2 = x1;
        x1 = sv;
      }
    }
    wave_lds_fence();
  }
}

// sum_i a_i x_i as one chain over i (a: global with stride lda, or x itself when null); the
// result in every lane
__device__ double dot_chain_wave(int l, const double* __restrict__ a, long lda, const lds_f64* x, lds_f64* stg) {
  const int lane = threadIdx.x & 63;
  double s = 0.0;
  double g = (a && lane < l) ? a[lane * lda] : 0.0;
  for (int kb = 0; kb < l; kb += 64) {
    const int n = l - kb < 64 ? l - kb : 64;
    const lds_f64 *xb = x + kb, *y = xb;
    if (a) {
      stg[lane] = g;
      wave_lds_fence();
      y = stg;
      if (kb + 64 + lane < l) g = a[(kb + 64 + lane) * lda];
    }
    if (lane == 0) {
      int h = 0;
      for (; h + 16 <= n; h += 16) {
        double p[16], q[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) { p[u] = y[h + u]; q[u] = xb[h + u]; }
#pragma unroll
        for (int u = 0; u < 16; ++u) s += p[u] * q[u];
      }
      for (; h < n; ++h) s += y[h] * xb[h];
    }
    wave_lds_fence();
  }
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(s)),
                          __builtin_amdgcn_readfirstlane(__double2loint(s)));
}

// members m0 .. m1 - 1 of one cluster (factors of member m at scr + 6 l m) into Z
__device__ void cluster_wave(int l, int nev, int m0, int m1, const double* __restrict__ scr, double* __restrict__ Z,
                             lds_f64* x, lds_f64* stg) {
  const int lane = threadIdx.x & 63;
  for (int m = m0; m < m1; ++m) {
    const double* base = scr + (size_t)6 * l * m;
    for (int i = lane; i < l; i += 64) x[i] = hash_unit((unsigned)m, (unsigned)i);
    wave_lds_fence();
    for (int it = 0; it < 4; ++it) {
      tri_apply_wave(l, base, base + l, base + 2 * l, base + 3 * l, (const int*)(base + 4 * l), x, stg);
      for (int mm = m0; mm < m; ++mm) {
        const double s = dot_chain_wave(l, Z + mm, nev, x, stg);
        for (int i = lane; i < l; i += 64) x[i] -= s * Z[(long)i * nev + mm];
        wave_lds_fence();
      }
      double nrm = sqrt(dot_chain_wave(l, nullptr, 0, x, stg));
      if (!(nrm > 0.0)) nrm = 1.0;
      for (int i = lane; i < l; i += 64) x[i] /= nrm;
      wave_lds_fence();
    }
    for (int i = lane; i < l; i += 64) Z[(long)i * nev + m] = x[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // later members read it from global memory
    wave_lds_fence();
  }
}

// Householder steps j0 <= j < j1 in one workgroup.  X(r, c) = X[r * ldx + c] holds the rows and
// columns j0, .. l - 1 of the matrix, in LDS or in global memory; reflector j goes to row j of W
// behind the diagonal (never read again by the reduction), where the back-transformation reads it
// coalesced.  X may be W itself: row j is then written through X in step j - 1 and through W in
// step j, with barriers between.  A wave takes RB rows and CB chunks of 64 columns at a time: a
// load's latency, not its bandwidth, bounds a step.
template <int RB, int CB, typename P>
__device__ __forceinline__ void hh_block_steps(P X, int ldx, int j0, int j1, int l, double* W,
                                               double* __restrict__ d, double* __restrict__ e,
                                               double* __restrict__ tau, lds_f64* sv, lds_f64* sp, double* sh) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
  for (int j = j0; j < j1; ++j) {
    const int n2 = l - j - 1;
    P X2 = X + (j + 1 - j0) * (ldx + 1);       // the trailing block
    double* refl = W + (long)j * l + j + 1;
    const double dj = X[(j - j0) * (ldx + 1)];
    double part = 0.0;
    for (int r = tid; r < n2; r += blockDim.x) {
      const double x = X2[r * ldx - 1];
      sv[r] = x;
      part += x * x;
    }
    const double alpha2 = blk_sum(part, sh);
    const double x0 = sv[0];
    __syncthreads();
    if (alpha2 <= 1e-300) {
      if (tid == 0) { tau[j] = 0.0; e[j] = 0.0; d[j] = dj; }
      for (int r = tid; r < n2; r += blockDim.x) refl[r] = 0.0;
      __syncthreads();
      continue;
    }
    const double alpha = sqrt(alpha2);
    const double beta = (x0 >= 0.0) ? -alpha : alpha;
    const double v0 = x0 - beta;
    const double vtv = alpha2 - x0 * x0 + v0 * v0;
    const double t = 2.0 / vtv;
    if (tid == 0) { sv[0] = v0; tau[j] = t; e[j] = beta; d[j] = dj; }
    __syncthreads();
    // p = t * A22 v  (lanes across columns)
    for (int r = RB * wv; r < n2; r += RB * nw) {
      double s[RB];
      int o[RB];
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        s[u] = 0.0;
        o[u] = (r + u < n2 ? r + u : n2 - 1) * ldx;
      }
      for (int c0 = lane; c0 < n2; c0 += 64 * CB) {
        double x[CB][RB];
#pragma unroll
        for (int q = 0; q < CB; ++q) {
          const int c = c0 + 64 * q < n2 ? c0 + 64 * q : c0;
#pragma unroll
          for (int u = 0; u < RB; ++u) x[q][u] = X2[o[u] + c];
        }
#pragma unroll
        for (int q = 0; q < CB; ++q)
          if (c0 + 64 * q < n2) {
            const double v = sv[c0 + 64 * q];
#pragma unroll
            for (int u = 0; u < RB; ++u) s[u] += x[q][u] * v;
          }
      }
#pragma unroll
      for (int u = 0; u < RB; ++u) s[u] = wave_sum(s[u]);
      if (lane == 0) {
#pragma unroll
        for (int u = 0; u < RB; ++u)
          if (r + u < n2) sp[r + u] = t * s[u];
      }
    }
    __syncthreads();
    part = 0.0;
    for (int r = tid; r < n2; r += blockDim.x) part += sp[r] * sv[r];
    const double K = 0.5 * t * blk_sum(part, sh);
    for (int r = tid; r < n2; r += blockDim.x) {
      refl[r] = sv[r];
      sp[r] -= K * sv[r];
    }
    __syncthreads();
    for (int r = RB * wv; r < n2; r += RB * nw) {
      double vr[RB], pr[RB];
      int o[RB];
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int q = r + u < n2 ? r + u : n2 - 1;
        vr[u] = sv[q];
        pr[u] = sp[q];
        o[u] = q * ldx;
      }
      for (int c0 = lane; c0 < n2; c0 += 64 * CB) {
        double x[CB][RB];
#pragma unroll
        for (int q = 0; q < CB; ++q) {
          const int c = c0 + 64 * q < n2 ? c0 + 64 * q : c0;
#pragma unroll
          for (int u = 0; u < RB; ++u) x[q][u] = X2[o[u] + c];
        }
#pragma unroll
        for (int q = 0; q < CB; ++q)
          if (c0 + 64 * q < n2) {
            const double vc = sv[c0 + 64 * q], pc = sp[c0 + 64 * q];
#pragma unroll
            for (int u = 0; u < RB; ++u)   // rows beyond the last repeat it: the same value again
              X2[o[u] + c0 + 64 * q] = x[q][u] - __builtin_fma(vr[u], pc, pr[u] * vc);
          }
      }
    }
    __syncthreads();
  }
}

// z <- H_0 ... H_{l-3} z, one wave per vector: entry i of vector n at Z[i * zi + n * zn], reflectors
// in the rows of W behind the diagonal, the next one's first 256 entries loaded ahead.
template <typename P>
__device__ __forceinline__ void hh_block_back(int l, int nev, const double* __restrict__ W,
                                              const double* __restrict__ tau, P Z, int zi, int zn) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int n = wv; n < nev; n += nw) {
    P z = Z + n * zn;
    double vn[4], tn = 0.0;
    auto fetch = [&](int j) {
      tn = tau[j];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = j + 1 + lane + 64 * q;
        vn[q] = i < l ? W[(long)j * l + i] : 0.0;
      }
    };
    if (l >= 3) fetch(l - 3);
    for (int j = l - 3; j >= 0; --j) {
      const int n2 = l - j - 1;
      const double t = tn;
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = vn[q];
      if (j > 0) fetch(j - 1);
      if (t == 0.0) continue;
      const double* vr = W + (long)j * l + j + 1;
      P zj = z + (j + 1) * zi;
      double s = 0.0, x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = lane + 64 * q;
        x[q] = r < n2 ? zj[r * zi] : 0.0;
        if (r < n2) s += v[q] * x[q];
      }
      for (int r = lane + 256; r < n2; r += 64) s += vr[r] * zj[r * zi];
      s = t * wave_sum(s);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = lane + 64 * q;
        if (r < n2) zj[r * zi] = x[q] - s * v[q];
      }
      for (int r = lane + 256; r < n2; r += 64) zj[r * zi] -= s * vr[r];
      wave_lds_fence();
    }
  }
}

__device__ __noinline__ void syevx_tridiag_vectors(int l, int nev, double* __restrict__ evals,
                                                   char* __restrict__ ws, double* sv, double* sp, double* sh,
                                                   double* s_bnd, int cap, double* stg);

// Lowest nev eigenpairs of the symmetric l x l matrix A (leading dim ld), one
// workgroup: Householder tridiagonalisation, Sturm bisection, inverse
// iteration (clusters re-orthogonalised), back-transformation.  sv, sp: LDS
// scratch of cap >= l doubles each; sh: >= blockDim/64 doubles; s_bnd: 2; stg:
// EIG_STAGE_WAVES * EIG_STAGE doubles of LDS; wl: nl x (nl | 1) doubles of LDS.
// The reduction runs on global memory until nl rows are left and on LDS from there, the
// back-transformation on LDS where l nev doubles fit.  In the ensemble (l up to 250, 17 solves
// of a C22H24 member) with everything on L2 and a row or an element at a time it took 61 ms,
// now 42: 20 in the steps on L2, 6 on LDS, 13 for the eigenpairs of T, 2 back.
__device__ __noinline__ void syevx_block(const double* __restrict__ A, int l, int ld, int nev,
                                         double* __restrict__ evals, double* __restrict__ evecs,
                                         char* __restrict__ ws, double* sv, double* sp, double* sh, double* s_bnd,
                                         int cap, double* stg, double* wl, int nl) {
  EigLayout Lo = eig_layout(l, nev);
  double* W = (double*)(ws + Lo.W);
  double* d = (double*)(ws + Lo.d);
  double* e = (double*)(ws + Lo.e);
  double* tau = (double*)(ws + Lo.tau);
  double* Z = (double*)(ws + Lo.z);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
  lds_f64 *lv = (lds_f64*)sv, *lp = (lds_f64*)sp, *X = (lds_f64*)wl;

  const int j0 = l > nl ? l - nl : 0, ldx = (l - j0) | 1;
  for (int r = wv; r < l; r += nw)
    for (int c = lane; c < l; c += 64) {
      const double a = 0.5 * (A[(long)r * ld + c] + A[(long)c * ld + r]);
      if (j0 > 0)
        W[(long)r * l + c] = a;
      else
        X[r * ldx + c] = a;
    }
  __syncthreads();
  if (j0 > 0) {
    hh_block_steps<8, 4>(W, l, 0, j0, l, W, d, e, tau, lv, lp, sh);
    for (int r = j0 + wv; r < l; r += nw)
      for (int c = j0 + lane; c < l; c += 64) X[(r - j0) * ldx + (c - j0)] = W[(long)r * l + c];
    __syncthreads();
  }
  if (l > 2) hh_block_steps<4, 2>(X, ldx, j0, l - 2, l, W, d, e, tau, lv, lp, sh);
  // the last 2 x 2 block
  if (tid < 4) {
    const int r = l - 1 - (tid >> 1), c = l - 1 - (tid & 1);
    if (r >= j0 && c >= j0) W[(long)r * l + c] = X[(r - j0) * ldx + (c - j0)];
  }
  __syncthreads();
  syevx_tridiag_vectors(l, nev, evals, ws, sv, sp, sh, s_bnd, cap, stg);
  if ((long)l * nev <= (long)nl * (nl | 1)) {
    for (int i = tid; i < l * nev; i += blockDim.x) {
      const int r = (unsigned)i / (unsigned)nev;
      X[(i - r * nev) * l + r] = Z[i];
    }
    __syncthreads();
    hh_block_back(l, nev, W, tau, X, 1, l);
    __syncthreads();
    for (int i = tid; i < l * nev; i += blockDim.x) {
      const int r = (unsigned)i / (unsigned)nev;
      evecs[i] = X[(i - r * nev) * l + r];
    }
  } else {
    hh_block_back(l, nev, W, tau, Z, nev, 1);
    __syncthreads();
    for (int i = tid; i < l * nev; i += blockDim.x) evecs[i] = Z[i];
  }
}

// Steps after the Householder reduction of W (reflectors below the first
// subdiagonal, d[0..l-3], e[0..l-3], tau set): last 2x2 block, bisection for
// the nev lowest eigenvalues and inverse iteration into Z (l x nev, row-major).
// sv, sp: LDS scratch of cap >= l doubles each (they hold d and e).
__device__ __noinline__ void syevx_tridiag_vectors(int l, int nev, double* __restrict__ evals,
                                                   char* __restrict__ ws, double* sv, double* sp, double* sh,
                                                   double* s_bnd, int cap, double* stg) {
  EigLayout Lo = eig_layout(l, nev);
  double* W = (double*)(ws + Lo.W);
  double* d = (double*)(ws + Lo.d);
  double* e = (double*)(ws + Lo.e);
  double* Z = (double*)(ws + Lo.z);
  double* scr = (double*)(ws + Lo.scratch);
  const int tid = threadIdx.x;
  if (tid == 0) {
    if (l >= 2) {
      d[l - 2] = W[(long)(l - 2) * l + (l - 2)];
      e[l - 2] = W[(long)(l - 1) * l + (l - 2)];
    }
    d[l - 1] = W[(long)(l - 1) * l + (l - 1)];
    if (l >= 1) e[l - 1] = 0.0;
  }
  __syncthreads();
  for (int i = tid; i < l; i += blockDim.x) {
    sv[i] = d[i];
    sp[i] = e[i];
  }
  __syncthreads();
  // Gershgorin bounds and the largest e^2 (minima and maxima: any order)
  double emax2 = 0.0;
  {
    double lo = 1e300, hi = -1e300;
    for (int i = tid; i < l; i += blockDim.x) {
      const double r = (i > 0 ? fabs(sp[i - 1]) : 0.0) + (i < l - 1 ? fabs(sp[i]) : 0.0);
      lo = fmin(lo, sv[i] - r);
      hi = fmax(hi, sv[i] + r);
      if (i + 1 < l) emax2 = fmax(emax2, sp[i] * sp[i]);
    }
    lo = -blk_max_any(-lo, sh);
    hi = blk_max_any(hi, sh);
    emax2 = blk_max_any(emax2, sh);
    if (tid == 0) {
      s_bnd[0] = lo;
      s_bnd[1] = hi;
    }
  }
  __syncthreads();
  const double* dl = sv;
  const double* el = sp;
  const lds_f64* ldl = (const lds_f64*)sv;   // the same LDS buffers, address-space typed
  const lds_f64* lel = (const lds_f64*)sp;
  const double lo0 = s_bnd[0], hi0 = s_bnd[1];
  const double tnorm = fmax(fabs(lo0), fabs(hi0));
  const double pivmin = 2.2250738585072014e-308 * fmax(1.0, emax2);
  const double eps = 1.1102230246251565e-16;

  // ---- 2. the nev lowest eigenvalues by Sturm counts.  With P = blockDim / nev >= 2
  // points per eigenvalue and round (multisection), every round narrows each
  // interval to one of its P + 1 parts; otherwise plain bisection per thread.
  // Both stop at b - a <= 2 eps max(|a|, |b|) + pivmin.
  // (the counts live in the 6 l nev doubles of scratch: P <= 12 l - 6 keeps them inside)
  const int P = min((int)blockDim.x / nev, 12 * l - 6);
  if (P < 2) {
    for (int m = tid; m < nev; m += blockDim.x) {
      double a = lo0 - 2.0 * eps * tnorm - pivmin, b = hi0 + 2.0 * eps * tnorm + pivmin;
      for (int it = 0; it < 200; ++it) {
        double mid = 0.5 * (a + b);
        if (sturm_count(ldl, lel, l, mid, pivmin) > m) b = mid; else a = mid;
        if (b - a <= 2.0 * eps * fmax(fabs(a), fabs(b)) + pivmin) break;
      }
      evals[m] = 0.5 * (a + b);
    }
  } else {
    double* ivl = scr;                          // [nev][2] intervals
    int* cnt = (int*)(scr + 2 * nev);           // [nev][P] counts
    int* flag = cnt + nev * P;                  // [nev] converged, then [1] all converged
    for (int m = tid; m < nev; m += blockDim.x) {
      ivl[2 * m] = lo0 - 2.0 * eps * tnorm - pivmin;
      ivl[2 * m + 1] = hi0 + 2.0 * eps * tnorm + pivmin;
      flag[m] = 0;
    }
    __syncthreads();
    for (int round = 0; round < 200; ++round) {
      if (tid < nev * P) {
        const int m = tid / P, k = tid % P;
        if (!flag[m]) {
          const double a = ivl[2 * m], b = ivl[2 * m + 1];
          const double x = a + (b - a) * (double)(k + 1) / (double)(P + 1);
          cnt[m * P + k] = sturm_count(ldl, lel, l, x, pivmin);
        }
      }
      __syncthreads();
      for (int m = tid; m < nev; m += blockDim.x) {
        if (flag[m]) continue;
        const double a = ivl[2 * m], b = ivl[2 * m + 1];
        double na = a, nb = b;
        for (int k = 0; k < P; ++k) {
          const double x = a + (b - a) * (double)(k + 1) / (double)(P + 1);
          if (cnt[m * P + k] > m) {
            nb = x;
            break;
          }
          na = x;
        }
        ivl[2 * m] = na;
        ivl[2 * m + 1] = nb;
        if (nb - na <= 2.0 * eps * fmax(fabs(na), fabs(nb)) + pivmin) flag[m] = 1;
      }
      __syncthreads();
      if (tid == 0) {
        int all = 1;
        for (int m = 0; m < nev; ++m) all &= flag[m];
        flag[nev] = all;
      }
      __syncthreads();
      if (flag[nev]) break;
    }
    for (int m = tid; m < nev; m += blockDim.x) evals[m] = 0.5 * (ivl[2 * m] + ivl[2 * m + 1]);
  }
  __syncthreads();

  // ---- 3. inverse iteration.  Clusters (gap < 1e-3 ||T||) of at most EIG_SMALL_CLUSTER
  // members are handled by one wave each; larger clusters
  // are processed by the whole workgroup with classical Gram-Schmidt (twice)
  // against the earlier members in every iteration.  Member m of a cluster
  // starting at m0 uses the shift evals[m] + 10 (m - m0) eps ||T||; its LU
  // factors (6 l doubles at scr + 6 l m: 1/u0, u1, u2, multipliers, pivots, x)
  // are formed once, for all members in parallel.
  const double ortol = 1.0e-3 * tnorm;
  const double tiny = eps * fmax(tnorm, 1e-300);
  double* coef = (double*)(ws + Lo.coef);
  for (int m = tid; m < nev; m += blockDim.x) {
    int m0 = m;
    while (m0 > 0 && evals[m0] - evals[m0 - 1] < ortol) --m0;
    const double lam = evals[m] + (double)(m - m0) * 10.0 * tiny;
    double* base = scr + (size_t)6 * l * m;
    tri_factor(dl, el, l, lam, tiny, base, base + l, base + 2 * l, base + 3 * l, (int*)(base + 4 * l));
  }
  __syncthreads();
  const int lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
  {
    // one wave per cluster; the iterates live in sv / sp (d and e are used up), so at
    // most 2 floor(cap / l) waves take part
    int nwl = 2 * (cap / l);
    if (nwl > nw) nwl = nw;
    if (nwl > EIG_STAGE_WAVES) nwl = EIG_STAGE_WAVES;
    if (wv < nwl) {
      lds_f64* x = (lds_f64*)((wv & 1 ? sp : sv) + (size_t)(wv >> 1) * l);
      lds_f64* st = (lds_f64*)(stg + wv * EIG_STAGE);
      int at = 0;                              // small clusters in order, dealt to the waves
      for (int m0 = 0; m0 < nev;) {
        int m1 = m0 + 1;
        while (m1 < nev && evals[m1] - evals[m1 - 1] < ortol) ++m1;
        if (m1 - m0 <= EIG_SMALL_CLUSTER && at++ % nwl == wv) cluster_wave(l, nev, m0, m1, scr, Z, x, st);
        m0 = m1;
      }
    }
  }
  __syncthreads();
  // large clusters, cooperatively.  The member's factors and iterate are staged in
  // the LDS buffers (free once the factors exist) when 4 l doubles fit, so the
  // serial solve runs on LDS; the Gram-Schmidt coefficients take one wave each.
  const bool stage = 4 * l <= cap;
  for (int m0 = 0; m0 < nev;) {
    int m1 = m0 + 1;
    while (m1 < nev && evals[m1] - evals[m1 - 1] < ortol) ++m1;
    if (m1 - m0 > EIG_SMALL_CLUSTER) {
      for (int m = m0; m < m1; ++m) {
        double* base = scr + (size_t)6 * l * m;
        const double *fu0 = base, *fu1 = base + l, *fu2 = base + 2 * l, *fml = base + 3 * l;
        const int* fpv = (const int*)(base + 4 * l);
        double* x = base + 5 * l;
        if (stage) {
          for (int i = tid; i < l; i += blockDim.x) {
            sv[i] = base[i];
            sv[l + i] = base[l + i];
            sv[2 * l + i] = base[2 * l + i];
            sv[3 * l + i] = base[3 * l + i];
            ((int*)(sp + l))[i] = ((const int*)(base + 4 * l))[i];
          }
          fu0 = sv; fu1 = sv + l; fu2 = sv + 2 * l; fml = sv + 3 * l;
          fpv = (const int*)(sp + l);
          x = sp;
        }
        for (int i = tid; i < l; i += blockDim.x) x[i] = hash_unit((unsigned)m, (unsigned)i);
        __syncthreads();
        for (int it = 0; it < 3; ++it) {
          if (tid == 0) {
            if (stage)
              tri_apply(l, (const lds_f64*)fu0, (const lds_f64*)fu1, (const lds_f64*)fu2, (const lds_f64*)fml,
                        (const lds_i32*)fpv, (lds_f64*)x);
            else
              tri_apply(l, fu0, fu1, fu2, fml, fpv, x);
          }
          __syncthreads();
          for (int pass = 0; pass < 2 && m > m0; ++pass) {
            for (int mm = m0 + wv; mm < m; mm += nw) {
              double s = 0.0;
              for (int i = lane; i < l; i += 64) s += Z[(long)i * nev + mm] * x[i];
              s = wave_sum(s);
              if (lane == 0) coef[mm] = s;
            }
            __syncthreads();
            for (int i = tid; i < l; i += blockDim.x) {
              double s = x[i];
              for (int mm = m0; mm < m; ++mm) s -= coef[mm] * Z[(long)i * nev + mm];
              x[i] = s;
            }
            __syncthreads();
          }
          double part = 0.0;
          for (int i = tid; i < l; i += blockDim.x) part += x[i] * x[i];
          double nrm = sqrt(blk_sum(part, sh));
          if (!(nrm > 0.0)) nrm = 1.0;
          for (int i = tid; i < l; i += blockDim.x) x[i] /= nrm;
          __syncthreads();
        }
        for (int i = tid; i < l; i += blockDim.x) Z[(long)i * nev + m] = x[i];
        __syncthreads();
      }
    }
    m0 = m1;
  }
  __syncthreads();
}

// ---- 4. back-transformation z <- H_0 ... H_{l-3} z in one workgroup (reflectors
// in the columns of W below the subdiagonal), evecs = Z.
__device__ __noinline__ void syevx_back_block(int l, int nev, double* __restrict__ evecs, char* __restrict__ ws,
                                              double* sv) {
  EigLayout Lo = eig_layout(l, nev);
  const double* W = (const double*)(ws + Lo.W);
  const double* tau = (const double*)(ws + Lo.tau);
  double* Z = (double*)(ws + Lo.z);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
  for (int j = l - 3; j >= 0; --j) {
    const int n2 = l - j - 1;
    const double t = tau[j];
    if (t == 0.0) continue;
    for (int r = tid; r < n2; r += blockDim.x) sv[r] = W[(long)(j + 1 + r) * l + j];
    __syncthreads();
    for (int n = wv; n < nev; n += nw) {
      double s = 0.0;
      for (int r = lane; r < n2; r += 64) s += sv[r] * Z[(long)(j + 1 + r) * nev + n];
      s = t * wave_sum(s);
      for (int r = lane; r < n2; r += 64) Z[(long)(j + 1 + r) * nev + n] -= s * sv[r];
    }
    __syncthreads();
  }
  for (long i = tid; i < (long)l * nev; i += blockDim.x) evecs[i] = Z[i];
}
