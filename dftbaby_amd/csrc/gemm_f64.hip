// FP64 MFMA GEMM for gfx950 without LDS staging.
//
// v_mfma_f64_16x16x4f64 occupies its SIMD for 64 cycles (78.6 TFLOP/s over 1024
// SIMDs), so a wave that multiplies TM x TN register tiles needs only
// (TM + TN) 2 KiB of operands per TM TN 256 cycles: 16 bytes per cycle and CU at
// 4 x 4 tiles, a quarter of what L2 delivers.  Each wave therefore loads its
// operand fragments straight from global memory (L1 / L2) into registers, KS
// 16-deep k chunks ahead of the MFMAs that use them; there is no LDS traffic and no
// barrier in the main loop, and 8-byte alignment is enough (odd leading dimensions).
// Small tiles are latency bound, not fed: they prefetch up to six chunks.
//
// Every result is one chain of fused multiply-adds over ascending k (the MFMA adds
// its four k in lane-group order), whatever the tile: results do not depend on the
// shape chosen.  MFMA step s of a chunk takes k = 16 c + 4 s + lane / 16; a
// K-contiguous operand is loaded as 16 bytes per lane and brought into that order by
// one v_permlane16_swap per register pair, an operand with K as the slow index as
// 16 consecutive elements per k row.
//
// Measured against the kernel this replaces (128 x 128 and narrower tiles staged
// through LDS with one barrier per 16 k; identical results), us, old -> new:
//   4096 x 4096 x 4096 NN            3140 -> 2030   (44 -> 68 TFLOP/s of 78.6)
//   392 x 1696 x 1696, batch 15, NT  1310 ->  700   (26 -> 48)
//   798 x 798 x 798 TN                170 ->   37   (49 workgroups before)
//   40 x 1557504 x 400 TN            1500 -> 1250   (4.5 TB/s)
//   10 x 10 Gram, 1568 deep           102 ->   25   (one chain of 392 MFMAs)
#include <math.h>
#include "common.h"
#include "gemm.h"

typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));

__device__ __forceinline__ void store_f64(const GemmArgs& p, long off, double val) {
  if (p.out_type == GEMM_OUT_F64) {
    double* C = (double*)p.C + off;
    if (p.beta != 0.0) val += p.beta * (*C);
    *C = val;
  } else if (p.out_type == GEMM_OUT_F32) {
    float* C = (float*)p.C + off;
    if (p.beta != 0.0) val += p.beta * (double)(*C);
    *C = (float)val;
  } else {  // bf16 hi/lo pair
    const float x = (float)val;
    const unsigned short hi = bf16_bits_rne(x);
    ((unsigned short*)p.C)[off] = hi;
    ((unsigned short*)p.C2)[off] = bf16_bits_rne(x - bf16_bits_to_float(hi));
  }
}

// (a, b) -> (a of even 16-lane rows beside b's, a of odd rows beside b's): exchanges the
// register index with the low bit of the lane group
__device__ __forceinline__ void swap16(double& a, double& b) {
  unsigned al = (unsigned)__double2loint(a), ah = (unsigned)__double2hiint(a);
  unsigned bl = (unsigned)__double2loint(b), bh = (unsigned)__double2hiint(b);
  const auto lo = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
  a = __hiloint2double((int)hi[0], (int)lo[0]);
  b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// Fragments of one operand: T tiles of 16 rows, the 4 KS k steps of KS chunks.
// KC: K contiguous (x[row * ld + k]); otherwise x[k * ld + row].
template <int T, bool KC, int KS>
struct Frag {
  const double* ptr[T];   // this lane's row (clamped into the matrix) at its first k
  long ld;
  __device__ __forceinline__ void init(const double* x, long ld_, long r0, long rows, int lane) {
    ld = ld_;
    const long g = lane >> 4, k = KC ? 2 * (((g & 1) << 1) | (g >> 1)) : g;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      long r = r0 + 16 * i + (lane & 15);
      if (r >= rows) r = rows - 1;       // its products land in rows that are not stored
      ptr[i] = KC ? x + r * ld + k : x + k * ld + r;
    }
  }
  // steps 2 h and 2 h + 1 (k0 + 8 h .. k0 + 8 h + 7) of the chunks at k0; a K-contiguous pair
  // still has to go through order()
  __device__ __forceinline__ void load(long k0, int h, double (&v)[T][4 * KS]) const {
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if constexpr (KC) {
        const d2u_t x = *(const d2u_t*)(ptr[i] + k0 + 8 * h);
        v[i][2 * h] = x.x;
        v[i][2 * h + 1] = x.y;
      } else {
        const double* q = ptr[i] + (k0 + 8 * h) * ld;
        v[i][2 * h] = q[0];
        v[i][2 * h + 1] = q[4 * ld];
      }
    }
  }
  // lane group (hi, lo) holds k = 4 lo + 2 hi + {0, 1}; after the swap k = 4 s + 2 hi + lo in step s
  __device__ __forceinline__ void order(int h, double (&v)[T][4 * KS]) const {
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < T; ++i) swap16(v[i][2 * h], v[i][2 * h + 1]);
    }
  }
  // the last, partial chunk: k >= kend reads as zero
  __device__ __forceinline__ void load_tail(long k0, long kend, int lane, double (&v)[T][4 * KS]) const {
    const long g = lane >> 4, kp = KC ? 2 * (((g & 1) << 1) | (g >> 1)) : g;
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const long k = k0 + 4 * s + g;
        v[i][s] = k < kend ? (KC ? ptr[i][k - kp] : ptr[i][(k - kp) * ld]) : 0.0;
      }
  }
};

template <int TM, int TN, int WM, int WN, int KS, bool AT, bool BT>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_f64_kernel(GemmArgs p) {
  // two buffers of KS chunks where they and the addresses fit 256 registers
  // (the streaming shapes, WN = 4, measured faster with refilled half chunks)
  constexpr bool DB = KS > 1 || (16 * (TM + TN) + 8 * TM * TN <= (AT && !BT ? 184 : 208) && WN != 4);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  unsigned tx, ty, tz;
  xcd_tile_grouped<4>(tx, ty, tz);
  const long m0 = ((long)ty * WM + wm) * (16 * TM), n0 = ((long)tx * WN + wn) * (16 * TN);
  const long M = p.M, N = p.N;
  if (m0 >= M || n0 >= N) return;
  const int ks = tz % p.ksplit;
  const long b = tz / p.ksplit;
  const long kbeg = (long)ks * p.kchunk;
  const long kend = min((long)p.K, kbeg + p.kchunk);

  Frag<TM, !AT, KS> fa;
  Frag<TN, BT, KS> fb;
  fa.init((const double*)p.A + b * p.sA, p.lda, m0, M, lane);
  fb.init((const double*)p.B + b * p.sB, p.ldb, n0, N, lane);

  d4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (d4_t)(0.0);
  auto mul = [&](double (&a)[TM][4 * KS], double (&bb)[TN][4 * KS], int h) {
    fa.order(h, a);
    fb.order(h, bb);
#pragma unroll
    for (int s = 2 * h; s < 2 * h + 2; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][s], bb[j][s], acc[i][j], 0, 0, 0);
  };
  auto load = [&](long k, double (&a)[TM][4 * KS], double (&bb)[TN][4 * KS]) {
#pragma unroll
    for (int h = 0; h < 2 * KS; ++h) {
      fa.load(k, h, a);
      fb.load(k, h, bb);
    }
  };
  auto mul_all = [&](double (&a)[TM][4 * KS], double (&bb)[TN][4 * KS]) {
#pragma unroll
    for (int h = 0; h < 2 * KS; ++h) mul(a, bb, h);
  };
  // one operand load between every few MFMAs of the region, up to a scheduling barrier
  auto spread = [&]() {
    constexpr int NL = KS * ((AT ? 4 : 2) * TM + (BT ? 2 : 4) * TN);
    constexpr int PER = 4 * KS * TM * TN / NL > 0 ? 4 * KS * TM * TN / NL : 1;
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);   // VMEM read
      __builtin_amdgcn_sched_group_barrier(0x8, PER, 0);  // MFMA
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  const int n = kend > kbeg ? (int)((kend - kbeg) / 16) : 0;   // whole chunks
  const int ns = n / KS;                                       // whole buffers
  double av[TM][4 * KS], bv[TN][4 * KS];
  if (ns > 0) {
    long k = kbeg;
    if constexpr (DB) {
      // two buffers: the loads of one are issued before the MFMAs of the other.  The odd
      // buffer goes first, so that the loop has one exit; its last prefetch repeats the
      // last chunks.
      double aw[TM][4 * KS], bw[TN][4 * KS];
      load(k, av, bv);
      if (ns & 1) {
        mul_all(av, bv);
        if (ns > 1) k += 16 * KS;
        load(k, av, bv);
      }
      for (int c = ns & 1; c < ns; c += 2) {
        k += 16 * KS;
        load(k, aw, bw);
        mul_all(av, bv);
        spread();
        if (c + 2 < ns) k += 16 * KS;
        load(k, av, bv);
        mul_all(aw, bw);
        spread();
      }
    } else {
      // one buffer: each half chunk's registers are refilled for the next chunk as soon as
      // its MFMAs are issued, so its loads have the other half's MFMAs to arrive; the
      // scheduling barriers keep that order.  The last prefetch repeats the last chunk.
      fa.load(k, 0, av);
      fb.load(k, 0, bv);
      __builtin_amdgcn_sched_barrier(0);
      fa.load(k, 1, av);
      fb.load(k, 1, bv);
      for (int c = 1; c <= ns; ++c) {
        if (c < ns) k += 16;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          __builtin_amdgcn_sched_barrier(0);
          mul(av, bv, h);
          __builtin_amdgcn_sched_barrier(0);
          fa.load(k, h, av);
          fb.load(k, h, bv);
        }
      }
    }
  }
  for (int c = ns * KS; c < n; ++c) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      fa.load(kbeg + 16L * c, h, av);
      fb.load(kbeg + 16L * c, h, bv);
    }
    mul(av, bv, 0);
    mul(av, bv, 1);
  }
  if (kend > kbeg + 16L * n) {
    // zeros beyond K leave the sums as they are
    fa.load_tail(kbeg + 16L * n, kend, lane, av);
    fb.load_tail(kbeg + 16L * n, kend, lane, bv);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i][s], bv[j][s], acc[i][j], 0, 0, 0);
  }

  // accumulator entry r of lane l: row l / 16 + 4 r, column l % 16
  const long cbase = b * p.sC + (long)ks * p.sCk;
  const bool had_on = p.had != nullptr;
  long coff[TN], hcol[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const long col = n0 + j * 16 + (lane & 15);
    coff[j] = gemm_col_part(p, col);
    hcol[j] = had_on ? gemm_had_col(p, col) : 0;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const long row = m0 + i * 16 + (lane >> 4) + 4 * r;
      if (row >= M) continue;
      const long ro = cbase + gemm_row_part(p, row);
      const long hr = had_on ? gemm_had_row(p, row) : 0;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const long col = n0 + j * 16 + (lane & 15);
        if (col < N) store_f64(p, ro + coff[j], p.alpha * (had_on ? p.had[hr + hcol[j]] : 1.0) * acc[i][j][r]);
      }
    }
}

template <int TM, int TN, int WM, int WN, int KS>
static void launch_f64(const GemmArgs& p, hipStream_t st) {
  dim3 grid(ceil_div(p.N, 16L * TN * WN), ceil_div(p.M, 16L * TM * WM), p.batch * p.ksplit);
  const dim3 blk(64 * WM * WN);
  if (!p.a_trans && !p.b_trans)
    hipLaunchKernelGGL((gemm_f64_kernel<TM, TN, WM, WN, KS, false, false>), grid, blk, 0, st, p);
  else if (p.a_trans && !p.b_trans)
    hipLaunchKernelGGL((gemm_f64_kernel<TM, TN, WM, WN, KS, true, false>), grid, blk, 0, st, p);
  else if (!p.a_trans && p.b_trans)
    hipLaunchKernelGGL((gemm_f64_kernel<TM, TN, WM, WN, KS, false, true>), grid, blk, 0, st, p);
  else
    hipLaunchKernelGGL((gemm_f64_kernel<TM, TN, WM, WN, KS, true, true>), grid, blk, 0, st, p);
}

struct F64Tile {
  int tm, tn, wm, wn, ks;
  void (*launch)(const GemmArgs&, hipStream_t);
};
#define F64_TILE(tm, tn, wm, wn, ks) {tm, tn, wm, wn, ks, launch_f64<tm, tn, wm, wn, ks>}
static const F64Tile f64_tiles[] = {
    F64_TILE(4, 4, 2, 2, 1), F64_TILE(2, 2, 2, 2, 1), F64_TILE(5, 3, 1, 1, 1), F64_TILE(4, 3, 1, 1, 1),
    F64_TILE(3, 3, 1, 1, 1), F64_TILE(2, 5, 1, 1, 1), F64_TILE(2, 3, 1, 1, 1), F64_TILE(2, 2, 1, 1, 2),
    F64_TILE(1, 4, 1, 1, 2), F64_TILE(1, 2, 1, 1, 4), F64_TILE(1, 1, 1, 1, 4), F64_TILE(1, 1, 1, 1, 6),
    F64_TILE(1, 4, 1, 4, 1), F64_TILE(2, 4, 1, 4, 1), F64_TILE(3, 4, 1, 4, 1)};

// Tile rule: the tile with the least estimated time, in cycles of the busiest SIMD.  A
// chunk costs the larger of its MFMAs (256 cycles per 16 x 16 tile) and its operands
// (2 KiB per tile row or column at the ~18 bytes per cycle and CU that L1 and L2 deliver
// to four waves); the waves of a SIMD (1024 SIMDs) share it, and a SIMD with few waves
// waits for memory between buffers; filling and draining a wave is a fixed part.  The
// constants are a fit to 89 products (20 x 20 x 42 up to 4992 x 4992 x 1248 x 2, Gram
// products of 1.6e6-long vectors) timed with every tile: the rule's choice takes 2.0%
// longer than the best of these tiles on average.
static double f64_cost(const F64Tile& t, const GemmArgs& p) {
  if (ceil_div(p.M, 16L * t.tm * t.wm) > 65535) return INFINITY;   // grid limit
  const double groups = (double)ceil_div(p.M, 16L * t.tm * t.wm) * ceil_div(p.N, 16L * t.tn * t.wn) *
                        ((double)p.batch * p.ksplit);
  const int chunks = ceil_div(p.kchunk < p.K ? p.kchunk : p.K, 16);
  const double mfma = 256.0 * t.tm * t.tn, operand = 447.0 * (t.tm + t.tn);
  const bool two = t.ks > 1 || (16 * (t.tm + t.tn) + 8 * t.tm * t.tn <= 208 && t.wn != 4);
  double w = (mfma > operand ? mfma : operand) + 133.0;
  // a split product streams its K-contiguous operands from HBM, where refilling half
  // chunks (64 bytes of a row at a time) costs more: 400 x 39 over 1557504, 1.61 ms with
  // the 80 x 48 tile, 1.43 ms with the 64 x 48 one
  if (p.ksplit > 1 && !two && !p.a_trans) w *= 1.28;
  const int regs = (two ? 16 : 8) * t.ks * (t.tm + t.tn) + 8 * t.tm * t.tn + 40;
  const double occ = 512 / regs < 8 ? 512 / regs : 8;
  double r = groups * (t.wm * t.wn) / 1024.0;             // waves per SIMD
  if (r < 14.0) r = ceil(r);
  const double o = r < occ ? r : occ, wait = r / o * (w + 226.0 / t.ks);
  return (r * w > wait ? r * w : wait) * chunks + (2023.0 + 484.0 * t.tm * t.tn) * (r > o ? r / o : 1.0) +
         (t.wm * t.wn > 1 ? 50.0 : 0.0);
}

int gemm_f64_launch(const GemmArgs& p, hipStream_t st, int* big) {
  const int nt = (int)(sizeof(f64_tiles) / sizeof(f64_tiles[0]));
  int best = 0;
  if (p.tile != 128) {
    double c = f64_cost(f64_tiles[0], p);
    for (int i = 1; i < nt; ++i) {
      const double ci = f64_cost(f64_tiles[i], p);
      if (ci < c) { c = ci; best = i; }
    }
  }
  f64_tiles[best].launch(p, st);
  *big = best == 0;
  DFTB_CHECK_LAUNCH();
  return DFTB_OK;
}
