// Persistent ensemble solver: many molecules of uneven size, one launch.
//
// One workgroup per molecule (with helpers, below) runs the complete non-Hermitian Davidson loop of
// DFTB/Solver.py:637-917 for one molecule on the device (no host round trip
// per iteration): MFMA matvecs on the molecule's own charges, subspace
// matrices, Newton-Schulz sqrtm(Mm), the lowest-root eigensolver, residuals,
// the Solver.py selection rule for new vectors, preconditioning and CGS2 +
// Cholesky-QR orthonormalisation.  The host orders molecules largest first so
// the big ones start first.  Everything is FP64 except the exchange
// contractions in precision 1 (FP32 operands and intermediates, FP32
// accumulation), which read FP32 copies of the charges.
#include "common.h"
#include "blockops.h"
#include "../../include/dftbaby_amd.h"

#define ENS_THREADS 512
#define ENS_MAXL 1024   // largest subspace (LDS scratch of the eigensolver)
#define ENS_EIG_LDS 120  // rows of the eigensolver's matrix in LDS (with the other buffers 154 of 160 KB)
#define ENS_MAXK 32     // largest number of states
#define ENS_BLOCKS 8    // most blocks per molecule
#define ENS_GRID 192    // most blocks of a launch with helpers

// --------------------------------------------------------------------------
// block-level MFMA GEMM on global operands
//   C = alpha op(A) op(B) + beta C; optional column remap of the output:
//   col -> (col / cdiv) * cstr + row * ldc + col % cdiv.
// The eight waves deal out tiles of TM x TN 16 x 16 blocks; a wave loads its operand
// fragments straight into registers, KS chunks of 16 k ahead of the MFMAs (two buffers).
// Every result is one chain over ascending k (an MFMA adds its four k in lane-group order),
// so the tile shape does not show in the results.  One CU sustains 614 GFLOP/s in FP32 and
// 307 in FP64; latency of the loads bounds these products.  With 32 x 32 tiles loaded and
// multiplied in turn the block products of a C22H24 member (FP32 exchange, 17 iterations) took
// 188 ms of one block and its Newton-Schulz products 91 ms; with these tiles 127 and 82 ms.
// --------------------------------------------------------------------------
typedef double ens_d2 __attribute__((ext_vector_type(2), aligned(8)));
typedef float ens_f2 __attribute__((ext_vector_type(2), aligned(4)));
template <typename T> struct EnsVec;
template <> struct EnsVec<double> { typedef ens_d2 pair; typedef d4_t acc; };
template <> struct EnsVec<float> { typedef ens_f2 pair; typedef f4_t acc; };

__device__ __forceinline__ void ens_swap16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap((unsigned)__float_as_uint(a), (unsigned)__float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void ens_swap16(double& a, double& b) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
  a = __hiloint2double((int)hi[0], (int)lo[0]);
  b = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ d4_t ens_mfma(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t ens_mfma(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// N 16-row fragments of one operand over KS chunks.  KC: K contiguous (x[row * ld + k]), loaded as
// pairs that one lane swap brings to k = 16 c + 4 s + lane / 16; otherwise x[k * ld + row].
// Rows beyond the operand repeat the last one (their results are not stored).
template <typename T, int N, int KS, bool KC>
struct EnsFrag {
  const T* ptr[N];
  long ld;
  __device__ __forceinline__ void init(const T* x, long ld_, int r0, int rows, int lane) {
    ld = ld_;
    const int g = lane >> 4, k = KC ? 2 * (((g & 1) << 1) | (g >> 1)) : g;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      int r = r0 + 16 * i + (lane & 15);
      if (r >= rows) r = rows - 1;
      ptr[i] = KC ? x + r * ld + k : x + k * ld + r;
    }
  }
  __device__ __forceinline__ void load(long k0, T (&v)[N][4 * KS]) const {
#pragma unroll
    for (int h = 0; h < 2 * KS; ++h)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if constexpr (KC) {
          const auto x = *(const typename EnsVec<T>::pair*)(ptr[i] + k0 + 8 * h);
          v[i][2 * h] = x.x;
          v[i][2 * h + 1] = x.y;
        } else {
          const T* q = ptr[i] + (k0 + 8 * h) * ld;
          v[i][2 * h] = q[0];
          v[i][2 * h + 1] = q[4 * ld];
        }
      }
  }
  __device__ __forceinline__ void order(T (&v)[N][4 * KS]) const {
    if constexpr (KC) {
#pragma unroll
      for (int h = 0; h < 2 * KS; ++h)
#pragma unroll
        for (int i = 0; i < N; ++i) ens_swap16(v[i][2 * h], v[i][2 * h + 1]);
    }
  }
  // one chunk at k0 with zeros from kend on, in MFMA order
  __device__ __forceinline__ void load_chunk(int k0, int kend, int lane, T (&v)[N][4 * KS]) const {
    const int g = lane >> 4, kp = KC ? 2 * (((g & 1) << 1) | (g >> 1)) : g;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = k0 + 4 * s + g;
        v[i][s] = k < kend ? (KC ? ptr[i][k - kp] : ptr[i][(k - kp) * ld]) : (T)0;
      }
  }
};

template <typename T, typename TC, int TM, int TN, int KS, bool AT, bool BT>
__device__ __forceinline__ void bgemm_tiles(int M, int N, int K, const T* __restrict__ A, long lda,
                                            const T* __restrict__ B, long ldb, TC* __restrict__ C, long ldc,
                                            double alpha, double beta, long cdiv, long cstr, int t0, int t1) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int tn = (N + 16 * TN - 1) / (16 * TN);
  constexpr bool F64 = sizeof(T) == 8;
  const int ns = K / (16 * KS);
  for (int t = t0 + wv; t < t1; t += nw) {
    const int m0 = (t / tn) * 16 * TM, n0 = (t % tn) * 16 * TN;
    EnsFrag<T, TM, KS, !AT> fa;
    EnsFrag<T, TN, KS, BT> fb;
    fa.init(A, lda, m0, M, lane);
    fb.init(B, ldb, n0, N, lane);
    typename EnsVec<T>::acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (typename EnsVec<T>::acc)((T)0);
    auto mul = [&](T (&a)[TM][4 * KS], T (&b)[TN][4 * KS], int steps) {
#pragma unroll
      for (int s = 0; s < 4 * KS; ++s)
        if (s < steps)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = ens_mfma(a[i][s], b[j][s], acc[i][j]);
    };
    T av[TM][4 * KS], bv[TN][4 * KS];
    if (ns > 0) {
      // two buffers; the odd one goes first, and the last prefetch repeats the last chunks
      T aw[TM][4 * KS], bw[TN][4 * KS];
      long k = 0;
      fa.load(k, av);
      fb.load(k, bv);
      if (ns & 1) {
        fa.order(av);
        fb.order(bv);
        mul(av, bv, 4 * KS);
        if (ns > 1) k += 16 * KS;
        fa.load(k, av);
        fb.load(k, bv);
      }
      for (int c = ns & 1; c < ns; c += 2) {
        k += 16 * KS;
        fa.load(k, aw);
        fb.load(k, bw);
        __builtin_amdgcn_sched_barrier(0);
        fa.order(av);
        fb.order(bv);
        mul(av, bv, 4 * KS);
        __builtin_amdgcn_sched_barrier(0);
        if (c + 2 < ns) k += 16 * KS;
        fa.load(k, av);
        fb.load(k, bv);
        __builtin_amdgcn_sched_barrier(0);
        fa.order(aw);
        fb.order(bw);
        mul(aw, bw, 4 * KS);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    for (int k = ns * 16 * KS; k < K; k += 16) {
      fa.load_chunk(k, K, lane, av);
      fb.load_chunk(k, K, lane, bv);
      mul(av, bv, 4);
    }
    long coff[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + 16 * j + (lane & 15);
      coff[j] = cdiv > 0 ? (col / (int)cdiv) * cstr + col % (int)cdiv : col;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // v_mfma_f64_16x16x4f64 holds rows (lane/16) + 4r, the f32 form rows 4(lane/16) + r
        const int row = m0 + 16 * i + (F64 ? ((lane >> 4) + 4 * r) : (4 * (lane >> 4) + r));
        if (row < M)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            if (n0 + 16 * j + (lane & 15) < N) {
              const long off = row * ldc + coff[j];
              double v = alpha * (double)acc[i][j][r];
              if (beta != 0.0) v += beta * (double)C[off];
              C[off] = (TC)v;
            }
      }
  }
}

// tiles of an M x N result
__device__ __forceinline__ int bgemm_count(int M, int N, int tm, int tn) {
  return ((M + 16 * tm - 1) / (16 * tm)) * ((N + 16 * tn - 1) / (16 * tn));
}

// tiles of an item where nb blocks share nt of them: few tiles go to as many blocks as there
// are, since the operand loads of a block's waves add up
__device__ __forceinline__ int bgemm_share(int nt, int nb) {
  const int g = (nt + nb - 1) / nb;
  return g < 8 ? g : 8;
}

// cycles of the product over the eight waves (two per SIMD) of nb blocks with TM x TN tiles:
// MFMA time of a SIMD, operands at about 40 bytes per cycle and CU, or memory latency per buffer
__device__ __forceinline__ float bgemm_cost(int M, int N, int K, int tm, int tn, int ks, int esz, int nb) {
  const int nt = bgemm_count(M, N, tm, tn);
  const int act = bgemm_share(nt, nb);
  const float mf = (esz == 8 ? 256.0f : 128.0f) * tm * tn, op = act * (tm + tn) * 256.0f * esz / 40.0f;
  float w = (act > 4 ? 2.0f : 1.0f) * mf;
  w = fmaxf(w, fmaxf(op, mf + 500.0f / ks));
  return ((nt + act * nb - 1) / (act * nb)) * (((K + 15) / 16) * w + 1500.0f + 60.0f * tm * tn);
}

// The cheapest tile over nb blocks (0: 16 x 16, 1: 16 x 32, 2: 32 x 32, 3: 32 x 64), its cost and
// how many of them there are.
__device__ __forceinline__ int bgemm_pick(int M, int N, int K, int esz, int nb, float* cost, int* nt) {
  const int kb = esz == 8 ? 2 : 4;            // chunks per buffer of the 32 x 32 tile
  const float c11 = bgemm_cost(M, N, K, 1, 1, 4, esz, nb), c12 = bgemm_cost(M, N, K, 1, 2, kb, esz, nb);
  const float c22 = bgemm_cost(M, N, K, 2, 2, kb, esz, nb), c24 = bgemm_cost(M, N, K, 2, 4, kb / 2, esz, nb);
  const float best = fminf(fminf(c11, c12), fminf(c22, c24));
  const int tile = best == c24 ? 3 : best == c22 ? 2 : best == c12 ? 1 : 0;
  *cost = best;
  *nt = bgemm_count(M, N, tile < 2 ? 1 : 2, tile == 0 ? 1 : tile == 3 ? 4 : 2);
  return tile;
}

// tiles t0 <= t < t1 of the product
template <typename T, typename TC, bool AT, bool BT>
__device__ __noinline__ void bgemm_t(int M, int N, int K, const T* __restrict__ A, long lda, const T* __restrict__ B,
                                     long ldb, TC* __restrict__ C, long ldc, double alpha, double beta, long cdiv,
                                     long cstr, int tile, int t0, int t1) {
  constexpr int KB = sizeof(T) == 8 ? 2 : 4;
  if (tile == 3)
    bgemm_tiles<T, TC, 2, 4, KB / 2, AT, BT>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, t0, t1);
  else if (tile == 2)
    bgemm_tiles<T, TC, 2, 2, KB, AT, BT>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, t0, t1);
  else if (tile == 1)
    bgemm_tiles<T, TC, 1, 2, KB, AT, BT>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, t0, t1);
  else
    bgemm_tiles<T, TC, 1, 1, 4, AT, BT>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, t0, t1);
}

// the three operand orders in use
template <typename T, typename TC>
__device__ __forceinline__ void bgemm_range(int M, int N, int K, const T* A, long lda, int at, const T* B, long ldb,
                                            int bt, TC* C, long ldc, double alpha, double beta, long cdiv, long cstr,
                                            int tile, int t0, int t1) {
  if (at)
    bgemm_t<T, TC, true, false>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, tile, t0, t1);
  else if (bt)
    bgemm_t<T, TC, false, true>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, tile, t0, t1);
  else
    bgemm_t<T, TC, false, false>(M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, cdiv, cstr, tile, t0, t1);
}

// by this block alone
template <typename T, typename TC>
__device__ __forceinline__ void bgemm(int M, int N, int K, const T* A, long lda, int at, const T* B, long ldb, int bt,
                                      TC* C, long ldc, double alpha, double beta, long cdiv, long cstr) {
  float cost;
  int nt;
  const int tile = bgemm_pick(M, N, K, sizeof(T), 1, &cost, &nt);
  bgemm_range<T, TC>(M, N, K, A, lda, at, B, ldb, bt, C, ldc, alpha, beta, cdiv, cstr, tile, 0, nt);
  __syncthreads();
}

// --------------------------------------------------------------------------
// Work shared between the blocks of a molecule.
// One block, the leader, runs the molecule's loop.  The large products and the exchange of a
// block of vectors are cut into items that its helpers (further blocks of the launch) take
// along with the leader, by tickets; the items are the same whoever takes them.  Nothing waits
// for a block that may not be running: the leader takes every item that no helper has taken and
// then waits only for items that running helpers hold; a helper whose leader has not started
// within 0.2 ms ends, and the others end when the leader says so.
// 24 members on one block each leave nine tenths of the chip idle: with up to eight blocks each
// 24 polyenes C8-C22 (8 states, FP32 exchange) take 131 ms instead of 326; of a C22H24 member's
// time the block products fell from 127 to 19 ms, the matrix square roots from 82 to 33.
// --------------------------------------------------------------------------
#define ENS_ITEM_BITS 24
#define ENS_STARTED (1ull << 62)
#define ENS_QUIT (1ull << 63)

struct EnsProduct {                        // C = alpha op(A) op(B) + beta C
  int M, N, K, at, bt;
  const double* A;
  long lda;
  const double* B;
  long ldb;
  double* C;
  long ldc;
  double alpha, beta;
  int tile, nt, share, end;                // tile shape, tiles, tiles per item, items up to here
};

#define ENS_PRODUCTS 4
struct EnsTask {
  int np;                                  // products; 0: the exchange of a block of vectors
  EnsProduct p[ENS_PRODUCTS];
  const double* V;
  double *outP, *outM;
};

struct EnsCtl {
  unsigned long long word;                 // flags, items of the current section, next item
  char pad0[120];
  unsigned long long done;                 // items finished by helpers since the launch began
  char pad1[120];
  unsigned long long here;                 // helpers that have started
  char pad2[120];
  EnsTask task;
};

struct EnsShare {                          // the leader's view
  EnsCtl* ctl;
  int nb;                                  // blocks at work on this molecule when last counted
  int cap;                                 // most of them
  int* s_item;                             // LDS
  unsigned long long done;                 // items that helpers have finished so far
};

__device__ __forceinline__ unsigned long long ens_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Every wave's stores have reached the L2 before the block goes on.  A barrier alone waits for LDS
// (within a CU stores stay in order), and a release by one thread for the stores of its own wave:
// another wave's could still be on their way when that thread writes the L2 back, and a block on
// another XCD would read what was there before.
__device__ __forceinline__ void ens_stores_done() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// One thread, after ens_stores_done(): the L2 is written back, and that has ended, before the word
// that hands the stores over.
__device__ __forceinline__ void ens_release() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// One thread, after reading such a word and before a barrier: L1 and L2 have dropped what is
// stale when the block's other waves read.
__device__ __forceinline__ void ens_acquire() {
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Counts the helpers: where none run (other work holds the CUs), products stay in one piece.
__device__ __forceinline__ void ens_count(EnsShare& sh) {
  if (sh.nb >= sh.cap) return;
  if (threadIdx.x == 0) *sh.s_item = (int)ens_load(&sh.ctl->here);
  __syncthreads();
  const int nb = 1 + *sh.s_item;
  __syncthreads();
  sh.nb = nb < sh.cap ? nb : sh.cap;
}

// next item of the current section, or -1
template <bool HELPER>
__device__ __forceinline__ int ens_take(EnsCtl* ctl, int* s_item) {
  if (threadIdx.x == 0) {
    const unsigned long long old =
        __hip_atomic_fetch_add(&ctl->word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long mask = (1ull << ENS_ITEM_BITS) - 1, idx = old & mask;
    *s_item = (old & ENS_QUIT) || idx >= ((old >> ENS_ITEM_BITS) & mask) ? -1 : (int)idx;
    if (HELPER) ens_acquire();
  }
  __syncthreads();
  const int item = *s_item;
  __syncthreads();
  return item;
}

template <typename F>
__device__ __forceinline__ void ens_section(EnsShare& sh, int items, F&& run) {
  // thread 0 has written the task
  ens_stores_done();
  if (threadIdx.x == 0) {
    ens_release();
    __hip_atomic_store(&sh.ctl->word, ENS_STARTED | ((unsigned long long)items << ENS_ITEM_BITS), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  int mine = 0;
  for (int i = ens_take<false>(sh.ctl, sh.s_item); i >= 0; i = ens_take<false>(sh.ctl, sh.s_item)) {
    run(i);
    ++mine;
  }
  sh.done += items - mine;
  if (threadIdx.x == 0) {
    while (ens_load(&sh.ctl->done) != sh.done) __builtin_amdgcn_s_sleep(1);
    ens_acquire();
  }
  __syncthreads();
}

// item i of a section of products
__device__ __noinline__ void ens_product_item(const EnsTask* t, int i) {
  int q = 0;
  while (i >= t->p[q].end) ++q;
  const EnsProduct& p = t->p[q];
  const int t0 = (i - (q > 0 ? t->p[q - 1].end : 0)) * p.share;
  bgemm_range<double, double>(p.M, p.N, p.K, p.A, p.lda, p.at, p.B, p.ldb, p.bt, p.C, p.ldc, p.alpha, p.beta, 0, 0,
                              p.tile, t0, t0 + p.share < p.nt ? t0 + p.share : p.nt);
}

// Independent products, by all blocks of the molecule where the estimate for them, with 12000
// cycles for handing a section out and collecting it, is the lower one.
template <int NP>
__device__ __noinline__ void pg(EnsShare& sh, EnsProduct (&p)[NP]) {
  float c1 = 0.0f, cn = 0.0f;
  int items = 0, t1[NP], n1[NP];
  for (int q = 0; q < NP; ++q) {
    float c;
    t1[q] = bgemm_pick(p[q].M, p[q].N, p[q].K, 8, 1, &c, &n1[q]);
    c1 += c;
    p[q].tile = bgemm_pick(p[q].M, p[q].N, p[q].K, 8, sh.nb, &c, &p[q].nt);
    cn += c;
    p[q].share = bgemm_share(p[q].nt, sh.nb);
    items += (p[q].nt + p[q].share - 1) / p[q].share;
    p[q].end = items;
  }
  if (sh.nb > 1 && cn + 12000.0f < c1) {
    EnsTask* t = &sh.ctl->task;
    if (threadIdx.x == 0) {
      t->np = NP;
      for (int q = 0; q < NP; ++q) t->p[q] = p[q];
    }
    ens_section(sh, items, [&](int i) { ens_product_item(t, i); });
  } else {
    for (int q = 0; q < NP; ++q)
      bgemm_range<double, double>(p[q].M, p[q].N, p[q].K, p[q].A, p[q].lda, p[q].at, p[q].B, p[q].ldb, p[q].bt,
                                  p[q].C, p[q].ldc, p[q].alpha, p[q].beta, 0, 0, t1[q], 0, n1[q]);
    __syncthreads();
  }
}

__device__ __forceinline__ void pg(EnsShare& sh, int M, int N, int K, const double* A, long lda, int at,
                                   const double* B, long ldb, int bt, double* C, long ldc, double alpha = 1.0,
                                   double beta = 0.0) {
  EnsProduct p[1] = {{M, N, K, at, bt, A, lda, B, ldb, C, ldc, alpha, beta, 0, 0, 0, 0}};
  pg(sh, p);
}

__device__ double bsum(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += sh[i];
  __syncthreads();
  return s;
}

__device__ double bmax(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s = fmax(s, sh[i]);
  __syncthreads();
  return s;
}

// --------------------------------------------------------------------------
// per-molecule workspace layout (host and device agree)
// --------------------------------------------------------------------------
struct EnsLayout {
  size_t TT, X1, X2, tv, gv, Sq, Sinv, H, Y2, Z2, P, Tns, eig, Tbv, Rb, Lb, R, L, PR, ML, W, nrm, w2, G, Li, ref,
      Qt, v32, keep, ctl, tt, total;
  int slots;  // blocks that have an expansion buffer TT
};

__host__ __device__ static long ens_mmax(const EnsMolecule& m) {
  long a = 2L * m.k, b = m.nguess;
  return a > b ? a : b;
}

// nb: blocks per molecule of the launch; only TT, at the end, depends on it
__host__ __device__ static EnsLayout ens_layout(const EnsMolecule& m, int nb) {
  EnsLayout L;
  const long N = (long)m.opad * m.vpad;
  const long rows = m.opad > m.vpad ? m.opad : m.vpad;
  const long mm = ens_mmax(m);
  const long cap = m.cap, k = m.k;
  // one TT per block while they stay within 256 MB
  L.tt = al256((size_t)m.nat * rows * m.vpad * 8);
  const size_t fit = L.tt > 0 ? ((size_t)1 << 28) / L.tt : 1;
  L.slots = fit < 1 ? 1 : fit > (size_t)nb ? nb : (int)fit;
  size_t o = 0;
  size_t* fields[] = {&L.X1, &L.X2, &L.tv, &L.gv, &L.Sq, &L.Sinv, &L.H, &L.Y2, &L.Z2, &L.P, &L.Tns, &L.eig,
                      &L.Tbv, &L.Rb, &L.Lb, &L.R, &L.L, &L.PR, &L.ML, &L.W, &L.nrm, &L.w2, &L.G, &L.Li,
                      &L.ref, &L.Qt, &L.v32, &L.keep, &L.ctl, &L.TT};
  const size_t sizes[] = {(size_t)mm * N * 8, (size_t)mm * N * 8,
                          (size_t)mm * m.nat * 8, (size_t)mm * m.nat * 8, (size_t)cap * cap * 8,
                          (size_t)cap * cap * 8, (size_t)cap * cap * 8, (size_t)cap * cap * 8,
                          (size_t)cap * cap * 8, (size_t)cap * cap * 8, (size_t)cap * cap * 8,
                          eig_layout((int)cap, (int)k).total, (size_t)cap * k * 8, (size_t)cap * k * 8,
                          (size_t)cap * k * 8, (size_t)k * N * 8, (size_t)k * N * 8, (size_t)k * N * 8,
                          (size_t)k * N * 8, (size_t)2 * k * N * 8, (size_t)2 * k * 8, (size_t)k * 8,
                          (size_t)mm * mm * 8, (size_t)mm * mm * 8, (size_t)mm * 8,
                          (size_t)mm * N * 8, (size_t)mm * N * 4, (size_t)mm * 4, sizeof(EnsCtl),
                          L.tt * L.slots};
  for (int i = 0; i < 30; ++i) {
    *fields[i] = o;
    o += al256(sizes[i]);
  }
  L.total = o;
  return L;
}

// Blocks per molecule of a launch of nmol.  Helpers leave a quarter of the chip to other streams.
// From ENS_GRID molecules on the leaders take the chip anyway, and helpers start as members end
// (256 polyenes C8-C40: 2.25 s without helpers, 1.18 so).
static int ens_blocks(int nmol) {
  const int nb = nmol >= ENS_GRID ? ENS_BLOCKS : ENS_GRID / (nmol < 1 ? 1 : nmol);
  return nb < 1 ? 1 : nb > ENS_BLOCKS ? ENS_BLOCKS : nb;
}

extern "C" size_t dftb_ensemble_workspace(const EnsMolecule* m) { return ens_layout(*m, ENS_BLOCKS).total; }

extern "C" size_t dftb_ensemble_workspace_of_launch(const EnsMolecule* m, int nmol) {
  return ens_layout(*m, ens_blocks(nmol)).total;
}

// --------------------------------------------------------------------------
// matvec of m vectors V (FP64, [m][N]) -> outP = (A+B)V, outM = (A-B)V
// --------------------------------------------------------------------------
// vector n: the exchange and the sum, in the buffer TT of the block that does it; outP holds the
// Coulomb part
template <typename T>
__device__ __noinline__ void ens_exchange(const EnsMolecule& Mo, char* ws, const EnsLayout& L, int slot,
                                          const double* Vd, int n, double* outP, double* outM) {
  const long N = (long)Mo.opad * Mo.vpad, nat = Mo.nat, op = Mo.opad, vp = Mo.vpad, o = n * N;
  double* X1 = (double*)(ws + L.X1) + o;
  double* X2 = (double*)(ws + L.X2) + o;
  for (long i = threadIdx.x; i < N; i += blockDim.x) {
    X1[i] = 0.0;
    X2[i] = 0.0;
  }
  const T* v = (const T*)Vd + o;
  if (sizeof(T) == 4) {
    float* v32 = (float*)(ws + L.v32) + o;
    for (long i = threadIdx.x; i < N; i += blockDim.x) v32[i] = (float)Vd[o + i];
    v = (const T*)v32;
  }
  __syncthreads();
  const T* qoo = (const T*)(sizeof(T) == 4 ? Mo.q32[0] : Mo.q_oo);
  const T* qov = (const T*)(sizeof(T) == 4 ? Mo.q32[1] : Mo.q_ov);
  const T* qfov = (const T*)(sizeof(T) == 4 ? Mo.q32[2] : Mo.qf_ov);
  const T* qfvv = (const T*)(sizeof(T) == 4 ? Mo.q32[3] : Mo.qf_vv);
  T* TT = (T*)(ws + L.TT + slot * L.tt);
  // K1 expand: T[A][j][a] = sum_b V[j][b] qf_vv[b][A][a]
  bgemm<T, T>((int)op, (int)(nat * vp), (int)vp, v, vp, 0, qfvv, nat * vp, 0, TT, vp, 1.0, 0.0, vp, op * vp);
  // K1 contract: X1[i][a] = sum_{A,j} q_oo[i][A][j] T[A][j][a]
  bgemm<T, double>(Mo.nocc, (int)vp, (int)(nat * op), qoo, nat * op, 0, TT, vp, 0, X1, vp, 1.0, 0.0, 0, 0);
  // K2 expand: U[A][b][a] = sum_j V[j][b] qf_ov[j][A][a]
  bgemm<T, T>((int)vp, (int)(nat * vp), Mo.nocc, v, vp, 1, qfov, nat * vp, 0, TT, vp, 1.0, 0.0, vp, vp * vp);
  // K2 contract: X2[i][a] = sum_{A,b} q_ov[i][A][b] U[A][b][a]
  bgemm<T, double>(Mo.nocc, (int)vp, (int)(nat * vp), qov, nat * vp, 0, TT, vp, 0, X2, vp, 1.0, 0.0, 0, 0);
  for (long i = threadIdx.x; i < N; i += blockDim.x) {
    const double ov = Mo.omega[i] * Vd[o + i];
    const double k1 = X1[i], k2 = X2[i];
    outP[o + i] = ov + outP[o + i] - k1 - k2;
    outM[o + i] = ov - k1 + k2;
  }
  __syncthreads();
}

template <typename T>
__device__ void ens_matvec(EnsShare& sh, const EnsMolecule& Mo, char* ws, const EnsLayout& L, const double* Vd, int m,
                           double* outP, double* outM) {
  const long N = (long)Mo.opad * Mo.vpad, nat = Mo.nat;
  double* tv = (double*)(ws + L.tv);
  double* gv = (double*)(ws + L.gv);
  // Coulomb: t = V q_c^T, g = t gamma, outP = 4 g q_c  (FP64)
  pg(sh, m, (int)nat, (int)N, Vd, N, 0, Mo.q_c, N, 1, tv, nat);
  pg(sh, m, (int)nat, (int)nat, tv, nat, 0, Mo.gamma, nat, 0, gv, nat);
  pg(sh, m, (int)N, (int)nat, gv, nat, 0, Mo.q_c, N, 0, outP, N, 4.0, 0.0);
  if (Mo.lc) {
    if (sh.nb > 1 && m > 1) {
      if (threadIdx.x == 0) {
        EnsTask* t = &sh.ctl->task;
        t->np = 0;
        t->V = Vd;
        t->outP = outP;
        t->outM = outM;
      }
      ens_section(sh, m, [&](int n) { ens_exchange<T>(Mo, ws, L, 0, Vd, n, outP, outM); });
    } else {
      for (int n = 0; n < m; ++n) ens_exchange<T>(Mo, ws, L, 0, Vd, n, outP, outM);
    }
    return;
  }
  for (int n = 0; n < m; ++n)
    for (long i = threadIdx.x; i < N; i += blockDim.x) {
      const double ov = Mo.omega[i] * Vd[n * N + i];
      outP[n * N + i] = ov + outP[n * N + i];
      outM[n * N + i] = ov;
    }
  __syncthreads();
}

// helper number slot of a molecule: items until the leader ends
template <typename T>
__device__ void ens_help(const EnsMolecule& Mo, int slot, int nb, int* s_item) {
  char* ws = (char*)Mo.work;
  const EnsLayout L = ens_layout(Mo, nb);
  EnsCtl* ctl = (EnsCtl*)(ws + L.ctl);
  if (slot >= L.slots) return;
  const unsigned long long mask = (1ull << ENS_ITEM_BITS) - 1;
  const unsigned long long t0 = wall_clock64();
  bool counted = false;
  for (;;) {
    if (threadIdx.x == 0) {
      // -1: the leader has ended, or did not start within 0.2 ms (100 MHz clock); 1: an item may be free
      int go = 0;
      while (!go) {
        const unsigned long long w = ens_load(&ctl->word);
        if ((w & ENS_STARTED) && !counted) {
          __hip_atomic_fetch_add(&ctl->here, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          counted = true;
        }
        if ((w & ENS_QUIT) || (!(w & ENS_STARTED) && wall_clock64() - t0 > 20000))
          go = -1;
        else if ((w & mask) < ((w >> ENS_ITEM_BITS) & mask))
          go = 1;
        else
          __builtin_amdgcn_s_sleep(8);
      }
      *s_item = go;
    }
    __syncthreads();
    const int go = *s_item;
    __syncthreads();
    if (go < 0) return;
    const int i = ens_take<true>(ctl, s_item);
    if (i < 0) continue;
    const EnsTask* t = &ctl->task;
    if (t->np == 0)
      ens_exchange<T>(Mo, ws, L, slot, t->V, i, t->outP, t->outM);
    else
      ens_product_item(t, i);
    ens_stores_done();
    if (threadIdx.x == 0) {
      ens_release();
      __hip_atomic_fetch_add(&ctl->done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// S = sqrt(A), Si = its inverse; both end in the buffers passed as S and Si
__device__ int ens_sqrtm(EnsShare& es, const double* A, int l, int ld, double* S, double* Si, double* T, double* P,
                         double* Y2, double* Z2, double* sh) {
  double *const S0 = S, *const Si0 = Si;
  double fro = 0.0;
  for (int i = threadIdx.x; i < l * l; i += blockDim.x) {
    double a = A[(long)((unsigned)i / (unsigned)l) * ld + (unsigned)i % (unsigned)l];
    fro += a * a;
  }
  const double c = fmax(sqrt(bsum(fro, sh)), 1e-300);
  for (int i = threadIdx.x; i < l * l; i += blockDim.x) {
    const int r = (unsigned)i / (unsigned)l, q = i - r * l;
    S[i] = 0.5 * (A[(long)r * ld + q] + A[(long)q * ld + r]) / c;
    Si[i] = (r == q) ? 1.0 : 0.0;
  }
  __syncthreads();
  double err = 1.0;
  int ok = 0;
  for (int it = 0; it < 100; ++it) {
    pg(es, l, l, l, Si, l, 0, S, l, 0, P, l);
    double m = 0.0;
    for (int i = threadIdx.x; i < l * l; i += blockDim.x) {
      const int r = (unsigned)i / (unsigned)l, q = i - r * l;
      double id = (r == q) ? 1.0 : 0.0;
      m = fmax(m, fabs(P[i] - id));
      T[i] = 0.5 * (3.0 * id - P[i]);
    }
    err = bmax(m, sh);
    if (!(err == err) || err > 1e6) break;
    if (err < 1e-14 * (l > 16 ? l : 16)) {
      ok = 1;
      break;
    }
    EnsProduct yz[2] = {{l, l, l, 0, 0, S, l, T, l, Y2, l, 1.0, 0.0}, {l, l, l, 0, 0, T, l, Si, l, Z2, l, 1.0, 0.0}};
    pg(es, yz);
    double* x = S;
    S = Y2;
    Y2 = x;
    x = Si;
    Si = Z2;
    Z2 = x;
  }
  if (!ok && err < 1e-10) ok = 1;
  const double f = sqrt(c);
  for (int i = threadIdx.x; i < l * l; i += blockDim.x) {
    S0[i] = S[i] * f;
    Si0[i] = Si[i] / f;
  }
  __syncthreads();
  return ok ? 0 : 1;
}

// --------------------------------------------------------------------------
// orthonormalise rows Q[0..m) (N) against B[0..l) and among themselves;
// dependent rows dropped (compacted); returns the number kept
// --------------------------------------------------------------------------
__device__ int ens_orthonormalize(EnsShare& es, const double* B, int l, double* Q, int m, long N, double tol, double* Cc, double* G,
                                  double* Lc, double* Li, double* ref, double* Qt, int* keep, double* sh) {
  for (int t = 0; t < m; ++t) {
    double s = 0.0;
    for (long i = threadIdx.x; i < N; i += blockDim.x) s += Q[(long)t * N + i] * Q[(long)t * N + i];
    s = bsum(s, sh);
    if (threadIdx.x == 0) {
      ref[t] = sqrt(s);
      keep[t] = 1;
    }
  }
  __syncthreads();
  for (int pass = 0; pass < 2 && l > 0; ++pass) {
    pg(es, l, m, (int)N, B, N, 0, Q, N, 1, Cc, m);            // Cc[p][t] = <B_p, Q_t>
    pg(es, m, (int)N, l, Cc, m, 1, B, N, 0, Q, N, -1.0, 1.0);  // Q -= Cc^T B
  }
  for (int pass = 0; pass < 2; ++pass) {
    pg(es, m, m, (int)N, Q, N, 0, Q, N, 1, G, m);
    // column by column, one row per thread (the factor's rows packed in LDS); then the inverse,
    // one column per thread
    for (int i = threadIdx.x; i < m * (m + 1) / 2; i += blockDim.x) Lc[i] = 0.0;
    for (int i = threadIdx.x; i < m * m; i += blockDim.x) Li[i] = 0.0;
    __syncthreads();
    for (int j = 0; j < m; ++j) {
      const double* Lj = Lc + j * (j + 1) / 2;
      if (threadIdx.x == 0) {
        double d = G[j * m + j];
        for (int q = 0; q < j; ++q) d -= Lj[q] * Lj[q];
        const double r = pass == 0 ? ref[j] * ref[j] : 1.0;
        const double t2 = pass == 0 ? tol * tol : 1e-24;
        const int ok = keep[j] && d > t2 * r && d > 1e-12 * G[j * m + j] && d > 0.0;
        keep[j] = ok;
        Lc[j * (j + 1) / 2 + j] = ok ? sqrt(d) : 1.0;
      }
      __syncthreads();
      if (keep[j])
        for (int i = j + 1 + threadIdx.x; i < m; i += blockDim.x) {
          double* Lr = Lc + i * (i + 1) / 2;
          double s = G[i * m + j];
          for (int q = 0; q < j; ++q) s -= Lr[q] * Lj[q];
          Lr[j] = s / Lj[j];
        }
      __syncthreads();
    }
    for (int c = threadIdx.x; c < m; c += blockDim.x)
      for (int i = c; i < m; ++i) {
        const double* Lr = Lc + i * (i + 1) / 2;
        double s = (i == c) ? 1.0 : 0.0;
        for (int q = c; q < i; ++q) s -= Lr[q] * Li[q * m + c];
        Li[i * m + c] = s / Lr[i];
      }
    __syncthreads();
    for (int i = threadIdx.x; i < m * m; i += blockDim.x)
      if (!keep[i / m]) Li[i] = 0.0;
    __syncthreads();
    pg(es, m, (int)N, m, Li, m, 0, Q, N, 0, Qt, N);
    for (long i = threadIdx.x; i < (long)m * N; i += blockDim.x) Q[i] = Qt[i];
    __syncthreads();
  }
  // compact kept rows to the front
  int kept = 0;
  for (int t = 0; t < m; ++t) {
    if (keep[t]) {
      if (kept != t)
        for (long i = threadIdx.x; i < N; i += blockDim.x) Q[(long)kept * N + i] = Q[(long)t * N + i];
      __syncthreads();
      ++kept;
    }
  }
  return kept;
}

// --------------------------------------------------------------------------
// the per-molecule Davidson
// --------------------------------------------------------------------------
template <typename T>
__device__ void ens_davidson(const EnsMolecule& Mo, double conv, int maxiter, double* sh, double* sv, double* sp,
                             double* bnd, int* s_sel, double* stg, double* wl, int nb) {
  char* ws = (char*)Mo.work;
  const EnsLayout L = ens_layout(Mo, nb);
  EnsShare es = {(EnsCtl*)(ws + L.ctl), 1, L.slots, s_sel + 2 * ENS_MAXK + 1, 0};
  if (threadIdx.x == 0)
    __hip_atomic_store(&es.ctl->word, ENS_STARTED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // hands nothing over
  const long N = (long)Mo.opad * Mo.vpad;
  const int k = Mo.k, cap = Mo.cap;
  const long kmax = (long)Mo.nocc * Mo.nvirt;
  double* bs = Mo.bs;
  double* bp = Mo.bp;
  double* bm = Mo.bm;
  double* Mp = Mo.Mp;
  double* Mm = Mo.Mm;
  double* Sq = (double*)(ws + L.Sq);
  double* Sinv = (double*)(ws + L.Sinv);
  double* H = (double*)(ws + L.H);
  double* Tb = (double*)(ws + L.Tbv);
  double* Rb = (double*)(ws + L.Rb);
  double* Lb = (double*)(ws + L.Lb);
  double* R = (double*)(ws + L.R);
  double* Lv = (double*)(ws + L.L);
  double* PR = (double*)(ws + L.PR);
  double* ML = (double*)(ws + L.ML);
  double* W = (double*)(ws + L.W);
  double* nrm = (double*)(ws + L.nrm);
  double* w2 = (double*)(ws + L.w2);
  double* w = Mo.w;
  int* status = Mo.status;
  // initial guess: unit vectors at the host-sorted lowest-omega indices
  int l = Mo.nguess;
  for (long i = threadIdx.x; i < (long)l * N; i += blockDim.x) bs[i] = 0.0;
  __syncthreads();
  for (int t = threadIdx.x; t < l; t += blockDim.x) bs[(long)t * N + Mo.guess[t]] = 1.0;
  __syncthreads();
  int new0 = 0;
  int code = 0, it = 0;
  for (it = 0; it < maxiter; ++it) {
    const int m = l - new0;
    ens_count(es);
    if (m > 0) {
      ens_matvec<T>(es, Mo, ws, L, bs + (long)new0 * N, m, bp + (long)new0 * N, bm + (long)new0 * N);
      // new columns/rows of M+- = bs^T (A+-B) bs
      const double* bn = bs + (long)new0 * N;
      EnsProduct cols[2] = {{l, m, (int)N, 0, 1, bs, N, bp + (long)new0 * N, N, Mp + new0, cap, 1.0, 0.0},
                            {l, m, (int)N, 0, 1, bs, N, bm + (long)new0 * N, N, Mm + new0, cap, 1.0, 0.0}};
      if (new0 > 0) {
        EnsProduct all[4] = {cols[0], cols[1],
                             {m, new0, (int)N, 0, 1, bn, N, bp, N, Mp + (long)new0 * cap, cap, 1.0, 0.0},
                             {m, new0, (int)N, 0, 1, bn, N, bm, N, Mm + (long)new0 * cap, cap, 1.0, 0.0}};
        pg(es, all);
      } else {
        pg(es, cols);
      }
    }
    if (sizeof(T) == 4) {
      // FP32 products: use the symmetric parts of M+-
      for (int i = threadIdx.x; i < l * l; i += blockDim.x) {
        const int r = (unsigned)i / (unsigned)l, c = i - r * l;
        if (c > r) {
          double a = 0.5 * (Mp[(long)r * cap + c] + Mp[(long)c * cap + r]);
          Mp[(long)r * cap + c] = a;
          Mp[(long)c * cap + r] = a;
          double b = 0.5 * (Mm[(long)r * cap + c] + Mm[(long)c * cap + r]);
          Mm[(long)r * cap + c] = b;
          Mm[(long)c * cap + r] = b;
        }
      }
      __syncthreads();
    }
    ens_count(es);
    // subspace step (Solver.py:759-798)
    if (ens_sqrtm(es, Mm, l, cap, Sq, Sinv, (double*)(ws + L.Tns), (double*)(ws + L.P), (double*)(ws + L.Y2),
                  (double*)(ws + L.Z2), sh)) {
      code = -3;
      break;
    }
    pg(es, l, l, l, Mp, cap, 0, Sq, l, 0, (double*)(ws + L.P), l);
    pg(es, l, l, l, Sq, l, 0, (double*)(ws + L.P), l, 0, H, l);
    double he = 0.0;
    for (int i = threadIdx.x; i < l * l; i += blockDim.x) {
      const int r = (unsigned)i / (unsigned)l, c = i - r * l;
      he += fabs(H[(long)r * l + c] - H[(long)c * l + r]);
    }
    he = bsum(he, sh);
    if (sizeof(T) == 8 && he > 1.0e-10) {
      code = -4;
      break;
    }
    const int nev = k < l ? k : l;
    syevx_block(H, l, l, nev, w2, Tb, ws + L.eig, sv, sp, sh, bnd, ENS_MAXL, stg, wl, ENS_EIG_LDS);
    __syncthreads();
    int bad = 0;
    for (int n = threadIdx.x; n < nev; n += blockDim.x)
      if (!(w2[n] > 0.0)) bad = 1;
    if (bsum((double)bad, sh) > 0.0) {
      code = -3;
      break;
    }
    for (int n = threadIdx.x; n < nev; n += blockDim.x) w[n] = sqrt(w2[n]);
    __syncthreads();
    pg(es, l, nev, l, Sq, l, 0, Tb, nev, 0, Rb, nev);
    for (int i = threadIdx.x; i < l * nev; i += blockDim.x) Rb[i] /= sqrt(w[(unsigned)i % (unsigned)nev]);
    __syncthreads();
    pg(es, l, nev, l, Mp, cap, 0, Rb, nev, 0, Lb, nev);
    for (int i = threadIdx.x; i < l * nev; i += blockDim.x) Lb[i] /= w[(unsigned)i % (unsigned)nev];
    __syncthreads();
    // R, L and their products
    EnsProduct ritz[4] = {{nev, (int)N, l, 1, 0, Rb, nev, bs, N, R, N, 1.0, 0.0},
                          {nev, (int)N, l, 1, 0, Lb, nev, bs, N, Lv, N, 1.0, 0.0},
                          {nev, (int)N, l, 1, 0, Rb, nev, bp, N, PR, N, 1.0, 0.0},
                          {nev, (int)N, l, 1, 0, Lb, nev, bm, N, ML, N, 1.0, 0.0}};
    pg(es, ritz);
    // residuals WL = (A+B)R - w L, WR = (A-B)L - w R
    for (int n = 0; n < nev; ++n) {
      double sL = 0.0, sR = 0.0;
      for (long i = threadIdx.x; i < N; i += blockDim.x) {
        double a = PR[(long)n * N + i] - w[n] * Lv[(long)n * N + i];
        double b = ML[(long)n * N + i] - w[n] * R[(long)n * N + i];
        W[(long)n * N + i] = a;
        W[(long)(k + n) * N + i] = b;
        sL += a * a;
        sR += b * b;
      }
      sL = bsum(sL, sh);
      sR = bsum(sR, sh);
      if (threadIdx.x == 0) {
        nrm[n] = sqrt(sL);
        nrm[k + n] = sqrt(sR);
      }
    }
    __syncthreads();
    // convergence and selection (thread 0; Solver.py:837-884)
    if (threadIdx.x == 0) {
      int all = 1;
      for (int n = 0; n < nev; ++n)
        if (!(nrm[n] + nrm[k + n] < conv)) all = 0;
      s_sel[0] = (all && it > 0) ? -1 : 0;
      if (!(all && it > 0)) {
        const long dkmax = (kmax - l < 2 * k) ? kmax - l : 2 * k;
        const double eps = 0.01 * conv;
        int ncL = 0, ncR = 0;
        for (int n = 0; n < nev; ++n) {
          ncL += nrm[n] > eps;
          ncR += nrm[k + n] > eps;
        }
        int dkR = (int)((dkmax + 1) / 2);
        if (dkR > ncL) dkR = ncL;
        int dkL = (int)(dkmax - dkR);
        if (dkL > ncR) dkL = ncR;
        const int dk = dkR + dkL;
        int nb = 0;
        for (int n = 0; n < nev && nb < dk; ++n)
          if (nrm[n] > eps) s_sel[1 + nb++] = n;
        for (int n = 0; n < nev && nb < dk; ++n)
          if (nrm[k + n] > eps) s_sel[1 + nb++] = k + n;
        if (l + nb > cap) nb = -2;
        s_sel[0] = nb;
      }
    }
    __syncthreads();
    const int dk = s_sel[0];
    if (dk == -1) {
      code = 1;
      break;
    }
    if (dk < 0) {
      code = -6;
      break;
    }
    if (dk == 0) {
      new0 = l;
      continue;
    }
    // precondition into bs[l .. l+dk)
    double* Q = bs + (long)l * N;
    for (int t = 0; t < dk; ++t) {
      const int src = s_sel[1 + t];
      const double wt = w[src % k];
      for (long e = threadIdx.x; e < N; e += blockDim.x) {
        const double om = Mo.omega[e];
        double d = wt - om;
        if (fabs(d) < 1.0e-6) d = 1.0e-6 * om;
        Q[t * N + e] = W[(long)src * N + e] / d;
      }
    }
    __syncthreads();
    const int kept = ens_orthonormalize(es, bs, l, Q, dk, N, 1.0e-8, (double*)(ws + L.Sq), (double*)(ws + L.G),
                                        stg, (double*)(ws + L.Li), (double*)(ws + L.ref),
                                        (double*)(ws + L.Qt), (int*)(ws + L.keep), sh);
    new0 = l;
    l += kept;
  }
  // outputs: C = bs Tb, X+Y = R, X-Y = L
  if (code == 1) {
    const int nev = k < l ? k : l;
    pg(es, nev, (int)N, l, Tb, nev, 1, bs, N, 0, Mo.C, N);
    for (long i = threadIdx.x; i < (long)nev * N; i += blockDim.x) {
      Mo.XpY[i] = R[i];
      Mo.XmY[i] = Lv[i];
    }
    for (int n = threadIdx.x; n < nev; n += blockDim.x) Mo.resid[n] = nrm[n] + nrm[k + n];
  }
  if (threadIdx.x == 0) {
    status[0] = it + 1;
    status[1] = code;
    status[2] = l;
    __hip_atomic_store(&es.ctl->word, ENS_STARTED | ENS_QUIT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
}

__global__ __launch_bounds__(ENS_THREADS) void ensemble_kernel(const EnsMolecule* __restrict__ mols, int nmol,
                                                               double conv, int maxiter) {
  __shared__ double sh[ENS_THREADS / 64];
  __shared__ double sv[ENS_MAXL];
  __shared__ double sp[ENS_MAXL];
  __shared__ double bnd[2];
  __shared__ int s_sel[2 + 2 * ENS_MAXK];  // the selection, and the item
  __shared__ double stg[EIG_STAGE_WAVES * EIG_STAGE];
  __shared__ double wl[ENS_EIG_LDS * (ENS_EIG_LDS | 1)];
  const int mi = blockIdx.x % nmol, slot = blockIdx.x / nmol, nb = gridDim.x / nmol;
  const EnsMolecule& Mo = mols[mi];
  if (slot > 0) {
    if (Mo.precision == 1)
      ens_help<float>(Mo, slot, nb, s_sel);
    else
      ens_help<double>(Mo, slot, nb, s_sel);
  } else if (Mo.precision == 1)
    ens_davidson<float>(Mo, conv, maxiter, sh, sv, sp, bnd, s_sel, stg, wl, nb);
  else
    ens_davidson<double>(Mo, conv, maxiter, sh, sv, sp, bnd, s_sel, stg, wl, nb);
}

__global__ void ensemble_begin_kernel(const EnsMolecule* __restrict__ mols, int nmol) {
  const int mi = blockIdx.x * blockDim.x + threadIdx.x;
  if (mi >= nmol) return;
  EnsCtl* ctl = (EnsCtl*)((char*)mols[mi].work + ens_layout(mols[mi], 1).ctl);
  ctl->word = 0;
  ctl->done = 0;
  ctl->here = 0;
}

extern "C" int dftb_ensemble_solve(const EnsMolecule* mols_dev, int nmol, double conv, int maxiter, void* stream) {
  if (!mols_dev || nmol <= 0 || maxiter <= 0) return DFTB_ERR_ARG;
  const int nb = ens_blocks(nmol);         // leaders come first in the grid
  hipLaunchKernelGGL(ensemble_begin_kernel, dim3((nmol + 63) / 64), dim3(64), 0, (hipStream_t)stream, mols_dev, nmol);
  DFTB_CHECK_LAUNCH();
  hipLaunchKernelGGL(ensemble_kernel, dim3(nmol * nb), dim3(ENS_THREADS), 0, (hipStream_t)stream, mols_dev, nmol, conv,
                     maxiter);
  DFTB_CHECK_LAUNCH();
  return DFTB_OK;
}
