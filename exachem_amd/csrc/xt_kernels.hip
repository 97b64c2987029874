// gfx950 kernels of the closed-shell CCSD(T) triples energy.
//
// Work decomposition (shared by the HBM-resident path and the per-task
// packed-buffer drop-in):
//   * a task (h1b,h2b,h3b,p4b,p5b,p6b) is cut into 4x4x4x4x4x4 sub-tiles of
//     the triples tile t3[h1,h2,h3,p4,p5,p6]; one 256-thread workgroup (4
//     wave64) owns one sub-tile at a time and keeps it in LDS (never in HBM);
//   * every d1 and d2 equation of the reference (ccsd_t_all_fused_cpu.hpp:
//     173-270, 331-428) is a GEMM into one of 9 bipartitions of the six
//     t3 indices: M = {single hole hs, particle pair (pA,pB)} and
//     N = {hole pair (hA,hB), single particle ps}.  Each bipartition g is
//     fed by exactly one d1 equation (K = h7) and one d2 equation (K = p7),
//     so the two run back to back into FP64 accumulators held in MFMA
//     registers (v_mfma_f64_16x16x4f64) and the result is added once into the
//     LDS t3 tile.  Up to 64 x 64, cut to the task tile: the 16 x 16 tiles that
//     are needed are dealt to the four waves (wave_share; quadrant in the
//     per-task kernel);
//   * operands are staged through LDS in K-chunks of 16 (aligned 16-byte
//     loads from zero-padded arrays) with a register prefetch of the next chunk;
//     a workgroup holds 53 KB of LDS, so three share a CU;
//   * s1 (ccsd_t_all_fused_cpu.hpp:472-578) and the denominator-weighted
//     energy (586-619) run on the LDS tile; the 256 partials are reduced
//     with wave64 shuffles and a fixed-order cross-wave sum.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstring>
#include <mutex>

#include "xt_device.h"
#include "xt_claim.h"
#include "xt_fixed.h"
#include "xt_queue.h"
#include "xt_tasksums.h"

namespace xt {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

constexpr int NT      = 256;       // threads per workgroup
constexpr int KC      = 16;        // K chunk staged per LDS round
constexpr int LDK     = KC + 2;    // padded row stride (doubles) of staged operands: 144 B, so
                                   // the 16x16 fragment reads (16 rows x 2 k per half-wave) hit
                                   // distinct banks
constexpr int T3N     = 4096;      // 4^6 sub-tile
constexpr int S1_T1   = 9 * 16;    // s1 T1 blocks in LDS
constexpr int STAGE_D = 2 * 64 * LDK;  // staging union: A,B chunks; then the s1 V blocks (9*256)
static_assert(STAGE_D >= 9 * 256, "staging too small for the s1 V blocks");

__device__ __forceinline__ int cdiv(int a, int b) { return (a + b - 1) / b; }
// parity sign of the single index at position x (0,1,2) within its triple:
// (x, others ascending) is even for x=0,2 and odd for x=1.
__device__ __forceinline__ double sgn_single(int x) { return x == 1 ? -1.0 : 1.0; }

__device__ __forceinline__ void pair_of(int s, int& a, int& b) {
  a = (s == 0) ? 1 : 0;
  b = (s == 2) ? 1 : 2;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for(int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Sum of a per-thread value over the workgroup in a fixed order; result valid
// in thread 0.
template<class SM>
__device__ __forceinline__ void block_sum2(SM& sm, double& a, double& b) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  a = wave_sum(a);
  b = wave_sum(b);
  if(lane == 0) {
    sm.red[wave]     = a;
    sm.red[4 + wave] = b;
  }
  __syncthreads();
  if(threadIdx.x == 0) {
    a = ((sm.red[0] + sm.red[1]) + sm.red[2]) + sm.red[3];
    b = ((sm.red[4] + sm.red[5]) + sm.red[6]) + sm.red[7];
  }
}

// A sub-tile at the edge of its task tile has fewer than four orbitals along
// some positions.  Rows (hs, pA, pB) and columns (hA, hB, ps) of a bipartition
// are numbered inside the tile only, first position fastest, so the 16-row and
// 16-column MFMA tiles that are needed shrink with it: over the uneven tiles
// of O=48, V=384 the 4^6 sub-tiles hold 1.79 times the tile's elements, the
// needed MFMA tiles 1.05 times.
__device__ __forceinline__ int small_div(int n, int e) {  // n / e, 0 <= n < 64, 1 <= e <= 4
  return (int) (((float) n + 0.5f) * __builtin_amdgcn_rcpf((float) e));
}
struct Item {
  int a, b, c;  // coordinates along the three positions of a side
};
__device__ __forceinline__ Item item_of(int n, int ea, int eb) {
  Item      x;
  const int t = small_div(n, ea);
  x.a         = n - t * ea;
  x.c         = small_div(t, eb);
  x.b         = t - x.c * eb;
  return x;
}

// The MFMA tiles of one wave: row tiles wm and wm + 2, column tiles wn and
// wn + 2 of the Mt x Nt that are needed; bit 2 i + j of mask is set for the
// needed ones.  Wave w takes quadrant (w + g) % 4, so that over the bipartitions
// every SIMD gets the larger quadrants in turn.
struct Quad {
  int wm, wn, mask;
};
__device__ __forceinline__ Quad quadrant(int g, int rows, int cols) {
  const int w = (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + g) & 3;
  const int mt = (rows + 15) >> 4, nt = (cols + 15) >> 4;
  Quad      q;
  q.wm   = w >> 1;
  q.wn   = w & 1;
  q.mask = 0;
#pragma unroll
  for(int i = 0; i < 2; i++)
#pragma unroll
    for(int j = 0; j < 2; j++)
      if(q.wm + 2 * i < mt && q.wn + 2 * j < nt) q.mask |= 1 << (2 * i + j);
  return q;
}

// Box index part of a row or column (sum_pos idx[pos] << 2*pos, pos 0..2 =
// h1..h3, 3..5 = p4..p6).  Padding ones get an index outside the tile (some
// extent of their side is short wherever there is one).
__device__ __forceinline__ unsigned short box_index(Item x, int e0, int e1, int e2, int q0, int q1, int q2) {
  if(x.c >= e2) {
    x.a = e0 < 4 ? e0 : 0;
    x.b = e0 < 4 ? 0 : e1 < 4 ? e1 : 0;
    x.c = e0 < 4 || e1 < 4 ? 0 : e2 & 3;
  }
  return (unsigned short) ((x.a << (2 * q0)) | (x.b << (2 * q1)) | (x.c << (2 * q2)));
}
// Those of the current bipartition of the per-task kernel, written by 128 threads.
struct Tables {
  unsigned short row[64], col[64];
};
__device__ __forceinline__ void fill_tables(Tables& t, const int* ext, int hs, int hA, int hB, int ps,
                                            int pA, int pB) {
  const int tid = threadIdx.x;
  if(tid >= 128) return;
  const bool row = tid < 64;
  const int  q0 = row ? hs : hA, q1 = row ? 3 + pA : hB, q2 = 3 + (row ? pB : ps);
  const int  e0 = ext[q0], e1 = ext[q1], e2 = ext[q2];
  const unsigned short v = box_index(item_of(tid & 63, e0, e1), e0, e1, e2, q0, q1, q2);
  if(row) t.row[tid] = v;
  else t.col[tid - 64] = v;
}

// c[i][j] += a_i b_j for the tiles of mask.  In assembly because of the
// branches (around builtins the compiler copies the accumulators per path).
// The nops in front cover a vector write of an operand just before; nothing is
// needed between matrix instructions on one accumulator; acc_ready() stands
// before a vector read or write of the accumulators.
__device__ __forceinline__ void mfma_step(int mask, double a0, double a1, double b0, double b1,
                                          v4d (&c)[2][2]) {
  asm volatile(
    "s_nop 1\n\t"
    "s_cmp_eq_u32 %[m], 15\n\t"
    "s_cbranch_scc0 .Lpart_%=\n\t"
    "v_mfma_f64_16x16x4_f64 %[c00], %[a0], %[b0], %[c00]\n\t"
    "v_mfma_f64_16x16x4_f64 %[c01], %[a0], %[b1], %[c01]\n\t"
    "v_mfma_f64_16x16x4_f64 %[c10], %[a1], %[b0], %[c10]\n\t"
    "v_mfma_f64_16x16x4_f64 %[c11], %[a1], %[b1], %[c11]\n\t"
    "s_branch .Ldone_%=\n"
    ".Lpart_%=:\n\t"
    "s_bitcmp1_b32 %[m], 0\n\t"
    "s_cbranch_scc0 .Ldone_%=\n\t"
    "v_mfma_f64_16x16x4_f64 %[c00], %[a0], %[b0], %[c00]\n\t"
    "s_bitcmp1_b32 %[m], 1\n\t"
    "s_cbranch_scc0 .Lrow_%=\n\t"
    "v_mfma_f64_16x16x4_f64 %[c01], %[a0], %[b1], %[c01]\n"
    ".Lrow_%=:\n\t"
    "s_bitcmp1_b32 %[m], 2\n\t"
    "s_cbranch_scc0 .Ldone_%=\n\t"
    "v_mfma_f64_16x16x4_f64 %[c10], %[a1], %[b0], %[c10]\n"
    ".Ldone_%=:\n"
    : [c00] "+v"(c[0][0]), [c01] "+v"(c[0][1]), [c10] "+v"(c[1][0]), [c11] "+v"(c[1][1])
    : [m] "s"(mask), [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1)
    : "scc");
}
__device__ __forceinline__ void acc_ready(v4d (&c)[2][2]) {
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(c[0][0]), "+v"(c[0][1]), "+v"(c[1][0]), "+v"(c[1][1]));
}

// The K step of one staged chunk over the wave's MFMA tiles.
template<int KCT = KC, int LDKT = LDK>
__device__ __forceinline__ void mfma_chunk(const double* __restrict__ As,
                                           const double* __restrict__ Bs, const Quad& q,
                                           v4d (&acc)[2][2], int len = KCT) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for(int kk = 0; kk < KCT / 4; kk++) {
    if(4 * kk >= len) break;
    const int    k  = 4 * kk + lk;
    const double a0 = As[(16 * q.wm + lr) * LDKT + k], a1 = As[(16 * q.wm + 32 + lr) * LDKT + k];
    const double b0 = Bs[(16 * q.wn + lr) * LDKT + k], b1 = Bs[(16 * q.wn + 32 + lr) * LDKT + k];
    mfma_step(q.mask, a0, a1, b0, b1, acc);
  }
}

// Adds the accumulators of a bipartition into the LDS t3 tile; the first one
// of a sub-tile stores instead (every bipartition covers every element of the
// tile).  D layout of v_mfma_f64_16x16x4f64: register r of lane l holds row
// 4*r + (l>>4), column l&15 (the four row groups are interleaved, unlike the
// 16-bit forms).
__device__ __forceinline__ void acc_to_t3(double* t3, const Tables& t, const Quad& q, bool store,
                                          v4d (&acc)[2][2]) {
  const int lane = threadIdx.x & 63;
  acc_ready(acc);
#pragma unroll
  for(int i = 0; i < 2; i++)
#pragma unroll
    for(int j = 0; j < 2; j++) {
      if(!((q.mask >> (2 * i + j)) & 1)) continue;
      const int n = t.col[16 * (q.wn + 2 * j) + (lane & 15)];
#pragma unroll
      for(int r = 0; r < 4; r++) {
        double* p = &t3[t.row[16 * (q.wm + 2 * i) + 4 * r + (lane >> 4)] | n];
        *p        = store ? acc[i][j][r] : *p + acc[i][j][r];
      }
    }
}

// Energy of the finished sub-tile: t3d in LDS, s1 operands staged in LDS (zero
// for slots that are off), denominators from sm.eps, ext the orbitals inside the
// tile.  Returns (E4, E5) partial sums in thread 0.
//   T1s[s][pa][hi] (16 per slot), V1s[s][hk + 4 hj + 16 pc + 64 pb] (256 per slot)
// A thread owns one (h1, h2, h3, p4) and runs over p5 and p6.  Bound by vector
// instructions: what depends on p6 or p5 alone is read once for it (99 reads for
// 16 elements, not 288).
template<class SM>
__device__ __forceinline__ void subtile_energy(SM& sm, const double* T1s, const double* V1s,
                                               const int* ext, double& e4, double& e5) {
  e4 = 0.0;
  e5 = 0.0;
  const int tid = threadIdx.x;
  int       h[3];
#pragma unroll
  for(int p = 0; p < 3; p++) h[p] = (tid >> (2 * p)) & 3;
  const int p4 = tid >> 6;
  const int n5 = __builtin_amdgcn_readfirstlane(ext[4]), n6 = __builtin_amdgcn_readfirstlane(ext[5]);
  if(h[0] < ext[0] && h[1] < ext[1] && h[2] < ext[2] && p4 < ext[3]) {
    // slot 3 pa + hi: T1(p, hi) V1(hj, hk, pb, pc)
    double    t0[3], t2[3][4], v1[3][4];
    const double *T[3], *V[3];
#pragma unroll
    for(int hi = 0; hi < 3; hi++) {
      int hj, hk;
      pair_of(hi, hj, hk);
      T[hi]  = T1s + hi * 16 + h[hi];
      V[hi]  = V1s + hi * 256 + h[hk] + 4 * h[hj];
      t0[hi] = T[hi][4 * p4];
#pragma unroll
      for(int p6 = 0; p6 < 4; p6++) {
        t2[hi][p6] = T[hi][6 * 16 + 4 * p6];
        v1[hi][p6] = V[hi][3 * 256 + 16 * p6 + 64 * p4];
      }
    }
    const double Dh = sm.eps[8 + h[2]] + sm.eps[4 + h[1]] + sm.eps[h[0]], D4 = sm.eps[12 + p4];
#pragma unroll 1
    for(int p5 = 0; p5 < n5; p5++) {
      double t1[3], v2[3];
#pragma unroll
      for(int hi = 0; hi < 3; hi++) {
        t1[hi] = T[hi][3 * 16 + 4 * p5];
        v2[hi] = V[hi][6 * 256 + 16 * p5 + 64 * p4];
      }
#pragma unroll
      for(int p6 = 0; p6 < 4; p6++) {
        if(p6 >= n6) break;
        const double d = sm.t3[tid + NT * (p5 + 4 * p6)];
        double       s = 0.0;
#pragma unroll
        for(int hi = 0; hi < 3; hi++) s += t0[hi] * V[hi][16 * p6 + 64 * p5];
#pragma unroll
        for(int hi = 0; hi < 3; hi++) s += t1[hi] * v1[hi][p6];
#pragma unroll
        for(int hi = 0; hi < 3; hi++) s += t2[hi][p6] * v2[hi];
        // denominator in the reference's order (ccsd_t_all_fused_cpu.hpp:612-614)
        const double D = Dh - sm.eps[20 + p6] - sm.eps[16 + p5] - D4;
        e4 += d * d / D;
        e5 += d * (d + s) / D;
      }
    }
  }
  block_sum2(sm, e4, e5);
}

// Rows and columns of a bipartition: index parts in the 4^6 box (as
// fill_tables), of it and the next one, and the rows of the d1 and d2 operand
// arrays, of the next one.
struct Rows {
  unsigned       r1[128], r2[128];
  unsigned short e[2][128];
};

// LDS of the persistent FP64 kernel, sized for three workgroups per CU.
struct __align__(16) Smem {
  double t3[T3N];
  double stage[STAGE_D];
  union {
    Rows   tab;
    double t1s[S1_T1];  // later: the s1 T1 blocks
  };
  double eps[24];
  double red[8];
  int    start[6], ext[6];  // current sub-tile: first orbitals, orbitals inside the tile
};

// ---------------------------------------------------------------------------
// HBM-resident path: operands are formed on the fly from spatial closed-shell
// tensors (spin-orbital antisymmetrised values of <pq||rs> and T2, exactly the
// numbers the reference's gathers would copy out of TAMM blocks).
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned uni(int x) { return (unsigned) __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  return (uint64_t) (unsigned) __builtin_amdgcn_readfirstlane((int) v) |
         (uint64_t) (unsigned) __builtin_amdgcn_readfirstlane((int) (v >> 32)) << 32;
}

// The MFMA tiles of one wave: row tiles i0 + is * i (i < ni) times column tiles
// j0 + js * j (j < nj) of the mt x nt that are needed, dealt out as evenly as
// four waves allow with at most four operand rows a lane.  Wave w takes the
// share (w + g) % 4, so that over the bipartitions every SIMD gets the larger
// ones in turn.
struct Share {
  int i0, is, ni, j0, js, nj;
};
__device__ __forceinline__ Share wave_share(int g, int rows, int cols) {
  const int w = (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + g) & 3;
  const int mt = (rows + 15) >> 4, nt = (cols + 15) >> 4, wm = w >> 1, wn = w & 1;
  if(mt == 1) return {0, 1, w < nt, w, 1, 1};
  if(nt == 1) return {w, 1, w < mt, 0, 1, 1};
  if(mt == 3 && nt == 3) return w == 0 ? Share{0, 1, 3, 0, 1, 1} : Share{w - 1, 1, 1, 1, 1, 2};
  if(mt == 3 && nt == 4) return {0, 1, 3, w, 1, 1};
  if(mt == 4 && nt == 3) return {w, 1, 1, 0, 1, 3};
  return {wm, 2, wm + 2 < mt ? 2 : 1, wn, 2, wn + 2 < nt ? 2 : 1};
}

// NI x NJ MFMA tiles of one wave over a bipartition's K, n1 units of 8 of d1 and
// n2 of d2, two units a chunk, a last odd one alone, then added into t3 (the
// first bipartition of a sub-tile stores instead: every bipartition covers
// every element of the tile).  refill() writes the chunk in flight to As and Bs
// and has the one after it loaded; refill_whole() does so for a whole chunk with
// at least another whole one of the family to load (left() units, skip() counts
// them off); ahead() runs before the sums are added.  neg1, neg2: signs of the
// families' products.  Every wave passes the same barriers, with NI = NJ = 0 for
// a wave without tiles.
// While an FP64 matrix instruction runs, no vector instruction of any wave
// issues on its SIMD (measured: a wave of additions beside one of matrix
// instructions stood still until that had ended; beside the 16-bit forms it ran
// at 80%), and waves that wait to prepare a chunk wait for the others' products.
// So the inner loop has none: fragments at fixed LDS addresses, a refill from
// scalar bases and fixed vector offsets, signs left to the sums.  With 30 vector
// and 40 scalar instructions a chunk here 12 tasks of O=40, V=300 took 65.8 ms,
// with none and 8 52.8 (FP64 matrix instructions 53% and 66% of the time).
// Operands straight from global memory into the fragments were slower (87 ms:
// neighbouring lanes are different rows, 64 cycles a load).
// Lane (lr, lk) takes k = 2 lk, 2 lk + 1 of each unit: the order of k inside a
// product is free as long as both sides agree, and this way a fragment is a
// 16-byte read for two instructions.  D layout of v_mfma_f64_16x16x4f64: register
// r of lane l holds row 4*r + (l>>4), column l&15 (the four row groups are
// interleaved, unlike the 16-bit forms).
template<int NI, int NJ, class Left, class Skip, class Whole, class Refill, class Ahead>
__device__ __forceinline__ void wave_tiles(double* t3, const double* As, const double* Bs, const unsigned short* te,
                                           const Share& q, bool store, int n1, int n2, bool neg1, bool neg2,
                                           Left&& left, Skip&& skip, Whole&& refill_whole, Refill&& refill, Ahead&& ahead) {
  constexpr int I = NI ? NI : 1, J = NJ ? NJ : 1;
  const int     lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  int pa[I], pb[J];  // fragment rows in As and Bs, kept out of the loop
#pragma unroll
  for(int i = 0; i < NI; i++) {
    pa[i] = (16 * (q.i0 + q.is * i) + lr) * LDK + 2 * lk;
    asm("" : "+v"(pa[i]));
  }
#pragma unroll
  for(int j = 0; j < NJ; j++) {
    pb[j] = (16 * (q.j0 + q.js * j) + lr) * LDK + 2 * lk;
    asm("" : "+v"(pb[j]));
  }
  v4d acc[I][J];
#pragma unroll
  for(int i = 0; i < NI; i++)
#pragma unroll
    for(int j = 0; j < NJ; j++) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  struct Frag {
    v2d a[I], b[J];
  };
  auto read = [&](Frag& f, int k) {
#pragma unroll
    for(int i = 0; i < NI; i++) f.a[i] = *reinterpret_cast<const v2d*>(&As[pa[i] + k]);
#pragma unroll
    for(int j = 0; j < NJ; j++) f.b[j] = *reinterpret_cast<const v2d*>(&Bs[pb[j] + k]);
  };
  auto mma = [&](const Frag& f) {
#pragma unroll
    for(int i = 0; i < NI; i++)
#pragma unroll
      for(int j = 0; j < NJ; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[i].x, f.b[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
    for(int i = 0; i < NI; i++)
#pragma unroll
      for(int j = 0; j < NJ; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[i].y, f.b[j].y, acc[i][j], 0, 0, 0);
  };
  refill();  // the staging is free: every wave has read the last chunk before
  bool d1 = n1 > 0;
#pragma unroll 1
  for(int n = d1 ? n1 : n2;;) {
    Frag f0, f1;
    // chunks that leave n and the load side in the middle of the family
    const int w = max(min(n - 2, left()), 0) >> 1;
#pragma unroll 1
    for(int c = w; c > 0; c--) {
      __syncthreads();
      read(f0, 0);
      read(f1, 8);
      __syncthreads();
      refill_whole();
      mma(f0);
      mma(f1);
    }
    n -= 2 * w;
    if(w) skip(2 * w);
    __syncthreads();
    read(f0, 0);
    read(f1, 8);
    __syncthreads();
    refill();
    mma(f0);
    if(n > 1) mma(f1);
    n -= 2;
    if(n > 0) continue;
    if(!d1 || n2 == 0) break;
    d1 = false;
    n  = n2;
    if(neg1 != neg2) {
#pragma unroll
      for(int i = 0; i < NI; i++)
#pragma unroll
        for(int j = 0; j < NJ; j++) acc[i][j] = -acc[i][j];
    }
  }
  ahead();
  const double sg = (n2 ? neg2 : neg1) ? -1.0 : 1.0;
#pragma unroll
  for(int i = 0; i < NI; i++)
#pragma unroll
    for(int j = 0; j < NJ; j++) {
      const int c = te[64 + 16 * (q.j0 + q.js * j) + lr];
      double*   p[4];
#pragma unroll
      for(int r = 0; r < 4; r++) p[r] = &t3[te[16 * (q.i0 + q.is * i) + 4 * r + lk] | c];
      if(store) {
#pragma unroll
        for(int r = 0; r < 4; r++) *p[r] = sg * acc[i][j][r];
      }
      else {
        double v[4];
#pragma unroll
        for(int r = 0; r < 4; r++) v[r] = *p[r];
#pragma unroll
        for(int r = 0; r < 4; r++) *p[r] = fma(sg, acc[i][j][r], v[r]);
      }
    }
}
template<class Left, class Skip, class Whole, class Refill, class Ahead>
__device__ __forceinline__ void share_tiles(double* t3, const double* As, const double* Bs, const unsigned short* te,
                                            const Share& q, bool store, int n1, int n2, bool neg1, bool neg2,
                                            Left&& left, Skip&& skip, Whole&& refill_whole, Refill&& refill, Ahead&& ahead) {
  switch(q.ni * 4 + q.nj) {
    case 4 + 1: wave_tiles<1, 1>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
    case 4 + 2: wave_tiles<1, 2>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
    case 4 + 3: wave_tiles<1, 3>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
    case 8 + 1: wave_tiles<2, 1>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
    case 8 + 2: wave_tiles<2, 2>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
    case 12 + 1: wave_tiles<3, 1>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
    default: wave_tiles<0, 0>(t3, As, Bs, te, q, store, n1, n2, neg1, neg2, left, skip, refill_whole, refill, ahead); break;
  }
}

// Operands of a bipartition for a sub-tile: of each family the addresses of the
// sub-tile's first M and N row, the units of K and the sign of the product.
// Rows c1*x - c2*y of the spin-orbital elements: both terms -> the
// antisymmetrised array; one term -> that array, its sign in the product's.
//   d1 M: t(pA,pB,hs,h7) - t(pA,pB,h7,hs) = t2h[pA,pB,hs,:] - t2h[pB,pA,hs,:]
//   d1 N: (hA h7|hB ps) - (hB h7|hA ps) = ovk[hB,ps,hA,:] - ovk[hA,ps,hB,:]
//   d2 M: (hs pA|p7 pB) - (hs pB|p7 pA) = xv[pB,pA,hs,:] - xv[pA,pB,hs,:]
//   d2 N: t(ps,p7,hA,hB) - t(p7,ps,hA,hB) = t2p[hA,hB,ps,:] - t2p[hB,hA,ps,:]
typedef const __attribute__((address_space(1))) char* GBytes;
struct Runs {
  GBytes a1, b1, a2, b2;
  int    n1, n2;  // 0: family off
  bool   neg1, neg2;
};
__device__ __forceinline__ Runs runs_of(const SpatialDev& S, const int* start, int g, unsigned c1, unsigned c2) {
  const int hs = g / 3, ps = g % 3;
  int       hA, hB, pA, pB;
  pair_of(hs, hA, hB);
  pair_of(ps, pA, pB);
  const unsigned HS = uni(start[hs]), HA = uni(start[hA]), HB = uni(start[hB]);
  const unsigned PS = uni(start[3 + ps]), PA = uni(start[3 + pA]), PB = uni(start[3 + pB]);
  const uint64_t O = S.O, V = S.V;
  auto           row = [](const double* p, uint64_t r, int K) { return (GBytes) (p + r * (unsigned) K); };
  Runs           R;
  R.a1   = row((c1 & 12) == 12 ? S.t2ha : S.t2h, (((c1 & 4) ? PA : PB) * V + ((c1 & 4) ? PB : PA)) * O + HS, S.Op);
  R.b1   = row((c1 & 48) == 48 ? S.ovka : S.ovk, (((c1 & 16) ? HB : HA) * V + PS) * O + ((c1 & 16) ? HA : HB), S.Op);
  R.a2   = row((c2 & 12) == 12 ? S.xva : S.xv, (((c2 & 4) ? PB : PA) * V + ((c2 & 4) ? PA : PB)) * O + HS, S.Vp);
  R.b2   = row((c2 & 48) == 48 ? S.t2pa : S.t2p, (((c2 & 16) ? HA : HB) * O + ((c2 & 16) ? HB : HA)) * V + PS, S.Vp);
  R.neg1 = ((c1 >> 1) ^ !(c1 & 4) ^ !(c1 & 16)) & 1;
  R.neg2 = ((c2 >> 1) ^ !(c2 & 4) ^ !(c2 & 16)) & 1;
  R.n1   = (c1 & 1) ? S.Op >> 3 : 0;
  R.n2   = (c2 & 1) ? S.Vp >> 3 : 0;
  return R;
}
// Tables of bipartition g, by 128 threads: rows relative to the sub-tile's first,
// at most three of the slowest coordinate, which takes less than 24 bits of any
// system whose operands fit the memory.
__device__ __forceinline__ void fill_rows(Rows& t, int tb, const int* ext, int g, unsigned c1, unsigned c2,
                                          unsigned O, unsigned V) {
  const int tid = threadIdx.x, hs = g / 3, ps = g % 3;
  if(tid >= 128) return;
  int hA, hB, pA, pB;
  pair_of(hs, hA, hB);
  pair_of(ps, pA, pB);
  const bool row = tid < 64;
  const int  q0 = row ? hs : hA, q1 = row ? 3 + pA : hB, q2 = 3 + (row ? pB : ps);
  const int  e0 = ext[q0], e1 = ext[q1], e2 = ext[q2];
  Item       x  = item_of(tid & 63, e0, e1);
  t.e[tb][tid]  = box_index(x, e0, e1, e2, q0, q1, q2);
  if(x.c >= e2) x.a = x.b = x.c = 0;
  const unsigned y0 = x.a, y1 = x.b, y2 = x.c;
  if(row) {  // (hs, pA, pB)
    t.r1[tid] = __umul24(__umul24((c1 & 4) ? y1 : y2, V) + ((c1 & 4) ? y2 : y1), O) + y0;
    t.r2[tid] = __umul24(__umul24((c2 & 4) ? y2 : y1, V) + ((c2 & 4) ? y1 : y2), O) + y0;
  }
  else {  // (hA, hB, ps)
    t.r1[tid] = __umul24(__umul24((c1 & 16) ? y1 : y0, V) + y2, O) + ((c1 & 16) ? y0 : y1);
    t.r2[tid] = __umul24(__umul24((c2 & 16) ? y0 : y1, O) + ((c2 & 16) ? y1 : y0), V) + y2;
  }
}

__device__ void spatial_subtile(Smem& sm, const SpatialDev& S, uint64_t d1code, uint64_t d2code,
                                uint64_t s1code, double& e4, double& e5) {
  const int      tid = threadIdx.x;
  const unsigned O = S.O, V = S.V;
  if(tid < 24) {
    const int p = tid >> 2, i = tid & 3;
    sm.eps[tid] = i < sm.ext[p] ? (p < 3 ? S.eo : S.ev)[sm.start[p] + i] : 0.0;
  }
  d1code = uniform64(d1code);
  d2code = uniform64(d2code);
  s1code = uniform64(s1code);
  auto code1 = [&](int g) { return (unsigned) (d1code >> (6 * g)) & 63u; };
  auto code2 = [&](int g) { return (unsigned) (d2code >> (6 * g)) & 63u; };
  auto next  = [&](int g) {  // first enabled bipartition from g on, or 9
    while(g < 9 && !((code1(g) | code2(g)) & 1)) g++;
    return g;
  };
  const int row = tid >> 2, kq = tid & 3;
  double*   As  = sm.stage;
  double*   Bs  = sm.stage + 64 * LDK;
  int       g   = next(0);
  bool      store = true;  // no bipartition has been added yet
  if(g < 9) fill_rows(sm.tab, 0, sm.ext, g, code1(g), code2(g), O, V);
  __syncthreads();

  // Chunk in flight: four k of this thread's M and N row (kq 0, 1: of the first
  // unit, or of the only one; kq 2, 3: of the second), loaded while the chunk
  // before is multiplied, also from one bipartition to the next.  Offsets from
  // the sub-tile's first row stay below 2^32 bytes: they span three rows of the
  // slowest coordinate of an array that fits the memory.
  Runs     R;
  GBytes   ba = nullptr, bb = nullptr;  // next chunk
  int      left = 0, tb = 0;            // units of the family to load
  bool     fam2 = false;
  unsigned oa = 0, ob = 0, oa2 = 0, ob2 = 0;
  const unsigned back = 64u * (kq >> 1);
  v2d      ax0 = {0.0, 0.0}, ax1 = ax0, bx0 = ax0, bx1 = ax0;
  typedef const __attribute__((address_space(1))) v2d* GD2;
  auto load = [&]() {
    asm("" : "+v"(oa), "+v"(ob));  // keeps scalar bases with vector offsets in the loop
    const GD2 a = (GD2) (ba + oa), b = (GD2) (bb + ob);
    ax0 = a[0];
    ax1 = a[1];
    bx0 = b[0];
    bx1 = b[1];
    ba += 8 * KC;
    bb += 8 * KC;
  };
  auto fetch = [&]() {
    if(left <= 0) {
      if(!fam2 && R.n2) {
        fam2 = true;
        ba   = R.a2;
        bb   = R.b2;
        oa   = oa2;
        ob   = ob2;
        left = R.n2;
      }
      else {  // the bipartition's last chunk is on its way: read it again
        ba -= 8 * KC;
        bb -= 8 * KC;
      }
    }
    if(left == 1) {
      oa -= back;
      ob -= back;
    }
    load();
    left -= 2;
  };
  v2d* const A = reinterpret_cast<v2d*>(&As[row * LDK + 4 * kq]);
  v2d* const B = reinterpret_cast<v2d*>(&Bs[row * LDK + 4 * kq]);
  auto       put = [&]() {
    A[0] = ax0;
    A[1] = ax1;
    B[0] = bx0;
    B[1] = bx1;
  };
  auto begin = [&]() {
    R = runs_of(S, sm.start, g, code1(g), code2(g));
    const unsigned K1 = S.Op, K2 = S.Vp;
    const Rows&    t = sm.tab;
    oa   = 8 * (__umul24(t.r1[row], K1) + 4 * kq);
    ob   = 8 * (__umul24(t.r1[64 + row], K1) + 4 * kq);
    oa2  = 8 * (__umul24(t.r2[row], K2) + 4 * kq);
    ob2  = 8 * (__umul24(t.r2[64 + row], K2) + 4 * kq);
    ba   = R.a1;
    bb   = R.b1;
    left = R.n1;
    fam2 = false;
    fetch();
  };
  if(g < 9) begin();
#pragma unroll 1
  while(g < 9) {
    const int             gn = next(g + 1), hs = g / 3, ps = g % 3;
    const unsigned short* te = sm.tab.e[tb];
    int                   hA, hB, pA, pB;
    pair_of(hs, hA, hB);
    pair_of(ps, pA, pB);
    const Share q = wave_share(g, __builtin_amdgcn_readfirstlane(sm.ext[hs] * sm.ext[3 + pA] * sm.ext[3 + pB]),
                               __builtin_amdgcn_readfirstlane(sm.ext[hA] * sm.ext[hB] * sm.ext[3 + ps]));
    auto left_units = [&]() { return left; };
    auto skip         = [&](int n) { left -= n; };
    auto refill_whole = [&]() {
      put();
      load();
    };
    auto refill = [&]() {
      put();
      fetch();
    };
    auto ahead = [&]() {
      tb ^= 1;
      g = gn;
      if(g < 9) begin();
    };
    __syncthreads();  // every wave has added the bipartition before: its tables are free
    if(gn < 9) fill_rows(sm.tab, tb ^ 1, sm.ext, gn, code1(gn), code2(gn), O, V);
    share_tiles(sm.t3, As, Bs, te, q, store, R.n1, R.n2, R.neg1, R.neg2, left_units, skip, refill_whole, refill, ahead);
    store = false;
  }
  if(store)
    for(int e = tid; e < T3N; e += NT) sm.t3[e] = 0.0;

  // ---- s1 operands: T1so(pa,hi) and <hk hj||pc pb> blocks of the sub-tile
  __syncthreads();
  double* T1s = sm.t1s;
  double* V1s = sm.stage;
  for(int x = tid; x < 9 * 16; x += NT) {
    const int      slot = x >> 4, pai = (x >> 2) & 3, hii = x & 3;
    const unsigned c    = (unsigned) (s1code >> (4 * slot)) & 15u;
    const int      pa = slot / 3, hi = slot % 3;
    double         v = 0.0;
    if((c & 1) && pai < sm.ext[3 + pa] && hii < sm.ext[hi]) {
      v = S.t1[(size_t) (sm.start[3 + pa] + pai) * O + sm.start[hi] + hii];
      if(c & 2) v = -v;
    }
    T1s[x] = v;
  }
  {
    // One element per slot and thread, every load in flight before the first
    // use; offsets from the sub-tile's first element stay below 2^32 bytes, as
    // the operand rows' do.
    const unsigned gk = tid & 3, gj = (tid >> 2) & 3, gc = (tid >> 4) & 3, gb = tid >> 6;
    const unsigned o1 = 8 * (__umul24(__umul24(__umul24(gc, V) + gb, O) + gk, O) + gj);
    const unsigned o2 = 8 * (__umul24(__umul24(__umul24(gb, V) + gc, O) + gk, O) + gj);
    double         x1[9], x2[9];
    typedef const __attribute__((address_space(1))) double* GD;
#pragma unroll
    for(int slot = 0; slot < 9; slot++) {
      const unsigned c  = (unsigned) (s1code >> (4 * slot)) & 15u;
      const int      pa = slot / 3, hi = slot % 3;
      int            hj, hk, pb, pc;
      pair_of(hi, hj, hk);
      pair_of(pa, pb, pc);
      x1[slot] = x2[slot] = 0.0;
      if((c & 1) && (int) gk < sm.ext[hk] && (int) gj < sm.ext[hj] && (int) gc < sm.ext[3 + pc] &&
         (int) gb < sm.ext[3 + pb]) {
        const uint64_t K = uni(sm.start[hk]), J = uni(sm.start[hj]), PC = uni(sm.start[3 + pc]),
                       PB = uni(sm.start[3 + pb]);
        if(c & 4) x1[slot] = *(GD) ((GBytes) (S.vvoo + ((PC * V + PB) * O + K) * O + J) + o1);  // (hk pc|hj pb)
        if(c & 8) x2[slot] = *(GD) ((GBytes) (S.vvoo + ((PB * V + PC) * O + K) * O + J) + o2);  // (hk pb|hj pc)
      }
    }
#pragma unroll
    for(int slot = 0; slot < 9; slot++) {
      const unsigned c = (unsigned) (s1code >> (4 * slot)) & 15u;
      V1s[slot * 256 + tid] = (c & 4) && (c & 8) ? x1[slot] - x2[slot] : ((c & 4) ? x1[slot] : -x2[slot]);
    }
  }
  __syncthreads();
  subtile_energy(sm, T1s, V1s, sm.ext, e4, e5);
}

// Persistent kernel: workgroup b serves queue b % kQueues first (dispatch is
// round-robin over the 8 XCDs, so that is its own XCD's queue), then steals
// from the others; one ticket = one sub-tile.  Thread 0 claims and decodes each
// ticket (its entry searched forward from its previous one) and keeps the
// running exact sums of the task its sub-tiles belong to (xt_tasksums.h).
__global__ void __launch_bounds__(NT, 3) k_spatial_fp64(SpatialDev S, RunDev R) {
  __shared__ Smem               sm;
  __shared__ int                s_task;
  __shared__ int                s_weight;  // thread 0: boxes that its box stands for
  __shared__ Claim              s_claim;   // thread 0; its task also for the others
  __shared__ int                s_cur;     // thread 0: task of the running sums
  __shared__ unsigned long long s_sum[4];  // thread 0: E4 lo, hi, E5 lo, hi of s_cur not yet added
  const int                     tid  = threadIdx.x;
  const int                     home = blockIdx.x % kQueues;
  if(tid == 0) {
    s_cur    = -1;
    s_sum[0] = s_sum[1] = s_sum[2] = s_sum[3] = 0ull;
  }
#pragma unroll 1
  for(int qi = 0; qi < kQueues; qi++) {
    const int q = (home + qi) % kQueues;
    if(tid == 0) claim_queue(s_claim, R, q);
#pragma unroll 1
    for(;;) {
      __syncthreads();  // previous sub-tile finished with LDS and s_task
      if(tid == 0) {
        int       sub[6], weight;
        const int ti = claim_box(s_claim, R, q, claim_ticket(R, q), false, sub, weight);
        if(ti >= 0) {
          s_weight         = weight;
          const TaskDev& T = s_claim.task;
#pragma unroll
          for(int p = 0; p < 6; p++) {
            sm.start[p] = T.off[p] + 4 * sub[p];
            sm.ext[p]   = min(4, T.dim[p] - 4 * sub[p]);
          }
        }
        s_task = ti;
      }
      __syncthreads();
      const int ti = s_task;
      if(ti < 0) break;
      const TaskDev&           T  = s_claim.task;
      const unsigned long long t0 = wall_clock64();
      double                   e4, e5;
      spatial_subtile(sm, S, T.d1code, T.d2code, T.s1code, e4, e5);
      if(tid == 0) {
        if(ti != s_cur) {
          sums_flush(R, s_cur, s_sum);
          s_cur = ti;
        }
        sums_add(R, s_sum, s_weight * e4, s_weight * e5);
        if(R.cost) atomicAdd(&R.cost[ti], wall_clock64() - t0);
      }
    }
  }
  if(tid == 0) sums_flush(R, s_cur, s_sum);
}

// Start of a run: clears the counters and sums and brings the queues from host
// memory; three fills and four copies in its place were a gap of about 10 us each.
// Bound by its launch, and by PCIe where the plan has many tasks: the first head
// words are copied as they are; behind them (task0, tick0: where the entries'
// tasks, two a word, and first tickets begin) only the entries in use, their count
// at the end of qbeg, which is read over PCIe first.  One task of 97,344: 24 us
// with every word copied.
__global__ void k_begin(unsigned long long* zero, long nz, unsigned long long* dst,
                        const unsigned long long* src, long n, long head, long task0, long tick0) {
  const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if(i < nz) zero[i] = 0ull;
  if(i >= n) return;
  if(i >= head) {
    const int ne = reinterpret_cast<const int*>(src + kQueues)[kQueues];
    if(i >= (i < tick0 ? task0 + (ne + 1) / 2 : tick0 + ne)) return;
  }
  dst[i] = src[i];
}

// Energy of task t from the fixed-point accumulators, scaled by the task's factor:
// to device memory and to host memory, as a copy back costs more than the sum.
__device__ __forceinline__ void task_energy(int t, const TaskDev* tasks, const unsigned long long* acc,
                                            double* task_e, double* task_h) {
  const double f  = tasks[t].factor;
  const double e4 = f * fx_value(&acc[4 * (size_t) t]), e5 = f * fx_value(&acc[4 * (size_t) t + 2]);
  task_e[2 * (size_t) t]     = task_h[2 * (size_t) t]     = e4;
  task_e[2 * (size_t) t + 1] = task_h[2 * (size_t) t + 1] = e5;
}
// Of the tasks that the queues list, or of all n in task order.
__global__ void __launch_bounds__(NT) k_task_energies(const TaskDev* tasks, int n, const int* qbeg, const int* qtask,
                                                     const unsigned long long* acc, double* task_e,
                                                     double* task_h) {
  const int ne = qbeg[kQueues];
  for(int x = blockIdx.x * NT + threadIdx.x; x < ne; x += gridDim.x * NT)
    task_energy(ne == n ? x : qtask[x], tasks, acc, task_e, task_h);
}

// Fixed-shape sum of the task energies in task order (one workgroup of NT threads):
// thread i sums tasks [i*per, (i+1)*per) in order, per = ceil(n/NT), then a
// halving tree over the threads.  CONVERT: the energies are formed here first, of
// all tasks; else k_task_energies has formed them, and there is no sum unless the
// queues list every task.  Bound by its launch and by what follows it.
// With k_begin and this, a whole mixed run of O=8, V=48 takes 0.37 ms (0.43 with
// fills, copies and two reduction kernels), an FP64 run of O=7, V=22 0.40 (0.47).
static_assert(NT == kReduceThreads, "the host repeats this reduction with kReduceThreads");
template<bool CONVERT>
__global__ void __launch_bounds__(NT) k_reduce(const TaskDev* tasks, int n, const int* qbeg,
                                              const unsigned long long* acc, const unsigned long long* err,
                                              double* task_e, double* task_h, double* e45) {
  __shared__ double ra[NT], rb[NT];
  if(CONVERT) {
    for(int t = threadIdx.x; t < n; t += NT) task_energy(t, tasks, acc, task_e, task_h);
    __syncthreads();
  }
  const int per = CONVERT || qbeg[kQueues] == n ? (n + NT - 1) / NT : 0;
  const int lo = threadIdx.x * per, hi = min(n, lo + per);
  double    a = 0.0, b = 0.0;
  for(int t = lo; t < hi; t++) {
    a += task_e[2 * (size_t) t];
    b += task_e[2 * (size_t) t + 1];
  }
  ra[threadIdx.x] = a;
  rb[threadIdx.x] = b;
  __syncthreads();
  for(int s = NT / 2; s >= 1; s >>= 1) {
    if((int) threadIdx.x < s) {
      ra[threadIdx.x] += ra[threadIdx.x + s];
      rb[threadIdx.x] += rb[threadIdx.x + s];
    }
    __syncthreads();
  }
  if(threadIdx.x == 0) {
    e45[0] = ra[0];
    e45[1] = rb[0];
    e45[2] = *err ? 1.0 : 0.0;
  }
}

// out[b*ldo + a] = in[a*lda + b] for a < rows, b < cols, batched over
// blockIdx.z with strides (in_bs, out_bs).  32x32 LDS tiles.
__global__ void k_transpose(const double* __restrict__ in, double* __restrict__ out, long rows,
                            long cols, long lda, long ldo, long in_bs, long out_bs) {
  __shared__ double tile[32][33];
  const long z  = blockIdx.z;
  const long a0 = (long) blockIdx.y * 32, b0 = (long) blockIdx.x * 32;
  const int  tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: 32 x 8
  for(int r = ty; r < 32; r += 8) {
    const long a = a0 + r, b = b0 + tx;
    tile[r][tx]  = (a < rows && b < cols) ? in[z * in_bs + a * lda + b] : 0.0;
  }
  __syncthreads();
  for(int r = ty; r < 32; r += 8) {
    const long b = b0 + r, a = a0 + tx;
    if(a < rows && b < cols) out[z * out_bs + b * ldo + a] = tile[tx][r];
  }
}

static int transpose(const double* in, double* out, long rows, long cols, long lda, long ldo,
                     long batch, long in_bs, long out_bs, hipStream_t st) {
  // grid.y and grid.z are limited to 65535
  const long max_yz = 65535;
  for(long z0 = 0; z0 < batch; z0 += max_yz) {
    const long nz = std::min(max_yz, batch - z0);
    for(long r0 = 0; r0 < rows; r0 += 32 * max_yz) {
      const long nr = std::min(32 * max_yz, rows - r0);
      dim3       grid((unsigned) ((cols + 31) / 32), (unsigned) ((nr + 31) / 32), (unsigned) nz);
      hipLaunchKernelGGL(k_transpose, grid, dim3(256), 0, st, in + z0 * in_bs + r0 * lda,
                         out + z0 * out_bs + r0, nr, cols, lda, ldo, in_bs, out_bs);
      if(hipGetLastError() != hipSuccess) return (int) hipErrorLaunchFailure;
    }
  }
  return 0;
}

// out[r][k] = in[r][k] for k < K, 0 for K <= k < Kp
__global__ void k_pad_rows(double* __restrict__ out, const double* __restrict__ in, long rows,
                           long K, long Kp) {
  const long n = rows * Kp;
  for(long i = (long) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long) gridDim.x * blockDim.x) {
    const long r = i / Kp, k = i % Kp;
    out[i]       = k < K ? in[r * K + k] : 0.0;
  }
}

// out[i0][i1][i2][k] = in[i0][i1][i2][k] - in[j0][j1][j2][k] with (j0,j1,j2) =
// (i1,i0,i2) (swap02 = 0) or (i2,i1,i0) (swap02 = 1); padding stays zero.
__global__ void k_antisym(double* __restrict__ out, const double* __restrict__ in, long n0,
                          long n1, long n2, long Kp, int swap02) {
  const long n = n0 * n1 * n2 * Kp;
  for(long i = (long) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long) gridDim.x * blockDim.x) {
    long       r  = i / Kp;
    const long k  = i % Kp;
    const long i2 = r % n2;
    r /= n2;
    const long i1 = r % n1, i0 = r / n1;
    const long j  = swap02 ? ((i2 * n1 + i1) * n2 + i0) * Kp + k : ((i1 * n1 + i0) * n2 + i2) * Kp + k;
    out[i]        = in[i] - in[j];
  }
}

// Blocks of 256 for n elements of a grid-stride kernel.  A dispatch's grid
// size is a 32-bit count of work-items, so the grid is capped (2^20 blocks
// keep every CU busy) and the kernels loop over the rest.
static unsigned nblk(long n) { return (unsigned) std::min<long>((n + 255) / 256, 1l << 20); }

int build_operands(int O, int V, double* t2, double* ovoo, double*& vvvo, SpatialBufs& B,
                   void* stream) {
  hipStream_t st = (hipStream_t) stream;
  const long  o = O, v = V, op = (O + 7) / 8 * 8, vp = (V + 7) / 8 * 8;
  auto        alloc = [](double** p, long n) { return (hipError_t) track_malloc((void**) p, sizeof(double) * n); };
  hipError_t  e;
  int         rc;
  // d1 operands (contraction over h7, padded to op)
  if((e = alloc(&B.t2h, v * v * o * op))) return (int) e;
  hipLaunchKernelGGL(k_pad_rows, dim3(nblk(v * v * o * op)), dim3(256), 0, st, B.t2h, t2, v * v * o,
                     o, op);
  if((e = alloc(&B.t2ha, v * v * o * op))) return (int) e;
  hipLaunchKernelGGL(k_antisym, dim3(nblk(v * v * o * op)), dim3(256), 0, st, B.t2ha, B.t2h, v, v,
                     o, op, 0);
  if((e = alloc(&B.ovk, o * v * o * op))) return (int) e;
  hipLaunchKernelGGL(k_pad_rows, dim3(nblk(o * v * o * op)), dim3(256), 0, st, B.ovk, ovoo,
                     o * v * o, o, op);
  if((e = alloc(&B.ovka, o * v * o * op))) return (int) e;
  hipLaunchKernelGGL(k_antisym, dim3(nblk(o * v * o * op)), dim3(256), 0, st, B.ovka, B.ovk, o, v,
                     o, op, 1);
  // d2 N side: t2p[i][j][a][b] = t2[a][b][i][j], padded in b
  double* tmp = nullptr;
  if((e = alloc(&tmp, o * o * v * v))) return (int) e;
  if((rc = transpose(t2, tmp, v * v, o * o, o * o, v * v, 1, 0, 0, st))) return rc;
  if((e = alloc(&B.t2p, o * o * v * vp))) return (int) e;
  hipLaunchKernelGGL(k_pad_rows, dim3(nblk(o * o * v * vp)), dim3(256), 0, st, B.t2p, tmp, o * o * v,
                     v, vp);
  if((e = alloc(&B.t2pa, o * o * v * vp))) return (int) e;
  hipLaunchKernelGGL(k_antisym, dim3(nblk(o * o * v * vp)), dim3(256), 0, st, B.t2pa, B.t2p, o, o, v,
                     vp, 0);
  if((e = hipStreamSynchronize(st))) return (int) e;
  track_free(tmp);
  if(!vvvo) return 0;  // xv comes from elsewhere (build_xv_cholesky), then build_xva
  // d2 M side: xv[c][b][i][a] = vvvo[a][c][b][i], padded in a
  if((e = alloc(&B.xv, v * v * o * vp))) return (int) e;
  if((e = hipMemsetAsync(B.xv, 0, sizeof(double) * v * v * o * vp, st))) return (int) e;
  if((rc = transpose(vvvo, B.xv, v, v * o, v * v * o, vp, v, v * o, v * o * vp, st))) return rc;
  if((e = hipStreamSynchronize(st))) return (int) e;
  track_free(vvvo);
  vvvo = nullptr;
  return build_xva(O, V, B, stream);
}

int build_xva(int O, int V, SpatialBufs& B, void* stream) {
  hipStream_t st = (hipStream_t) stream;
  const long  o = O, v = V, vp = (V + 7) / 8 * 8;
  hipError_t  e;
  if((e = (hipError_t) track_malloc((void**) &B.xva, sizeof(double) * v * v * o * vp))) return (int) e;
  hipLaunchKernelGGL(k_antisym, dim3(nblk(v * v * o * vp)), dim3(256), 0, st, B.xva, B.xv, v, v, o,
                     vp, 0);
  if((e = hipGetLastError())) return (int) e;
  return (int) hipStreamSynchronize(st);
}

// out[a][b][i][j] = in[((a * O + i) * V + b) * O + j]: the (ai|bj) GEMM result,
// rows (a,i) and columns (b,j), in the vvoo order.
__global__ void k_vvoo_order(const double* __restrict__ in, double* __restrict__ out, long O, long V) {
  const long n = V * V * O * O;
  for(long x = (long) blockIdx.x * blockDim.x + threadIdx.x; x < n; x += (long) gridDim.x * blockDim.x) {
    const long j = x % O, i = (x / O) % O, b = (x / (O * O)) % V, a = x / (O * O * V);
    out[x]       = in[((a * O + i) * V + b) * O + j];
  }
}

int launch_vvoo_order(const double* in, double* out, int O, int V, void* stream) {
  const long n = (long) V * V * O * O;
  hipLaunchKernelGGL(k_vvoo_order, dim3(nblk(n)), dim3(256), 0, (hipStream_t) stream, in, out,
                     (long) O, (long) V);
  return (int) hipGetLastError();
}

// Largest |(ai|bj) - (bj|ai)| and largest |(ai|bj)| over the pairs a <= b of each
// workgroup, to out[2 w] and out[2 w + 1] in host memory; an element that
// cannot be compared (NaN, or two infinities) counts as an infinite difference.
// A wave takes one pair at a time.  Bound: one read of vvoo (O=40, V=300: 0.26 ms).
__global__ void __launch_bounds__(256) k_vvoo_asym(const double* __restrict__ vvoo, long O, long V,
                                                   double* out) {
  const unsigned o = (unsigned) O, oo = o * o, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double         d = 0.0, m = 0.0;
  for(long p = 4l * blockIdx.x + wave; p < V * V; p += 4l * gridDim.x) {
    const long a = p / V, b = p - a * V;
    if(a > b) continue;
    const double* x = vvoo + p * oo;
    const double* y = vvoo + (b * V + a) * oo;
    for(unsigned q = lane; q < oo; q += 64) {
      const unsigned i = q / o, j = q - i * o;
      const double   u = x[q], v = y[j * o + i], e = fabs(u - v);
      m                = fmax(m, fmax(fabs(u), fabs(v)));
      if(!(e <= d)) d = e == e ? e : __builtin_inf();
    }
  }
  __shared__ double rd[4], rm[4];
#pragma unroll
  for(int k = 32; k >= 1; k >>= 1) {
    d = fmax(d, __shfl_xor(d, k, 64));
    m = fmax(m, __shfl_xor(m, k, 64));
  }
  if(lane == 0) {
    rd[wave] = d;
    rm[wave] = m;
  }
  __syncthreads();
  if(threadIdx.x == 0) {
    out[2 * blockIdx.x]     = fmax(fmax(rd[0], rd[1]), fmax(rd[2], rd[3]));
    out[2 * blockIdx.x + 1] = fmax(fmax(rm[0], rm[1]), fmax(rm[2], rm[3]));
  }
}
int launch_vvoo_asym(const double* vvoo, int O, int V, double* out, int* groups, void* stream) {
  *groups = (int) std::min<long>(((long) V * V + 3) / 4, kAsymGroups);
  hipLaunchKernelGGL(k_vvoo_asym, dim3((unsigned) *groups), dim3(256), 0, (hipStream_t) stream, vvoo,
                     (long) O, (long) V, out);
  return (int) hipGetLastError();
}

// Plans of more tasks bring only the queue entries in use and convert the task
// energies with many workgroups (wall time in us with one and with many: a whole
// run of 148 tasks 201.5 and 202.3, of 920 164.3 and 164.8, of 2,000 224.5 and 221.7,
// of 3,700 320 and 314; one task of 148 88.4 and 89.5, of 920 74.6 and 74.4, of 2,000
// 82.6 and 76.2, of 3,700 88.8 and 78.5).  One task of 97,344 takes 87 us, 505 where
// one workgroup walked the plan.
constexpr long kManyTasks = 1024;

int launch_begin(unsigned long long* zero, long nz, unsigned long long* dst,
                 const unsigned long long* src, long n, long task0, long tick0, void* stream) {
  const long head = n - tick0 <= kManyTasks ? n : task0;
  hipLaunchKernelGGL(k_begin, dim3((unsigned) ((std::max(nz, n) + 255) / 256)), dim3(256), 0,
                     (hipStream_t) stream, zero, nz, dst, src, n, head, task0, tick0);
  return (int) hipGetLastError();
}

int launch_spatial_fp64(const SpatialDev& S, const RunDev& R, int grid, void* stream) {
  hipLaunchKernelGGL(k_spatial_fp64, dim3(grid), dim3(NT), 0, (hipStream_t) stream, S, R);
  return (int) hipGetLastError();
}

int launch_reduce(const TaskDev* tasks, int n_tasks, const int* qbeg, const int* qtask,
                  const unsigned long long* acc, const unsigned long long* err, double* task_e,
                  double* task_h, double* e45, void* stream) {
  const bool many = n_tasks > kManyTasks;
  if(many) {
    hipLaunchKernelGGL(k_task_energies, dim3((unsigned) std::min((n_tasks + NT - 1) / NT, 1024)), dim3(NT), 0,
                       (hipStream_t) stream, tasks, n_tasks, qbeg, qtask, acc, task_e, task_h);
    const hipError_t e = hipGetLastError();
    if(e != hipSuccess) return (int) e;
  }
  hipLaunchKernelGGL(many ? k_reduce<false> : k_reduce<true>, dim3(1), dim3(NT), 0, (hipStream_t) stream, tasks,
                     n_tasks, qbeg, acc, err, task_e, task_h, e45);
  return (int) hipGetLastError();
}

// ---------------------------------------------------------------------------
// Per-task drop-in: operands come from the reference's packed buffers
// (ccsd_t_data_{s1,d1,d2}_new layouts, ccsd_t_all_fused_cpu.hpp index
// arithmetic), one workgroup per 4^6 block, partials per block.
// ---------------------------------------------------------------------------
// LDS of the per-task kernel, sized for three workgroups per CU (12 waves): the
// 4^6 tile, one staged K chunk of 16 (rows padded to 18 doubles, so the 16x16x4
// fragment reads of a half-wave hit distinct banks), which later holds the s1 V
// blocks.  Two forms of the K chunks (packed_ends in xt_host.cpp chooses): a chunk of
// one K tile has its addresses from scalars and one row pointer a thread; with
// the tiles of a family end to end there are fewer chunks where tiles are
// short, and each thread looks its k up in the list of tiles, which the LDS of the
// s1 T1 blocks holds until then.
constexpr int PKC  = kPackedKC;
constexpr int PLDK = PKC + 2;
static_assert(2 * 64 * PLDK >= 9 * 256, "staging too small for the s1 V blocks");
struct __align__(16) PSmem {
  double t3[T3N];
  double stage[2 * 64 * PLDK];
  union {
    int2   klist[kMaxNoab + kMaxNvab + 1];  // (family | exec slot << 1, K - 1 | first k << 12)
    double t1s[S1_T1];                      // later: the s1 T1 blocks
  };
  double eps[24];
  double red[8];
  Tables tab;
  int    ext[6];  // orbitals of the block inside the tile
};
static_assert((kMaxNoab + kMaxNvab) * 4096 + kPackedKC < (1 << 20), "first k must fit 20 bits");

template<bool ENDS>
__global__ void __launch_bounds__(NT, 3) k_packed_fp64(PackedArgs A) {
  __shared__ PSmem sm;
  const int        tid = threadIdx.x;
  const int*       dim = A.dim;
  int              nsub[6], sub[6];
#pragma unroll
  for(int p = 0; p < 6; p++) nsub[p] = cdiv(dim[p], 4);
  {
    long q = blockIdx.x;
#pragma unroll
    for(int p = 0; p < 6; p++) {
      sub[p] = (int) (q % nsub[p]);
      q /= nsub[p];
    }
  }
  const int* d1_size = A.meta;
  const int* d1_exec = d1_size + 7 * A.noab;
  const int* d2_size = d1_exec + 9 * A.noab;
  const int* d2_exec = d2_size + 7 * A.nvab;
  const int* s1_exec = d2_exec + 9 * A.nvab + 6;
  // the host's K tile lists of the nine bipartitions (packed_klists)
  const int*  k_n    = s1_exec + 9;
  const int4* k_list = reinterpret_cast<const int4*>(k_n + kKlistCountInts);

  if(tid < 24) {
    const int p = tid >> 2, i = tid & 3, g = 4 * sub[p] + i;
    sm.eps[tid] = g < dim[p] ? A.evl[p][g] : 0.0;
  }
  if(tid < 6) sm.ext[tid] = min(4, dim[tid] - 4 * sub[tid]);
  bool store = true;  // no bipartition has been added yet
  __syncthreads();
  double* As = sm.stage;
  double* Bs = sm.stage + 64 * PLDK;
  const int kk = tid & 15, rs = tid >> 4, n1 = tid & 63;
  const int kq = __builtin_amdgcn_readfirstlane(tid >> 6);

  int first = 0;  // first list entry of the bipartition
#pragma unroll 1
  for(int g = 0; g < 9; g++) {
    const int   nk   = k_n[g] & 0xffff, nd1 = k_n[g] >> 16;
    const int4* list = k_list + first;
    first += nk;
    if(nk == 0) continue;
    const int hs = g / 3, ps = g % 3;
    int       hA, hB, pA, pB;
    pair_of(hs, hA, hB);
    pair_of(ps, pA, pB);
    const bool neg = sgn_single(hs) * sgn_single(ps) > 0;  // the equations' sign, put on A
    const long DHS = dim[hs], DPA = dim[3 + pA], DPB = dim[3 + pB];
    const long DHA = dim[hA], DHB = dim[hB], DPS = dim[3 + ps];
    v4d        acc[2][2];
#pragma unroll
    for(int i = 0; i < 2; i++)
#pragma unroll
      for(int j = 0; j < 2; j++) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
    // A row of either operand is (item of the first two positions of its side,
    // third position): thread rs takes the item rs of up to 16 and j is the
    // third position, so row rs + per * j, per the items the tile holds.
    // Items and third positions outside the block read the nearest one inside.
    const int eHS = sm.ext[hs], ePA = sm.ext[3 + pA], ePB = __builtin_amdgcn_readfirstlane(sm.ext[3 + pB]);
    const int eHA = sm.ext[hA], eHB = sm.ext[hB], ePS = __builtin_amdgcn_readfirstlane(sm.ext[3 + ps]);
    const int aper = __builtin_amdgcn_readfirstlane(eHS * ePA), bper = __builtin_amdgcn_readfirstlane(eHA * eHB);
    const Quad quad = quadrant(g, aper * ePB, bper * ePS);
    const bool aok = rs < aper, bok = rs < bper;
    const int  ar = aok ? rs : 0, br = bok ? rs : 0;
    const int  ax = small_div(ar, eHS), bx = small_div(br, eHA);
    const int  aHS = 4 * sub[hs] + ar - ax * eHS, aPA = 4 * sub[3 + pA] + ax, aPB = 4 * sub[3 + pB];
    const int  bHA = 4 * sub[hA] + br - bx * eHA, bHB = 4 * sub[hB] + bx, bPS = 4 * sub[3 + ps];
    const long a1 = aPA + (aPB + aHS * DPB) * DPA;  // d1_t2 row of j = 0: [hs][pB][pA]
    const long a2 = aHS + (aPB + aPA * DPB) * DHS;  // d2_v2 row: [pA][pB][hs]
    const long b2 = bPS + (bHA + bHB * DHA) * DPS;  // d2_t2 row: [hB][hA][ps]
    const Item y   = item_of(n1 < bper * ePS ? n1 : 0, eHA, eHB);
    const int  gHA = 4 * sub[hA] + y.a, gHB = 4 * sub[hB] + y.b, gPS = 4 * sub[3 + ps] + y.c;
    const long rB1   = gHB + (gHA + gPS * DHA) * DHB;  // d1_v2 element of k = rB1 + k * bstr1
    const long bstr1 = DPS * DHA * DHB;

    // Walk over the chunks.  Current tile: it of nk, family d2, K; kt = first k
    // of the chunk to load; pa, pb the thread's pointers there, sa, sb the
    // strides of j.
    int           it = 0, kt = 0, K = 0;
    bool          d2 = false;
    const double *pa = nullptr, *pb = nullptr;
    long          sa = 0, sb = 0;
    auto          tile = [&]() {
      const int  fam = __builtin_amdgcn_readfirstlane(list[it].x);
      const long ex  = __builtin_amdgcn_readfirstlane(list[it].y);
      K  = __builtin_amdgcn_readfirstlane(list[it].z);
      kt = 0;
      d2 = fam != 0;
      if(d2) {
        pa = A.d2_v2 + A.max_d2_v2 * ex + a2 * K;
        sa = DHS * K;
        pb = A.d2_t2 + A.max_d2_t2 * ex + b2 * K;
        sb = K;
      }
      else {
        pa = A.d1_t2 + A.max_d1_t2 * ex + a1 * K;
        sa = DPA * K;
        pb = A.d1_v2 + A.max_d1_v2 * ex + rB1;
        sb = bstr1;
      }
    };
    double av[4], bv[4];
    int    clen = 0;      // k of the loaded chunk
    bool   cd2  = false;  // its family
    // ENDS: k1 k of d1 from 0 on, the d2 ones from the chunk kd2 / PKC on; chunk c of
    // nc; the tile of the thread's k (ia, la; na: the next one's first k) and, for the
    // d1 <ij||ka> block, of its wave's (ib, lb, nb).
    int  c = 0, nc = 0, k1 = 0, kd2 = 0, kall = 0, ia = 0, ib = 0, na = 0, nb = 0;
    int2 la = {};
    int4 lb = {};
    auto end_of = [&](int i) { return __builtin_amdgcn_readfirstlane(list[i].z + list[i].w); };
    auto next_b = [&]() { return ib + 1 < nk ? __builtin_amdgcn_readfirstlane(list[ib + 1].w) : INT_MAX; };
    if(ENDS) {
      k1   = nd1 ? end_of(nd1 - 1) : 0;
      kd2  = cdiv(k1, PKC) * PKC;
      kall = nk > nd1 ? end_of(nk - 1) : kd2;
      nc   = cdiv(kall, PKC);
      __syncthreads();  // every thread is done with the list before
      for(int x = tid; x <= nk; x += NT) {
        const int4 e = x < nk ? list[x] : make_int4(0, 0, 1, (1 << 20) - 1);
        sm.klist[x]  = make_int2(e.x | e.y << 1, (int) ((unsigned) (e.z - 1) | (unsigned) e.w << 12));
      }
      __syncthreads();
      la = sm.klist[0];
      na = (int) ((unsigned) sm.klist[1].y >> 12);
      lb = list[0];
      nb = next_b();
    }
    auto load_ends = [&]() {
      cd2  = c * PKC >= kd2;
      clen = min(PKC, (cd2 ? kall : k1) - c * PKC);
      const int k = c * PKC + min(kk, clen - 1);
      while(k >= na) {
        la = sm.klist[++ia];
        na = (int) ((unsigned) sm.klist[ia + 1].y >> 12);
      }
      const long ex = la.x >> 1, Kt = (la.y & 0xfff) + 1, kl = k - (int) ((unsigned) la.y >> 12);
      // third positions j outside the block read the last one inside
      auto row = [&](const double* q, long s, int n, double(&v)[4]) {
        v[0] = *q;
#pragma unroll
        for(int j = 1; j < 4; j++) {
          if(j < n) q += s;
          v[j] = *q;
        }
      };
      row(cd2 ? A.d2_v2 + A.max_d2_v2 * ex + a2 * Kt + kl : A.d1_t2 + A.max_d1_t2 * ex + a1 * Kt + kl,
          (cd2 ? DHS : DPA) * Kt, ePB, av);
      if(cd2) row(A.d2_t2 + A.max_d2_t2 * ex + b2 * Kt + kl, Kt, ePS, bv);
      else {
#pragma unroll
        for(int j = 0; j < 4; j++) {
          const int kj = c * PKC + min(4 * kq + j, clen - 1);
          while(kj >= nb) {
            lb = list[++ib];
            nb = next_b();
          }
          bv[j] = A.d1_v2[A.max_d1_v2 * (long) lb.y + rB1 + (kj - lb.w) * bstr1];
        }
      }
      c++;
    };
    // Issues every load of the next chunk, so that they are in flight together
    // while the previous chunk is multiplied; k past the tile's end reads its
    // last one.
    auto load = [&]() {
      if(kt == K) {
        it++;
        tile();
      }
      clen = min(PKC, K - kt);
      cd2  = d2;
      const double* qa = pa + kt + min(kk, clen - 1);
#pragma unroll
      for(int j = 0; j < 4; j++) av[j] = qa[min(j, ePB - 1) * sa];
      if(d2) {
        const double* qb = pb + kt + min(kk, clen - 1);
#pragma unroll
        for(int j = 0; j < 4; j++) bv[j] = qb[min(j, ePS - 1) * sb];
      }
      else {
#pragma unroll
        for(int j = 0; j < 4; j++) bv[j] = pb[(kt + min(4 * kq + j, clen - 1)) * sb];
      }
      kt += clen;
    };
    if(ENDS) load_ends();
    else {
      tile();
      load();
    }
    bool more = true, lead = true;
#pragma unroll 1
    while(more) {
      const int len = clen;
      __syncthreads();
      if(lead) fill_tables(sm.tab, sm.ext, hs, hA, hB, ps, pA, pB);
      lead = false;
      const bool kin = kk < len;
      if(aok) {
#pragma unroll
        for(int j = 0; j < 4; j++)
          if(j < ePB) As[(rs + aper * j) * PLDK + kk] = kin ? (neg ? -av[j] : av[j]) : 0.0;
      }
      if(cd2) {
        if(bok) {
#pragma unroll
          for(int j = 0; j < 4; j++)
            if(j < ePS) Bs[(rs + bper * j) * PLDK + kk] = kin ? bv[j] : 0.0;
        }
      }
      else {
#pragma unroll
        for(int j = 0; j < 4; j++) Bs[n1 * PLDK + 4 * kq + j] = 4 * kq + j < len ? bv[j] : 0.0;
      }
      __syncthreads();
      more = ENDS ? c < nc : kt < K || it + 1 < nk;
      if(more) {
        if(ENDS) load_ends();
        else load();
      }
      mfma_chunk<PKC, PLDK>(As, Bs, quad, acc, len);
    }
    acc_to_t3(sm.t3, sm.tab, quad, store, acc);
    store = false;
  }
  if(store)
    for(int e = tid; e < T3N; e += NT) sm.t3[e] = 0.0;

  // s1 operands from the packed buffers: t1 [hi][pa], v2 [pb][pc][hj][hk]
  __syncthreads();  // every thread is done with the tile list and the staged chunk
  double* T1s = sm.t1s;
  double* V1s = sm.stage;
  for(int x = tid; x < 9 * 16; x += NT) {
    const int slot = x >> 4, pai = (x >> 2) & 3, hii = x & 3;
    const int pa = slot / 3, hi = slot % 3;
    const int gp = 4 * sub[3 + pa] + pai, gh = 4 * sub[hi] + hii;
    double    v  = 0.0;
    if(s1_exec[slot] >= 0 && gp < dim[3 + pa] && gh < dim[hi])
      v = sgn_single(pa) * sgn_single(hi) *
          A.s1_t1[A.max_s1_t1 * (long) s1_exec[slot] + gp + (long) gh * dim[3 + pa]];
    T1s[x] = v;
  }
  {
    // one element per slot and thread, every load in flight before the first use
    const int w = tid;
    double    v[9];
#pragma unroll
    for(int slot = 0; slot < 9; slot++) {
      const int pa = slot / 3, hi = slot % 3;
      int       hj, hk, pb, pc;
      pair_of(hi, hj, hk);
      pair_of(pa, pb, pc);
      const int gk = 4 * sub[hk] + (w & 3), gj = 4 * sub[hj] + ((w >> 2) & 3),
                gc = 4 * sub[3 + pc] + ((w >> 4) & 3), gb = 4 * sub[3 + pb] + (w >> 6);
      v[slot] = 0.0;
      if(s1_exec[slot] >= 0 && gk < dim[hk] && gj < dim[hj] && gc < dim[3 + pc] && gb < dim[3 + pb])
        v[slot] = A.s1_v2[A.max_s1_v2 * (long) s1_exec[slot] + gk +
                          (gj + (gc + (long) gb * dim[3 + pc]) * dim[hj]) * dim[hk]];
    }
#pragma unroll
    for(int slot = 0; slot < 9; slot++) V1s[slot * 256 + tid] = v[slot];
  }
  __syncthreads();
  double e4, e5;
  subtile_energy(sm, T1s, V1s, sm.ext, e4, e5);
  if(tid == 0) {
    A.partial[blockIdx.x]                = e4;
    A.partial[blockIdx.x + A.num_blocks] = e5;
  }
}

int launch_packed_fp64(const PackedArgs& A, void* stream) {
  hipLaunchKernelGGL(A.ends ? k_packed_fp64<true> : k_packed_fp64<false>, dim3((unsigned) A.num_blocks), dim3(NT), 0,
                     (hipStream_t) stream, A);
  return (int) hipGetLastError();
}

// ---------------------------------------------------------------------------
// Allocation-free form of the per-task launch.  The launcher metadata lives in
// `scratch`, one fixed array per GPU for the life of the process.  In host
// code the name `scratch` is only a stand-in for the symbol, so every host use
// goes through the device address hipGetSymbolAddress returns, looked up once
// per device (with that device current) and kept in scratch_ptr.  The host
// arrays reach it through the arguments of k_store_meta launches on the
// caller's stream: ordered with the caller's work, captured by value at
// launch (the caller may reuse its arrays at once), and no allocation, copy
// engine or memset node involved.  Calls that overlap on one GPU race on it.
// ---------------------------------------------------------------------------
static __device__ __align__(256) int scratch[kPackedMetaInts];

namespace {
constexpr int kMetaChunk = 960;  // ints per copy launch (3.8 KB of kernel arguments)
struct MetaChunk {
  int off, n;
  int v[kMetaChunk];
};

__global__ void __launch_bounds__(256) k_store_meta(int* dst, MetaChunk c) {
  for(int i = threadIdx.x; i < c.n; i += blockDim.x) dst[c.off + i] = c.v[i];
}

constexpr int kMaxDevices = 64;
std::mutex    g_scratch_mu;
int*          scratch_ptr[kMaxDevices] = {};

// Device address of this GPU's scratch; nullptr on failure (*err set).
int* scratch_on_current_device(int* err) {
  int dev = 0;
  if((*err = (int) hipGetDevice(&dev))) return nullptr;
  if(dev < 0 || dev >= kMaxDevices) {
    *err = (int) hipErrorInvalidDevice;
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if(!scratch_ptr[dev]) {
    void* p = nullptr;
    if((*err = (int) hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)))) return nullptr;
    scratch_ptr[dev] = static_cast<int*>(p);
  }
  return scratch_ptr[dev];
}
}  // namespace

int launch_packed_fp64_noalloc(PackedArgs& A, const int* host_meta, int n_meta, void* stream,
                               void* after_copy) {
  if(n_meta < 0 || n_meta > kPackedMetaInts) return (int) hipErrorInvalidValue;
  int  err = 0;
  int* dst = scratch_on_current_device(&err);
  if(!dst) return err ? err : (int) hipErrorInvalidSymbol;
  hipStream_t st = (hipStream_t) stream;
  MetaChunk   c  = {};
  for(int off = 0; off < n_meta; off += kMetaChunk) {
    c.off = off;
    c.n   = std::min(kMetaChunk, n_meta - off);
    std::memcpy(c.v, host_meta + off, sizeof(int) * (size_t) c.n);
    hipLaunchKernelGGL(k_store_meta, dim3(1), dim3(256), 0, st, dst, c);
    if((err = (int) hipGetLastError())) return err;
  }
  if(after_copy && (err = (int) hipEventRecord((hipEvent_t) after_copy, st))) return err;
  A.meta = dst;
  return launch_packed_fp64(A, stream);
}

}  // namespace xt
