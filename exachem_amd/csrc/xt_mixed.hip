// Mixed-precision (T) kernel for gfx950.
//
// Same task / bipartition decomposition as the FP64 kernel, with larger
// workgroup boxes and 16-bit matrix cores:
//   * a workgroup owns a (4,4,4 | 8,8,8) box of t3[h1,h2,h3,p4,p5,p6]
//     (32768 elements, FP32 in LDS, never in HBM), cut to the task tile at its
//     edges;
//   * each bipartition g (single hole hs + particle pair | hole pair +
//     single particle ps) is a GEMM of up to 256 x 128: M = (hs,pA,pB),
//     N = (ps,hA,hB), K = h7 (d1) then p7 (d2).  Only rows and columns inside
//     the tile are numbered, so an edge box has fewer 32-row and 32-column
//     MFMA tiles (wave_tiles);
//   * operands are pre-split FP16 pairs y = hi + lo of x * 2^e, with one
//     power-of-two exponent per (tile, tile, tile) block of rows (per-tile
//     amplitude scaling: the block's max |y| lies in [2^13, 2^14)); every
//     product is hi*hi + hi*lo + lo*hi on v_mfma_f32_32x32x16_f16 with FP32
//     accumulation (~22-bit products).  All rows of one contraction part of a
//     task lie in one block per operand, so the part's scale (both exponents
//     and the spin-orbital signs) is one number, applied when the part ends and
//     its result is added into the FP32 box;
//   * eight waves (two per SIMD); in a whole box wave w owns the 32 M rows of
//     particle pB = w, loaded from L2/HBM straight into registers in the MFMA
//     operand layout.  The B panel (shared by all waves) goes through a
//     double-buffered LDS stage.  A register ring keeps PF chunks of loads in
//     flight across part and bipartition boundaries; every thread issues the
//     same loads for every chunk, so the compiler's wait counts follow the
//     ring; one barrier per K chunk;
//   * what bounds the K loop: the L1 takes one cycle per cache line that a
//     wave's load touches.  With each row's K run contiguous a load of 32 rows
//     touched 64 (67 cycles measured, against 18 where four lanes share a
//     line), 1,200 L1 cycles per 16-k chunk beside 768 of MFMA.  The split
//     arrays therefore hold the rows of one (x, y) pair side by side per 8 k
//     (SplitBufs), so that the four hs of a quad of lanes, and the eight ps of
//     a B column group, are one run.  With that, a wave's own instruction
//     stream was the next bound (one instruction per four cycles: the loop's
//     tests, cursor moves and late fragment reads added to the MFMAs instead
//     of running under them).  Both and the numbering of rows inside the tile:
//     24 tasks of O=40, V=300 26.8 -> 24.6 ms, 40 uneven tasks of O=48, V=384
//     124 -> 105.7 ms.  What is left beside the MFMAs of a whole box (about
//     1,440 cycles per chunk): 240 of loads that hit L1, 200 of L2 misses,
//     200 of fragment reads, each by timing a build without it;
//   * the flush into the box adds per-row and per-column offsets from LDS
//     tables; the box index xors the particle bits into the hole bits (swz) so
//     that the lanes of every bipartition's flush, and those of the energy
//     sweeps, fall on 64 distinct banks; the d1 part of a bipartition carries
//     its accumulators into the d2 part, so a bipartition flushes once;
//   * energy: one FP64 reciprocal of the denominator per element (from
//     separable hole and particle sums), E4 in FP64, then t3/D is kept in
//     place for the s1 sweeps (FP32 products, FP64 sums); task partials are
//     accumulated exactly like the FP64 kernel.
#include <hip/hip_runtime.h>

#include "xt_device.h"
#include "xt_claim.h"
#include "xt_fixed.h"
#include "xt_queue.h"
#include "xt_tasksums.h"

namespace xt {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float    f16v __attribute__((ext_vector_type(16)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
// an operand base read from LDS is a generic pointer to the compiler, whose
// flat loads would also count as LDS operations
typedef const __attribute__((address_space(1))) u4v* global_u4;

constexpr int NT  = 512;
constexpr int NW  = NT / 64;  // waves
constexpr int NM  = 256;      // bipartition rows (hs, pA, pB) of a whole box
constexpr int NN  = 128;      // bipartition columns (ps, hA, hB) of a whole box
constexpr int KC  = 16;       // K per chunk (one MFMA K step)
constexpr int BOX = 32768;
constexpr int PF  = 4;        // ring depth: chunks whose loads are in flight per thread
constexpr int S1P = 3;        // s1 slots staged per sweep
// the unrolled ring loop picks stage and fragment buffers by s & 1, which is
// the chunk's parity only when the ring depth is even
static_assert(PF % 2 == 0, "ring depth must be even");
// while chunk it is multiplied from slot it % PF, chunk it+2's B piece is staged
// and the A loads of chunk it+PF-1 go to another slot
static_assert(PF >= 4, "the ring must hold the current chunk, the next two and one in flight");

struct __align__(16) MSmem {
  float t3[BOX];
  union {
    struct {
      uint4 hi[2][2][NN];  // [buffer][k half][column]: FP16 hi of 8 k (planes 0, 1 of read_frags)
      uint4 lo[2][2][NN];  // FP16 lo of the same 8 k (planes 2, 3)
    } g;
    struct {
      double dp[512];  // e_p4 + e_p5 + e_p6 over the box's particles (p4 | p5<<3 | p6<<6)
    } d;
    struct {
      float t1[S1P][32];    // [slot][pa*4 + hi]
      float v1[S1P][1088];  // [slot][hk + 4 hj + 16 pc + 128 pb]; p4 slots (hk + 4 hj) * 68 + 8 pc + pb
    } s;
  } u;
  unsigned short rowt[9][NM];  // box index part of row m of bipartition g
  unsigned short colt[9][NN];  // box index part of column n
  double eps[36];  // h1,h2,h3 (4 each) at 0,4,8; p4,p5,p6 (8 each) at 12,20,28
  double red[2 * NW];
  float  scale[18];  // scale of each contraction part of the box's task
  int    start[6];   // first orbital of the box per position
  int    ext[6];     // orbitals of the box inside the task tile
  int    rc[9];      // rows | columns << 16 of bipartition g
  struct {
    uint64_t a, b;              // addresses of the operand rows of the box's first orbitals
    unsigned             a1, a2, b1, b2;  // bytes per orbital of pA, pB, hA, hB
  } part[18];
};

// bit position of each t3 index in the box layout (2 bits per hole, 3 per particle)
__host__ __device__ constexpr int sh(int pos) { return pos < 3 ? 2 * pos : 6 + 3 * (pos - 3); }
__host__ __device__ constexpr int ext(int pos) { return pos < 3 ? 4 : 8; }
__host__ __device__ constexpr int pair_a(int s) { return s == 0 ? 1 : 0; }
__host__ __device__ constexpr int pair_b(int s) { return s == 2 ? 1 : 2; }

// Storage index of box element e = sum idx << sh: the particle bits are xored
// into the six hole bits (the LDS bank).  A flush's 64 lanes differ in the
// three ps bits, two hA bits and the low pA bit; these masks make the six
// independent for every bipartition (hA is h1 or h2: masks 5 and 10 have a bit
// in both), and the energy sweeps' lanes differ in the hole bits alone.  The
// map is linear, so a row's part and a column's part combine by xor.
__host__ __device__ constexpr int swz(int e) {
  const int p4 = (e >> 6) & 7, p56 = ((e >> 9) ^ (e >> 12)) & 7, x = p4 ^ p56;
  return e ^ ((p56 & 1) ? 5 : 0) ^ ((x & 2) ? 10 : 0) ^ ((x & 4) ? 16 : 0) ^ ((p4 & 1) ? 32 : 0);
}

__device__ __forceinline__ void pair_of(int s, int& a, int& b) {
  a = pair_a(s);
  b = pair_b(s);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for(int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ h8 as_h8(uint4 u) { return __builtin_bit_cast(h8, u); }
// The thread index as a value the compiler cannot see through: what a phase
// derives from it is computed in that phase instead of being held in registers
// (or spilled) through the others.
__device__ __forceinline__ int thread_id() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// n / e for 0 <= n < 256 and 1 <= e <= 8 (the half keeps the product at least
// 1/16 from an integer, far beyond the reciprocal's error)
__device__ __forceinline__ int small_div(int n, int e) {
  return (int) (((float) n + 0.5f) * __builtin_amdgcn_rcpf((float) e));
}
// Coordinates of item n of a (fast a, then b, then c) numbering of extents ea, eb.
__device__ __forceinline__ void split3(int n, int ea, int eb, int& a, int& b, int& c) {
  const int t = small_div(n, ea);
  a           = n - t * ea;
  c           = small_div(t, eb);
  b           = t - c * eb;
}

// Operand array and first-term flag of the term c1*x - c2*y of a spin-orbital
// element (bits bx, by of the part code): both terms -> the antisymmetrised
// array (holding x - y), one term -> the plain array.
__host__ __device__ __forceinline__ void choose_term(unsigned c, unsigned bx, unsigned by, int both,
                                                     int single, int& arr, bool& first, float& coef) {
  const bool hx = (c & bx) != 0, hy = (c & by) != 0;
  arr   = hx && hy ? both : single;
  first = hx;
  coef  = (hx || hy) ? (hx ? 1.f : -1.f) : 0.f;
}

// MFMA tiles of one wave in a bipartition of R rows and C columns: row tile
// rt and column tiles ct .. ct + nj - 1 (32 each).  Five to eight row tiles:
// one each, all columns.  Up to four (two): two (four) waves share a row tile
// and split its columns, so that every SIMD has work (waves w and w + 4 share
// one).
struct WaveTiles {
  int nj, rt, ct;
};
__device__ __forceinline__ WaveTiles wave_tiles(int rc, int wave) {
  const int mt = ((rc & 0xffff) + 31) >> 5, nt = ((rc >> 16) + 31) >> 5;
  const int lg = mt > 4 ? 3 : mt > 2 ? 2 : mt > 1 ? 1 : 0;  // row tiles rounded up to 2^lg
  const int rt = wave & ((1 << lg) - 1), part = wave >> lg;  // 2^(3-lg) shares of the columns
  const int per = (nt + (1 << (3 - lg)) - 1) >> (3 - lg);
  WaveTiles W;
  W.rt = rt;
  W.ct = part * per;
  W.nj = rt < mt ? max(0, min(per, nt - W.ct)) : 0;
  return W;
}

// Entry of the box's part table: where the operand rows of part gp start and
// what the pair coordinates add (a row's neighbour along hs or ps is 32 bytes
// away).
__device__ __forceinline__ void part_entry(MSmem& sm, const MixedDev& M, int gp, unsigned code) {
  const int g = gp >> 1, d2 = gp & 1, hs = g / 3, ps = g % 3;
  int       hA, hB, pA, pB, arr;
  bool      first;
  float     coef;
  pair_of(hs, hA, hB);
  pair_of(ps, pA, pB);
  const long O = M.O, V = M.V, K = d2 ? M.Kv : M.Ko;
  {
    // t2h[a][b][i]: pairs (pA,pB) or (pB,pA); xv[c][b][i]: (pB,pA) or (pA,pB); row hs
    choose_term(code, 4, 8, d2 ? 5 : 1, d2 ? 4 : 0, arr, first, coef);
    const bool pa_slow = first == (d2 == 0);
    const long PA = sm.start[3 + pA], PB = sm.start[3 + pB], one = K * O * 4;
    sm.part[gp].a  = (uint64_t) M.v[arr] + (pa_slow ? PA * V + PB : PB * V + PA) * one + 32l * sm.start[hs];
    sm.part[gp].a1 = (unsigned) (pa_slow ? V * one : one);
    sm.part[gp].a2 = (unsigned) (pa_slow ? one : V * one);
  }
  {
    // ovk: pairs (hB,hA) or (hA,hB); t2p: (hA,hB) or (hB,hA); row ps
    choose_term(code, 16, 32, d2 ? 7 : 3, d2 ? 6 : 2, arr, first, coef);
    const bool ha_slow = first == (d2 != 0);
    const long HA = sm.start[hA], HB = sm.start[hB], one = K * V * 4;
    sm.part[gp].b  = (uint64_t) M.v[arr] + (ha_slow ? HA * O + HB : HB * O + HA) * one + 32l * sm.start[3 + ps];
    sm.part[gp].b1 = (unsigned) (ha_slow ? O * one : one);
    sm.part[gp].b2 = (unsigned) (ha_slow ? one : O * one);
  }
}

// This thread's source of one operand in part d2 of bipartition g, as a base
// shared by the workgroup and a 32-bit offset (the pair strides times seven
// stay below 2^32 for arrays that fit the device): the A row of its lane (row
// 32 rt + lane%32, k half lane/32), or its 16-byte piece of a B column (column
// tid%128, piece tid/128 = [hi k0-7 | lo k0-7 | hi k8-15 | lo k8-15]).  Rows
// and columns past the last read the last one: their products are never
// flushed.
struct Src {
  uint64_t base;
  unsigned off;
  __device__ __forceinline__ global_u4 at() const { return (global_u4) (base + off); }
};
__device__ __forceinline__ uint64_t uni64(uint64_t u) {
  return (uint64_t) (unsigned) uni((int) (u >> 32)) << 32 | (uint64_t) (unsigned) uni((int) (unsigned) u);
}
__device__ __forceinline__ Src src_a(const MSmem& sm, const MixedDev& M, int g, int d2) {
  const int   tid = thread_id(), lane = tid & 63, wave = uni(tid >> 6);
  const int   hs = g / 3, ps = g % 3, pA = pair_a(ps), pB = pair_b(ps);
  const auto& E  = sm.part[2 * g + d2];
  const int   rc = uni(sm.rc[g]);
  const int   v  = sm.rowt[g][min(32 * wave_tiles(rc, wave).rt + (lane & 31), (rc & 0xffff) - 1)];
  Src         S;
  S.base = uni64(E.a);
  S.off  = ((v >> sh(3 + pA)) & 7) * E.a1 + ((v >> sh(3 + pB)) & 7) * E.a2 +
          ((swz(v) >> sh(hs)) & 3) * 32u + (unsigned) (lane >> 5) * 32u * (unsigned) M.O;
  return S;
}
__device__ __forceinline__ Src src_b(const MSmem& sm, const MixedDev& M, int g, int d2) {
  const int   tid = thread_id(), piece = uni(tid >> 7);
  const int   hs = g / 3, ps = g % 3, hA = pair_a(hs), hB = pair_b(hs);
  const auto& E = sm.part[2 * g + d2];
  const int   v = sm.colt[g][min(tid & 127, (uni(sm.rc[g]) >> 16) - 1)], h = swz(v);
  Src         S;
  S.base = uni64(E.b);
  S.off  = ((h >> sh(hA)) & 3) * E.b1 + ((h >> sh(hB)) & 3) * E.b2 + ((v >> sh(3 + ps)) & 7) * 32u +
          (unsigned) (piece >> 1) * 32u * (unsigned) M.V + 16u * (piece & 1);
  return S;
}

// Writes a chunk's B piece into LDS buffer `buf` (a wave writes 64 consecutive
// columns of one plane).
__device__ __forceinline__ void stage(MSmem& sm, u4v b, int buf) {
  const int tid = threadIdx.x, n = tid & 127, piece = tid >> 7;
  uint4*    plane = (piece & 1) ? &sm.u.g.lo[buf][piece >> 1][n] : &sm.u.g.hi[buf][piece >> 1][n];
  *plane          = __builtin_bit_cast(uint4, b);
}

struct Frags {
  h8 bhi[4], blo[4];
};

// Fragment of one column tile: plane 0, 1 hi of buffer 0, 1; planes 2, 3 lo.
__device__ __forceinline__ h8 read_frag(const uint4* col, int plane) { return as_h8(col[2 * NN * plane]); }

// acc[j] += ahi bhi[j], then ahi blo[j] (mfma_hi); acc[j] += alo bhi[j]
// (mfma_lo), for j < nj.  In assembly because of the branch: around builtins
// the compiler kept a copy of the 64 accumulators per path (up to 691 spilled
// registers).  The blocks are closed towards the rest of the code: the nops in
// front cover a vector write of the accumulators before them (flush),
// acc_ready() a read after them; matrix instructions on the same accumulators
// need none between them.
__device__ __forceinline__ void mfma_hi(int nj, h8 a, const h8 (&bh)[4], const h8 (&bl)[4], f16v (&acc)[4]) {
  asm volatile(
    "s_nop 1\n\t"
    "s_cmp_lt_i32 %[nj], 4\n\t"
    "s_cbranch_scc1 .Lnj3_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c0], %[a], %[h0], %[c0]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c1], %[a], %[h1], %[c1]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c2], %[a], %[h2], %[c2]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c3], %[a], %[h3], %[c3]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c0], %[a], %[l0], %[c0]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c1], %[a], %[l1], %[c1]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c2], %[a], %[l2], %[c2]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c3], %[a], %[l3], %[c3]\n\t"
    "s_branch .Lnj0_%=\n"
    ".Lnj3_%=:\n\t"
    "s_cmp_lt_i32 %[nj], 1\n\t"
    "s_cbranch_scc1 .Lnj0_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c0], %[a], %[h0], %[c0]\n\t"
    "s_cmp_lt_i32 %[nj], 2\n\t"
    "s_cbranch_scc1 .Lnj1_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c1], %[a], %[h1], %[c1]\n\t"
    "s_cmp_lt_i32 %[nj], 3\n\t"
    "s_cbranch_scc1 .Lnj2_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c2], %[a], %[h2], %[c2]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c2], %[a], %[l2], %[c2]\n"
    ".Lnj2_%=:\n\t"
    "v_mfma_f32_32x32x16_f16 %[c1], %[a], %[l1], %[c1]\n"
    ".Lnj1_%=:\n\t"
    "v_mfma_f32_32x32x16_f16 %[c0], %[a], %[l0], %[c0]\n"
    ".Lnj0_%=:\n"
    : [c0] "+v"(acc[0]), [c1] "+v"(acc[1]), [c2] "+v"(acc[2]), [c3] "+v"(acc[3])
    : [nj] "s"(nj), [a] "v"(a), [h0] "v"(bh[0]), [h1] "v"(bh[1]), [h2] "v"(bh[2]), [h3] "v"(bh[3]),
      [l0] "v"(bl[0]), [l1] "v"(bl[1]), [l2] "v"(bl[2]), [l3] "v"(bl[3])
    : "scc");
}
__device__ __forceinline__ void mfma_lo(int nj, h8 a, const h8 (&bh)[4], f16v (&acc)[4]) {
  asm volatile(
    "s_nop 1\n\t"
    "s_cmp_lt_i32 %[nj], 4\n\t"
    "s_cbranch_scc1 .Lnj3_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c0], %[a], %[h0], %[c0]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c1], %[a], %[h1], %[c1]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c2], %[a], %[h2], %[c2]\n\t"
    "v_mfma_f32_32x32x16_f16 %[c3], %[a], %[h3], %[c3]\n\t"
    "s_branch .Lnj0_%=\n"
    ".Lnj3_%=:\n\t"
    "s_cmp_lt_i32 %[nj], 1\n\t"
    "s_cbranch_scc1 .Lnj0_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c0], %[a], %[h0], %[c0]\n\t"
    "s_cmp_lt_i32 %[nj], 2\n\t"
    "s_cbranch_scc1 .Lnj0_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c1], %[a], %[h1], %[c1]\n\t"
    "s_cmp_lt_i32 %[nj], 3\n\t"
    "s_cbranch_scc1 .Lnj0_%=\n\t"
    "v_mfma_f32_32x32x16_f16 %[c2], %[a], %[h2], %[c2]\n"
    ".Lnj0_%=:\n"
    : [c0] "+v"(acc[0]), [c1] "+v"(acc[1]), [c2] "+v"(acc[2]), [c3] "+v"(acc[3])
    : [nj] "s"(nj), [a] "v"(a), [h0] "v"(bh[0]), [h1] "v"(bh[1]), [h2] "v"(bh[2]), [h3] "v"(bh[3])
    : "scc");
}

// Waits until vector instructions may read or write the accumulators (19 wait
// states cover the longest matrix instruction in flight).
__device__ __forceinline__ void acc_ready(f16v (&acc)[4]) {
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
}

// Adds the scaled accumulators of a bipartition into the box (the first
// bipartition of a box stores instead) and clears them.  D layout of
// v_mfma_f32_32x32x16_f16: register q of lane l holds row 8*(q/4) + 4*(l/32)
// + q%4, column l%32.  Rows and columns past the last have table entries
// outside the tile (nothing reads those elements).
__device__ __forceinline__ void flush(MSmem& sm, int g, const WaveTiles& W, float sc, bool store,
                                      f16v (&acc)[4]) {
  const int tid = thread_id();
  const int lane = tid & 63;
  int       ro[4][4];
#pragma unroll
  for(int qq = 0; qq < 4; qq++) {
    const ushort4 r = *reinterpret_cast<const ushort4*>(&sm.rowt[g][32 * W.rt + 8 * qq + 4 * (lane >> 5)]);
    ro[qq][0]       = r.x;
    ro[qq][1]       = r.y;
    ro[qq][2]       = r.z;
    ro[qq][3]       = r.w;
  }
#pragma unroll
  for(int j = 0; j < 4; j++) {
    if(j < W.nj) {
      const int co = sm.colt[g][32 * (W.ct + j) + (lane & 31)];
      if(store) {
#pragma unroll
        for(int q = 0; q < 16; q++) sm.t3[ro[q >> 2][q & 3] ^ co] = acc[j][q] * sc;
      }
      else {
        float v[16];
#pragma unroll
        for(int q = 0; q < 16; q++) v[q] = sm.t3[ro[q >> 2][q & 3] ^ co];
#pragma unroll
        for(int q = 0; q < 16; q++) sm.t3[ro[q >> 2][q & 3] ^ co] = v[q] + acc[j][q] * sc;
      }
    }
  }
#pragma unroll
  for(int j = 0; j < 4; j++)
#pragma unroll
    for(int q = 0; q < 16; q++) acc[j][q] = 0.f;
}

__device__ __forceinline__ bool part_on(uint64_t d1, uint64_t d2, int gp) {
  const uint64_t c = (gp & 1) ? d2 : d1;
  return (c >> (6 * (gp >> 1))) & 1;
}
__device__ __forceinline__ unsigned part_code(uint64_t d1, uint64_t d2, int gp) {
  const uint64_t c = (gp & 1) ? d2 : d1;
  return (unsigned) (c >> (6 * (gp >> 1))) & 63u;
}

// Row and column tables of the nine bipartitions of a box of extents sm.ext.
// Padding rows (columns) of the last 32 get an index outside the tile: some
// extent of their side is short wherever there is one.
__device__ __forceinline__ void box_tables(MSmem& sm) {
  for(int x = thread_id(); x < 9 * (NM + NN); x += NT) {
    const int  g = x / (NM + NN), y = x - g * (NM + NN), hs = g / 3, ps = g % 3;
    const bool row = y < NM;
    int        hA, hB, pA, pB;
    pair_of(hs, hA, hB);
    pair_of(ps, pA, pB);
    const int q0 = row ? hs : 3 + ps, q1 = row ? 3 + pA : hA, q2 = row ? 3 + pB : hB;
    const int e0 = sm.ext[q0], e1 = sm.ext[q1], e2 = sm.ext[q2], n = row ? y : y - NM;
    int       a, b, c;
    split3(n, e0, e1, a, b, c);
    if(c >= e2) {
      a = e0 < ext(q0) ? e0 : 0;
      b = e0 < ext(q0) ? 0 : e1 < ext(q1) ? e1 : 0;
      c = e0 < ext(q0) || e1 < ext(q1) ? 0 : e2 & (ext(q2) - 1);
    }
    const int v = swz((a << sh(q0)) | (b << sh(q1)) | (c << sh(q2)));
    if(row) sm.rowt[g][n] = (unsigned short) v;
    else sm.colt[g][n] = (unsigned short) v;
    if(y == 0) sm.rc[g] = e0 * e1 * e2 | (sm.ext[3 + ps] * sm.ext[hA] * sm.ext[hB]) << 16;
  }
}

__device__ __forceinline__ void box_contract(MSmem& sm, const MixedDev& M, uint64_t d1, uint64_t d2) {
  // the d1 and d2 equations of a bipartition are enabled together (both
  // contract an index of the same spin), n1 chunks of h7 and then n2 of p7
  unsigned on = 0;
#pragma unroll
  for(int g = 0; g < 9; g++) on |= (unsigned) ((d1 >> (6 * g)) & 1) << g;
  on = uni(on);
  if(on == 0) {
    for(int e = threadIdx.x; e < BOX; e += NT) sm.t3[e] = 0.f;
    return;
  }
  const int n1 = M.Ko / KC, n2 = M.Kv / KC, nb = n1 + n2;
  // chunk count padded to a multiple of the ring depth, so the loop body is
  // the same for every chunk; the chunks past the end repeat the last loads
  // and are not flushed
  const int total_pad = (__builtin_popcount(on) * nb + PF - 1) / PF * PF;
  const int tid = thread_id(), wave = uni(tid >> 6), lane = tid & 63;
  const long sa = 64l * M.O, sb = 64l * M.V;  // bytes per chunk
  auto next = [&](int g) {  // enabled bipartition after g, or 9
    const unsigned rest = g < 8 ? on >> (g + 1) : 0u;
    return rest ? g + 1 + __builtin_ctz(rest) : 9;
  };
  f16v acc[4];
#pragma unroll
  for(int j = 0; j < 4; j++)
#pragma unroll
    for(int q = 0; q < 16; q++) acc[j][q] = 0.f;
  const int g0 = __builtin_ctz(on);
  // load cursors, one per operand: A runs PF - 1 chunks ahead of the MFMAs (a
  // slot is free once its chunk is multiplied), B runs PF ahead (its slot is
  // free once its piece is in LDS), so that a piece is loaded two iterations
  // before it is staged.  Past the last bipartition a cursor repeats its last
  // chunk.
  struct Cursor {
    Src src;
    int g, d2, left;  // bipartition, part, chunks left in the part
  };
  auto advance = [&](Cursor& c, bool isa, long step) {
    if(--c.left) {
      c.src.base += step;
      return;
    }
    c.d2 ^= 1;
    if(!c.d2) {
      const int ng = next(c.g);
      if(ng == 9) {
        c.d2   = 1;
        c.left = 1;
        return;
      }
      c.g = ng;
    }
    c.left = c.d2 ? n2 : n1;
    c.src  = isa ? src_a(sm, M, c.g, c.d2) : src_b(sm, M, c.g, c.d2);
  };
  Cursor ca = {src_a(sm, M, g0, 0), g0, 0, n1}, cb = {src_b(sm, M, g0, 0), g0, 0, n1};
  u4v    ra[PF][2], rb[PF];  // hi, lo of this lane's 8 k; this thread's B piece
  auto   load_a = [&](u4v(&a)[2]) {
    a[0] = ca.src.at()[0];
    a[1] = ca.src.at()[1];
    advance(ca, true, sa);
  };
  auto load_b = [&](u4v& b) {
    b = *cb.src.at();
    advance(cb, false, sb);
  };
#pragma unroll
  for(int s = 0; s < PF; s++) {
    load_b(rb[s]);
    if(s < PF - 1) load_a(ra[s]);
  }
  // compute cursor, and the position of the chunk whose fragments are read next
  int          cg = g0, cd2 = 0, cleft = n1, rleft = nb;
  bool         store = true;
  WaveTiles    W = wave_tiles(uni(sm.rc[cg]), wave);
  const uint4* col0 = &sm.u.g.hi[0][lane >> 5][lane & 31];
  const uint4* col[4];
  auto         set_cols = [&](int ct) {
#pragma unroll
    for(int j = 0; j < 4; j++) col[j] = col0 + 32 * ((ct + j) & 3);
  };
  set_cols(W.ct);
  Frags F[2];
  // prologue: chunks 0 and 1 staged, fragments of chunk 0 read
  stage(sm, rb[0], 0);
  stage(sm, rb[1], 1);
  __syncthreads();
#pragma unroll
  for(int j = 0; j < 4; j++) {
    F[0].bhi[j] = read_frag(col[j], 0);
    F[0].blo[j] = read_frag(col[j], 2);
  }
  __syncthreads();
  // iteration it (chunk it: A in ra[it % PF], B fragments in F[it & 1]): stage
  // chunk it+2 into buffer it&1 (its fragments were read before the previous
  // barrier), read the fragments of chunk it+1 (buffer (it+1)&1) and issue the
  // loads into the slots that became free, around the twelve MFMAs; flush at
  // the end of a bipartition; one barrier.  A wave issues one instruction per
  // four cycles and two waves share a SIMD, so beside 768 cycles of MFMA the
  // loop has room for few others: the cursors count down to their next part,
  // and everything else about a part sits behind those four tests (the tests
  // and cursor moves took 62 scalar instructions and 25 branches a chunk).
#pragma unroll 1
  for(int it0 = 0; it0 < total_pad; it0 += PF) {
#pragma unroll
    for(int s = 0; s < PF; s++) {
      if(--rleft == 0) {
        rleft        = nb;
        const int ng = next(cg);
        set_cols(wave_tiles(uni(sm.rc[ng < 9 ? ng : cg]), wave).ct);
      }
      Frags &Fc = F[s & 1], &Fn = F[(s + 1) & 1];
      const h8 ahi = __builtin_bit_cast(h8, ra[s][0]), alo = __builtin_bit_cast(h8, ra[s][1]);
      stage(sm, rb[(s + 2) % PF], s & 1);
#pragma unroll
      for(int j = 0; j < 4; j++) Fn.bhi[j] = read_frag(col[j], (s + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
      mfma_hi(W.nj, ahi, Fc.bhi, Fc.blo, acc);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for(int j = 0; j < 4; j++) Fn.blo[j] = read_frag(col[j], 2 + ((s + 1) & 1));
      load_b(rb[s]);
      load_a(ra[(s + PF - 1) % PF]);
      __builtin_amdgcn_sched_barrier(0);
      mfma_lo(W.nj, alo, Fc.bhi, acc);
      __builtin_amdgcn_sched_barrier(0);
      if(--cleft == 0) {
        // The d1 part of a bipartition carries its accumulators into the d2
        // part (the same box elements), rescaled by the ratio of the two part
        // scales (both +-2^k, so the ratio is exact).  Ratios outside 2^+-60
        // flush instead, keeping the FP32 range.
        const float sc    = sm.scale[2 * cg + cd2];
        bool        carry = false;
        acc_ready(acc);
        if(!cd2) {
          const float r = sc / sm.scale[2 * cg + 1];
          carry         = uni(fabsf(r) >= 0x1p-60f && fabsf(r) <= 0x1p60f);
          if(carry)
#pragma unroll
            for(int j = 0; j < 4; j++)
#pragma unroll
              for(int q = 0; q < 16; q++) acc[j][q] *= r;
        }
        if(!carry) {
          flush(sm, cg, W, sc, store, acc);
          store = false;
        }
        cd2 ^= 1;
        cleft = n2;
        if(!cd2) {
          const int ng = next(cg);
          cleft        = ng < 9 ? n1 : total_pad;  // past the last one only padding chunks are left
          if(ng < 9) {
            cg = ng;
            W  = wave_tiles(uni(sm.rc[cg]), wave);
          }
        }
      }
      __syncthreads();
    }
  }
  acc_ready(acc);  // the padding chunks' instructions are done with the registers
}

// Denominator reciprocal in FP64: hardware estimate refined by two Newton
// steps (error below one ulp; |D| is bounded away from zero by the gap).
__device__ __forceinline__ double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  double e = fma(-d, r, 1.0);
  r        = fma(r, e, r);
  e        = fma(-d, r, 1.0);
  return fma(r, e, r);
}

// s1 term of S1P slots starting at S0, staged in LDS: returns this thread's
// sum over its elements of (t3/D) * s.  W = t3/D is already in sm.t3 for the
// threads inside the tile (zero where p5 is outside), T1 and V blocks are zero
// outside the tile.
//
// The thread's elements are every (p5, p6) for its own (h1, h2, h3, p4) (the
// bits of tid; tb is their storage index), and the slots of one sweep share
// their particle position pa = S0/3.  So a sweep needs one T1 value and
// 64 V values per slot (pa = p4), or 8 and 8 (pa = p5, p6): each is read from
// LDS once instead of once per element.  Per element the slots are summed in
// FP32 in slot order and the products W*s added in FP64 in element order, as
// an element-by-element loop would.
template<int S0>
__device__ __forceinline__ double s1_sweep(const MSmem& sm, int tb, int n6) {
  static_assert(S0 % 3 == 0 && S1P == 3, "a sweep covers the three slots of one pa");
  constexpr int pa = S0 / 3;
  const int     tid = thread_id();
  const int     hidx[3] = {tid & 3, (tid >> 2) & 3, (tid >> 4) & 3};
  const int     p4 = (tid >> 6) & 7;
  int           vb[S1P], th[S1P];  // per slot: h part of the V index, T1 hole index
#pragma unroll
  for(int q = 0; q < S1P; q++) {
    const int hi = (S0 + q) % 3;
    int       hj, hk;
    pair_of(hi, hj, hk);
    vb[q] = hidx[hk] + 4 * hidx[hj];
    th[q] = hidx[hi];
  }
  double es = 0.0;
  if constexpr(pa == 0) {  // T1 by p4 (one value per slot); V by (pc, pb) = (p6, p5)
    float t[S1P];
#pragma unroll
    for(int q = 0; q < S1P; q++) t[q] = sm.u.s.t1[q][p4 * 4 + th[q]];
    // these slots are stored with pb (= p5) contiguous: the 8 values of one p6
    // are two 16-byte reads
#pragma unroll 1
    for(int p6 = 0; p6 < n6; p6++) {
      const int tp = tb ^ swz(p6 << 12);
      float4    v[S1P][2];
#pragma unroll
      for(int q = 0; q < S1P; q++) {
        const float4* r = reinterpret_cast<const float4*>(&sm.u.s.v1[q][vb[q] * 68 + 8 * p6]);
        v[q][0]         = r[0];
        v[q][1]         = r[1];
      }
#pragma unroll
      for(int p5 = 0; p5 < 8; p5++) {
        float sv = 0.f;
#pragma unroll
        for(int q = 0; q < S1P; q++) {
          const float4 h = v[q][p5 >> 2];
          const int    i = p5 & 3;
          sv += t[q] * (i == 0 ? h.x : i == 1 ? h.y : i == 2 ? h.z : h.w);
        }
        es += (double) (sm.t3[tp ^ swz(p5 << 9)] * sv);
      }
    }
  }
  else {
    // pa = p5: T1 by p5, V by (pc, pb) = (p6, p4); pa = p6: T1 by p6, V by (p5, p4).
    // The operand indexed by p5 is held for the whole sweep (constant indices
    // in the unrolled p5 loop); the one indexed by p6 is read per p6.
    float hold[S1P][8];
#pragma unroll
    for(int q = 0; q < S1P; q++)
#pragma unroll
      for(int k = 0; k < 8; k++)
        hold[q][k] = pa == 1 ? sm.u.s.t1[q][k * 4 + th[q]] : sm.u.s.v1[q][vb[q] + 16 * k + 128 * p4];
#pragma unroll 1
    for(int p6 = 0; p6 < n6; p6++) {
      const int tp = tb ^ swz(p6 << 12);
      float     per[S1P];
#pragma unroll
      for(int q = 0; q < S1P; q++)
        per[q] = pa == 1 ? sm.u.s.v1[q][vb[q] + 16 * p6 + 128 * p4] : sm.u.s.t1[q][p6 * 4 + th[q]];
#pragma unroll
      for(int p5 = 0; p5 < 8; p5++) {
        float sv = 0.f;
#pragma unroll
        for(int q = 0; q < S1P; q++) sv += pa == 1 ? hold[q][p5] * per[q] : per[q] * hold[q][p5];
        es += (double) (sm.t3[tp ^ swz(p5 << 9)] * sv);
      }
    }
  }
  return es;
}

// Loads (into registers) the T1 entries and <hk hj||pc pb> blocks of slots
// S0..S0+S1P-1.  Consecutive threads read consecutive hj, the contiguous index
// of vvoo[c][b][k][j].
constexpr int S1V = 1024 / NT;  // block elements per thread and slot
struct S1Regs {
  double v[S1P][S1V];
  double t[S1P];
};

template<int S0>
__device__ __forceinline__ void s1_load(const MSmem& sm, const MixedDev& M, uint64_t s1code,
                                        S1Regs& R) {
  const int  tid = thread_id();
  const long O = M.O, V = M.V;
#pragma unroll
  for(int q = 0; q < S1P; q++) {
    const int slot = S0 + q;
    R.t[q]         = 0.0;
#pragma unroll
    for(int j = 0; j < S1V; j++) R.v[q][j] = 0.0;
    if(slot >= 9) continue;
    const unsigned c  = (unsigned) (s1code >> (4 * slot)) & 15u;
    const int      pa = slot / 3, hi = slot % 3;
    int            hj, hk, pb, pc;
    pair_of(hi, hj, hk);
    pair_of(pa, pb, pc);
    if(!(c & 1)) continue;
    if(tid < 32) {
      const int gp = tid >> 2, gh = tid & 3;
      if(gp < sm.ext[3 + pa] && gh < sm.ext[hi]) {
        const double t = M.t1[(long) (sm.start[3 + pa] + gp) * O + sm.start[hi] + gh];
        R.t[q]         = (c & 2) ? -t : t;
      }
    }
#pragma unroll
    for(int j = 0; j < S1V; j++) {
      const int w  = tid + NT * j;
      const int gj = w & 3, gk = (w >> 2) & 3, gc = (w >> 4) & 7, gb = w >> 7;
      if(gk < sm.ext[hk] && gj < sm.ext[hj] && gc < sm.ext[3 + pc] && gb < sm.ext[3 + pb]) {
        const long K = sm.start[hk] + gk, J = sm.start[hj] + gj, PC = sm.start[3 + pc] + gc,
                   PB = sm.start[3 + pb] + gb;
        double x = 0.0;
        if(c & 4) x = M.vvoo[((PC * V + PB) * O + K) * O + J];
        if(c & 8) x -= M.vvoo[((PB * V + PC) * O + K) * O + J];
        R.v[q][j] = x;
      }
    }
  }
}

// Stores S1P slots starting at S0.  The slots of particle position p4 (S0 = 0)
// go to (k + 4 j) * 68 + 8 c + b, so that their sweep reads b (= p5) runs;
// 68 rather than 64 keeps the stores of a wave on distinct banks but for pairs.
template<int S0>
__device__ __forceinline__ void s1_store(MSmem& sm, const S1Regs& R) {
  const int tid = thread_id();
#pragma unroll
  for(int q = 0; q < S1P; q++) {
    if(tid < 32) sm.u.s.t1[q][tid] = (float) R.t[q];
#pragma unroll
    for(int j = 0; j < S1V; j++) {
      const int w = tid + NT * j;  // (j, k, c, b) -> stored as k + 4 j + 16 c + 128 b
      const int o = S0 == 0 ? (((w >> 2) & 3) + 4 * (w & 3)) * 68 + 8 * ((w >> 4) & 7) + (w >> 7)
                            : ((w >> 2) & 3) + 4 * (w & 3) + (w & ~15);
      sm.u.s.v1[q][o] = (float) R.v[q][j];
    }
  }
}

// Energy of the box: E4 = sum t3^2/D and E5 = E4 + sum t3*s/D over the tile
// elements of the box (FP64 sums of per-element terms; t3 and s in FP32).
__device__ __forceinline__ void box_energy(MSmem& sm, const MixedDev& M, uint64_t s1code, double& e4,
                           double& e5) {
  const int tid = thread_id();
  S1Regs    R;
  s1_load<0>(sm, M, s1code, R);  // in flight during the E4 sweep
  // separable denominators, in the order of the reference's sum
  for(int y = tid; y < 512; y += NT)
    sm.u.d.dp[y] = (sm.eps[28 + (y >> 6)] + sm.eps[20 + ((y >> 3) & 7)]) + sm.eps[12 + (y & 7)];
  __syncthreads();
  const int    h1 = tid & 3, h2 = (tid >> 2) & 3, h3 = (tid >> 4) & 3, p4 = tid >> 6;
  const int    n5 = uni(sm.ext[4]), n6 = uni(sm.ext[5]), tb = swz(tid);
  const double dh = (sm.eps[8 + h3] + sm.eps[4 + h2]) + sm.eps[h1];
  const bool   in = h1 < sm.ext[0] && h2 < sm.ext[1] && h3 < sm.ext[2] && p4 < sm.ext[3];
  e4              = 0.0;
  auto elem       = [&](int at, int y) {
    const double d  = (double) sm.t3[at];
    const double di = d * recip(dh - sm.u.d.dp[y]);
    e4 += d * di;
    sm.t3[at] = (float) di;
  };
  if(in)
    for(int p6 = 0; p6 < n6; p6++) {
      const int tp = tb ^ swz(p6 << 12), y = p4 + 64 * p6;
      if(n5 == 8) {
#pragma unroll
        for(int p5 = 0; p5 < 8; p5++) elem(tp ^ swz(p5 << 9), y + 8 * p5);
      }
      else {
        for(int p5 = 0; p5 < n5; p5++) elem(tp ^ swz(p5 << 9), y + 8 * p5);
        for(int p5 = n5; p5 < 8; p5++) sm.t3[tp ^ swz(p5 << 9)] = 0.f;
      }
    }
  double es = 0.0;
  if(s1code & 0x111111111ull) {
    __syncthreads();  // denominators no longer needed; W complete
    s1_store<0>(sm, R);
    s1_load<S1P>(sm, M, s1code, R);
    __syncthreads();
    if(in) es += s1_sweep<0>(sm, tb, n6);
    __syncthreads();
    s1_store<S1P>(sm, R);
    s1_load<2 * S1P>(sm, M, s1code, R);
    __syncthreads();
    if(in) es += s1_sweep<S1P>(sm, tb, n6);
    __syncthreads();
    s1_store<2 * S1P>(sm, R);
    __syncthreads();
    if(in) es += s1_sweep<2 * S1P>(sm, tb, n6);
  }
  e5                  = e4 + es;
  const int lane = tid & 63, wave = tid >> 6;
  e4 = wave_sum(e4);
  e5 = wave_sum(e5);
  if(lane == 0) {
    sm.red[wave]      = e4;
    sm.red[NW + wave] = e5;
  }
  __syncthreads();
  if(tid == 0) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for(int w = 0; w < NW; w++) {
      a += sm.red[w];
      b += sm.red[NW + w];
    }
    e4 = a;
    e5 = b;
  }
}

// Persistent kernel: workgroup b serves queue b % kQueues first (dispatch is
// round-robin over the 8 XCDs, so that is its own XCD's queue), then steals
// from the others; one ticket = one box.  Thread 0 claims and decodes each
// ticket (its entry searched forward from its previous one) and keeps the
// running exact sums of the task its boxes belong to, which go to the task's
// global accumulator when the task changes and when the workgroup leaves.
__global__ void __launch_bounds__(NT) k_spatial_mixed(MixedDev M, RunDev R) {
  __shared__ MSmem              sm;
  __shared__ int                s_task;
  __shared__ int                s_retable; // thread 0: the box's extents differ from the last one's
  __shared__ int                s_weight;  // thread 0: boxes that its box stands for
  __shared__ Claim              s_claim;   // thread 0; its task also for the others
  __shared__ int                s_cur;     // thread 0: task of the running sums
  __shared__ unsigned long long s_sum[4];  // thread 0: E4 lo, hi, E5 lo, hi of s_cur not yet added
  const int                     tid  = threadIdx.x;
  const int                     home = blockIdx.x % kQueues;
  if(tid == 0) {
    s_cur    = -1;
    s_sum[0] = s_sum[1] = s_sum[2] = s_sum[3] = 0ull;
#pragma unroll
    for(int p = 0; p < 6; p++) sm.ext[p] = 0;
  }
#pragma unroll 1
  for(int qi = 0; qi < kQueues; qi++) {
    const int q = (home + qi) % kQueues;
    if(tid == 0) claim_queue(s_claim, R, q);
#pragma unroll 1
    for(;;) {
      __syncthreads();
      if(tid == 0) {
        int       sub[6], weight;
        const int ti = claim_box(s_claim, R, q, claim_ticket(R, q), true, sub, weight);
        s_retable    = 0;
        if(ti >= 0) {
          s_weight         = weight;
          const TaskDev& T = s_claim.task;
#pragma unroll
          for(int p = 0; p < 6; p++) {
            const int x = min(ext(p), T.dim[p] - ext(p) * sub[p]);
            if(x != sm.ext[p]) s_retable = 1;
            sm.start[p] = T.off[p] + ext(p) * sub[p];
            sm.ext[p]   = x;
          }
        }
        s_task = ti;
      }
      __syncthreads();
      const int ti = s_task;
      if(ti < 0) break;
      if(tid >= 64 && tid < 64 + 18) sm.scale[tid - 64] = M.pscale[18 * (size_t) ti + tid - 64];
      if(s_retable) box_tables(sm);
      if(tid >= 128 && tid < 128 + 18) {
        const TaskDev& T = s_claim.task;
        part_entry(sm, M, tid - 128, part_code(T.d1code, T.d2code, tid - 128));
      }
      if(tid < 36) {
        const int p = tid < 12 ? tid / 4 : 3 + (tid - 12) / 8;
        const int i = tid < 12 ? tid % 4 : (tid - 12) % 8;
        sm.eps[tid] = i < sm.ext[p] ? (p < 3 ? M.eo : M.ev)[sm.start[p] + i] : 0.0;
      }
      __syncthreads();
      const TaskDev&           T  = s_claim.task;
      const unsigned long long t0 = wall_clock64();
      box_contract(sm, M, T.d1code, T.d2code);
      __syncthreads();
      double e4, e5;
      box_energy(sm, M, T.s1code, e4, e5);
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

// Per-row exponent: one wave per row, e = 13 - floor(log2(max|x|)); an
// all-zero row puts no constraint on its block (kNoRow).
constexpr int kNoRow = 200;

__global__ void k_row_exp(const double* __restrict__ x, long rows, long Kin, short* __restrict__ e) {
  const long row  = (long) blockIdx.x * 4 + (threadIdx.x >> 6);
  const int  lane = threadIdx.x & 63;
  if(row >= rows) return;
  double m = 0.0;
  for(long k = lane; k < Kin; k += 64) m = fmax(m, fabs(x[row * Kin + k]));
#pragma unroll
  for(int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  if(lane == 0) {
    int ex = kNoRow;
    if(m > 0.0) ex = 13 - ilogb(m);
    ex     = ex > kNoRow ? kNoRow : (ex < -kNoRow ? -kNoRow : ex);
    e[row] = (short) ex;
  }
}

// Row r = (x*D2 + y)*D3 + z of an operand array; each coordinate is an
// occupied (type 0) or virtual (type 1) orbital.  Its block is the tile
// triple of (x, y, z) in the same order.
struct BlockMap {
  long       D2, D3;
  int        n2, n3;                  // tiles of coordinates 2 and 3
  const int* t1;
  const int* t2;
  const int* t3;                      // orbital -> tile maps of the three coordinates
  __device__ long operator()(long r) const {
    const long z = r % D3, y = (r / D3) % D2, x = r / (D2 * D3);
    return ((long) t1[x] * n2 + t2[y]) * n3 + t3[z];
  }
};

__global__ void k_fill_i32(int* p, long n, int v) {
  const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) p[i] = v;
}

// Block exponent = min over the block's rows (the largest row sets it).
__global__ void k_block_exp(const short* __restrict__ er, long rows, BlockMap bm, int* eb) {
  const long r = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if(r >= rows) return;
  const int e = er[r];
  if(e < kNoRow) atomicMin(&eb[bm(r)], e);
}

// Split: y = x * 2^e[block(row)] = hi + lo (FP16), in the order of SplitBufs:
// one thread per 8 k of a row, neighbouring threads on neighbouring rows of a
// pair, so that a wave writes one run of 2 KB and reads 64-byte runs.  `mid`:
// the pair is (x, z) and the row y (the ovk arrays), else (x, y) and z.
__global__ void __launch_bounds__(256) k_split(const double* __restrict__ x, long rows, long Kin,
                                               long Kout, BlockMap bm, int mid,
                                               const int* __restrict__ eb, uint4* __restrict__ out) {
  const long R = mid ? bm.D2 : bm.D3, k8 = Kout / 8, n = rows * k8;
  for(long i = (long) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long) gridDim.x * blockDim.x) {
    const long q = i / R, r = i - q * R, pair = q / k8, k = 8 * (q - pair * k8);
    const long row = mid ? ((pair / bm.D3) * bm.D2 + r) * bm.D3 + pair % bm.D3 : pair * R + r;
    const int  e   = eb[bm(row)];
    h8         hi, lo;
#pragma unroll
    for(int j = 0; j < 8; j++) {
      const double y = k + j < Kin ? ldexp(x[row * Kin + k + j], e) : 0.0;
      hi[j]          = (_Float16) y;
      lo[j]          = (_Float16) (y - (double) hi[j]);
    }
    out[2 * i]     = __builtin_bit_cast(uint4, hi);
    out[2 * i + 1] = __builtin_bit_cast(uint4, lo);
  }
}

// One thread per (task, part): the part's sign and term coefficients times
// 2^-(eA + eB), eA and eB the exponents of the (tile, tile, tile) blocks of
// the two operands (the same for every row of the part).
__global__ void k_part_scales(const TaskDev* __restrict__ tasks, int n_tasks, MixedDev M,
                              float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= 18 * n_tasks) return;
  const TaskDev& T  = tasks[i / 18];
  const int      gp = i % 18;
  if(!part_on(T.d1code, T.d2code, gp)) {
    out[i] = 0.f;
    return;
  }
  const unsigned code = part_code(T.d1code, T.d2code, gp);
  const int      g = gp >> 1, d2 = gp & 1, hs = g / 3, ps = g % 3;
  const int      hA = pair_a(hs), hB = pair_b(hs), pA = pair_a(ps), pB = pair_b(ps);
  const int      no = M.nto, nv = M.ntv;
  const int      tHS = T.tile[hs], tHA = T.tile[hA], tHB = T.tile[hB];
  const int      tPS = T.tile[3 + ps], tPA = T.tile[3 + pA], tPB = T.tile[3 + pB];
  int            aa, ka, ab, kb;
  bool           fa, fb;
  float          ca, cb;
  if(!d2) {  // t2h blocks (V,V,O): (pA,pB,hs) / (pB,pA,hs); ovk (O,V,O): (hB,ps,hA) / (hA,ps,hB)
    choose_term(code, 4, 8, 1, 0, aa, fa, ca);
    ka = ((fa ? tPA : tPB) * nv + (fa ? tPB : tPA)) * no + tHS;
    choose_term(code, 16, 32, 3, 2, ab, fb, cb);
    kb = ((fb ? tHB : tHA) * nv + tPS) * no + (fb ? tHA : tHB);
  }
  else {  // xv blocks (V,V,O): (pB,pA,hs) / (pA,pB,hs); t2p (O,O,V): (hA,hB,ps) / (hB,hA,ps)
    choose_term(code, 4, 8, 5, 4, aa, fa, ca);
    ka = ((fa ? tPB : tPA) * nv + (fa ? tPA : tPB)) * no + tHS;
    choose_term(code, 16, 32, 7, 6, ab, fb, cb);
    kb = ((fb ? tHA : tHB) * no + (fb ? tHB : tHA)) * nv + tPS;
  }
  const float sg = (code & 2) ? -1.f : 1.f;
  out[i]         = sg * ca * cb * ldexpf(1.f, -(M.eblk[aa][ka] + M.eblk[ab][kb]));
}

}  // namespace

int build_part_scales(const TaskDev* tasks, int n_tasks, const MixedDev& M, float* out,
                      void* stream) {
  if(n_tasks <= 0) return 0;
  hipLaunchKernelGGL(k_part_scales, dim3((unsigned) ((18l * n_tasks + 255) / 256)), dim3(256), 0,
                     (hipStream_t) stream, tasks, n_tasks, M, out);
  return (int) hipGetLastError();
}

int build_split(const SpatialBufs& B, int O, int V, const int* tile_o, int nto, const int* tile_v,
                int ntv, SplitBufs& S, void* stream) {
  hipStream_t   st = (hipStream_t) stream;
  const long    o = O, v = V, op = (O + 7) / 8 * 8, vp = (V + 7) / 8 * 8;
  const long    ko = (O + 15) / 16 * 16, kv = (V + 15) / 16 * 16;
  const double* src[kOperands] = {B.t2h, B.t2ha, B.ovk, B.ovka, B.xv, B.xva, B.t2p, B.t2pa};
  // row coordinates of each array (0 occupied, 1 virtual), slowest first
  const int types[kOperands][3] = {{1, 1, 0}, {1, 1, 0}, {0, 1, 0}, {0, 1, 0},
                                   {1, 1, 0}, {1, 1, 0}, {0, 0, 1}, {0, 0, 1}};
  int *      dto = nullptr, *dtv = nullptr;
  short*     er  = nullptr;
  hipError_t err = hipSuccess;
  auto       done = [&](hipError_t e) {
    if(dto) (void) hipFree(dto);
    if(dtv) (void) hipFree(dtv);
    if(er) (void) hipFree(er);
    return (int) e;
  };
  if((err = hipMalloc((void**) &dto, sizeof(int) * o)) || (err = hipMalloc((void**) &dtv, sizeof(int) * v)))
    return done(err);
  if((err = hipMemcpyAsync(dto, tile_o, sizeof(int) * o, hipMemcpyHostToDevice, st)) ||
     (err = hipMemcpyAsync(dtv, tile_v, sizeof(int) * v, hipMemcpyHostToDevice, st)))
    return done(err);
  const long rows_max = v * v * o > o * o * v ? v * v * o : o * o * v;
  // k_row_exp runs one wave per row: 64 * rows work-items in one dispatch
  if(rows_max * 64 > (long) UINT32_MAX) return done(hipErrorInvalidConfiguration);
  if((err = hipMalloc((void**) &er, sizeof(short) * rows_max))) return done(err);
  for(int j = 0; j < kOperands; j++) {
    const int* const tmap[2] = {dto, dtv};
    const long       dim[2]  = {o, v};
    const int        nt[2]   = {nto, ntv};
    const int*       ty      = types[j];
    BlockMap         bm;
    bm.D2 = dim[ty[1]];
    bm.D3 = dim[ty[2]];
    bm.n2 = nt[ty[1]];
    bm.n3 = nt[ty[2]];
    bm.t1 = tmap[ty[0]];
    bm.t2 = tmap[ty[1]];
    bm.t3 = tmap[ty[2]];
    const long rows   = dim[ty[0]] * dim[ty[1]] * dim[ty[2]];
    const long blocks = (long) nt[ty[0]] * nt[ty[1]] * nt[ty[2]];
    const long kin = j < 4 ? op : vp, kout = j < 4 ? ko : kv;
    S.rows[j]      = rows;
    if((err = hipMalloc((void**) &S.eblk[j], sizeof(int) * blocks))) return done(err);
    if((err = hipMalloc((void**) &S.v[j], 4 * rows * kout))) return done(err);
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned) ((blocks + 255) / 256)), dim3(256), 0, st,
                       S.eblk[j], blocks, kNoRow);
    hipLaunchKernelGGL(k_row_exp, dim3((unsigned) ((rows + 3) / 4)), dim3(256), 0, st, src[j], rows,
                       kin, er);
    hipLaunchKernelGGL(k_block_exp, dim3((unsigned) ((rows + 255) / 256)), dim3(256), 0, st, er,
                       rows, bm, S.eblk[j]);
    // grid-stride: a dispatch's grid size is a 32-bit count of work-items
    const long n = rows * (kout / 8);
    hipLaunchKernelGGL(k_split, dim3((unsigned) std::min<long>((n + 255) / 256, 1l << 20)), dim3(256), 0, st, src[j], rows,
                       kin, kout, bm, j == 2 || j == 3, S.eblk[j], reinterpret_cast<uint4*>(S.v[j]));
    if((err = hipGetLastError())) return done(err);
  }
  return done(hipStreamSynchronize(st));
}

int launch_spatial_mixed(const MixedDev& M, const RunDev& R, int grid, void* stream) {
  hipLaunchKernelGGL(k_spatial_mixed, dim3(grid), dim3(NT), 0, (hipStream_t) stream, M, R);
  return (int) hipGetLastError();
}

}  // namespace xt
