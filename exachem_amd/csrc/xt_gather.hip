// Device-side gather of the per-task packed operand buffers: the work of the
// reference's host gathers ccsd_t_data_s1_new (ccsd_t_all_fused_singles.hpp:34-391),
// ccsd_t_data_d1_new (ccsd_t_all_fused_doubles1.hpp:37-307) and ccsd_t_data_d2_new
// (ccsd_t_all_fused_doubles2.hpp:37-360), which read TAMM blocks (Tensor::get)
// and permute them with hptt, done here from the device-resident closed-shell
// inputs.  The host plans the list of blocks (xt_gather.cpp); this kernel
// writes every element of every block.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "xt_device.h"

namespace xt {
namespace {

// The spin-orbital elements the gathers read, from the spatial closed-shell
// inputs (spin-orbital order is [alpha, beta] per space), as c1*x - c2*y:
//   T1   t1(a,i)        = [sa=si] t1[A][I]
//   T2   t2(a,b,i,j)    = [sa=si][sb=sj] t2[A][B][I][J] - [sa=sj][sb=si] t2[A][B][J][I]
//   IJAB <ij||ab>       = [si=sa][sj=sb] (ai|bj) - [si=sb][sj=sa] (bi|aj)          (vvoo)
//   IJKA <ij||ka>       = [si=sk][sj=sa] (ja|ik) - [sj=sk][si=sa] (ia|jk)          (ovoo)
//   IABC <ia||bc>       = [si=sb][sa=sc] (ac|bi) - [si=sc][sa=sb] (ab|ci)          (vvvo)
// with t2 read from t2h[a][b][i][Op] or t2p[i][j][a][Vp], ovoo from
// ovk[i][a][j][Op] and vvvo from xv[c][b][i][Vp] = vvvo[a][c][b][i].

// n / d of the block's index arithmetic: a multiply by ceil(2^32 / d) where
// that is exact (n d < 2^32, checked once per block), else a division.
struct Div {
  unsigned d, m;
  bool     mul;
  __device__ __forceinline__ Div(unsigned d_, bool mul_): d(d_), m(d_ > 1 ? 0xffffffffu / d_ + 1u : 0u), mul(mul_) {}
  __device__ __forceinline__ unsigned operator()(unsigned n) const {
    return mul ? (d > 1 ? __umulhi(n, m) : n) : n / d;
  }
};

constexpr int GT   = 256;      // threads per gather workgroup
constexpr int SLAB = 48 * 49;  // LDS slab (doubles): extents up to 48 with one pad column

// blockIdx.y = block.  Destination element e has (row-major, last fastest)
// coordinates i[k] over the permuted extents size[perm[k]]; source coordinate
// perm[k] is i[k] (hptt's row-major permutation), and the value is alpha
// times the element.
//
// Where the destination's fastest dimension is also the source's contiguous
// one, threads stride over destination elements directly.  Otherwise the block
// goes through LDS in slabs over (destination position of the source's
// contiguous dimension) x (destination's fastest position), one slab per pair
// of the two other positions: the slab is read along the source's contiguous
// dimension and written along the destination's, so both sides run through
// whole rows instead of one element per row.
//
// Bound: memory.  Per element the spin tests, the array's index rule and four
// 32-bit divisions used to cost more than the copy: the host works the rules
// out once per block (plan_gather), the divisions are multiplies, and T2 blocks
// that run over a virtual index are read from t2p, whose rows are virtual.
__global__ __launch_bounds__(GT) void k_gather(const GatherDesc* __restrict__ blocks, GatherSrc S,
                                               GatherDst D) {
  __shared__ double slab[SLAB];
  const GatherDesc& B = blocks[blockIdx.y];
  const unsigned    n = (unsigned) B.n;  // a block holds fewer than 2^31 doubles (host check)
  double* __restrict__ dst       = D.buf[B.buf] + B.dst;
  const double* __restrict__ src = S.a[B.src];
  const double* __restrict__ x0  = src + B.px;
  const double* __restrict__ y0  = src + B.py;
  const double al  = B.alpha;
  const bool   on1 = B.on1 != 0, on2 = B.on2 != 0;
  auto         value = [&](long px, long py) {
    const double x = on1 ? x0[px] : 0.0, y = on2 ? y0[py] : 0.0;
    return al * (on1 && on2 ? x - y : on1 ? x : on2 ? -y : 0.0);
  };
  const int      kS = B.kS;
  const unsigned E[4]  = {B.ext[0], B.ext[1], B.ext[2], B.ext[3]};
  const long     sx[4] = {B.sx[0], B.sx[1], B.sx[2], B.sx[3]}, sy[4] = {B.sy[0], B.sy[1], B.sy[2], B.sy[3]};
  const unsigned emax = max(max(E[0], E[1]), max(E[2], E[3]));
  const bool     mul  = (unsigned long long) n * emax < (1ull << 32);
  const unsigned ES = B.ext[kS], EF = E[3], ld = EF + 1;
  if(kS == 3 || ES * ld > (unsigned) SLAB) {
    const Div q3(E[3], mul), q2(E[2], mul), q1(E[1], mul);
    for(unsigned e = blockIdx.x * GT + threadIdx.x; e < n; e += gridDim.x * GT) {
      const unsigned r2 = q3(e), i3 = e - r2 * E[3], r1 = q2(r2), i2 = r2 - r1 * E[2], i0 = q1(r1),
                     i1 = r1 - i0 * E[1];
      dst[e]            = value(i0 * sx[0] + i1 * sx[1] + i2 * sx[2] + i3 * sx[3],
                                i0 * sy[0] + i1 * sy[1] + i2 * sy[2] + i3 * sy[3]);
    }
    return;
  }
  // the two other positions o1 < o2 index the slabs; st: destination steps
  const int      o1 = kS == 0 ? 1 : 0, o2 = kS == 2 ? 1 : 2;
  const unsigned st2 = E[3], st1 = st2 * E[2], st0 = st1 * E[1];
  const unsigned E1 = o1 ? E[1] : E[0], E2 = o2 == 1 ? E[1] : E[2], nslab = E1 * E2, nel = ES * EF;
  const Div      qs(ES, mul), qf(EF, mul), qe(E2, mul);
  const long     sxS = B.sx[kS], syS = B.sy[kS], sxF = sx[3], syF = sy[3];
  const long     sx1 = o1 ? sx[1] : sx[0], sy1 = o1 ? sy[1] : sy[0];
  const long     sx2 = o2 == 1 ? sx[1] : sx[2], sy2 = o2 == 1 ? sy[1] : sy[2];
  const unsigned d1 = o1 ? st1 : st0, d2 = o2 == 1 ? st1 : st2, dS = kS == 0 ? st0 : kS == 1 ? st1 : st2;
  // every thread of the workgroup runs the same slab loop, so the barriers
  // below are reached by all of them
  for(unsigned sl = blockIdx.x; sl < nslab; sl += gridDim.x) {
    const unsigned a = qe(sl), b = sl - a * E2;
    const long     px = a * sx1 + b * sx2, py = a * sy1 + b * sy2;
    __syncthreads();  // the previous slab's LDS reads are done
    for(unsigned e = threadIdx.x; e < nel; e += GT) {
      const unsigned f = qs(e), s = e - f * ES;
      slab[s * ld + f] = value(px + s * sxS + f * sxF, py + s * syS + f * syF);
    }
    __syncthreads();
    const unsigned base = a * d1 + b * d2;
    for(unsigned e = threadIdx.x; e < nel; e += GT) {
      const unsigned s = qf(e), f = e - s * EF;
      dst[base + s * dS + f] = slab[s * ld + f];
    }
  }
}

// Element [a][i] of the spin-orbital T1.
__device__ __forceinline__ double t1_so_value(const GatherSrc& S, long a, long i) {
  return a / S.V == i / S.O ? S.a[kArrT1][(a % S.V) * S.O + i % S.O] : 0.0;
}

// Dense spin-orbital amplitudes, [alpha, beta] per space:
//   t1_so[A][I] (2V x 2O), t2_so[A][B][I][J] ((2V)^2 (2O)^2), A = spin * V + a.
// blockIdx.y strides over rows (A for T1, the (A, B) pair for T2), threads
// over the occupied index (pair) of the row.
__global__ void k_expand_t(GatherSrc S, double* __restrict__ t1_so, double* __restrict__ t2_so) {
  const long    nv = 2 * S.V, no = 2 * S.O;
  const double* t2h = S.a[kArrT2h];
  if(t1_so)
    for(long a = blockIdx.y; a < nv; a += gridDim.y)
      for(long i = (long) blockIdx.x * blockDim.x + threadIdx.x; i < no; i += (long) gridDim.x * blockDim.x) {
        t1_so[a * no + i] = t1_so_value(S, a, i);
      }
  if(t2_so) {
    // spin = index >= n, spatial = index - spin * n: no divide per element
    // but the 32-bit one that splits the occupied pair
    const unsigned uo = (unsigned) S.O, uno = (unsigned) no, nq = uno * uno;
    for(long p = blockIdx.y; p < nv * nv; p += gridDim.y) {
      const long a = p / nv, b = p % nv;
      const int  sa = a >= S.V, sb = b >= S.V;
      double*    row = t2_so + p * (long) nq;
      for(unsigned q = blockIdx.x * blockDim.x + threadIdx.x; q < nq; q += gridDim.x * blockDim.x) {
        const unsigned i = q / uno, j = q - i * uno;
        const int      si = i >= uo, sj = j >= uo;
        const long     ab = ((a - sa * S.V) * S.V + (b - sb * S.V)) * S.O, i0 = i - si * uo, j0 = j - sj * uo;
        const bool     on1 = sa == si && sb == sj, on2 = sa == sj && sb == si;
        const double   u = on1 ? t2h[(ab + i0) * S.Op + j0] : 0.0, w = on2 ? t2h[(ab + j0) * S.Op + i0] : 0.0;
        row[q]           = on1 && on2 ? u - w : on1 ? u : on2 ? -w : 0.0;
      }
    }
  }
}

// The same T2 for occupied spaces whose O x O block fits LDS: a workgroup holds
// t2(a, b) of one spatial pair and writes its four spin rows, each one run of
// 16-byte stores of two elements.  Bound: the write of 8 (2V)^2 (2O)^2 bytes
// (an element-wise kernel made two dependent reads behind spin tests per
// element: 2.3 TB/s at O=20, V=120).  t2_so must be 16-byte aligned.  Workgroups
// beyond the `pairs` ones write T1: as a second kernel it took a small system's
// expansion (O=7, V=22) from 4.6 to 7.6 us.
constexpr int kExpandMaxO = 84;  // O (O + 1) doubles of LDS

__global__ void __launch_bounds__(256) k_expand_t2(GatherSrc S, double* __restrict__ t1_so,
                                                   double* __restrict__ t2_so, unsigned pairs) {
  extern __shared__ double t[];
  if(blockIdx.x >= pairs) {
    const long no = 2 * S.O, n = 2 * S.V * no;
    for(long x = (blockIdx.x - pairs) * 256l + threadIdx.x; x < n; x += (gridDim.x - pairs) * 256l)
      t1_so[x] = t1_so_value(S, x / no, x % no);
    return;
  }
  const unsigned O = (unsigned) S.O, ld = O + 1, oo = O * O, np = 2 * oo;  // pairs of elements per row
  const long     V = S.V, nv = 2 * V;
  const Div      q(O, true);
  for(long p = blockIdx.x; p < V * V; p += pairs) {
    const long a = p / V, b = p - a * V;
    __syncthreads();  // the previous pair's reads are done
    for(unsigned x = threadIdx.x; x < oo; x += 256) {
      const unsigned i = q(x), j = x - i * O;
      t[i * ld + j] = S.a[kArrT2h][(p * O + i) * S.Op + j];
    }
    __syncthreads();
    double2* row[4];
#pragma unroll
    for(int s = 0; s < 4; s++)
      row[s] = reinterpret_cast<double2*>(t2_so + (((s >> 1) * V + a) * nv + (s & 1) * V + b) * (4l * oo));
    for(unsigned x = threadIdx.x; x < np; x += 256) {
      const unsigned I = q(x), J = 2 * (x - I * O), si = I >= O, i = I - si * O;  // O pairs per I
      double         v[4][2];
#pragma unroll
      for(int k = 0; k < 2; k++) {
        const unsigned sj = J + k >= O, j = J + k - sj * O;
        const double   u = t[i * ld + j], w = t[j * ld + i];
        v[0][k] = !si && !sj ? u - w : 0.0;
        v[3][k] = si && sj ? u - w : 0.0;
        v[1][k] = !si && sj ? u : si && !sj ? -w : 0.0;
        v[2][k] = si && !sj ? u : !si && sj ? -w : 0.0;
      }
#pragma unroll
      for(int s = 0; s < 4; s++) row[s][x] = make_double2(v[s][0], v[s][1]);
    }
  }
}

}  // namespace

int launch_expand_t(const GatherSrc& S, double* t1_so, double* t2_so, void* stream) {
  if(t2_so && S.O <= kExpandMaxO && ((uintptr_t) t2_so & 15) == 0) {
    const unsigned pairs = (unsigned) std::min<long>(S.V * S.V, 1l << 16);
    const unsigned more  = t1_so ? (unsigned) std::min<long>((4 * S.V * S.O + 255) / 256, 64) : 0;
    hipLaunchKernelGGL(k_expand_t2, dim3(pairs + more), dim3(256), (unsigned) (sizeof(double) * S.O * (S.O + 1)),
                       (hipStream_t) stream, S, t1_so, t2_so, pairs);
    return (int) hipGetLastError();
  }
  const long     no = 2 * S.O, nv = 2 * S.V;
  const unsigned gx = (unsigned) std::min<long>(((t2_so ? no * no : no) + 255) / 256, 64);
  const unsigned gy = (unsigned) std::min<long>(t2_so ? nv * nv : nv, 65535);
  hipLaunchKernelGGL(k_expand_t, dim3(gx, gy), dim3(256), 0, (hipStream_t) stream, S, t1_so, t2_so);
  return (int) hipGetLastError();
}

int launch_gather(const GatherDesc* blocks, int n_blocks, long max_elems, const GatherSrc& S,
                  const GatherDst& D, void* stream) {
  if(n_blocks <= 0) return 0;
  if(n_blocks > 65535) return (int) hipErrorInvalidConfiguration;
  const long     per = (max_elems + 255) / 256;
  const unsigned gx  = (unsigned) (per < 512 ? (per > 0 ? per : 1) : 512);
  hipLaunchKernelGGL(k_gather, dim3(gx, (unsigned) n_blocks), dim3(GT), 0, (hipStream_t) stream,
                     blocks, S, D);
  return (int) hipGetLastError();
}

}  // namespace xt
