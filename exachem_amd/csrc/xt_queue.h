// Work-queue tickets of the persistent kernels: which queue entry owns a
// ticket, and which box of the task's box grid a ticket names.  Shared by the
// kernels (xt_kernels.hip, xt_mixed.hip), the host planner (xt_host.cpp) and
// the host emulation of the claim loop (tests/host/queue_emu.cpp), so the
// emulation runs the kernels' own decode.
#pragma once
#include "xt_device.h"

#if defined(__HIPCC__)
#define XT_HD __host__ __device__
#else
#define XT_HD
#endif

namespace xt {

// Tickets of a task whose box grid is nbox[0..5] boxes along (h1,h2,h3,p4,p5,p6):
// one per box (a group of the grid cut into 2^glog[p] boxes along each
// position has fewer tickets where it overhangs the grid's edge).
XT_HD inline long long task_ticket_count(const int* nbox, const int* glog) {
  (void) glog;  // the count does not depend on the shape; callers hold it beside the grid
  long long n = 1;
  for(int p = 0; p < 6; p++) n *= nbox[p];
  return n;
}

// Entry of queue q that owns ticket t: the last entry e of qbeg[q]..qbeg[q+1]-1
// with qtick[e] <= t (qtick ascends within a queue; the caller checks
// t < qtotal[q], which makes the queue non-empty).
XT_HD inline int queue_entry(const int* qbeg, const long long* qtick, int q, long long t) {
  int lo = qbeg[q], hi = qbeg[q + 1] - 1;
  while(lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if(qtick[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// The same entry, searched from entry `from` of queue q, which must be at or
// before the answer (the entry of the caller's previous ticket on this queue:
// a workgroup's tickets on one queue only grow): two steps forward, then a
// binary search over the rest.  A workgroup's next ticket is usually in the
// same entry or the next, so this reads one or two qtick values instead of
// the dozen dependent reads of a search over the whole queue.
XT_HD inline int queue_entry_from(const int* qbeg, const long long* qtick, int q, long long t,
                                  int from) {
  int       lo   = from < qbeg[q] ? qbeg[q] : from;
  const int last = qbeg[q + 1] - 1;
  for(int s = 0; s < 2; s++) {
    if(lo >= last || qtick[lo + 1] > t) return lo;
    lo++;
  }
  int hi = last;
  while(lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if(qtick[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Box named by a task's local ticket, groups of boxes one after the other
// (h1's group index fastest) and inside a group the boxes with h1 fastest.  An
// edge group is cut to the grid, so every ticket names a box: with whole
// groups of 64 a task of few boxes (tiles of one or two boxes) had several
// times as many tickets as boxes, each with its atomic, its decode and two
// barriers (O=7, V=22, uneven tiles, every spin block: 40,960 tickets for 5,120
// boxes).  Along position p
// (p6 down to h1) a slab of 2^glog[p] boxes holds L = 2^glog[p] * (boxes of
// the faster positions) * (this group's extents along the slower ones)
// tickets, and only the last slab is shorter.  Returns false only for a
// ticket outside the task.  32-bit arithmetic: the host runs no task of 2^31
// or more tickets.
XT_HD inline bool ticket_box(long long local, const int* nbox, const int* glog, int* sub) {
  unsigned below[7];  // boxes of the positions before p
  below[0] = 1;
#pragma unroll
  for(int p = 0; p < 6; p++) below[p + 1] = below[p] * (unsigned) nbox[p];
  if(local < 0 || (unsigned long long) local >= below[6]) return false;
  unsigned rem = (unsigned) local, above = 1, ext[6];
#pragma unroll
  for(int p = 5; p >= 0; p--) {
    const int      gl = glog[p];
    const unsigned nb = (unsigned) nbox[p], per = below[p] * above;  // tickets per box row
    const unsigned first = ((rem / per) >> gl) << gl;                // < nb
    rem -= first * per;
    ext[p] = nb - first < (1u << gl) ? nb - first : 1u << gl;
    sub[p] = (int) first;
    above *= ext[p];
  }
#pragma unroll
  for(int p = 0; p < 6; p++) {
    const unsigned q = rem / ext[p];
    sub[p] += (int) (rem - q * ext[p]);
    rem = q;
  }
  return true;
}

// Antisymmetry of the triples: where two holes (or two particles) of a task
// lie on the same spin-orbital tile, exchanging them changes only the sign of
// t3 and of the singles term, so boxes whose positions are a permutation of
// another's add the same energy.  eq holds bit 0 for h1b = h2b, 1 for
// h2b = h3b, 2 for p4b = p5b, 3 for p5b = p6b (tiles ascend within each
// triple, so h1b = h3b implies both).  Returns how many boxes the ascending
// one stands for (its energy is multiplied by that), 0 for the others, which
// are skipped.  Summed over a grid the weights give its box count.
// The copies' rounding errors differed, so a box that stands for them brings its
// own w times where they used to average: in the mixed kernel the rms error of a
// task's energy (relative, against FP64; six tilings of O=12 V=60 to O=32 V=160)
// stays within 2% where up to two neighbours share a tile, grows by up to 7% where
// three do (4.2e-10 to 1.7e-9) and by up to 25% on the few tasks whose holes and
// particles are all equal (2.8e-10 to 2.3e-9).  Whole runs and shares keep their
// error (3.6e-10 to 1e-9, within 3%).  FP64 keeps its last-place errors.
XT_HD inline int fold_triple(int e, int a, int b, int c) {
  if((e & 1) && a > b) return 0;
  if((e & 2) && b > c) return 0;
  if(e == 3) return a == b ? (b == c ? 1 : 3) : (b == c ? 3 : 6);
  if(e == 1) return a == b ? 1 : 2;
  if(e == 2) return b == c ? 1 : 2;
  return 1;
}
XT_HD inline int fold_weight(int eq, const int* sub) {
  return fold_triple(eq & 3, sub[0], sub[1], sub[2]) *
         fold_triple((eq >> 2) & 3, sub[3], sub[4], sub[5]);
}

}  // namespace xt
