// Claiming boxes from the ticket queues in the persistent kernels (device code).
#pragma once
#include "xt_device.h"
#include "xt_queue.h"

namespace xt {

// State of a workgroup's thread 0 between claims, in LDS.
struct Claim {
  long long lo, hi;  // tickets of the cached entry
  long long total;   // of the current queue
  int       entry, ti;
  TaskDev   task;  // of the cached entry
};

__device__ __forceinline__ void claim_queue(Claim& c, const RunDev& R, int q) {
  c.lo = c.hi = 0;
  c.total     = R.qtotal[q];
  c.entry     = R.qbeg[q];
}

__device__ __forceinline__ long long claim_ticket(const RunDev& R, int q) {
  return (long long) atomicAdd(&R.qctr[q], 1ull);
}

// Next box of queue q to run, from ticket t on: its task, box coordinates and
// weight (the boxes that it stands for), or -1 when the queue is exhausted.
// Copies under the exchange of equal tiles are passed over, a claim each
// (claims of several tickets left workgroups idle at the end: O=8, V=48 took
// 0.92 ms, not 0.43).  The task's record is read when the entry changes, not
// with each ticket: O=20, V=120 in mixed precision 68.2 -> 66.2 ms, O=16, V=96 in
// FP64 59.1 -> 58.8 ms.
__device__ __forceinline__ int claim_box(Claim& c, const RunDev& R, int q, long long t, bool mixed, int* sub,
                                         int& weight) {
  for(;; t = claim_ticket(R, q)) {
    // progress mirror in host memory (tickets taken so far, approximate)
    if(R.prog)
      __hip_atomic_store(&R.prog[q], (unsigned long long) t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if(t >= c.total) return -1;
    if(t < c.lo || t >= c.hi) {
      const int e = queue_entry_from(R.qbeg, R.qtick, q, t, c.entry);
      c.entry     = e;
      c.lo        = R.qtick[e];
      c.hi        = e + 1 < R.qbeg[q + 1] ? R.qtick[e + 1] : c.total;
      c.ti        = R.qtask[e];
      c.task      = R.tasks[c.ti];
    }
    const bool in = ticket_box(t - c.lo, mixed ? c.task.nsubm : c.task.nsub, R.glog, sub);
    weight        = !in ? 0 : R.fold ? fold_weight(c.task.eq, sub) : 1;
    if(weight) return c.ti;
  }
}

}  // namespace xt
