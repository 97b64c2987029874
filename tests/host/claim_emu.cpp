// Host emulation of the persistent kernels' claims with their own claim_box
// (exachem_amd/csrc/xt_claim.h): the cached entry range and task record, the
// forward search, and tickets of copies passed over.  Queues of made-up tasks;
// workgroup b serves queue b % 8 first, then the others in turn.  The order of the
// atomics is drawn at random: which workgroup claims next, and, at each ticket
// taken, whether others claim whole boxes in between.  Checks: every box that runs
// (fold_weight) of every listed task is claimed once, by the task's own record, with
// its weight, no other box is, and every workgroup finds every queue exhausted.
// Built and run by tests/test_claim_emulation.py.
//
//   claim_emu <workgroups> <fold 0|1> <mixed 0|1> <seed>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <random>
#include <tuple>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))
static std::function<void()> between;  // what other workgroups do before a ticket is taken
static unsigned long long    atomicAdd(unsigned long long* p, unsigned long long v) {
  if(between) between();
  const unsigned long long old = *p;
  *p += v;
  return old;
}
#include "../../exachem_amd/csrc/xt_claim.h"

int main(int argc, char** argv) {
  if(argc != 5) return std::printf("claim_emu: usage\n"), 1;
  const int  grid = std::atoi(argv[1]);
  const bool fold = std::atoi(argv[2]) != 0, mixed = std::atoi(argv[3]) != 0;
  std::mt19937_64 rng(std::strtoull(argv[4], nullptr, 10));
  auto draw = [&](int lo, int hi) { return lo + (int) (rng() % (unsigned) (hi - lo + 1)); };
  // tasks: some listed, in a drawn order, over the eight queues, some of them empty
  const int                nt = 40;
  std::vector<xt::TaskDev> tasks(nt);
  for(int t = 0; t < nt; t++) {
    xt::TaskDev& T = tasks[t];
    T.eq           = draw(0, 15);
    for(int p = 0; p < 6; p++) {
      const bool same = p % 3 && ((T.eq >> (p < 3 ? p - 1 : p - 2)) & 1);
      T.nsub[p]       = same ? T.nsub[p - 1] : draw(1, 3);
      T.nsubm[p]      = same ? T.nsubm[p - 1] : draw(1, 2);
    }
    T.off[0] = t;  // names the record
  }
  int glog[6] = {0, 0, 0, 0, 0, 0};
  for(int k = 0; k < xt::kGroupLog2; k++) glog[draw(0, 5)]++;
  std::vector<int>       order, qbeg(1, 0), qtask;
  std::vector<long long> qtick, qtotal;
  for(int t = 0; t < nt; t++)
    if(rng() % 4) order.push_back(t);
  std::shuffle(order.begin(), order.end(), rng);
  const int empty = draw(0, xt::kQueues - 1);
  std::vector<std::vector<int>> per(xt::kQueues);
  for(int t: order) {
    int q = draw(0, xt::kQueues - 2);
    per[q + (q >= empty)].push_back(t);
  }
  for(int q = 0; q < xt::kQueues; q++) {
    long long tk = 0;
    for(int t: per[q]) {
      qtask.push_back(t);
      qtick.push_back(tk);
      tk += xt::task_ticket_count(mixed ? tasks[t].nsubm : tasks[t].nsub, glog);
    }
    qbeg.push_back((int) qtask.size());
    qtotal.push_back(tk);
  }
  std::vector<unsigned long long> qctr(xt::kQueues, 0), prog(xt::kQueues, 0);
  xt::RunDev R = {};
  R.tasks      = tasks.data();
  R.qtask      = qtask.data();
  R.qtick      = qtick.data();
  R.qbeg       = qbeg.data();
  R.qtotal     = qtotal.data();
  R.qctr       = qctr.data();
  R.prog       = prog.data();
  R.fold       = fold;
  for(int p = 0; p < 6; p++) R.glog[p] = glog[p];

  struct Workgroup {
    xt::Claim c;
    int       qi = 0;
    bool      busy = false;
  };
  std::vector<Workgroup> wg(grid);
  std::map<std::tuple<int, int, int, int, int, int, int>, int> got;  // task and box -> weight
  bool ok   = true;
  int  left = grid, depth = 0;
  for(int b = 0; b < grid; b++) xt::claim_queue(wg[b].c, R, b % xt::kQueues);
  std::function<void(int)> claim = [&](int b) {  // one claim of workgroup b
    Workgroup& w = wg[b];
    if(w.busy || w.qi == xt::kQueues) return;
    w.busy = true;
    depth++;
    const int q = (b + w.qi) % xt::kQueues;
    int       sub[6], weight = -1;
    const int ti = xt::claim_box(w.c, R, q, xt::claim_ticket(R, q), mixed, sub, weight);
    if(ti < 0) {
      if(++w.qi == xt::kQueues) left--;
      else xt::claim_queue(w.c, R, (b + w.qi) % xt::kQueues);
    }
    else {
      ok = ok && w.c.task.off[0] == ti && weight > 0;
      ok = ok && got.insert({{ti, sub[0], sub[1], sub[2], sub[3], sub[4], sub[5]}, weight}).second;
    }
    depth--;
    w.busy = false;
  };
  between = [&] {
    if(depth < 4)
      while(rng() % 3 == 0) claim(draw(0, grid - 1));
  };
  while(left && ok) claim(draw(0, grid - 1));
  if(!ok) return std::printf("claim_emu: a box twice, or by another task's record\n"), 1;
  size_t want = 0;
  for(int t: qtask) {
    const int* n = mixed ? tasks[t].nsubm : tasks[t].nsub;
    int        s[6];
    long long  weights = 0, boxes = 1;
    for(int p = 0; p < 6; p++) boxes *= n[p];
    for(long long k = 0; k < boxes; k++) {
      long long r = k;
      for(int p = 0; p < 6; p++) {
        s[p] = (int) (r % n[p]);
        r /= n[p];
      }
      const int  w  = fold ? xt::fold_weight(tasks[t].eq, s) : 1;
      const auto it = got.find({t, s[0], s[1], s[2], s[3], s[4], s[5]});
      if((it == got.end() ? 0 : it->second) != w) return std::printf("claim_emu: weight of a box\n"), 1;
      want += w != 0;
      weights += w;
    }
    if(weights != boxes) return std::printf("claim_emu: weights of a task\n"), 1;
  }
  if(want != got.size()) return std::printf("claim_emu: a box outside the queues\n"), 1;
  for(int q = 0; q < xt::kQueues; q++)
    if((long long) qctr[q] < qtotal[q] + grid) return std::printf("claim_emu: a queue left early\n"), 1;
  std::printf("claim_emu: ok %zu boxes\n", got.size());
  return 0;
}
