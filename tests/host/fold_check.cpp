// Host check of the box folding of equal tiles (fold_weight in
// exachem_amd/csrc/xt_queue.h): over every grid of a task whose equal
// positions have equal box counts, each orbit of boxes under the exchange of
// equal positions has exactly one box of non-zero weight, the ascending one,
// and that weight is the orbit's size.  Tickets decode to every box once for
// group shapes whose groups overhang the grid.  Built and run by
// tests/test_fold.py.
#include <algorithm>
#include <array>
#include <cstdio>
#include <map>

#include "../../exachem_amd/csrc/xt_queue.h"

int main() {
  const int shapes[4][6] = {{1, 1, 1, 1, 1, 1}, {2, 2, 2, 0, 0, 0}, {0, 0, 2, 2, 2, 0}, {6, 0, 0, 0, 0, 0}};
  const int grids[5][6] = {{1, 1, 1, 1, 1, 1}, {2, 2, 2, 3, 3, 3}, {3, 3, 3, 1, 2, 2}, {1, 5, 5, 4, 4, 2}, {2, 3, 1, 5, 5, 5}};
  long checked = 0;
  for(auto& nb: grids)
    for(int eq = 0; eq < 16; eq++) {
      bool ok = true;  // equal tiles have equal box counts
      for(int b = 0; b < 4; b++) {
        const int p = b < 2 ? b : b + 1;
        if((eq >> b) & 1) ok = ok && nb[p] == nb[p + 1];
      }
      if(!ok) continue;
      for(auto& gl: shapes) {
        std::map<std::array<int, 6>, std::array<int, 3>> orbit;  // canonical box: size, weight, bearers
        const long long n = xt::task_ticket_count(nb, gl);
        std::map<std::array<int, 6>, int> seen;
        for(long long t = 0; t < n; t++) {
          std::array<int, 6> s, c;
          if(!xt::ticket_box(t, nb, gl, s.data())) return std::printf("fold_check: ticket without a box\n"), 1;
          if(seen[s]++) return std::printf("fold_check: box decoded twice\n"), 1;
          c = s;
          for(int k = 0; k < 6; k += 3) {
            const int e = (eq >> (k ? 2 : 0)) & 3;
            if(e == 3) std::sort(c.begin() + k, c.begin() + k + 3);
            else if(e == 1) std::sort(c.begin() + k, c.begin() + k + 2);
            else if(e == 2) std::sort(c.begin() + k + 1, c.begin() + k + 3);
          }
          const int w = xt::fold_weight(eq, s.data());
          auto&     o = orbit[c];
          o[0]++;
          o[1] += w;
          o[2] += w != 0;
          if((w != 0) != (c == s)) return std::printf("fold_check: weight on the wrong box\n"), 1;
        }
        if(xt::ticket_box(n, nb, gl, std::array<int, 6>{}.data())) return std::printf("fold_check: past the end\n"), 1;
        for(auto& [c, o]: orbit)
          if(o[0] != o[1] || o[2] != 1) return std::printf("fold_check: orbit weight\n"), 1;
        checked += (long) orbit.size();
      }
    }
  std::printf("fold_check: ok %ld orbits\n", checked);
  return 0;
}
