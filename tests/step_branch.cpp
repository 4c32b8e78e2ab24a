// Prints, for caterpillar and balanced trees of 2 to 40 leaves, the leaves, the
// tree's branches and the highest branch that a step of its program reads.
#include <algorithm>
#include <cstdio>
#include <utility>

#include "host/program.hpp"

int main() {
  for (int nl = 2; nl <= 40; ++nl)
    for (int balanced = 0; balanced < 2; ++balanced) {
      std::vector<int> lc(2 * nl - 1, -1), rc(lc), todo;
      for (int i = 0; i < nl; ++i) todo.push_back(i);
      for (int i = nl; i < 2 * nl - 1; ++i) {  // the two oldest nodes, or the newest and the oldest
        lc[i] = todo.front();
        todo.erase(todo.begin());
        auto at = balanced ? todo.begin() : todo.end() - 1;
        rc[i] = *at;
        todo.erase(at);
        todo.push_back(i);
      }
      const pcsf::Program p = pcsf::make_program(lc, rc, nl, false);
      int top = 0;
      for (size_t k = 1; k + 1 < p.ops.size() / kOpWords; k += 2)  // every second op of a step
        top = std::max(top, step_branch(p.ops[kOpWords * k], p.ops[kOpWords * k + 1]));
      std::printf("%d %d %d\n", nl, 2 * nl - 2, top);
    }
}
