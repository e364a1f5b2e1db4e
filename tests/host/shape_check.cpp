// Prints what the launch-shape rules of shape.hpp and batch_items.hpp pick, one line per line of
// standard input (a rule's name and its arguments).
#include <cstdio>
#include <cstring>

#include "../../symphas_amd/csrc/batch_items.hpp"
#include "../../symphas_amd/csrc/shape.hpp"

int main() {
  char rule[32];
  int X, Y, Z, esize;
  while (std::scanf("%31s", rule) == 1) {
    if (!std::strcmp(rule, "one_site") && std::scanf("%d%d%d%d", &X, &Y, &Z, &esize) == 4)
      std::printf("%d\n", sps::one_site_step3d(X, Y, Z, esize) ? 1 : 0);
    else if (!std::strcmp(rule, "radius_two") && std::scanf("%d%d%d%d", &X, &Y, &Z, &esize) == 4) {
      const sps::StreamShape s = sps::radius_two_shape3d(X, Y, Z, esize);
      std::printf("%d %d %d\n", s.steps, s.rows, s.planes);
    } else if (!std::strcmp(rule, "batch") && std::scanf("%d", &X) == 1) {
      std::vector<sps::BatchSides> inst(X);
      for (sps::BatchSides& i : inst)
        if (std::scanf("%d%d%d", &i.X, &i.Y, &i.R) != 3) return 1;
      std::printf("%d\n", sps::batch_rows(inst, 4));
    } else if (!std::strcmp(rule, "launch_cost") && std::scanf("%d%d%d", &Y, &Z, &X) == 3) {
      // steps per launch, item height, number of instances: the launch's cost by
      // the rule and by its lists
      std::vector<sps::BatchSides> inst(X);
      for (sps::BatchSides& i : inst)
        if (std::scanf("%d%d%d", &i.X, &i.Y, &i.R) != 3) return 1;
      double most = 0;
      for (const auto& x : sps::batch_lists(inst, Y, Z)) {
        long long simd[128] = {};
        for (size_t p = 0; p < x.size(); ++p) {
          const int c = sps::batch_item_cost(Y, inst[x[p].inst].R, x[p].ty);
          simd[p % 128] += c;
          most = std::max(most, std::max((double)simd[p % 128], 1.5 * c));
        }
      }
      std::printf("%.0f %.0f\n", 2 * sps::batch_launch_cost(inst, Y, Z), 2 * most);
    } else
      return 1;
  }
  return 0;
}
