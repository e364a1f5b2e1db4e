// Prints what the launch-shape rules of shape.hpp pick, one line per line of
// standard input (a rule's name and its arguments).
#include <cstdio>
#include <cstring>

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
    } else
      return 1;
  }
  return 0;
}
