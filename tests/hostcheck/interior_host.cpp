/*
 * interior_host.cpp -- the cells that the reductions visit (Interior from
 * reduce_common.h, compiled for the host): for each "nx ny pad" on stdin the
 * number of cells and, where there are few, every cell's row and column.
 */
#include <cstdio>

#include "../../flow_amd/csrc/kernels/reduce_common.h"

int main() {
  int nx, ny, pad;
  while (std::scanf("%d %d %d", &nx, &ny, &pad) == 3) {
    const flowhip::Interior in(nx, ny, pad);
    std::printf("%u", in.n);
    for (unsigned int k = 0; k < in.n && in.n <= 4096; ++k)
      std::printf(" %d,%d", in.row(k), in.col(k));
    std::printf("\n");
  }
  return 0;
}
