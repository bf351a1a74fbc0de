// The shape of the single-pass 2D step's strips (march2d_shape) on a GPU of 256 CUs.
//
// Usage: march_shape nx ny [nx ny ...]; prints per grid: columns per strip, output rows per strip,
// strips along x, strips along y
#include <cstdio>
#include <cstdlib>

#include "kernels.hpp"

int main(int argc, char **argv) {
  for (int a = 1; a + 1 < argc; a += 2) {
    ppk::DevParams p{};
    p.dim = 2;
    p.nx = std::atoi(argv[a]);
    p.ny = std::atoi(argv[a + 1]);
    p.nz = 1;
    ppk::march2d_shape(p, 256);
    std::printf("%d %d %d %d\n", p.march_lw, p.march_rows,
                (p.nx + p.march_lw - 5) / (p.march_lw - 4),
                (p.ny + p.march_rows - 1) / p.march_rows);
  }
  return 0;
}
