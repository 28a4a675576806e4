// Host build of the GEMMs' tile order (csrc/kernels/common.h) for tests/test_tile_plan.py.
#include "common.h"

extern "C" void order(unsigned gx, unsigned gy, unsigned gz, unsigned gn, unsigned* out) {
  for (unsigned i = 0; i < gx * gy * gz; ++i) {
    const TilePos p = tile_order(i, gx, gy, gz, gn);
    out[3 * i] = p.row, out[3 * i + 1] = p.col, out[3 * i + 2] = p.kz;
  }
}
