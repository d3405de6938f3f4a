// map_blocks' double solves for 8 < n <= 64 (map_blocks_seg.h).
#include "map_blocks_seg.h"

int map_blocks_seg(nmx_ctx* ctx, int kind, int n, int64_t batch, const double* xs, double* ys) {
  return map_blocks_seg_any<double>(ctx, kind, n, batch, xs, ys);
}
