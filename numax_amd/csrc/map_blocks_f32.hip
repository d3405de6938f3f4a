// map_blocks' float solves for 8 < n <= 64 (map_blocks_seg.h).
#include "map_blocks_seg.h"

int map_blocks_seg(nmx_ctx* ctx, int kind, int n, int64_t batch, const float* xs, float* ys) {
  return map_blocks_seg_any<float>(ctx, kind, n, batch, xs, ys);
}
