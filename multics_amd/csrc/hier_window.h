// The key frames that a query of the frame-window attention sees: key frame kf
// is visible to query frame qf when
//   kf / n_block <= qf / n_block  and  (local_attn < 0 or qf - kf < local_attn)
// with divisions towards zero, as the host's integer division of non-negative
// frames.  That is an interval of frames, [first, first + span]: the block rule
// bounds it above, the window below, and it always holds the query's own frame.
// INT_MAX is no frame: it marks a row past the last key, which nobody sees.
//
// Plain C++ (no HIP types) so that the host test suite compiles this header
// and checks it without a GPU.
#pragma once

#include <limits.h>
#include <stdint.h>

#include "hier_launch.h"

namespace hier {

struct Window {
  int first;
  uint32_t span;
  HIER_HD void init(int qf, int n_block, int local_attn) {
    const int b = qf / n_block;
    const int64_t end = (int64_t)b * n_block + (b >= 0 ? n_block - 1 : 0);
    const int64_t last = end < (int64_t)INT_MAX - 1 ? end : (int64_t)INT_MAX - 1;
    const int64_t f0 = local_attn < 0 ? (int64_t)INT_MIN : (int64_t)qf - local_attn + 1;
    first = (int)(f0 > (int64_t)INT_MIN ? f0 : (int64_t)INT_MIN);
    span = (uint32_t)(last - first);
  }
  // (unsigned: without a window kf - first does not fit an int)
  HIER_HD bool sees(int kf) const { return (uint32_t)kf - (uint32_t)first <= span; }
};

}  // namespace hier
