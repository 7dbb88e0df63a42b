// Host rules of the launches: which kernel form, tile or piece a call takes, from its sizes alone. No HIP
// here, so that tests/test_launch_rules.py builds and checks them without a GPU.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace fo {

// f(first, count) for each launch of a kernel over `rows` rows: a launch's threads have to fit 32 bits.
// The pieces are equal powers of two but for the last, so a block's rows never straddle two.
template <typename F>
void for_row_pieces(int64_t rows, int64_t threads_per_row, F&& f) {
  const int64_t per = (1ll << 31) / threads_per_row;
  for (int64_t first = 0; first < rows; first += per) f(first, std::min(per, rows - first));
}

}  // namespace fo
