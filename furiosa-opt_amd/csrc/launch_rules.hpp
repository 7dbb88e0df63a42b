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

// Attention without a given row max: 2 groups of 32 queries x 4 of keys a workgroup, 4 x 2, or 256 queries.
// By the workgroups each would have (WG64 and WG128: one per 64 or 128 queries of a head). Kernel alone in
// a recorded graph, D = 128, us (one box), causal / not:
//     heads, seq   WG64    2 x 4 groups   WG128    4 x 2 groups    256 queries
//     1, 600         10    14.1 / -           5    16.3 / -        22.4 / -
//     16, 600       160    15.5 / -          80    17.3 / -        23.2 / -
//     16, 1024      256    21.0 / -         128    24.9 / -        34.5 / -
//     32, 600       320    - / -            160    17.3 / -        24.0 / -
//     64, 600       640    29.5 / 41.4      320    19.7 / 33.8     24.5 / 25.9
//     100, 300      500    19.0 / 24.0      300    19.5 / 23.8     16.2 / 17.6
//     32, 1200      608    38.0 / 63.3      320    28.9 / 54.0     39.0 / 39.6
//     32, 2048     1024    78.2 / 129       512    53.7 / 91.7     62.7 / 74.6
//     300, 100      600    21.7 / 21.6      300    15.8 / 16.0     18.6 / 18.6
// and D = 64 alike. A second, partly filled round of 4 x 2 workgroups costs what a full one does, so past
// one a CU they are taken only where their work is uneven and long (causal, past 384 keys), or where one
// query block covers the head.
enum class AttnForm { kKeys4, kKeys2, kQueries256 };
inline AttnForm attention_form(int64_t heads, int64_t seq, bool causal) {
  const int64_t wg64 = heads * ((seq + 63) / 64), wg128 = heads * ((seq + 127) / 128);
  if (wg64 <= 256 && seq > 64) return AttnForm::kKeys4;
  if (wg128 <= 256 || (wg128 <= 320 && (seq <= 128 || (causal && seq > 384))) || (wg128 <= 512 && causal && seq >= 1024))
    return AttnForm::kKeys2;
  return AttnForm::kQueries256;
}

}  // namespace fo
