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

// RMSNorm -> softmax of aligned rows: whether the persistent DMA form (k_rmsnorm_softmax_dma, 4096 rows a round of
// the chip) takes them from the row kernel. It hides a round's loads behind the last one's work but pays a whole
// round for a part of one. Kernel alone in a recorded graph, one box, us, DMA / row kernel:
//     rows         3500          4000          4096          4500          6000          8000          8192
//     2048      8.2 / 6.7     8.3 / 7.1     8.3 / 7.1    11.6 / 7.9    11.6 / 10.1   12.5 / 13.3   12.8 / 13.4
//     4096     14.0 / 12.9   12.8 / 14.2   12.8 / 14.5   19.9 / 15.1   22.0 / 19.4       -         25.7 / 26.8
//     rows         9000         11000         12288         14000         16384         20000         32768
//     2048     16.2 / 14.2   17.9 / 17.1   18.6 / 19.2   23.4 / 21.6   25.6 / 26.8   30.2 / 31.7   48.7 / 49.7
// and of 1024 columns and fewer the row kernel is the faster one at every number of rows.
inline bool norm_dma(int64_t rows, int64_t cols) {
  const int64_t last = (rows - 1) % 4096 + 1;  // rows of the last round
  if (cols == 4096) return rows >= 6144 || (rows > 3840 && rows <= 4096);
  return cols == 2048 && rows > 4096 && rows <= 32768 && last > 3400;
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

// Output tiles of a matrix product, by how many of each size it has on the 256 CUs (T64, T128, T256;
// batches included). Kernel alone in a recorded graph, one box, us:
//     types, M, N, K               64x64   128x128 4 stages   128x128 2 stages   256x256
//     bf16  500, 3072, 1024         10.0        12.9               15.3             38
//     bf16  512, 4096, 4096         30.7        32.3               42.6             75      T64 = 512
//     bf16  1024, 4096, 4096        58          39.3               48.6             76      T128 = 256
//     bf16  2048, 4096, 4096       104          75.0               66.9             80      T128 = 512, T256 = 128
//     f8    2048, 4096, 4096        58          45.7               36.6             52
//     bf16  1500, 5500, 1024        37.9        39.9               35.2             44      T128 = 516, T256 = 132
//     bf16  2304, 3840, 1024        36.0        36.4               31.3             29.5    T128 = 540, T256 = 135
//     bf16  2304, 3840, 4096       115         104                 99.9             81.5
//     i8    1500, 5500, 1024        25.5        29.1               24.1             26.2
//     i8    1500, 5500, 4096        66.8        61.4               57.9             49.3
//     f8    1500, 5500, 2048        34.9        39.4               35.0             32.0
//     bf16  2048, 8192, 1024        68          54                 44.8             37.5    T256 = 256
// Hence: 64x64 (32 KiB of LDS a stage pair, two blocks a CU) up to two tiles a CU; 128x128 with four stages
// in flight while one block a CU covers them and K has stages enough to pay for filling four (deep_stages); with two
// stages, two blocks a CU, up to 512; past that 256x256, but for the first, mostly empty round of them over a short K (1024 elements; 512 of the 8-bit
// floats, whose 256x256 form is the faster one). An output side of up to 32, 64 or 128 keeps the tile as small
// at any number of tiles, the rest of a larger one being padding (batch x M, N, K):
//     types                       32x64   64x64   128x128 2 stages   256x256
//     bf16  16, 155648, 1024       60.1    65.2         70.2           87.3
//     bf16  32, 65536, 256          9.2     9.4          9.3           16.2
//     bf16  64, 40000, 1024          -     18.1         19.4           34.2
//     bf16  128, 65536, 1024         -     37.4         26.5           36.2
//     i8    100, 40000, 1024         -     20.0         16.1           24.9
//     bf16  520 x 16, 64, 256        5.8    7.7         11.2           34.2
//     f8    600 x 64, 64, 512        -     10.9         16.0           27.3
//     bf16  300 x 100, 100, 256      -     16.3         10.7           45.3
//
// Stages of k from which 128x128 tiles keep four in flight, not two. A number of tiles that the 8 XCDs don't divide
// is walked in launch order, neighbours on different XCDs' caches, and waits longer for each stage. us, two / four,
// by stages of 128 bytes of k:
//     types, M, N (tiles)         5            7            9           11           13           15           17
//     bf16  777, 4096 (224)   7.1 / 7.4    7.9 / 8.4    8.7 / 9.2    9.5 / 9.9   10.2 / 10.6  11.0 / 11.3  11.9 / 12.2
//     bf16  1024, 3000 (192)  7.3 / 7.7    8.2 / 8.7    9.0 / 9.4    9.7 / 10.2  10.5 / 10.8  11.6 / 11.5  12.9 / 12.3
//       K off 128 bytes       7.5 / 7.9    8.4 / 8.8    9.3 / 9.4   10.3 / 10.2  11.4 / 11.1  12.4 / 11.7  13.8 / 12.6
//     i8    777, 4096 (224)   8.1 / 8.4    8.9 / 9.5    9.8 / 10.2  10.6 / 11.0  11.3 / 11.7  12.2 / 12.4  14.3 / 13.5
//     i8    900, 3000 (192)   8.0 / 8.6    8.9 / 9.4    9.8 / 10.1  10.9 / 10.9  11.9 / 11.7  13.2 / 12.3  14.4 / 13.2
//     f8    900, 3000 (192)   7.9 / 8.2    8.8 / 9.1    9.7 / 9.8   10.9 / 10.6  12.1 / 11.6  13.5 / 12.3  14.8 / 13.2
//     bf16  583, 5384 (215)   8.4 / 8.6    9.2 / 9.2   11.3 / 10.3  13.2 / 11.8  14.8 / 13.2  16.3 / 14.4  17.8 / 15.8
//     bf16  343, 5584 (132)   7.1 / 7.4    7.9 / 8.5    8.8 / 9.2   11.1 / 10.1  12.5 / 10.8  14.7 / 11.8  16.2 / 12.5
//       K off 128 bytes       7.2 / 7.5    8.1 / 8.4   10.0 / 9.5   10.7 / 10.3  14.1 / 12.0  15.8 / 13.1  17.4 / 14.4
//     i8    640, 3300 (130)   8.1 / 8.3    9.5 / 9.6   10.7 / 10.4  12.2 / 11.3  14.2 / 12.1  16.0 / 12.9  17.4 / 13.8
//     f8    583, 5384 (215)   9.1 / 9.1   10.5 / 10.1  12.4 / 11.1  14.3 / 12.4  16.0 / 13.8  17.5 / 14.8  19.1 / 16.1
enum GemmTile { kTile32x64 = 32, kTile64 = 64, kTile128 = 128, kTile128Deep = 1284, kTile256 = 256 };
inline int64_t tiles_of(int64_t m, int64_t n, int64_t batch, int64_t tm, int64_t tn) {
  return ((m + tm - 1) / tm) * ((n + tn - 1) / tn) * batch;
}
inline int64_t deep_stages(int64_t tiles, int elem_bytes, bool f8) {
  if (tiles % 8) return elem_bytes == 2 ? 9 : 8;
  return elem_bytes == 2 ? 15 : f8 ? 10 : 13;
}
inline GemmTile gemm_tile(int64_t m, int64_t n, int64_t k, int64_t batch, int elem_bytes, bool f8) {
  const int64_t t64 = tiles_of(m, n, batch, 64, 64), t128 = tiles_of(m, n, batch, 128, 128), side = std::min(m, n);
  // Batches are the launch's second dimension; the first one's threads have to fit 32 bits.
  auto fits = [&](int64_t tm, int64_t tn, int64_t threads) { return tiles_of(m, n, 1, tm, tn) * threads < (1ll << 32); };
  if (m <= 32 && fits(32, 64, 128)) return kTile32x64;
  if ((t64 <= 512 || side <= 64) && fits(64, 64, 256)) return kTile64;
  if (t128 <= 256 && (k * elem_bytes + 127) / 128 >= deep_stages(tiles_of(m, n, 1, 128, 128), elem_bytes, f8)) return kTile128Deep;
  if ((t128 <= 512 || side <= 128) && fits(128, 128, 256)) return kTile128;
  if (tiles_of(m, n, batch, 256, 256) < 144 && k <= (f8 ? 512 : 1024)) return kTile128;
  return kTile256;
}

// Operands whose rows or K are off 16 bytes: 64x64 or 128x128 tiles staged through registers. As above, a
// side of up to 64 keeps the smaller tile at any number of tiles (2000 x 32, 32, 63: 12.8 us against 28 bf16,
// 14.1 against 34 i8, and 17-18 for the vector-unit fold that took it before). 0: the vector-unit fold, for what no
// launch of these tiles holds and for a K so short that the tiles' fixed 4 us (i8: 5) are not paid back. Kernel
// alone in a recorded graph, one box, us, fold / tiles:
//     batch x M, N           K = 2         7            14           20           31           47
//     i8    1 x 8, 8       2.8 / 4.7    3.0 / 4.7    3.2 / 4.7    3.4 / 4.9    3.7 / 4.8    4.7 / 4.9
//     i8    1 x 100, 100   3.5 / 4.9    3.8 / 4.9    4.0 / 4.8    4.1 / 5.1    4.5 / 5.1    5.5 / 5.1
//     i8    1 x 500, 500   4.0 / 5.1    4.3 / 5.1    4.5 / 5.1    4.7 / 5.3    5.1 / 5.3    6.2 / 5.3
//     i8    1 x 700, 700   4.5 / 5.3    4.8 / 5.2    5.2 / 5.2    5.4 / 5.5    5.8 / 5.5    7.1 / 5.5
//     i8    1000 x 16, 16  5.4 / 6.8    5.8 / 6.8    6.3 / 7.0    6.7 / 6.9    7.6 / 7.6   10.0 / 7.6
//     i8    5000 x 8, 8     12 / 24      13 / 24      15 / 24      16 / 25      19 / 26      26 / 27
//     i8    1 x 8, 30000   5.7 / 5.3    6.2 / 5.4    6.7 / 5.4    7.2 / 5.5    8.0 / 5.6   10.5 / 5.6
//     bf16  1 x 8, 8       3.2 / 3.8    3.4 / 3.9    3.7 / 4.0    3.8 / 3.9    4.2 / 4.1    5.5 / 4.2
//     bf16  1 x 100, 100   3.9 / 4.3    4.2 / 4.3    4.5 / 4.4    4.6 / 4.5    5.1 / 4.5    6.4 / 4.6
//     bf16  1 x 500, 500   4.3 / 4.5    4.6 / 4.5    4.9 / 4.6    5.2 / 4.7    5.7 / 4.7    6.9 / 4.8
//     bf16  5000 x 8, 8     15 / 19      16 / 19      18 / 19      19 / 19      22 / 21      30 / 23
inline int64_t gemm_any_min_k(int64_t m, int64_t n, int64_t batch, bool i8) {
  const int64_t cells = m * n * batch;
  if (cells <= 128 * tiles_of(m, n, batch, 64, 64)) return i8 ? 48 : 20;  // tiles nearly empty
  if (!i8) return cells <= (1 << 17) ? 8 : 0;
  if (std::min(m, n) < 16) return cells <= (1 << 16) ? 32 : 0;
  return cells <= (1 << 18) ? 32 : cells <= (1 << 19) ? 16 : 0;
}
inline int gemm_any_tile(int64_t m, int64_t n, int64_t k, int64_t batch, bool i8) {
  auto fits = [&](int64_t t) { return tiles_of(m, n, 1, t, t) * 256 < (1ll << 32); };
  if (k < gemm_any_min_k(m, n, batch, i8)) return 0;
  if ((tiles_of(m, n, batch, 64, 64) <= 512 || std::min(m, n) <= 64) && fits(64)) return 64;
  return fits(128) ? 128 : 0;
}

// The MLP's forms: a row a block with a thread per fold (k_mlp) or, where the shape fits them, producer and
// folder waves (k_mlp_split, `split`); or several rows a block (k_mlp_rows). Kernel alone in a recorded graph, one
// box, us, one row a block / k_mlp_rows:
//     k_mlp_split, batch:         257           320-400         512          513
//     64, 65, 10                6.7 / 7.6      7.2 / 7.7      7.3 / 7.8        -
//     400, 72, 10              13.8 / 15.4    14.3 / 15.5    14.4 / 15.5       -
//     64, 88, 10                8.7 / 7.9      9.2 / 8.0      9.3 / 8.0        -
//     784, 100, 10             22.3 / 22.9    23.0 / 23.0    23.1 / 23.0       -
//     256, 112, 10             12.1 / 12.3    12.6 / 12.4    12.7 / 12.5       -
//     64, 128, 10               7.6 / 8.1      8.0 / 8.1      8.2 / 8.2        -
//     784, 128, 10             23.5 / 22.5    24.2 / 22.5    24.4 / 22.6   34.4 / 26.0
//     1024, 136, 10            31.2 / 33.4    32.1 / 33.2    32.3 / 33.3       -
//     784, 160, 10             27.9 / 28.3    28.8 / 28.6    29.1 / 28.6   41.2 / 30.2
//     64, 16, 10                6.7 / -        7.2 / -        7.3 / -       9.4 / 6.7
// so a second block a CU still pays, but for 105 to 128 units (the widest two folder waves hold) of a long row, or
// with more than 16 units past whole runs of 32 (the second layer adds those one LDS read at a time).
//     k_mlp, batch:               1             64-256         320-512       600-1024     1500      2048
//     75, 25, 10                5.7 / -        6.4 / -        6.7 / 7.8     6.4 / 8.1   8.1 / 8.4   7.7 / 8.4
//     105, 16, 10               6.1 / -        7.0 / -        9.0 / 8.4     7.1 / 8.7   8.5 / 9.1   8.2 / 9.2
//     34, 102, 10               6.9 / 8.1      7.7 / 8.6      9.7 / 8.9     8.1 / 9.0  10.4 / 9.4  10.8 / 9.5
//     75, 75, 50                8.4 / 9.5      9.0 / 10.0    10.0 / 10.5   10.0 / 11.4 12.9 / 11.3 13.8 / 11.4
//     134, 16, 10               7.3 / 8.2      8.3 / 8.7     10.8 / 9.0     8.4 / 9.1  10.0 / 9.5   9.6 / 9.5
//     100, 100, 50              9.6 / 10.4    10.1 / 10.9    11.4 / 11.4   11.7 / 12.5 15.4 / 12.6 16.6 / 12.8
//     50, 150, 10               8.7 / 9.8      9.7 / 10.4    12.5 / 10.6   11.0 / 10.8 14.4 / 12.3 16.6 / 12.4
//     164, 16, 10               8.1 / 8.7      9.2 / 9.1     12.1 / 9.5     9.4 / 9.7  11.0 / 10.2 10.7 / 10.3
//     70, 200, 5               10.5 / 11.5    11.9 / 11.9       -             -           -           -
//     195, 65, 10              11.9 / 10.1    12.6 / 10.6    14.1 / 11.4   14.0 / 12.2 19.6 / 12.6 21.0 / 12.7
// k_mlp's time is its two serial folds, an input costing about two hidden values; k_mlp_rows pays about 0.55 us
// a chunk of 32 of either, and more past 32 outputs (362 x 123 x 17 x 50 8.4 / 9.7; 512 x 130 x 130 x 50 13.4 / 14.1).
enum class MlpForm { kThread, kSplit, kRows };
inline MlpForm mlp_form(int64_t batch, int64_t in_f, int64_t hidden, int64_t out_f, bool split) {
  if (split) {
    const bool wide = (hidden > 104 && hidden <= 128 && in_f >= 256) || hidden % 32 > 16;
    return batch <= (wide && hidden > 64 && hidden <= 128 ? 256 : 512) ? MlpForm::kSplit : MlpForm::kRows;
  }
  const int64_t folds = 2 * in_f + hidden;
  const bool thread = batch <= 256    ? folds <= 344 && hidden <= 256
                      : batch <= 512  ? (out_f > 32 ? folds <= 400 && hidden <= 130 : folds <= 240 && hidden <= 80)
                      : batch <= 1024 ? folds <= 315 && hidden <= 128
                                      : batch <= 2048 && folds <= 260 && hidden <= 64;
  return thread ? MlpForm::kThread : MlpForm::kRows;
}

// Cells a block of the folded GEMV (K up to 4096): 16 or 32 with three producer waves, or 64 with six. Fewer cells
// leave the LDS pipe to the fold and spread a small N over more CUs; but a CU holds three blocks of 32 (by their
// LDS: 24576 rows a round of the chip) or two of 64 (32768 rows), and a second block on a CU slows the first.
// Kernel alone in a recorded graph, one box, us, 16 / 32 / 64:
//     N             K = 64              512                 1024                2048                4096
//     4097      3.0 / 3.2 / 3.3     4.3 / 4.5 / 4.8     5.9 / 5.9 / 6.6     9.8 / 9.7 / 10.6   17.2 / 16.0 / 18.7
//     8192      3.2 / 3.2 / 3.3     4.7 / 4.6 / 4.9     6.4 / 6.3 / 7.0    11.0 / 10.1 / 11.2  18.9 / 17.2 / 19.0
//     10000     3.3 / 3.4 / 3.3     5.4 / 5.1 / 4.9     7.4 / 7.1 / 7.0    12.7 / 12.1 / 11.9  21.0 / 21.3 / 19.3
//     16384     3.5 / 3.4 / 3.4     5.9 / 5.3 / 5.3     8.8 / 7.7 / 7.3    15.7 / 13.5 / 12.8  25.3 / 29.2 / 21.7
//     18000     4.5 / 3.7 / 3.8     7.7 / 6.2 / 6.7    12.4 / 9.7 / 10.0   21.0 / 16.8 / 18.5  35.9 / 36.2 / 33.7
//     24576     4.8 / 3.8 / 3.9     8.9 / 6.3 / 6.9    14.6 / 10.2 / 10.3  23.8 / 19.3 / 19.6  40.3 / 36.8 / 34.6
//     32768     5.2 / 5.1 / 4.0    10.5 / 9.2 / 7.1    16.9 / 14.1 / 13.3  27.9 / 24.3 / 21.8  47.8 / 48.3 / 41.1
//     40000     6.4 / 5.6 / 5.4    13.7 / 12.2 / 10.9  20.0 / 16.5 / 17.0  34.2 / 27.7 / 29.3          -
//     49152     7.1 / 5.9 / 5.5    15.5 / 13.2 / 11.8  23.0 / 18.7 / 17.7  39.9 / 32.9 / 30.4          -
//     65536     8.8 / 7.7 / 6.3    19.4 / 16.4 / 15.1  29.3 / 23.5 / 22.6  51.3 / 43.0 / 40.1          -
//     98304    12.2 / 10.0 / 9.7   26.9 / 21.6 / 21.6  41.0 / 31.6 / 33.7          -                   -
//     155648   18.2 / 15.3 / 13.7  39.4 / 31.2 / 30.3  66.2 / 54.3 / 55.9          -                   -
inline int gemv_cells(int64_t n, int64_t k) {
  if (n <= 4096) return 16;
  if (n <= 8192) return 32;
  if (n <= 16384) return 64;
  if (n <= 24576) return k <= 3584 ? 32 : 64;
  if (n <= 32768 || k < 768) return 64;
  return n <= 45056 || n > 90112 ? 32 : 64;
}

}  // namespace fo
