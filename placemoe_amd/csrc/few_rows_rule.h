// Which kernel a grouped GEMM over copies with few rows runs on.
//
// The host knows the average rows per copy, rows / copies, not the counts; the
// kernels of few_rows.h come in two tilings, 64 x 128 with two blocks per CU and
// 128 x 256 with one.  Against the 256-row kernels (fc1 and fc2 dgrad: four
// waves; fc2 and fc1 dgrad: register-staged), 2048 x 768 layer, row counts
// log-normal with sigma 0.5 or Zipf(1.0), us (64 x 128 / 128 x 256 / 256-row):
//   copies rows      fc1             fc2             fc2 dgrad       fc1 dgrad
//   160    4.8 ln    177 / 174 / 256  91 /  93 / 105  96 /  96 / 136 185 / 170 / 182
//   160    25  ln    205 / 203 / 262 104 / 104 / 106 113 / 112 / 139 202 / 187 / 191
//   160    40  Zipf  -               -               127 / 157 / 141 241 / 209 / 238
//   128    96  ln    226 / 213 / 228 125 / 111 / 105 136 / 127 / 143 223 / 185 / 180
//   128    96  Zipf  234 / 222 / 241 130 / 120 / 122 146 / 157 / 143 250 / 202 / 204
//   128    128 ln    254 / 234 / 276 144 / 125 / 125 159 / 167 / 147 253 / 205 / 220
// Up to some tens of rows the call is bound by reading the weights, and the small
// tiles keep more of them in flight.  Beyond, the number of rounds of tiles
// decides: a persistent block that takes one tile more than the others adds a
// whole tile's time, and copies past 64 or 128 rows have more of the small tiles
// than of 256-row ones.  16 copies of 72 rows of 7168 x 2048, one round of 256-row
// tiles: fc1 254 us with 128 x 256 tiles against 213; 40 of 120 rows of 2048 x
// 1408: fc2 dgrad 99 against 75.  So a tiling is taken up to its line where its
// rounds are no more than those of one 256-row tile per copy and column strip.
// Three relaxations:
//  - up to the `always` line hardly any copy has a second tile, and the rounds are
//    not asked;
//  - the 64 x 128 tiles of fc1 and the fc2 dgrad may take half as many rounds
//    more, as theirs last about half as long as a 256-row tile's (their 256-row
//    kernel's loads have one K-tile to land, those of the register-staged one,
//    which runs fc2 and the fc1 dgrad, two);
//  - the 128 x 256 tiles of fc1 may be half as many more over three rounds or
//    more of K >= 1536 (2048 x 768, 128 copies of 96 rows: 203-213 us against
//    225; at K = 1280 they would be slower, 145 against 135).
// The dgrads' [K][N] weights prefer the 512-byte row segments of 128 x 256 tiles:
// the 64 x 128 ones serve the fc1 dgrad, and the fc2 dgrad up to its `always`
// line, only where 256-wide tiles would be fewer than the CUs.
//
// Over 37 layers (8 to 256 copies, 1024 to 7168 wide), 1 to 120 rows, even,
// log-normal and Zipf(1.0) counts, 1082 calls of each kind, the kernel this rule
// takes was at most 5% slower than the 256-row kernels (fc2 dgrad: 7% once);
// geometric means: fc1 0.79, fc2 0.89, fc1 dgrad 0.92, fc2 dgrad 0.71 of their
// time.
//
// Plain C++, so that the rule is unit-tested on the host.
#pragma once

#include <stdint.h>

namespace pmx {

struct FewRowsLines {
  int64_t max64, always64;  // rows per copy, 64 x 128 tiles
  int64_t half_rounds64;    // half rounds of them allowed per round of 256-row tiles
  int64_t max128;           // rows per copy, 128 x 256 tiles (0: not for this kind)
};
// fc1, fc2, fc1 dgrad, fc2 dgrad
constexpr FewRowsLines kFewRowsLines[4] = {{56, 40, 3, 120}, {48, 8, 2, 0}, {40, 8, 2, 40}, {56, 40, 3, 120}};
constexpr int64_t kFewRowsAlways128 = 8;

// The m-tile height of the few-rows kernel for `rows` rows over `copies` copies,
// N output columns, K deep, on `cus` CUs: 64, 128, or 0 for the 256-row kernels.
// kind: 0 fc1, 1 fc2, 2 fc1 dgrad, 3 fc2 dgrad.
inline int few_rows_tiling(int kind, int64_t rows, int64_t copies, int64_t N, int64_t K, int64_t cus) {
  const FewRowsLines& l = kFewRowsLines[kind];
  const auto div_up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t active = rows < copies ? rows : copies;  // copies with rows, at most
  // a copy's last tile whole, rows past the first as half a tile each tile height
  // (between even and Zipf(1.0) counts)
  const auto tiles = [&](int64_t bm, int64_t bn) { return (active + rows / (2 * bm)) * div_up(N, bn); };
  const int64_t tiles256 = active * div_up(N, 256), rounds256 = div_up(tiles256, cus);
  const bool narrow = kind < 2 || tiles256 < cus;
  if (rows <= l.max64 * copies) {
    if (narrow && rows <= l.always64 * copies) return 64;
    if ((narrow || kind == 3) && 2 * div_up(tiles(64, 128), 2 * cus) <= l.half_rounds64 * rounds256) return 64;
  }
  if (rows <= l.max128 * copies) {
    if (rows <= kFewRowsAlways128 * copies || div_up(tiles(128, 256), cus) <= rounds256) return 128;
    if (kind == 0 && K >= 1536 && rounds256 >= 3 && 2 * tiles(128, 256) <= 3 * rounds256 * cus) return 128;
  }
  return 0;
}

}  // namespace pmx
