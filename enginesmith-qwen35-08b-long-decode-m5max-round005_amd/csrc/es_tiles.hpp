// Which tile a GEMM block works on: plain C++, used by the kernels and by the
// CPU test of the deal.
#pragma once

namespace es {

struct GemmTile {
  int bx, by;
};

// Block b of nb column tiles x mb row tiles. The dispatcher sends block b to
// XCD b % 8. Row tiles in groups of eight go one to an XCD, whose L2 then holds
// one copy of the tile's X for all its columns; the mb % 8 that are left go
// column by column over all XCDs. (Dealt whole as well, they load as many XCDs
// and leave the others idle: 9 row tiles of the MLP's 56 column tiles put 112
// blocks on one XCD and 56 on each other, and 1030 rows took 44 us instead of
// 27.)
constexpr unsigned gemm_grid(unsigned nb, unsigned mb) { return nb * mb; }
constexpr GemmTile gemm_tile(unsigned b, unsigned nb, unsigned mb) {
  const unsigned whole = mb & ~7u;
  if (b < nb * whole) {
    const unsigned i = b >> 3;
    return {(int)(i % nb), (int)((b & 7) + 8 * (i / nb))};
  }
  const unsigned r = b - nb * whole;
  return {(int)(r % nb), (int)(whole + r / nb)};
}

}  // namespace es
