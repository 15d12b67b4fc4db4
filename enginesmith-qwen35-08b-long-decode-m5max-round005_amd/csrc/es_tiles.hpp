// Which form of a kernel a call takes and which tile a block works on: plain C++,
// used by the kernels, their launchers and a CPU test.
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

// Whether a GEMM without residual goes to the kernel of 256 x 256 tiles: each
// of its blocks has a CU to itself, so it is the faster one where the tiles fill
// the 256 CUs in whole rounds, nearly (one round alone needs fewer: what it is
// compared with is then two and a part), and where K is long enough for its
// start and end, which nothing else on the CU covers, not to weigh. us, it and
// the other kernel, rows x N x K:
//   192 tiles, one round     3035 x 4096 x 3584 124 and 115   1499 x 8192 x 2048  73 and  66
//   196 to 208, one round    3547 x 3584 x 3584 116 and 129   3291 x 4096 x 3584 119 and 128
//   256, one round           4059 x 4096 x 3584 132 and 144   2011 x 8192 x 4096 144 and 161
//   448 of 512               7131 x 4096 x 3584 248 and 238   3547 x 8192 x 2048 156 and 146
//   480 of 512               5083 x 6144 x 3584 256 and 273   3803 x 8192 x 4096 277 and 301
//   704 of 768              11227 x 4096 x 3584 375 and 373   2779 x 16384 x 2048 225 and 214
//   728 of 768              13275 x 3584 x 3584 368 and 391
//   K = 1024                 4096 x 6144 x 1024  81 and  67
constexpr bool gemm_wide(int n, int k, int m) {
  const long tiles = (long)((n + 255) / 256) * ((m + 255) / 256), rounds = (tiles + 255) / 256;
  return k >= 2048 && k % 128 == 0 && tiles >= (rounds == 1 ? 196 : 240 * rounds);
}

// Whether the matvec of several token rows gives a wave four weight rows (per
// half-wave where K = 1024, half_wave) instead of one (two): outputs = token rows
// x weight rows. A wave unpacks and sums its slices of x once for its weight rows
// (about 100 instructions a slice, more than a row's dot product over it), so
// four pay once their waves fill the 1024 SIMDs. Whole waves: at one a SIMD, not
// where a few SIMDs get a second, and again from one and a half. Half-waves,
// whose small form already has four weight rows a wave: from two and a half. us
// with the small form and with four, outputs:
//   K = 2048  4096 4.0 and 3.8   5120  4.5 and  4.7    6144  4.9 and  4.7   8192  5.8 and 4.7
//   K = 1536  4096 3.7 and 3.7   5120  4.2 and  4.6    6144  4.7 and  4.7   8192  5.4 and 4.7
//   K = 3584  4096 4.2 and 3.8   5120  4.7 and  4.8    6144  5.4 and  4.9  11264  8.3 and 6.4
//   K = 1024 12288 3.2 and 3.5  18432  3.8 and  4.0   20480  3.8 and  4.0  21504  4.1 and 4.0   32768 4.9 and 4.5
// Eight rows are slower again.
constexpr bool qmv_four_rows(bool half_wave, long outputs) {
  const long simds = 1024, waves = outputs / (half_wave ? 8 : 4);
  return half_wave ? 8 * simds * 5 / 2 < outputs : waves == simds || 2 * waves >= 3 * simds;
}

// Whether the attention's output gate takes eight elements a thread (where the
// pointers allow it) instead of one: below, fewer blocks finish later than more
// do. us with one and with eight, rows: 64 1.9 and 2.1, 160 2.1 and 2.15, 203 2.2
// and 2.15, 500 3.1 and 2.7, 4096 20.4 and 11.2.
constexpr bool gate_eight(int rows) { return rows >= 192; }

}  // namespace es
