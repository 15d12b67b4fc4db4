// Batched prefill kernels (Model::encode_forward with rows > 1,
// model.rs:228-350): the row-batched forms of the decode path's operators.
//
// k_q4_gemm: Y[M,N] = bf16(X[M,K] . dequant(W)[N,K]^T), optionally
//   Y = bf16(R + that), as qmm_q4_nax (linear_nax.metal:1096-1139) computes
//   it: each weight is dequantised to bf16, bf16(scale*q + bias), and the
//   products accumulate in fp32 (v_mfma_f32_32x32x16_bf16 over K in increasing
//   order, one chain per output whatever the tiling, so every kernel and tile
//   height gives the same bits).
//   Operand layouts (32x32x16 bf16): lane l holds A[l%32][8(l/32)..+7] and
//   B[8(l/32)..+7][l%32]; result element r of lane l is
//   D[8(r/4) + 4(l/32) + r%4][l%32].
#include <type_traits>

#include "es_kernels.hpp"
#include "es_tiles.hpp"

namespace es {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Wait until at most N vector-memory operations of this wave are pending.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Two values -> packed bf16 pair (lo in bits 0..15), one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack_bf2(lo, hi); }

// The 8 nibbles of one code word (element j = bits 4j..4j+3) as
// fma(scale, q, bias), packed to four bf16 pairs. The even nibbles are the
// bytes of word & 0x0F0F0F0F and the odd ones the bytes of
// (word >> 4) & 0x0F0F0F0F, so each converts with one v_cvt_f32_ubyteN (the
// masked words are hidden from known-bits analysis, which would otherwise
// extract every nibble separately).
__device__ __forceinline__ u32x4 dequant8(uint32_t word, float sc, float bi) {
  uint32_t lo = word & 0x0F0F0F0Fu;
  uint32_t hi = (word >> 4) & 0x0F0F0F0Fu;
  asm("" : "+v"(lo));
  asm("" : "+v"(hi));
  float v[8];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    v[2 * b] = fmaf(sc, (float)((lo >> (8 * b)) & 0xffu), bi);
    v[2 * b + 1] = fmaf(sc, (float)((hi >> (8 * b)) & 0xffu), bi);
  }
  return u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
}

// ---- GEMM: 32 MT x 128 block tiles, weights dequantised in registers ----
//
// Block = four waves side by side along N, each 32 MT rows x 32 columns. A
// lane's 8 values of an MFMA's weight operand are the 8 nibbles of one code
// word, so a wave dequantises its own columns straight into the operand: no
// dequantised weight goes through LDS or is made twice in a block. The weights
// are the MFMA's A operand, so a lane's results are one row and groups of four
// consecutive columns. X goes through LDS (the four waves read all of it), 64
// columns of K a step, two stages, one barrier a step; global loads run four
// steps ahead in registers.
//
// A step's arithmetic is 4 MT MFMAs (32 cycles each) and about 115 vector
// instructions of dequantisation (4 cycles each) that issue in their shadow:
// MT = 4 balances them, smaller MT repeat the dequantisation for fewer rows.
// Measured against a 128 x 128 kernel that staged both operands one step ahead
// and stored its results one by one (us a launch in a graph's replay; the third
// and the last on 256 x 256 tiles before; under the profiler, whose runs clock
// lower, the present kernel's first, second, fourth and last take 26, 47, 89 and
// 71):
//   rows x N x K  203 x 1024 x 3584  4096 x 1024 x 3584  1000 x 4096 x 1024  4096 gate/up  4096 x 6144 x 1024
//   before              56                 81                  40               103              84
//   now                 26                 45                  18                82              68
constexpr int kGemmBK = 64, kGemmAhead = 4;

// 16-byte chunk c of 64-column row r: chunk slot c ^ ((r >> 1) & 7), so the 16
// rows that one 16-lane group of a fragment read touches cover all banks once.
__device__ __forceinline__ int tile_slot(int r, int c) { return ((c ^ ((r >> 1) & 7)) << 3) + (r << 6); }

// Barrier for LDS data alone: unlike __syncthreads it does not wait for global
// loads still in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The code word of slice kk (16 columns of K) for every lane: word 2 kk in
// lanes 0..31 and word 2 kk + 1 in lanes 32..63.
__device__ __forceinline__ u32x4 slice_words(const u32x4 c) {
  const auto p = __builtin_amdgcn_permlane32_swap(c[0], c[1], false, false);  // {w0|w1}, {w4|w5}
  const auto q = __builtin_amdgcn_permlane32_swap(c[2], c[3], false, false);  // {w2|w3}, {w6|w7}
  return u32x4{p[0], q[0], p[1], q[1]};
}

// act = bf16(bf16(g * sigmoid_bf(g)) * u) of the bf16-rounded gate and up
__device__ __forceinline__ float swiglu(float g, float u) {
  const float gb = rbf(g), ub = rbf(u);
  return rbf(rbf(gb * sigmoid_bf(gb)) * ub);
}

// GATEUP: segment 0 is the gate matrix and segment 1 the up matrix of the MLP;
// a wave's 32 weight rows are 16 rows of gate and the same 16 of up, so a lane
// holds both of a column and writes swiglu(g, u) (swiglu_bf16 after the two
// linears) to y[0] [m, N]. Otherwise the
// output columns span the stacked segments of a, each written to its own
// [m][n_s] output; residual (one segment only) may alias y[0].
//
// Weights are fetched four steps (256 columns of K, one 128-byte line of codes
// a row) at a time, eight lanes to a row, and laid down in the wave's own LDS,
// from which each lane takes its column's words step by step: fetching them a
// step at a time straight into the lanes that use them touches a line four
// times, after other rows' lines have evicted it from the L1, and one more line
// a step for two bytes of scale. LINES: K is a multiple of 256 and the scales
// allow four-byte accesses; otherwise the loads stay within the row one by one.
template <int MT, bool GATEUP, bool LINES>
__global__ __launch_bounds__(256, 2) void k_q4_gemm(GemmArgs a, const uint16_t* residual) {
  constexpr int kRows = 32 * MT, D = kGemmAhead, kCols = GATEUP ? 16 : 32;  // output columns of a wave
  __shared__ __attribute__((aligned(16))) uint16_t xs[2][kRows * kGemmBK];
  __shared__ __attribute__((aligned(16))) uint16_t wl[4][32 * kGemmBK];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int fr = lane & 31, fh = lane >> 5;
  const int K = a.w[0].k, m = a.m, nk = K / kGemmBK;
  const int ncols = GATEUP ? a.w[0].n : a.nstart[a.nseg];
  int bx = blockIdx.x, by = blockIdx.y;
  if (a.by_xcd) {
    const GemmTile tile = gemm_tile(blockIdx.x, (ncols + 4 * kCols - 1) / (4 * kCols), (m + kRows - 1) / kRows);
    bx = tile.bx;
    by = tile.by;
  }
  const int m0 = by * kRows;

  // Weight rows: lane l fetches chunk l % 8 of rows 8 i + l / 8 (i = 0..3) of
  // its wave's 32, and the scales (lanes 0..31) or biases (32..63) of row
  // l % 32. Rows past the end read row 0 and are not stored.
  const int wn0 = (bx * 4 + wave) * kCols;
  auto locate = [&](int n, int& seg) {  // n of the wave's 32 -> segment and row in it
    const int c = wn0 + (GATEUP ? n & 15 : n);
    seg = GATEUP ? n >> 4 : 0;
    if (GATEUP) return c < ncols ? c : 0;
#pragma unroll
    for (int q = 1; q < 4; ++q)
      if (q < a.nseg && c < ncols && c >= a.nstart[q]) seg = q;
    return c < ncols ? c - a.nstart[seg] : 0;
  };
  const uint32_t* cptr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int seg;
    const int row = locate(8 * i + (lane >> 3), seg);
    const uint32_t* w = seg == 0 ? a.w[0].w : seg == 1 ? a.w[1].w : seg == 2 ? a.w[2].w : a.w[3].w;
    cptr[i] = w + (size_t)row * (K >> 3) + (LINES ? (lane & 7) * 4 : 0);
  }
  const uint16_t* sptr;
  {
    int seg;
    const int row = locate(fr, seg);
    const uint16_t* w = fh ? (seg == 0 ? a.w[0].b : seg == 1 ? a.w[1].b : seg == 2 ? a.w[2].b : a.w[3].b)
                           : (seg == 0 ? a.w[0].s : seg == 1 ? a.w[1].s : seg == 2 ? a.w[2].s : a.w[3].s);
    sptr = w + (size_t)row * (K >> 6);
  }
  // four steps' weights in flight, and the scales and biases of the four at hand
  u32x4 cq[4];
  uint2 sq;
  uint32_t sc4[2], bi4[2];
  auto load_w = [&](int grp) {
    // LINES: whole groups only; otherwise a chunk past the row's end repeats its last one
#pragma unroll
    for (int i = 0; i < 4; ++i)
      cq[i] = *reinterpret_cast<const u32x4*>(cptr[i] + (LINES ? grp * 32 : min(grp * 8 + (lane & 7), 2 * nk - 1) * 4));
    if (LINES) {
      sq = *reinterpret_cast<const uint2*>(sptr + grp * 4);
    } else {
      uint32_t v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = sptr[min(grp * 4 + i, nk - 1)];
      sq = make_uint2(v[0] | v[1] << 16, v[2] | v[3] << 16);
    }
  };
  // the fetched four steps become the ones at hand
  auto turn_w = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x4*>(&wl[wave][tile_slot(8 * i + (lane >> 3), lane & 7)]) = cq[i];
    const auto p = __builtin_amdgcn_permlane32_swap(sq.x, sq.x, false, false);  // {scales|scales}, {biases|biases}
    const auto q = __builtin_amdgcn_permlane32_swap(sq.y, sq.y, false, false);
    sc4[0] = p[0]; bi4[0] = p[1];
    sc4[1] = q[0]; bi4[1] = q[1];
  };
  // the lane's words, scale and bias of step u of the four
  auto words = [&](int u) { return slice_words(*reinterpret_cast<const u32x4*>(&wl[wave][tile_slot(fr, 2 * u + fh)])); };
  auto scale = [&](int u) { return (u & 1) ? bf_hi(sc4[u >> 1]) : bf_lo(sc4[u >> 1]); };
  auto bias = [&](int u) { return (u & 1) ? bf_hi(bi4[u >> 1]) : bf_lo(bi4[u >> 1]); };

  // X: thread t moves chunk t & 7 of rows t / 8 + 32 i
  const int xc = t & 7, xr = t >> 3;
  const uint16_t* xbase = a.x + (size_t)m0 * K;
  uint32_t xoff[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xoff[i] = (uint32_t)min(xr + 32 * i, m - 1 - m0) * (uint32_t)K + xc * 8;
  auto load_x = [&](int kb, u32x4 (&r)[MT]) {
#pragma unroll
    for (int i = 0; i < MT; ++i) r[i] = *reinterpret_cast<const u32x4*>((xbase + kb * kGemmBK) + xoff[i]);
  };
  auto store_x = [&](int buf, const u32x4 (&r)[MT]) {
#pragma unroll
    for (int i = 0; i < MT; ++i) *reinterpret_cast<u32x4*>(&xs[buf][tile_slot(xr + 32 * i, xc)]) = r[i];
  };

  f32x16 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;

  // Loads are issued in the loop's order, which its waits count: the fences
  // keep it.
  const int ngrp = (nk + 3) / 4;
  u32x4 xq[D][MT];
  u32x4 bq[4];  // weight operands of a step's four slices
  load_w(0);
  issue_fence();
  load_x(0, xq[0]);
  issue_fence();
  turn_w();
  issue_fence();
  load_w(min(1, ngrp - 1));
  issue_fence();
#pragma unroll
  for (int u = 1; u < D; ++u) {
    load_x(min(u, nk - 1), xq[u]);
    issue_fence();
  }
  store_x(0, xq[0]);
  load_x(min(D, nk - 1), xq[0]);
  issue_fence();
  {
    const u32x4 wd = words(0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) bq[kk] = dequant8(wd[kk], scale(0), bias(0));
  }
  lds_barrier();
  // Step kb = 4 i + u. No step branches, so every wait counts the loads issued
  // since its own: the loads past the last step repeat it and the X they would
  // bring goes to a stage nobody reads.
  auto step = [&](int kb, auto uc) {
    constexpr int u = decltype(uc)::value, un = (u + 1) % 4;
    issue_fence();
    if (u == 3) {
      turn_w();
      issue_fence();
      load_w(min(kb / 4 + 2, ngrp - 1));
    }
    // the next step's X to the other stage, whose readers passed the last barrier
    store_x((u + 1) & 1, xq[un]);
    load_x(min(kb + 1 + D, nk - 1), xq[un]);
    const u32x4 wd = words(un);
    issue_fence();
    bf16x8 xf[2][MT];
    auto read_x = [&](int kk) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
        xf[kk & 1][i] = *reinterpret_cast<const bf16x8*>(&xs[u & 1][tile_slot(32 * i + fr, 2 * kk + fh)]);
    };
    read_x(0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk + 1 < 4) read_x(kk + 1);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bq[kk]), xf[kk & 1][i], acc[i], 0, 0, 0);
      bq[kk] = dequant8(wd[kk], scale(un), bias(un));  // the same slice of the next step
    }
    // Issue order: the next slice's fragment reads, then MFMAs each followed by
    // its share of the dequantisation, which runs in the MFMA's shadow.
    __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk + 1 < 4) __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 24 / MT, 0);
      }
    }
    issue_fence();
    lds_barrier();
  };
  int k0 = 0;
  for (; k0 + 4 <= nk; k0 += 4) {
    step(k0, std::integral_constant<int, 0>{});
    step(k0 + 1, std::integral_constant<int, 1>{});
    step(k0 + 2, std::integral_constant<int, 2>{});
    step(k0 + 3, std::integral_constant<int, 3>{});
  }
  if (!LINES) {
    if (k0 < nk) step(k0, std::integral_constant<int, 0>{});
    if (k0 + 1 < nk) step(k0 + 1, std::integral_constant<int, 1>{});
    if (k0 + 2 < nk) step(k0 + 2, std::integral_constant<int, 2>{});
  }

  // Lane l holds row l % 32 of each row tile and, for g = 0..3, weight rows
  // 8 g + 4 (l / 32) .. + 3 of the wave's 32.
  auto column = [&](int n, uint16_t*& y, int& ld) {  // output column n -> its matrix and column there
    int sg = 0;
    if (!GATEUP) {
#pragma unroll
      for (int q = 1; q < 4; ++q)
        if (q < a.nseg && n >= a.nstart[q]) sg = q;
    }
    y = sg == 0 ? a.y[0] : sg == 1 ? a.y[1] : sg == 2 ? a.y[2] : a.y[3];
    ld = GATEUP ? ncols : a.nstart[sg + 1] - a.nstart[sg];
    return n - (GATEUP ? 0 : a.nstart[sg]);
  };
  auto value = [&](int i, int r) { return GATEUP ? swiglu(acc[i][r], acc[i][(r + 8) & 15]) : acc[i][r]; };
  uint16_t* y;
  int ld;
  if (a.vec) {  // 8 columns and one 16-byte store a lane: the halves of a pair of groups change lanes
#pragma unroll
    for (int p = 0; p < kCols / 16; ++p) {
      const int n = wn0 + 16 * p + 8 * fh;
      const int col = column(n, y, ld);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = value(i, 8 * p + e);
        const auto c01 = __builtin_amdgcn_permlane32_swap(pack2(v[0], v[1]), pack2(v[4], v[5]), false, false);
        const auto c23 = __builtin_amdgcn_permlane32_swap(pack2(v[2], v[3]), pack2(v[6], v[7]), false, false);
        const int row = m0 + 32 * i + fr;
        if (row >= m || n >= ncols) continue;
        u32x4 o = u32x4{c01[0], c23[0], c01[1], c23[1]};
        const size_t at = (size_t)row * ld + col;
        if (residual) {
          const u32x4 rs = *reinterpret_cast<const u32x4*>(residual + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = pack2(bf_lo(rs[e]) + bf_lo(o[e]), bf_hi(rs[e]) + bf_hi(o[e]));
        }
        *reinterpret_cast<u32x4*>(y + at) = o;
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < kCols / 2; ++r) {
      const int row = m0 + 32 * i + fr, n = wn0 + 8 * (r >> 2) + 4 * fh + (r & 3);
      if (row >= m || n >= ncols) continue;
      const int col = column(n, y, ld);
      const size_t o = (size_t)row * ld + col;
      float v = rbf(value(i, r));
      if (residual) v = bf2f(residual[o]) + v;
      y[o] = (uint16_t)f2bf(v);
    }
}

// ---- wide GEMM: 256 x 256 block tiles for a long K and many tiles (gemm_wide) ----
//
// k_q4_gemm_wide computes the same products as k_q4_gemm, bit for bit: the
// same bf16 operands (weights dequantised as bf16(fma(scale, q, bias))) and,
// for every output element, the same sequence of 32x32x16 MFMAs over K in
// increasing order. Only the tiling differs. A block of 256 threads owns a
// 256 x 256 output tile; each wave a 128 x 128 quarter (16 MFMA accumulators
// in the accumulation registers), so every 16-byte fragment read from LDS
// feeds four MFMAs instead of two. X reaches LDS by DMA (global_load_lds, no
// registers); each thread dequantises one weight row per 64-column step.
// LDS rows are 128 bytes with no padding; the 16-byte chunk c of row r sits
// at slot c ^ ((r >> 1) & 7), so the 16 rows that one 16-lane group of a
// fragment read touches cover all 64 banks once. The X DMA applies the same
// permutation on the source side (lane l of an instruction fetches the chunk
// that belongs in its slot).
// A block holds a whole CU (128 KB of LDS, all registers), so nothing covers
// its start and end: it is the faster kernel for a long K only.
constexpr int kWideM = 256, kWideN = 256, kWideK = 64;
static_assert(kWideM == 256 && kWideN == 256 && kWideK == 64, "gemm_wide counts these tiles, K in pairs of steps");

// Fragment reads as inline assembly: the compiler treats an LDS read after a
// DMA into LDS as dependent on it and would wait for every DMA in flight
// (including the next stage's) before the first read of a step. Four reads
// of one operand: rows r, r+32, r+64, r+96 share the slot, 4096 bytes apart.
__device__ __forceinline__ void wide_read4(uint32_t addr, u32x4& f0, u32x4& f1, u32x4& f2, u32x4& f3) {
  asm volatile(
      "ds_read_b128 %0, %4\n\t"
      "ds_read_b128 %1, %4 offset:4096\n\t"
      "ds_read_b128 %2, %4 offset:8192\n\t"
      "ds_read_b128 %3, %4 offset:12288"
      : "=&v"(f0), "=&v"(f1), "=&v"(f2), "=&v"(f3)
      : "v"(addr));
}
__device__ __forceinline__ void wide_wait8(u32x4 (&a)[4], u32x4 (&b)[4]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
}

// One 64-column step of the MFMA loop over the staged tiles at LDS byte
// addresses xt (X) and wt (W): the fragments of slice kk + 1 are read while
// the 16 MFMAs of slice kk run.
__device__ __forceinline__ void wide_step(uint32_t xt, uint32_t wt, int xrow, int wrow, f32x16 (&acc)[4][4],
                                          int fh) {
  // byte address of slot c of rows xrow (+32i) and wrow (+32j)
  auto xaddr = [&](int c) { return xt + (uint32_t)(tile_slot(xrow, c) * 2); };
  auto waddr = [&](int c) { return wt + (uint32_t)(tile_slot(wrow, c) * 2); };
  u32x4 fa[2][4], fb[2][4];
  wide_read4(xaddr(fh), fa[0][0], fa[0][1], fa[0][2], fa[0][3]);
  wide_read4(waddr(fh), fb[0][0], fb[0][1], fb[0][2], fb[0][3]);
  wide_wait8(fa[0], fb[0]);
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int cur = kk & 1;
    if (kk + 1 < 4) {
      const int c = 2 * (kk + 1) + fh;
      wide_read4(xaddr(c), fa[cur ^ 1][0], fa[cur ^ 1][1], fa[cur ^ 1][2], fa[cur ^ 1][3]);
      wide_read4(waddr(c), fb[cur ^ 1][0], fb[cur ^ 1][1], fb[cur ^ 1][2], fb[cur ^ 1][3]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[cur][i]),
                                                            __builtin_bit_cast(bf16x8, fb[cur][j]), acc[i][j], 0,
                                                            0, 0);
    if (kk + 1 < 4) wide_wait8(fa[cur ^ 1], fb[cur ^ 1]);
  }
}

// The two stages are four separate LDS arrays (not one indexed array), so the
// compiler can see that the DMA into one stage does not write the other and
// does not wait for it before reading fragments.
__shared__ __attribute__((aligned(16))) uint16_t g_wide_x0[kWideM * kWideK];
__shared__ __attribute__((aligned(16))) uint16_t g_wide_x1[kWideM * kWideK];
__shared__ __attribute__((aligned(16))) uint16_t g_wide_w0[kWideN * kWideK];
__shared__ __attribute__((aligned(16))) uint16_t g_wide_w1[kWideN * kWideK];

__global__ __launch_bounds__(256, 1) void k_q4_gemm_wide(Q4 w, const uint16_t* x, int m, uint16_t* y) {
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int K = w.k;
  const int m0 = blockIdx.y * kWideM;
  const int nk = K / kWideK;

  // this thread's weight row
  const int n_row = blockIdx.x * kWideN + t;
  const bool wok = n_row < w.n;
  const int r_ok = wok ? n_row : 0;
  const u32x4* cptr = reinterpret_cast<const u32x4*>(w.w + (size_t)r_ok * (K >> 3));
  const uint16_t* sptr = w.s + (size_t)r_ok * (K >> 6);
  const uint16_t* bptr = w.b + (size_t)r_ok * (K >> 6);

  // X DMA: instruction i of this wave fills LDS rows 8(8w+i) .. +7, lane l
  // the slot l & 7 of row l >> 3
  const int xr_lane = lane >> 3, xslot = lane & 7;
  auto issue_x = [&](int kb, uint16_t* xt) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = (wave * 8 + i) * 8 + xr_lane;
      const int c = xslot ^ ((r >> 1) & 7);
      const int gr = min(m0 + r, m - 1);
      const uint16_t* g = x + (size_t)gr * K + kb * kWideK + c * 8;
      __builtin_amdgcn_global_load_lds(g, (lds_ptr_t)&xt[(wave * 8 + i) * 512], 16, 0, 0);
    }
  };
  // Weight loads and the dequantised stores are inline assembly as well, so
  // the compiler inserts no waits of its own in the loop; each wait below is
  // counted by hand (the order of the vector-memory operations of a step:
  // the previous step's 4 weight loads, 8 X DMA, this step's 4 weight loads).
  struct WRegs {
    u32x4 c0, c1;
    uint32_t s, b;
  };
  auto load_w = [&](int kb, WRegs& r) {
    const u32x4* cp = cptr + kb * 2;
    const uint16_t* sp = sptr + kb;
    const uint16_t* bp = bptr + kb;
    asm volatile(
        "global_load_dwordx4 %0, %4, off\n\t"
        "global_load_dwordx4 %1, %4, off offset:16\n\t"
        "global_load_ushort %2, %5, off\n\t"
        "global_load_ushort %3, %6, off"
        : "=&v"(r.c0), "=&v"(r.c1), "=&v"(r.s), "=&v"(r.b)
        : "v"(cp), "v"(sp), "v"(bp));
  };
  // dequantise 64 weights (bf16(fma(scale, q, bias)); rows past N are 0);
  // the caller has waited for the set's loads
  auto store_w = [&](uint32_t wt, const WRegs& r) {
    const float sc = wok ? bf2f(r.s) : 0.0f, bi = wok ? bf2f(r.b) : 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const u32x4 o = dequant8(c < 4 ? r.c0[c] : r.c1[c - 4], sc, bi);
      asm volatile("ds_write_b128 %0, %1" ::"v"(wt + (uint32_t)(tile_slot(t, c) * 2)), "v"(o));
    }
  };
  // waits for a weight set with N vector-memory operations issued after it
  auto wait_set12 = [](WRegs& r) { asm volatile("s_waitcnt vmcnt(12)" : "+v"(r.c0), "+v"(r.c1), "+v"(r.s), "+v"(r.b)); };
  auto wait_set4 = [](WRegs& r) { asm volatile("s_waitcnt vmcnt(4)" : "+v"(r.c0), "+v"(r.c1), "+v"(r.s), "+v"(r.b)); };

  const int wm = (wave >> 1) * 128, wn = (wave & 1) * 128;
  const int fr = lane & 31, fh = lane >> 5;
  f32x16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Weights are loaded two steps ahead (register sets wa, wb) and dequantised
  // into the stage being filled while the MFMAs of the other stage run; the
  // end-of-step wait covers the X DMA but not the four weight loads issued
  // after it.
  auto lds_addr = [](const uint16_t* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)p;
  };
  const uint32_t lx0 = lds_addr(g_wide_x0), lx1 = lds_addr(g_wide_x1);
  const uint32_t lw0 = lds_addr(g_wide_w0), lw1 = lds_addr(g_wide_w1);
  // Weights are loaded two steps ahead (register set wa for even steps, wb
  // for odd) and dequantised into the stage being filled after the MFMAs of
  // the other stage are issued. Every step issues the same operations, so the
  // loop has no branch between a load and its wait: the X DMA of step s + 1
  // (8 operations) and the weight loads of step s + 2 (4), with the step
  // clamped to the last one (those loads fill the stage nobody reads again).
  // At the start of step s only the loads of weight set s + 1 are in flight;
  // it waits for them with 12 operations issued after them, and for its DMA
  // with 4.
  WRegs wa, wb;
  issue_x(0, g_wide_x0);
  load_w(0, wa);
  load_w(1, wb);
  wait_set4(wa);
  store_w(lw0, wa);
  lds_barrier();
  auto run_step = [&](int st, uint32_t lx, uint32_t lw, uint16_t* x_next, uint32_t lw_next, WRegs& w_next,
                      WRegs& w_after) {
    issue_x(min(st + 1, nk - 1), x_next);
    load_w(min(st + 2, nk - 1), w_after);
    issue_fence();
    wide_step(lx, lw, wm + fr, wn + fr, acc, fh);
    wait_set12(w_next);
    store_w(lw_next, w_next);
    wait_vmcnt<4>();
    lds_barrier();
  };
  for (int kb = 0; kb < nk; kb += 2) {  // K is a multiple of 128: nk even
    run_step(kb, lx0, lw0, g_wide_x1, lw1, wb, wa);
    run_step(kb + 1, lx1, lw1, g_wide_x0, lw0, wa, wb);
  }
  // The last step's weight loads (into wb) are still in flight: wait with
  // both sets as operands, so the compiler keeps their registers until the
  // data has landed instead of giving them to the epilogue.
  asm volatile("s_waitcnt vmcnt(0)"
               : "+v"(wa.c0), "+v"(wa.c1), "+v"(wa.s), "+v"(wa.b), "+v"(wb.c0), "+v"(wb.c1), "+v"(wb.s), "+v"(wb.b));

#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = blockIdx.x * kWideN + wn + 32 * j + fr;
    if (n >= w.n) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * fh + (r & 3);
        if (row < m) y[(size_t)row * w.n + n] = (uint16_t)f2bf(acc[i][j][r]);
      }
  }
}

// ---- row kernels: the decode operators' arithmetic, one row per token ----

// Embedding rows (embedding_q4, linear.metal:11-24): h = bf16(scale*q + bias).
// Half-wave per row, 32 elements per lane.
__global__ __launch_bounds__(256) void k_embed_rows(Q4 e, const uint32_t* tokens, int m, uint16_t* h) {
  const int row = blockIdx.x * 8 + (threadIdx.x >> 5), sl = threadIdx.x & 31;
  if (row >= m) return;
  uint32_t tok = tokens[row];
  if (tok >= (uint32_t)e.n) tok = 0;
  const u32x4 c = *reinterpret_cast<const u32x4*>(e.w + (size_t)tok * 128 + sl * 4);
  const float sc = bf2f(e.s[(size_t)tok * 16 + sl / 2]), bi = bf2f(e.b[(size_t)tok * 16 + sl / 2]);
  float xv[32];
#pragma unroll
  for (int w = 0; w < 4; ++w)
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[8 * w + j] = rbf(fmaf(sc, (float)((c[w] >> (4 * j)) & 15u), bi));
  store_bf16x32(h + (size_t)row * 1024 + sl * 32, xv);
}

// RMSNorm rows (rms_norm_bf16 rounding points, the decode kernels' order).
__global__ __launch_bounds__(256) void k_rmsnorm_rows(const uint16_t* x, const uint16_t* gain, int m,
                                                      uint16_t* out) {
  const int row = blockIdx.x * 8 + (threadIdx.x >> 5), sl = threadIdx.x & 31;
  if (row >= m) return;
  const Raw64 xr = load_raw64(x + (size_t)row * 1024 + sl * 32);
  const Raw64 gr = load_raw64(gain + sl * 32);
  float xv[32], xn[32];
  unpack_bf16x32(xr, xv);
  norm_slice_1024(xv, gr, xn);
  store_bf16x32(out + (size_t)row * 1024 + sl * 32, xn);
}

// SwiGLU (swiglu_bf16, linear.metal:382-398): silu = bf16(g*sigmoid_bf(g)),
// act = bf16(silu*up), over bf16 gate and up.
__global__ __launch_bounds__(256) void k_swiglu_rows(const uint16_t* gate, const uint16_t* up, int count,
                                                     uint16_t* act) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  const float gb = bf2f(gate[i]), ub = bf2f(up[i]);
  const float silu = rbf(gb * sigmoid_bf(gb));
  act[i] = (uint16_t)f2bf(silu * ub);
}

// GDN prepare rows (gdn_conv + gdn_prepare, gdn.metal:33-120, with the decode
// kernels' arithmetic): one wave per (4 consecutive rows, head), which loads
// the 7 input rows the 4 rows' taps span once. Lane i takes channels i and
// 64+i of the head's q, k and v: causal conv over taps (pos-3 .. pos) whose
// inputs are the chunk's raw rows, or the ring for positions before the
// chunk; SiLU; q and k L2-normalised (sum of squares tree64 over channels
// 0..63 plus tree64 over 64..127) and scaled (q by 1/128, k by bf16(128^-1/2));
// the gates are g = exp(-exp(A_log)*softplus(bf16(a+dt))), beta =
// sigmoid_bf(b). Outputs bf16 q, k, v [m,16,128] and fp32 g, beta [m,16].
// Bound by its arithmetic (24 convolutions and SiLUs a lane): 4096 rows take
// 49 us (86 us with a branch around every load and exponential, and the norms'
// reciprocals and the gates computed a row at a time).
constexpr int kPrepRows = 4;  // rows per wave: their taps span kPrepRows + 3 input rows
__global__ __launch_bounds__(256) void k_gdn_prep_rows(const uint16_t* raw, const uint16_t* ring,
                                                       const uint16_t* conv_w, const uint16_t* a_proj,
                                                       const uint16_t* b_proj, const float* a_log,
                                                       const uint16_t* dt_bias, int pos0, int m,
                                                       uint16_t* q, uint16_t* k, uint16_t* v, float* g,
                                                       float* beta) {
  const int lane = threadIdx.x & 63, h = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int t0 = blockIdx.x * kPrepRows;
  if (t0 >= m) return;
  const int nr = min(kPrepRows, m - t0);
  // input rows t0-3 .. t0+kPrepRows-1: the chunk's raw rows, or the ring for
  // positions before the chunk; those past the chunk (its last row here) enter
  // only outputs that are not stored
  const uint16_t* rows[kPrepRows + 3];
#pragma unroll
  for (int i = 0; i < kPrepRows + 3; ++i) {
    const int tt = t0 - 3 + i;
    rows[i] = tt >= 0 ? raw + (size_t)min(tt, m - 1) * kConv : ring + (size_t)((pos0 + tt) & 3) * kConv;
  }
  float out[3][2][kPrepRows];
#pragma unroll
  for (int part = 0; part < 3; ++part)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int c = part * 2048 + h * 128 + half * 64 + lane;
      uint32_t x[kPrepRows + 3];
#pragma unroll
      for (int i = 0; i < kPrepRows + 3; ++i) x[i] = rows[i][c];
      const uint2 w = *reinterpret_cast<const uint2*>(conv_w + (size_t)c * 4);
#pragma unroll
      for (int r = 0; r < kPrepRows; ++r) out[part][half][r] = conv4_silu(x + r, w);
    }
  // Lane 2 r + part takes the square-root reciprocal of row r's q (part 0) or k
  // (part 1), and lane r row r's gates: once for all rows instead of a row at a
  // time on a wave whose other lanes idle.
  float tot = 0.0f;
#pragma unroll
  for (int r = 0; r < kPrepRows; ++r)
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      const float s2 = tree64(out[part][0][r] * out[part][0][r]) + tree64(out[part][1][r] * out[part][1][r]);
      tot = lane == 2 * r + part ? s2 : tot;
    }
  const float inv_all = 1.0f / sqrtf(tot / 128.0f + 1.0e-6f / 128.0f);
  if (lane < nr) {
    const int t = t0 + lane;
    const float ax = rbf(bf2f(a_proj[(size_t)t * 16 + h]) + bf2f(dt_bias[h]));
    g[(size_t)t * 16 + h] = es_exp(-es_exp(a_log[h]) * softplus_bf(ax));
    beta[(size_t)t * 16 + h] = sigmoid_bf(bf2f(b_proj[(size_t)t * 16 + h]));
  }
#pragma unroll
  for (int r = 0; r < kPrepRows; ++r) {
    if (r >= nr) break;
    const size_t o = ((size_t)(t0 + r) * 16 + h) * 128;
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      const float inv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(inv_all), 2 * r + part));
      const float scale = part == 0 ? 0.0078125f : rbf(0.08838834764831845f);
      uint16_t* dst = part == 0 ? q : k;
      dst[o + lane] = (uint16_t)f2bf(rbf(out[part][0][r] * inv) * scale);
      dst[o + 64 + lane] = (uint16_t)f2bf(rbf(out[part][1][r] * inv) * scale);
    }
    v[o + lane] = (uint16_t)f2bf(out[2][0][r]);
    v[o + 64 + lane] = (uint16_t)f2bf(out[2][1][r]);
  }
}

// History after a chunk (gdn_history, gdn.metal:56-73, as the decode ring):
// the raw rows of the chunk's last min(m, 4) positions go to slot pos & 3.
__global__ __launch_bounds__(256) void k_ring_update(const uint16_t* raw, int pos0, int m, uint16_t* ring) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int r = i / kConv, c = i % kConv;
  const int t = m - 4 + r;
  if (r >= 4 || t < 0) return;
  ring[(size_t)((pos0 + t) & 3) * kConv + c] = raw[(size_t)t * kConv + c];
}

// The reference's GDN interface kernels over a history [3, 6144] (oldest row
// first, GDN_INTERFACE.md:12-18), with the arithmetic of the kernels above.
// gdn_conv (gdn.metal:31-51): conv [T,6144] = SiLU(bf16(4-tap conv)), taps
// before the first row from the history.
__global__ __launch_bounds__(256) void k_gdn_conv_hist(const uint16_t* raw, const uint16_t* history,
                                                       const uint16_t* conv_w, int rows, uint16_t* conv) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * kConv) return;
  const int t = i / kConv, c = i % kConv;
  uint32_t x[4];
#pragma unroll
  for (int tap = 0; tap < 4; ++tap) {
    const int r = t + tap - 3;
    x[tap] = r < 0 ? history[(size_t)(r + 3) * kConv + c] : raw[(size_t)r * kConv + c];
  }
  conv[i] = (uint16_t)f2bf(conv4_silu(x, *reinterpret_cast<const uint2*>(conv_w + (size_t)c * 4)));
}

// gdn_history (gdn.metal:53-73): the history takes the last three raw rows,
// keeping older history rows when rows < 3.
__global__ __launch_bounds__(256) void k_gdn_history(const uint16_t* raw, int rows, uint16_t* history) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= kConv) return;
  const uint16_t h0 = history[c], h1 = history[kConv + c], h2 = history[2 * kConv + c];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int r = rows + j - 3;  // row j of the new history; r < 0 keeps history row r + 3
    const uint16_t keep = r == -3 ? h0 : r == -2 ? h1 : h2;
    history[(size_t)j * kConv + c] = r < 0 ? keep : raw[(size_t)r * kConv + c];
  }
}

// gdn_prepare (gdn.metal:75-114): one wave per (row, head) normalises the
// head's q and k in place in conv (lane i: channels i and 64 + i, sum of
// squares tree64 + tree64, as k_gdn_prep_rows) and lane 0 forms g (fp32) and
// beta (bf16).
__global__ __launch_bounds__(256) void k_gdn_prepare_hist(uint16_t* conv, const uint16_t* a_proj,
                                                          const uint16_t* b_proj, const float* a_log,
                                                          const uint16_t* dt_bias, int rows, float* g,
                                                          uint16_t* beta) {
  const int lane = threadIdx.x & 63;
  const int wid = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid >= rows * 16) return;
  const int t = wid >> 4, h = wid & 15;
#pragma unroll
  for (int part = 0; part < 2; ++part) {
    uint16_t* p = conv + (size_t)t * kConv + part * 2048 + h * 128;
    const float x0 = bf2f(p[lane]), x1 = bf2f(p[64 + lane]);
    const float tot = tree64(x0 * x0) + tree64(x1 * x1);
    const float inv = 1.0f / sqrtf(tot / 128.0f + 1.0e-6f / 128.0f);
    const float scale = part == 0 ? 0.0078125f : rbf(0.08838834764831845f);
    p[lane] = (uint16_t)f2bf(rbf(x0 * inv) * scale);
    p[64 + lane] = (uint16_t)f2bf(rbf(x1 * inv) * scale);
  }
  if (lane == 0) {
    const float ax = rbf(bf2f(a_proj[wid]) + bf2f(dt_bias[h]));
    g[wid] = es_exp(-es_exp(a_log[h]) * softplus_bf(ax));
    beta[wid] = (uint16_t)f2bf(sigmoid_bf(bf2f(b_proj[wid])));
  }
}

// GDN recurrence over the rows of a chunk (gdn_recur with rows > 1,
// gdn.metal:176-228), the decode kernel's arithmetic and order per token:
// block = (16 value rows, head), four walking waves with thread = (row, 8
// keys) and the state in registers for the whole chunk, and four staging waves
// that bring the tokens to LDS as fp32 in tiles of 16, three tiles deep, one
// barrier per tile.
//
// The tokens are a serial chain, so the bound is the walking wave's own
// instruction stream: per token 8 decays, 8 memory and 8 readout fmas, 8
// updates, the 4 steps of the memory sum, and 4 LDS reads of k and q. A DPP
// step that reads a register written by the instruction before it costs two
// idle issue slots, so the 8 readout fmas of token t - 1 fill those of token
// t's memory sum (recur_sum_and_readout). The readout needs its own sum
// across the 16 lanes only once it is stored: 16 tokens' partial sums are
// reduced together by a transposing tree (33 instructions for 16 tokens
// instead of 64 plus the selects), which leaves token t's total in one lane.
// For that tree lane l holds the 8 keys of group recur_group(l), so that the
// first two of its levels join lanes 8 and 4 apart, where DPP's bank mask
// selects the token for free; every sum still joins the same key groups in the
// same order ((0+1)+(2+3))+..., so the bits are the decode kernel's.
// 4096 tokens: 377 us in a graph's replay, 219 cycles a token (566 us with the
// readout after the update and its own sum per token, and the walking waves
// staging the tiles; under the profiler 388 us).
// A copy without the LDS reads takes 340 us: the arithmetic's issue is what is
// left.
constexpr int kRecurTile = 16;
// lane of the 16 that hold a row -> key group (8 keys) it holds
__device__ __forceinline__ int recur_group(int l) {
  const int hi = (l >> 2) & 1, x = hi ? 3 - (l & 3) : l & 3;
  return 4 * (((x & 1) << 1) | (x >> 1)) + 2 * hi + (l >> 3);
}
// key group -> lane (the inverse)
__device__ __forceinline__ int recur_lane(int grp) {
  const int b = grp >> 2, x = ((b & 1) << 1) | (b >> 1);
  return ((grp & 2) ? 7 - x : x) + 8 * (grp & 1);
}
// q, k, v rows are `ld` elements apart (2048 for [m,16,128] arrays, 6144 for
// the reference's normalised conv buffer [T,6144]); beta is fp32 or, when
// beta_bf is set, the reference's bf16 [T,16].
struct RecurIn {
  const uint16_t *q, *k, *v;
  int ld;
  const float* g;
  const float* beta;
  const uint16_t* beta_bf;
};
// LDS tile rows of q and k: 132 floats apart (the tokens a store instruction
// covers fall in different banks); the keys of lane l's group sit at 4l (first
// four) and 64 + 4l (last four), so each 16-byte read of a row's 16 lanes
// covers 256 contiguous bytes. v is kept by row (20 floats apart) and the
// gates by token, so one 16-byte read fetches four tokens' values.
constexpr int kRecurRow = 132, kRecurVRow = 20, kRecurRing = 3;
struct RecurTile {
  float q[kRecurTile][kRecurRow], k[kRecurTile][kRecurRow];
  float v[16][kRecurVRow];
  float g[kRecurTile], beta[kRecurTile];
};
// A staging thread's part of a tile: key group t & 15 of q and k of token
// t >> 4; threads 0..63 four v of token t >> 2; threads 64..95 one gate. Its
// pointers step a tile at a time; the tokens of a last, partial tile that do
// not exist repeat the chunk's last token.
struct RecurStage {
  const uint16_t *q, *k, *v;
  size_t gate;  // index into g or beta
  u32x4 qr, kr;
  uint2 vr;
  float gr;
};
__device__ __forceinline__ void recur_load(const RecurIn& in, int t, RecurStage& R) {
  R.qr = *reinterpret_cast<const u32x4*>(R.q);
  R.kr = *reinterpret_cast<const u32x4*>(R.k);
  if (t < 64)
    R.vr = *reinterpret_cast<const uint2*>(R.v);
  else if (t < 96)
    R.gr = t < 80 ? in.g[R.gate] : in.beta_bf ? bf2f(in.beta_bf[R.gate]) : in.beta[R.gate];
}
// moves R from tile i to tile i + 1 of m tokens
__device__ __forceinline__ void recur_next(const RecurIn& in, int i, int m, int t, RecurStage& R) {
  const int first = (i + 1) * kRecurTile, last = m - 1;
  int dq = kRecurTile, dv = kRecurTile, dg = kRecurTile;
  if (first + kRecurTile > m) {  // steps that end at the last token
    dq = min(first + (t >> 4), last) - (i * kRecurTile + (t >> 4));
    dv = min(first + ((t >> 2) & 15), last) - (i * kRecurTile + ((t >> 2) & 15));
    dg = min(first + (t & 15), last) - (i * kRecurTile + (t & 15));
  }
  R.q += (ptrdiff_t)dq * in.ld;
  R.k += (ptrdiff_t)dq * in.ld;
  R.v += (ptrdiff_t)dv * in.ld;
  R.gate += (ptrdiff_t)dg * 16;
}
__device__ __forceinline__ void recur_store(const RecurStage& R, int t, RecurTile& T) {
  const int l = recur_lane(t & 15);
  float *qd = &T.q[t >> 4][4 * l], *kd = &T.k[t >> 4][4 * l];
  *reinterpret_cast<float4*>(qd) = make_float4(bf_lo(R.qr[0]), bf_hi(R.qr[0]), bf_lo(R.qr[1]), bf_hi(R.qr[1]));
  *reinterpret_cast<float4*>(qd + 64) = make_float4(bf_lo(R.qr[2]), bf_hi(R.qr[2]), bf_lo(R.qr[3]), bf_hi(R.qr[3]));
  *reinterpret_cast<float4*>(kd) = make_float4(bf_lo(R.kr[0]), bf_hi(R.kr[0]), bf_lo(R.kr[1]), bf_hi(R.kr[1]));
  *reinterpret_cast<float4*>(kd + 64) = make_float4(bf_lo(R.kr[2]), bf_hi(R.kr[2]), bf_lo(R.kr[3]), bf_hi(R.kr[3]));
  if (t < 64) {
    const int tt = t >> 2, rr = (t & 3) * 4;
    T.v[rr][tt] = bf_lo(R.vr.x);
    T.v[rr + 1][tt] = bf_hi(R.vr.x);
    T.v[rr + 2][tt] = bf_lo(R.vr.y);
    T.v[rr + 3][tt] = bf_hi(R.vr.y);
  } else if (t < 96) {
    (t < 80 ? T.g : T.beta)[t & 15] = R.gr;
  }
}
// Sum of mem over the 16 lanes of a row, in all of them (levels: lanes 8
// apart, the two quads of a half, lanes 2 and 1 apart), with the readout chain
// o = fma(S[i], q[i], o) from 0 in the slots between its steps: two
// instructions separate the write of a register from the DPP step that reads
// it, as the hardware requires.
__device__ __forceinline__ float recur_sum_and_readout(float& mem, const float (&S)[8], const float (&q)[8]) {
  float o;
  asm("v_fma_f32 %1, %2, %10, 0\n\t"
      "v_fmac_f32 %1, %3, %11\n\t"
      "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32 %1, %4, %12\n\t"
      "v_fmac_f32 %1, %5, %13\n\t"
      "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32 %1, %6, %14\n\t"
      "v_fmac_f32 %1, %7, %15\n\t"
      "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32 %1, %8, %16\n\t"
      "v_fmac_f32 %1, %9, %17\n\t"
      "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "+v"(mem), "=&v"(o)
      : "v"(S[0]), "v"(S[1]), "v"(S[2]), "v"(S[3]), "v"(S[4]), "v"(S[5]), "v"(S[6]), "v"(S[7]), "v"(q[0]),
        "v"(q[1]), "v"(q[2]), "v"(q[3]), "v"(q[4]), "v"(q[5]), "v"(q[6]), "v"(q[7]));
  return o;
}
// The updates S[i] = fma(k[i], delta, D[i]) (S holds D) with the same sum of the
// readout o in the slots between them.
__device__ __forceinline__ void recur_update_and_sum(float (&S)[8], const float (&k)[8], float delta, float& o) {
  asm("v_fmac_f32 %0, %9, %17\n\t"
      "v_fmac_f32 %1, %10, %17\n\t"
      "v_add_f32_dpp %8, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32 %2, %11, %17\n\t"
      "v_fmac_f32 %3, %12, %17\n\t"
      "v_add_f32_dpp %8, %8, %8 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32 %4, %13, %17\n\t"
      "v_fmac_f32 %5, %14, %17\n\t"
      "v_add_f32_dpp %8, %8, %8 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32 %6, %15, %17\n\t"
      "v_fmac_f32 %7, %16, %17\n\t"
      "v_add_f32_dpp %8, %8, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "+v"(S[0]), "+v"(S[1]), "+v"(S[2]), "+v"(S[3]), "+v"(S[4]), "+v"(S[5]), "+v"(S[6]), "+v"(S[7]), "+v"(o)
      : "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]), "v"(k[4]), "v"(k[5]), "v"(k[6]), "v"(k[7]), "v"(delta));
}
// The same sum alone.
__device__ __forceinline__ float recur_sum(float v) {
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "+v"(v));
  return v;
}
// The same sums of 16 tokens' values p: lane l of the row gets the total of
// token recur_token(l). A level halves the values: the lanes on one side keep
// the even token of a pair, those on the other side the odd one.
__device__ __forceinline__ int recur_token(int l) {
  return (l >> 3) | ((l >> 1) & 2) | ((l << 1) & 4) | ((l & 1) << 3);
}
__device__ __forceinline__ float recur_sum16(const float (&p)[16], int l) {
  float a[8], b[4], c[2];
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %1, %10, %10 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %2, %12, %12 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %3, %14, %14 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %4, %16, %16 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %5, %18, %18 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %6, %20, %20 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %7, %22, %22 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
      "v_add_f32_dpp %0, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %1, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %2, %13, %13 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %3, %15, %15 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %4, %17, %17 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %5, %19, %19 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %6, %21, %21 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
      "v_add_f32_dpp %7, %23, %23 row_ror:8 row_mask:0xf bank_mask:0xc"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(a[4]), "=&v"(a[5]), "=&v"(a[6]), "=&v"(a[7])
      : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]), "v"(p[8]),
        "v"(p[9]), "v"(p[10]), "v"(p[11]), "v"(p[12]), "v"(p[13]), "v"(p[14]), "v"(p[15]));
  asm("s_nop 1\n\t"
      "v_add_f32_dpp %0, %4, %4 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %1, %6, %6 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %2, %8, %8 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %3, %10, %10 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %0, %5, %5 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %1, %7, %7 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %2, %9, %9 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %3, %11, %11 row_half_mirror row_mask:0xf bank_mask:0xa"
      : "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]));
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float keep = (l & 2) ? b[2 * i + 1] : b[2 * i], give = (l & 2) ? b[2 * i] : b[2 * i + 1];
    c[i] = keep + dpp_xor2(give);
  }
  const float keep = (l & 1) ? c[1] : c[0], give = (l & 1) ? c[0] : c[1];
  return keep + dpp_xor1(give);
}
__device__ __forceinline__ void recur_read8(const float* row, int l, float (&x)[8]) {
  const float4 lo = *reinterpret_cast<const float4*>(row + 4 * l), hi = *reinterpret_cast<const float4*>(row + 64 + 4 * l);
  x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w;
  x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
}
__device__ __forceinline__ void recur_read4(const float* p, float (&x)[4]) {
  const float4 r = *reinterpret_cast<const float4*>(p);
  x[0] = r.x; x[1] = r.y; x[2] = r.z; x[3] = r.w;
}
// The walking wave's operands in flight: k of the token at hand and the next,
// q of the token before and the one at hand, four tokens' gates and v twice,
// and the readouts not yet reduced.
struct RecurWalk {
  float S[8], k[2][8], q[2][8], g[2][4], be[2][4], v[2][4], p[16];
};
// Walks the full tile T; `next` is the tile after it (its first operands are
// read here). While token u runs, token u + 1's k and token u's q (which the
// readout uses during token u + 1) are in flight; the fences keep the reads
// ahead of the arithmetic, and one wait per token covers them all (the
// compiler's own placement waits three times a token: 4% slower).
// The tile's own outputs but the last are complete at its end; yprev (when not
// null) gets the 16 of the tile before.
__device__ __forceinline__ void recur_walk_tile(const RecurTile& T, const RecurTile& next, int rl, int l, RecurWalk& W,
                                                uint16_t* yprev) {
#pragma unroll
  for (int u = 0; u < kRecurTile; ++u) {
    const int c = u & 1, f = (u >> 2) & 1;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads issued a token ago
    recur_read8(u + 1 < kRecurTile ? T.k[u + 1] : next.k[0], l, W.k[c ^ 1]);
    if ((u & 3) == 0) {
      const RecurTile& from = u + 4 < kRecurTile ? T : next;
      const int u4 = (u + 4) % kRecurTile;
      recur_read4(&from.g[u4], W.g[f ^ 1]);
      recur_read4(&from.v[rl][u4], W.v[f ^ 1]);
      recur_read4(&from.beta[u4], W.be[f ^ 1]);
    }
    recur_read8(T.q[u], l, W.q[c]);
    __builtin_amdgcn_sched_barrier(0);
    float D[8], mem = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      D[i] = W.S[i] * W.g[f][u & 3];
      mem = fmaf(D[i], W.k[c][i], mem);
    }
    W.p[(u + 15) & 15] = recur_sum_and_readout(mem, W.S, W.q[c ^ 1]);
    const float delta = (W.v[f][u & 3] - mem) * W.be[f][u & 3];
#pragma unroll
    for (int i = 0; i < 8; ++i) W.S[i] = fmaf(W.k[c][i], delta, D[i]);
    if (u == 0 && yprev) yprev[(size_t)recur_token(l) * 2048] = (uint16_t)f2bf(recur_sum16(W.p, l));
  }
}
__global__ __launch_bounds__(512, 1) void k_gdn_recur_rows(RecurIn in, int m, float* state, uint16_t* y) {
  __shared__ __attribute__((aligned(16))) RecurTile tile[kRecurRing];
  // blockIdx.x = head, blockIdx.y = block of 16 value rows: the dispatcher
  // deals consecutive blocks to the 8 XCDs in turn, so the 8 row blocks of a
  // head land on one XCD and share its L2 copy of the head's q and k
  const int h = blockIdx.x, r0 = blockIdx.y * 16;
  const int nfull = m / kRecurTile, ntile = (m + kRecurTile - 1) / kRecurTile;
  // Tile i is walked between barriers i and i + 1, while the staging waves
  // store tile i + 2 where tile i - 1 was and load tile i + 3; tile i + 1 is
  // complete, so its first operands are read ahead.
  if (threadIdx.x >= 256) {  // staging waves
    const int t = threadIdx.x - 256;
    RecurStage R;
    const size_t row = (size_t)min(t >> 4, m - 1) * in.ld + h * 128;
    R.q = in.q + row + (t & 15) * 8;
    R.k = in.k + row + (t & 15) * 8;
    R.v = in.v + (size_t)min((t >> 2) & 15, m - 1) * in.ld + h * 128 + r0 + (t & 3) * 4;
    R.gate = (size_t)min(t & 15, m - 1) * 16 + h;
    recur_load(in, t, R);
    int slot = 0;
    for (int i = 0; i < ntile; ++i) {  // tile i
      recur_store(R, t, tile[slot]);
      slot = slot == kRecurRing - 1 ? 0 : slot + 1;
      if (i + 1 < ntile) {
        recur_next(in, i, m, t, R);
        recur_load(in, t, R);
      }
      if (i > 0) __syncthreads();  // barrier i - 1
    }
    __syncthreads();  // barrier ntile - 1
    __syncthreads();  // barrier ntile
    return;
  }
  const int t = threadIdx.x, rl = t >> 4, row = r0 + rl, l = t & 15;
  float* sp = state + ((size_t)(h * 128 + row)) * 128 + 8 * recur_group(l);
  RecurWalk W;
  recur_read4(sp, *reinterpret_cast<float(*)[4]>(&W.S[0]));
  recur_read4(sp + 4, *reinterpret_cast<float(*)[4]>(&W.S[4]));
#pragma unroll
  for (int i = 0; i < 8; ++i) W.q[1][i] = 0.0f;
  uint16_t* yrow = y + h * 128 + row;
  __syncthreads();  // barrier 0
  int cur = 0;
  if (nfull > 0) {
    recur_read8(tile[0].k[0], l, W.k[0]);
    recur_read4(&tile[0].g[0], W.g[0]);
    recur_read4(&tile[0].v[rl][0], W.v[0]);
    recur_read4(&tile[0].beta[0], W.be[0]);
    // The loop starts 44 bytes past a multiple of 256: where it falls in the
    // instruction fetch counts 1% (4096 tokens, in turn: 377 us here, 380.5
    // where it fell by itself).
    asm volatile(".p2align 8\n\t.rept 9\n\ts_nop 0\n\t.endr");
    for (int i = 0; i < nfull; ++i) {
      const int nxt = cur == kRecurRing - 1 ? 0 : cur + 1;
      recur_walk_tile(tile[cur], tile[nxt], rl, l, W, i > 0 ? yrow + (size_t)(i - 1) * kRecurTile * 2048 : nullptr);
      cur = nxt;
      __syncthreads();  // barrier i + 1
    }
    float o = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) o = fmaf(W.S[i], W.q[1][i], o);
    W.p[15] = o;
    yrow[(size_t)((nfull - 1) * kRecurTile + recur_token(l)) * 2048] = (uint16_t)f2bf(recur_sum16(W.p, l));
  }
  // The last m % 16 tokens, with operands in flight and readouts a token late as
  // above (15 and 31 tokens: 5.2 and 7.1 us; with both sums alone after their
  // products and each token's operands read when it starts, 5.6 and 7.7).
  if (nfull < ntile) {
    const RecurTile& T = tile[cur];
    const int rest = m - nfull * kRecurTile;  // < 16: the token after the last has a place in the tile
    uint16_t* yt = yrow + (size_t)nfull * kRecurTile * 2048;
    float g[2] = {T.g[0], 0.0f}, v[2] = {T.v[rl][0], 0.0f}, be[2] = {T.beta[0], 0.0f};
    recur_read8(T.k[0], l, W.k[0]);
    auto token = [&](int u, auto cc) {
      constexpr int c = decltype(cc)::value;
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads issued a token ago
      recur_read8(T.k[u + 1], l, W.k[c ^ 1]);
      recur_read8(T.q[u], l, W.q[c]);
      g[c ^ 1] = T.g[u + 1];
      v[c ^ 1] = T.v[rl][u + 1];
      be[c ^ 1] = T.beta[u + 1];
      __builtin_amdgcn_sched_barrier(0);
      float D[8], mem = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        D[i] = W.S[i] * g[c];
        mem = fmaf(D[i], W.k[c][i], mem);
      }
      float o = recur_sum_and_readout(mem, W.S, W.q[c ^ 1]);
      const float delta = (v[c] - mem) * be[c];
#pragma unroll
      for (int i = 0; i < 8; ++i) W.S[i] = D[i];
      recur_update_and_sum(W.S, W.k[c], delta, o);
      if (u > 0 && l == 0) yt[(size_t)(u - 1) * 2048] = (uint16_t)f2bf(o);
      if (u == rest - 1) {
        o = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) o = fmaf(W.S[i], W.q[c][i], o);
        o = recur_sum(o);
        if (l == 0) yt[(size_t)u * 2048] = (uint16_t)f2bf(o);
      }
    };
    for (int u = 0; u < rest; u += 2) {
      token(u, std::integral_constant<int, 0>{});
      if (u + 1 < rest) token(u + 1, std::integral_constant<int, 1>{});
    }
    __syncthreads();  // barrier ntile
  }
  reinterpret_cast<float4*>(sp)[0] = make_float4(W.S[0], W.S[1], W.S[2], W.S[3]);
  reinterpret_cast<float4*>(sp)[1] = make_float4(W.S[4], W.S[5], W.S[6], W.S[7]);
}

// GDN gated norm rows (gdn_norm_gate, gdn.metal:230-255, the decode kernels'
// arithmetic): 16 lanes per (row, head), 8 channels per lane: sum of squares
// as an fma chain per lane then tree16; out = bf16(SiLU_fp32(z) *
// bf16(bf16(y*inv)*w)). One block per row (16 heads).
__global__ __launch_bounds__(256) void k_gdn_norm_gate_rows(const uint16_t* y, const uint16_t* z,
                                                            const uint16_t* norm_w, int m, uint16_t* out) {
  const int t = blockIdx.x, h = threadIdx.x >> 4, li = threadIdx.x & 15;
  if (t >= m) return;
  const size_t o = (size_t)t * 2048 + h * 128 + li * 8;
  const uint4 yr = *reinterpret_cast<const uint4*>(y + o);
  const uint4 zr = *reinterpret_cast<const uint4*>(z + o);
  const uint4 wr = *reinterpret_cast<const uint4*>(norm_w + li * 8);
  const uint32_t yw[4] = {yr.x, yr.y, yr.z, yr.w}, zw[4] = {zr.x, zr.y, zr.z, zr.w}, ww[4] = {wr.x, wr.y, wr.z, wr.w};
  float yv[8], zv[8], wv[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    yv[2 * i] = bf_lo(yw[i]); yv[2 * i + 1] = bf_hi(yw[i]);
    zv[2 * i] = bf_lo(zw[i]); zv[2 * i + 1] = bf_hi(zw[i]);
    wv[2 * i] = bf_lo(ww[i]); wv[2 * i + 1] = bf_hi(ww[i]);
  }
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(yv[i], yv[i], ss);
  ss = tree16(ss);
  const float ginv = 1.0f / sqrtf(ss / 128.0f + 1e-6f);
  uint32_t res[4];
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float r2[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float norm = rbf(rbf(yv[i + u] * ginv) * wv[i + u]);
      const float gz = zv[i + u];
      const float sy = 1.0f / (1.0f + es_exp(fabsf(gz)));
      const float sig = gz < 0.0f ? sy : 1.0f - sy;
      r2[u] = rbf((gz * sig) * norm);
    }
    res[i / 2] = pack_bf2(r2[0], r2[1]);
  }
  *reinterpret_cast<uint4*>(out + o) = make_uint4(res[0], res[1], res[2], res[3]);
}

// Attention prepare rows (attn_prepare_q / attn_prepare_kv,
// attention.metal:72-131, with the decode kernel's arithmetic): one wave per
// (row, q head) for q, per (row, kv head) for k (RMSNorm, RoPE at position
// pos0 + row) and v; k and v rows go to the cache. Block = one row, 12 waves.
__global__ __launch_bounds__(768) void k_attn_prep_rows(const uint16_t* qg, const uint16_t* kp,
                                                        const uint16_t* vp, const uint16_t* q_gain,
                                                        const uint16_t* k_gain, const float* inv_freq,
                                                        int pos0, int m, uint16_t* qr, uint16_t* kcache,
                                                        uint16_t* vcache, int capacity) {
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (t >= m) return;
  const int pos = pos0 + t;
  if (wave >= 10) {  // v rows of the two kv heads
    const int kvh = wave - 10;
    const uint2 xv = *reinterpret_cast<const uint2*>(vp + (size_t)t * 512 + kvh * 256 + lane * 4);
    *reinterpret_cast<uint2*>(vcache + ((size_t)kvh * capacity + pos) * 256 + lane * 4) = xv;
    return;
  }
  uint2 xv, gv;
  if (wave < 8) {
    xv = *reinterpret_cast<const uint2*>(qg + (size_t)t * 4096 + wave * 512 + lane * 4);
    gv = *reinterpret_cast<const uint2*>(q_gain + lane * 4);
  } else {
    xv = *reinterpret_cast<const uint2*>(kp + (size_t)t * 512 + (wave - 8) * 256 + lane * 4);
    gv = *reinterpret_cast<const uint2*>(k_gain + lane * 4);
  }
  // rope_at with one sine and cosine a lane (frequency lane & 31), fetched by
  // the 16 lanes that hold the rotated dims: a lane would form its four dims'
  // own, one after another, with 48 lanes idle. 4096 rows: 21.4 -> 15.5 us.
  float sn, cs;
  es_sincos((float)pos * inv_freq[lane & 31], &sn, &cs);
  float o4[4], r[4];
  head_norm4(xv, gv, o4);
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int f = ((lane * 4) & 31) + x;
    const float s1 = __shfl(sn, f), c1 = __shfl(cs, f), p1 = dpp_row_ror8(o4[x]);
    r[x] = lane < 8 ? fmaf(o4[x], c1, -(p1 * s1)) : lane < 16 ? fmaf(p1, s1, o4[x] * c1) : o4[x];
  }
  const uint2 packed = make_uint2(pack_bf2(r[0], r[1]), pack_bf2(r[2], r[3]));
  if (wave < 8)
    *reinterpret_cast<uint2*>(qr + ((size_t)t * 8 + wave) * 256 + lane * 4) = packed;
  else
    *reinterpret_cast<uint2*>(kcache + ((size_t)(wave - 8) * capacity + pos) * 256 + lane * 4) = packed;
}

// Output gate rows (attn_gate, attention.metal:133-151): gated =
// bf16(o * sigmoid_bf(gate)) with o the bf16 attention output and gate the
// second half of each head's q_proj row.
// V elements a thread: 8 where gate_eight says so and every pointer takes 16-byte
// accesses (4096 rows 20.4 -> 11.2 us, 4.5 TB/s over 50 MB), else 1.
template <int V>
__global__ __launch_bounds__(256) void k_attn_gate_rows(const uint16_t* o, const uint16_t* qg, int m,
                                                        uint16_t* gated) {
  const int i = (blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= m * 2048) return;
  const int t = i >> 11, hd = i & 2047, h = hd >> 8, d = hd & 255;
  const uint16_t* gp = qg + (size_t)t * 4096 + h * 512 + 256 + d;
  if constexpr (V == 8) {
    const u32x4 ov = *reinterpret_cast<const u32x4*>(o + i), gv = *reinterpret_cast<const u32x4*>(gp);
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      r[e] = pack2(bf_lo(ov[e]) * sigmoid_bf(bf_lo(gv[e])), bf_hi(ov[e]) * sigmoid_bf(bf_hi(gv[e])));
    *reinterpret_cast<u32x4*>(gated + i) = r;
  } else {
    gated[i] = (uint16_t)f2bf(bf2f(o[i]) * sigmoid_bf(bf2f(*gp)));
  }
}

// Causal GQA attention of m consecutive queries (positions pos0 .. pos0+m-1)
// over the cache (attn_prefill, attention_prefill.metal:2256; model.rs:337-343):
// o = bf16(softmax(q.K^T / 16) . V), fp32 softmax, MFMA products.
// Block = (32 queries, KV head), 8 waves, two per SIMD: wave w serves query
// head 4*kvh + (w & 3) for all 32 queries and keys 16(w >> 2) .. +15 of every
// block of 32 keys, with a softmax state of its own; the two halves are
// combined at the end. Every K and V fragment a wave reads from LDS so feeds
// two products: with 16 queries and all 32 keys to a wave the LDS reads (256 KB
// a key block, 2048 cycles at 128 bytes a cycle) took twice the products' 1024.
// 4096 queries over 32768 keys: 1141 -> 1020 us in a graph's replay, 1.0
// PFLOP/s (1211 us after under the profiler, whose runs clock lower).
// S^T = K . Q^T on 16x16x32 MFMAs (16 keys x two groups of 16 queries, K from
// LDS, Q fragments in registers); a row swap per score leaves lane l with query
// l % 32 and keys 8(l / 32) .. +7, so the online-softmax max and sum combine
// two lanes and the exp'ed scores, rounded to bf16, are directly the B operand
// of O^T += V^T . P^T on 32x32x16 MFMAs. Exponentials are base 2 on scores
// scaled by log2(e)/16.
//
// K and V blocks reach LDS by DMA (global_load_lds, 16 bytes a lane, no
// registers), kFaStages blocks deep: block kb + kFaStages - 1 is issued while
// block kb is computed. One DMA instruction moves one 512-byte row (32
// lanes); K rows sit 528 bytes apart and V rows 576 bytes apart, strides at
// which the K reads (16 rows x 4 chunks) and the transposing V reads
// (ds_read_b64_tr_b16: 4 rows x 64 bytes a half-wave) spread evenly over the
// banks. The transposing read gives lane i of each 16-lane group element i of
// the 4 rows x 16 columns its lanes address: lane l gets V[4 keys][d = 32t +
// l%32]. It is issued as inline assembly with its own lgkmcnt wait, which keeps
// the compiler from waiting for every DMA in flight before it.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kFaQ = 32, kFaStages = 4, kFaKs = 264, kFaVs = 288;
constexpr int kFaStageHalves = 32 * kFaKs + 32 * kFaVs;
constexpr int kFaMerge = 64 * 66;  // floats a wave leaves for the other: 64 sums, the reference and the sum a lane
constexpr int kFaQRow = 136;  // bf16 elements between 128-element Q rows in LDS: spread over the banks as the K rows
typedef u32x4 __attribute__((aligned(8))) u32x4_a8;
static_assert(kFaStageHalves >= 8 * 16 * kFaQRow, "the waves' Q rows fit a stage");
// Eight transposing reads from one base: keys 0..3 and 4..7 of the lane's eight
// for four 32-dim tiles at OFF + 64 t. Every read completes before the
// statement ends.
constexpr int kFaHi = 2 * 4 * kFaVs;  // bytes from a key row to the fourth after it
template <int OFF>
__device__ __forceinline__ void lds_read_tr16_x8(uint32_t a, u32x4 (&v)[4]) {
  uint64_t x0, x1, x2, x3, y0, y1, y2, y3;
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%9\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:%10\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:%9+64\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:%10+64\n\t"
      "ds_read_b64_tr_b16 %2, %8 offset:%9+128\n\t"
      "ds_read_b64_tr_b16 %6, %8 offset:%10+128\n\t"
      "ds_read_b64_tr_b16 %3, %8 offset:%9+192\n\t"
      "ds_read_b64_tr_b16 %7, %8 offset:%10+192\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x0), "=&v"(x1), "=&v"(x2), "=&v"(x3), "=&v"(y0), "=&v"(y1), "=&v"(y2), "=&v"(y3)
      : "v"(a), "n"(OFF), "n"(kFaHi + OFF)
      : "memory");
  const uint64_t x[4] = {x0, x1, x2, x3}, y[4] = {y0, y1, y2, y3};
#pragma unroll
  for (int t = 0; t < 4; ++t)
    v[t] = u32x4{(uint32_t)x[t], (uint32_t)(x[t] >> 32), (uint32_t)y[t], (uint32_t)(y[t] >> 32)};
}
// max of two scores by v_max_f32 alone: scores are never NaN, so the operand
// canonicalisation that fmaxf adds changes nothing and is left out
__device__ __forceinline__ float max_raw(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__global__ __launch_bounds__(512, 1) void k_attn_prefill(const uint16_t* qr, const uint16_t* kcache,
                                                         const uint16_t* vcache, int pos0, int m,
                                                         int capacity, uint16_t* o) {
  __shared__ __attribute__((aligned(16))) uint16_t kv[kFaStages][kFaStageHalves];
  __shared__ uint32_t merged[8];
  static_assert(sizeof(kv) >= 8 * kFaMerge * sizeof(float), "the merge fits the staging memory");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform: scalar DMA addressing
  if (t < 8) merged[t] = 0;
  // 1-D grid dealt to the 8 XCDs in turn (block b on XCD b % 8): XCDs
  // 0, 2, 4, 6 take KV head 0 and 1, 3, 5, 7 head 1, so the query tiles that
  // stream one head's K and V share an XCD's L2
  const int b = blockIdx.x, xcd = b & 7;
  const int tile = 4 * (b >> 3) + (xcd >> 1);
  if (tile * kFaQ >= m) return;
  const int t0 = tile * kFaQ, kvh = xcd & 1, hq = 4 * kvh + (wave & 3), kh = wave >> 2;
  const int qi = lane & 15, g = lane >> 4;
  const int qrow = t0 + (lane & 31);  // the lane's query once the scores are swapped
  const bool qvalid = qrow < m;
  const int qpos = pos0 + (qvalid ? qrow : m - 1);
  const int last_key = pos0 + min(t0 + kFaQ, m) - 1;
  const int nkb = last_key / 32 + 1;
  // Q by whole lines, four rows of 256 bytes an instruction: fetched straight
  // into the fragments' lanes (64 bytes of 16 rows an instruction) the block's
  // 128 loads took 8,500 cycles to issue. A query past m reads the last one; its
  // results are not stored.
  u32x4 qv[2][2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int hd = 0; hd < 2; ++hd)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        qv[u][hd][j] = *reinterpret_cast<const u32x4*>(
            qr + ((size_t)min(t0 + 16 * u + 4 * j + g, m - 1) * 8 + hq) * 256 + 128 * hd + 8 * qi);
  // DMA of one block of 32 keys: wave w moves rows 4w .. 4w+3 of K and V,
  // one row per instruction, lane L < 32 the row's 16-byte chunk L
  // Buffer resources over this KV head's rows of both caches: the row's byte
  // offset is a scalar operand and the lane's 16-byte chunk a fixed vector
  // offset, so a DMA takes no per-lane address arithmetic. Rows are clamped
  // to the capacity below, which the launcher keeps at most 2^22 (byte
  // offsets up to 2^31), so the resources set no range of their own.
  const size_t head_off = (size_t)kvh * capacity * 256;
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)(kcache + head_off), 0, -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)(vcache + head_off), 0, -1, 0x00020000);
  const uint32_t lane_off = (uint32_t)lane * 16u;
  auto issue = [&](int kb) {
    uint16_t* stage = kv[kb % kFaStages];
    if (lane < 32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * wave + i;
        const int key = min(kb * 32 + r, capacity - 1);
        const uint32_t row = (uint32_t)key * 512u;  // uniform byte offset
        __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (__attribute__((address_space(3))) void*)(stage + r * kFaKs), 16,
                                             lane_off, row, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (__attribute__((address_space(3))) void*)(stage + 32 * kFaKs + r * kFaVs),
                                             16, lane_off, row, 0, 0);
      }
    }
  };
  for (int kb = 0; kb < min(kFaStages - 1, nkb); ++kb) issue(kb);
  f32x16 ot[8];  // O^T: dims 32t + 8(r/4) + 4(l/32) + r%4 of query l % 32
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) ot[dt][r] = 0.0f;
  // cleared here, while the loads are on their way
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) asm volatile("" : "+v"(ot[dt]));
  __builtin_amdgcn_sched_barrier(0);
  // Q fragments: B operand of k-step s for query group u holds Q[16u + q][32s + 8g .. +7],
  // through the wave's own part of the last stage, which the loop fills only
  // after its first barrier (a group without queries repeats the other)
  bf16x8 qf[2][8];
  {
    uint16_t* const ql = &kv[kFaStages - 1][wave * (16 * kFaQRow)];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int hd = 0; hd < 2; ++hd) {
        if (u == 1 && t0 + 16 >= m) {
#pragma unroll
          for (int s2 = 0; s2 < 4; ++s2) qf[u][4 * hd + s2] = qf[0][4 * hd + s2];
          continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4*>(ql + (4 * j + g) * kFaQRow + 8 * qi) = qv[u][hd][j];
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
          qf[u][4 * hd + s2] = *reinterpret_cast<const bf16x8*>(ql + qi * kFaQRow + 32 * s2 + 8 * g);
      }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int s2 = 0; s2 < 8; ++s2) asm volatile("" : "+v"(qf[u][s2]));
  // The running reference starts below every score but finite: a row may have
  // no key in this wave's half of its blocks (or none before them), and
  // -inf - -inf would be NaN.
  float mrun = -3.0e38f, lrun = 0.0f;
  const float c = 0.0625f * 1.4426950408889634f;  // 1/16 * log2(e)
  const uint32_t kv_base =
      (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) uint16_t*)(&kv[0][0]));
  // V reads (see above): 16-lane group g takes dims 16(g & 1) .. of a tile and
  // keys 8(g / 2) .. of the wave's 16
  const uint32_t v_lane =
      (uint32_t)(2 * (32 * kFaKs + (16 * kh + 8 * (g >> 1) + (qi >> 2)) * kFaVs + 16 * (g & 1) + 4 * (qi & 3)));
  // The loop starts 44 bytes past a multiple of 256: where it falls in the
  // instruction fetch counts up to 1% (4096 queries at 28672, in turn: 1019 us
  // here, 1028 at 16 or 32 bytes).
  asm volatile(".p2align 8\n\t.rept 7\n\ts_nop 0\n\t.endr");
  for (int kb = 0;; ++kb) {
    // blocks issued after kb and still in flight: min(kFaStages - 2, nkb-1-kb),
    // 8 DMA instructions each per wave
    const int ahead = min(kFaStages - 2, nkb - 1 - kb);
    if (ahead >= 2)
      wait_vmcnt<16>();
    else if (ahead == 1)
      wait_vmcnt<8>();
    else
      wait_vmcnt<0>();
    __syncthreads();  // block kb visible; every wave is past block kb-1
    if (kb == nkb) break;  // every wave is past the last block: the staging memory is free
    const uint16_t* ks = kv[kb % kFaStages] + 16 * kh * kFaKs;
    const uint32_t vs_addr = kv_base + (uint32_t)(2 * kFaStageHalves * (kb % kFaStages)) + v_lane;
    // scores S^T[key][q] for the two groups of 16 queries. The K fragments of
    // k-steps s2 .. s2 + 3 are in flight while step s2's two products run
    // (fences keep the order), so each pair of products waits for its own read
    // only.
    f32x4 st[2];
    {
      bf16x8 kf[8];
      auto read_k = [&](int s2) { kf[s2] = *reinterpret_cast<const bf16x8*>(ks + qi * kFaKs + 32 * s2 + 8 * g); };
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2) read_k(s2);
      // block kb + 3 goes to the stage every wave finished before the barrier;
      // its DMA is issued while the first K reads are in flight
      if (kb + kFaStages - 1 < nkb) issue(kb + kFaStages - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) st[u][r] = 0.0f;
#pragma unroll
      for (int s2 = 0; s2 < 8; ++s2) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          st[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s2], qf[u][s2], st[u], 0, 0, 0);
        if (s2 + 4 < 8) read_k(s2 + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // lane l: keys 4g + r of query l % 16 of both groups -> keys 8(l / 32) + e
    // of query l % 32
    float x[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(st[0][r]), __float_as_uint(st[1][r]), false, false);
      x[r] = __uint_as_float(p[0]);
      x[4 + r] = __uint_as_float(p[1]);
    }
    // causal mask (only blocks that reach past the tile's first query),
    // online softmax for the lane's query; the maximum is taken on the raw
    // scores (scaling by c > 0 keeps the order) and the exponent is
    // fma(s, c, -max)
    if (kb * 32 + 31 > pos0 + t0) {
      const int key0 = kb * 32 + 16 * kh + 8 * (lane >> 5);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = key0 + e <= qpos ? x[e] : -INFINITY;
    }
    float mloc = x[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mloc = fmaxf(mloc, x[e]);
    const float2 m32 = rows_xor32(mloc);
    // The exponent's reference value moves only when the block's maximum
    // exceeds it by more than 8 (probabilities stay below 2^8; the output is
    // normalised by a sum taken against the same reference, so the softmax is
    // unchanged). The choice is per row, so a row's result depends on its own
    // scores only.
    const float mblk = max_raw(m32.x, m32.y) * c;
    const float mnew = mblk > mrun + 8.0f ? mblk : mrun;
    const float factor = __builtin_amdgcn_exp2f(mrun - mnew);
    float pv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) pv[e] = __builtin_amdgcn_exp2f(fmaf(x[e], c, -mnew));
    // ((p0 + p1) + p2) + ...: the same sum as from 0, since p0 >= +0
    float psum = pv[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) psum += pv[e];
    const float2 s32 = rows_xor32(psum);
    lrun = lrun * factor + (s32.x + s32.y);
    const float mrun_old = mrun;
    mrun = mnew;
    // factor is exactly 1 where the reference did not move: the rescale is
    // skipped unless some lane's reference moved
    if (__any(mnew > mrun_old)) {
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) ot[dt][r] *= factor;
    }
    // O^T += V^T . P^T: one 16-key step per 32-dim tile
    const u32x4 pb = u32x4{pack2(pv[0], pv[1]), pack2(pv[2], pv[3]), pack2(pv[4], pv[5]), pack2(pv[6], pv[7])};
    const bf16x8 pf = __builtin_bit_cast(bf16x8, pb);
#pragma unroll
    for (int d4 = 0; d4 < 2; ++d4) {
      u32x4 vf[4];
      if (d4 == 0)
        lds_read_tr16_x8<0>(vs_addr, vf);
      else
        lds_read_tr16_x8<256>(vs_addr, vf);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        ot[4 * d4 + i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[i]), pf, ot[4 * d4 + i], 0, 0, 0);
    }
  }
  // The two waves of a head each finish half of the dims, in their first four
  // tiles: a wave leaves the sums of the other four and its softmax state in the
  // staging memory, raises its flag and waits for the other's (both run on this
  // CU and raise before they wait, so the wait ends). Key 0 is in the lower
  // half, so the larger reference is a score's and the sum is not 0; an upper
  // half without keys has weight 0. This and Q are the fixed cost of a tile,
  // which shows where there are few keys (kernel us at position 0 for 8, 32,
  // 128, 400 and 1000 queries: 16 queries and all keys to a wave 7.0, 11.1,
  // 14.5, 23.5, 44.5; halves with Q straight into the fragments and one wave
  // finishing all dims 9.5, 14.3, 17.2, 25.0, 43.4; this 8.4, 10.4, 13.7, 21.5,
  // 39.7; at position 28672 853, 854, 857, 875, 894 against 967 .. 1012).
  if (kh) {
    asm volatile("s_nop 15\n\ts_nop 15");  // past the last products' latency, which the compiler does not see here
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float lo = ot[dt][r], hi = ot[4 + dt][r];
        asm volatile("v_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
        ot[dt][r] = lo;
        ot[4 + dt][r] = hi;
      }
  }
  float* const mine = reinterpret_cast<float*>(&kv[0][0]) + wave * kFaMerge;
  const float* const theirs = reinterpret_cast<const float*>(&kv[0][0]) + (wave ^ 4) * kFaMerge;
  if (qvalid) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<float4*>(mine + ((4 * dt + r) * 64 + lane) * 4) =
            make_float4(ot[4 + dt][4 * r], ot[4 + dt][4 * r + 1], ot[4 + dt][4 * r + 2], ot[4 + dt][4 * r + 3]);
    mine[64 * 64 + lane] = mrun;
    mine[64 * 65 + lane] = lrun;
  }
  __hip_atomic_store(&merged[wave], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  while (__hip_atomic_load(&merged[wave ^ 4], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
    __builtin_amdgcn_s_sleep(1);
  const float mo = theirs[64 * 64 + lane], lo = theirs[64 * 65 + lane];
  const float m0 = kh ? mo : mrun, m1 = kh ? mrun : mo, l0 = kh ? lo : lrun, l1 = kh ? lrun : lo;
  const float mx = fmaxf(m0, m1), f0 = __builtin_amdgcn_exp2f(m0 - mx), f1 = __builtin_amdgcn_exp2f(m1 - mx);
  const float inv = 1.0f / (l0 * f0 + l1 * f1), i0 = f0 * inv, i1 = f1 * inv;
  uint16_t* op = o + ((size_t)qrow * 8 + hq) * 256 + 128 * kh + 8 * (lane >> 5);
  auto finish = [&](auto upper) {
    constexpr bool U = decltype(upper)::value;  // own sums are the upper half's
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      uint32_t w[4];  // dims 16 i + 4 (l / 32) .. + 3, and 8 further
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const float4 u4 = *reinterpret_cast<const float4*>(theirs + ((2 * i + r) * 64 + lane) * 4);
        const float u[4] = {u4.x, u4.y, u4.z, u4.w};
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float own = ot[i >> 1][4 * (2 * (i & 1) + r) + e];
          v[e] = U ? fmaf(u[e], i0, own * i1) : fmaf(own, i0, u[e] * i1);
        }
        w[2 * r] = pack2(v[0], v[1]);
        w[2 * r + 1] = pack2(v[2], v[3]);
      }
      // the halves of the wave exchange, so that a lane holds 8 dims in a row
      const auto c01 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
      const auto c23 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
      if (qvalid) *reinterpret_cast<u32x4_a8*>(op + 16 * i) = u32x4{c01[0], c23[0], c01[1], c23[1]};
    }
  };
  // two bodies, kept apart: merged they select both operands of every product
  if (kh) {
    asm volatile("; upper half");
    finish(std::true_type{});
    asm volatile("; upper half done");
  } else {
    asm volatile("; lower half");
    finish(std::false_type{});
    asm volatile("; lower half done");
  }
}

}  // namespace

template <int MT, bool GATEUP>
static hipError_t launch_gemm_tiles(GemmArgs a, const uint16_t* residual, int nb, hipStream_t s) {
  const int mb = (a.m + 32 * MT - 1) / (32 * MT);
  a.by_xcd = mb >= 8;  // fewer row tiles than XCDs: blocks in column order reach them all
  a.vec = ((uintptr_t)residual & 15) == 0;
  bool lines = a.w[0].k % 256 == 0;
  for (int i = 0; i < a.nseg; ++i) {
    a.vec = a.vec && ((uintptr_t)a.y[i] & 15) == 0 && (a.nstart[i + 1] - a.nstart[i]) % 8 == 0;
    lines = lines && (((uintptr_t)a.w[i].s | (uintptr_t)a.w[i].b) & 3) == 0;
  }
  const dim3 grid = a.by_xcd ? dim3(gemm_grid(nb, mb)) : dim3(nb, mb);
  if (lines)
    hipLaunchKernelGGL((k_q4_gemm<MT, GATEUP, true>), grid, dim3(256), 0, s, a, residual);
  else
    hipLaunchKernelGGL((k_q4_gemm<MT, GATEUP, false>), grid, dim3(256), 0, s, a, residual);
  return hipGetLastError();
}
// The smallest row tile whose blocks fit one to a CU (256): below that the
// chip has CUs to spare and the time is one block's serial walk over K, which
// a taller tile lengthens; past it the tallest tile dequantises least.
template <bool GATEUP>
static hipError_t launch_gemm(const GemmArgs& a, const uint16_t* residual, hipStream_t s) {
  const int n = GATEUP ? a.w[0].n : a.nstart[a.nseg], cols = GATEUP ? 64 : 128;
  const int nb = (n + cols - 1) / cols;
  auto blocks = [&](int rows) { return (long)nb * ((a.m + rows - 1) / rows); };
  if (blocks(32) <= 256) return launch_gemm_tiles<1, GATEUP>(a, residual, nb, s);
  if (blocks(64) <= 256) return launch_gemm_tiles<2, GATEUP>(a, residual, nb, s);
  return launch_gemm_tiles<4, GATEUP>(a, residual, nb, s);
}

hipError_t launch_q4_gemm_stacked(const Q4* w, uint16_t* const* y, int nseg, const uint16_t* x, int m,
                                  hipStream_t s) {
  if (!w || !y || nseg < 1 || nseg > 4 || !x || m < 1) return hipErrorInvalidValue;
  GemmArgs a{};
  int n = 0;
  for (int i = 0; i < nseg; ++i) {
    if (!w[i].w || !w[i].s || !w[i].b || !y[i] || w[i].n < 1 || w[i].k != w[0].k || w[i].k < kGemmBK ||
        w[i].k % kGemmBK != 0)
      return hipErrorInvalidValue;
    a.w[i] = w[i];
    a.y[i] = y[i];
    a.nstart[i] = n;
    n += w[i].n;
  }
  for (int i = nseg; i < 4; ++i) {
    a.w[i] = w[0];
    a.y[i] = y[0];
  }
  a.nstart[nseg] = n;
  for (int i = nseg + 1; i < 5; ++i) a.nstart[i] = n;
  a.nseg = nseg;
  a.x = x;
  a.m = m;
  return launch_gemm<false>(a, nullptr, s);
}

hipError_t launch_q4_gemm(const Q4& w, const uint16_t* x, int m, const uint16_t* residual, uint16_t* y,
                          hipStream_t s) {
  if (!w.w || !w.s || !w.b || w.n < 1 || w.k < kGemmBK || w.k % kGemmBK != 0 || !x || !y || m < 1)
    return hipErrorInvalidValue;
  if (!residual && gemm_wide(w.n, w.k, m)) {
    const dim3 grid((w.n + kWideN - 1) / kWideN, (m + kWideM - 1) / kWideM);
    hipLaunchKernelGGL(k_q4_gemm_wide, grid, dim3(256), 0, s, w, x, m, y);
    return hipGetLastError();
  }
  const GemmArgs a{{w, w, w, w}, {y, y, y, y}, {0, w.n, w.n, w.n, w.n}, 1, x, m};
  return launch_gemm<false>(a, residual, s);
}

hipError_t launch_q4_gemm_swiglu(const Q4& gate, const Q4& up, const uint16_t* x, int m, uint16_t* act,
                                 hipStream_t s) {
  if (!gate.w || !gate.s || !gate.b || !up.w || !up.s || !up.b || gate.n != up.n || gate.k != up.k ||
      gate.n < 1 || gate.k < kGemmBK || gate.k % kGemmBK != 0 || !x || !act || m < 1)
    return hipErrorInvalidValue;
  const GemmArgs a{{gate, up, gate, up}, {act, act, act, act}, {0, gate.n, 2 * gate.n, 2 * gate.n, 2 * gate.n}, 2, x, m};
  return launch_gemm<true>(a, nullptr, s);
}

}  // namespace es

namespace es {

hipError_t launch_embed_rows(const Q4& e, const uint32_t* tokens, int m, uint16_t* h, hipStream_t s) {
  if (!e.w || m < 1 || !tokens || !h || e.k != 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_embed_rows, dim3((m + 7) / 8), dim3(256), 0, s, e, tokens, m, h);
  return hipGetLastError();
}

hipError_t launch_rmsnorm_rows(const uint16_t* x, const uint16_t* gain, int m, uint16_t* out, hipStream_t s) {
  if (!x || !gain || !out || m < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rmsnorm_rows, dim3((m + 7) / 8), dim3(256), 0, s, x, gain, m, out);
  return hipGetLastError();
}

hipError_t launch_swiglu_rows(const uint16_t* gate, const uint16_t* up, int count, uint16_t* act,
                              hipStream_t s) {
  if (!gate || !up || !act || count < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_swiglu_rows, dim3((count + 255) / 256), dim3(256), 0, s, gate, up, count, act);
  return hipGetLastError();
}

hipError_t launch_gdn_prep_rows(const GdnPrepRowsArgs& a, hipStream_t s) {
  if (!a.raw || !a.ring || !a.conv_w || !a.a_proj || !a.b_proj || !a.a_log || !a.dt_bias || a.m < 1 ||
      a.pos0 < 0 || !a.q || !a.k || !a.v || !a.g || !a.beta)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gdn_prep_rows, dim3((a.m + kPrepRows - 1) / kPrepRows, 4), dim3(256), 0, s, a.raw, a.ring,
                     a.conv_w, a.a_proj, a.b_proj, a.a_log, a.dt_bias, a.pos0, a.m, a.q, a.k, a.v, a.g, a.beta);
  if (hipGetLastError() != hipSuccess) return hipErrorLaunchFailure;
  hipLaunchKernelGGL(k_ring_update, dim3((4 * kConv + 255) / 256), dim3(256), 0, s, a.raw, a.pos0, a.m,
                     a.ring);
  return hipGetLastError();
}

hipError_t launch_gdn_recur_rows(const uint16_t* q, const uint16_t* k, const uint16_t* v, const float* g,
                                 const float* beta, int m, float* state, uint16_t* y, hipStream_t s) {
  if (!q || !k || !v || !g || !beta || !state || !y || m < 1) return hipErrorInvalidValue;
  const RecurIn in{q, k, v, 2048, g, beta, nullptr};
  hipLaunchKernelGGL(k_gdn_recur_rows, dim3(kGdnHeads, 8), dim3(512), 0, s, in, m, state, y);
  return hipGetLastError();
}

hipError_t launch_gdn_conv_hist(const uint16_t* raw, const uint16_t* history, const uint16_t* conv_w,
                                int rows, uint16_t* conv, hipStream_t s) {
  if (!raw || !history || !conv_w || !conv || rows < 1 || rows > (1 << 18)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gdn_conv_hist, dim3((rows * kConv + 255) / 256), dim3(256), 0, s, raw, history, conv_w,
                     rows, conv);
  return hipGetLastError();
}

hipError_t launch_gdn_history(const uint16_t* raw, int rows, uint16_t* history, hipStream_t s) {
  if (!raw || !history || rows < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gdn_history, dim3(kConv / 256), dim3(256), 0, s, raw, rows, history);
  return hipGetLastError();
}

hipError_t launch_gdn_prepare_hist(uint16_t* conv, const uint16_t* a_proj, const uint16_t* b_proj,
                                   const float* a_log, const uint16_t* dt_bias, int rows, float* g,
                                   uint16_t* beta, hipStream_t s) {
  if (!conv || !a_proj || !b_proj || !a_log || !dt_bias || !g || !beta || rows < 1 || rows > (1 << 24))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gdn_prepare_hist, dim3((rows * 16 + 3) / 4), dim3(256), 0, s, conv, a_proj, b_proj, a_log,
                     dt_bias, rows, g, beta);
  return hipGetLastError();
}

hipError_t launch_gdn_recur_conv(const uint16_t* conv, const float* g, const uint16_t* beta, int rows,
                                 float* state, uint16_t* y, hipStream_t s) {
  if (!conv || !g || !beta || !state || !y || rows < 1) return hipErrorInvalidValue;
  const RecurIn in{conv, conv + 2048, conv + 4096, kConv, g, nullptr, beta};
  hipLaunchKernelGGL(k_gdn_recur_rows, dim3(kGdnHeads, 8), dim3(512), 0, s, in, rows, state, y);
  return hipGetLastError();
}

hipError_t launch_gdn_norm_gate_rows(const uint16_t* y, const uint16_t* z, const uint16_t* norm_w, int m,
                                     uint16_t* out, hipStream_t s) {
  if (!y || !z || !norm_w || !out || m < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gdn_norm_gate_rows, dim3(m), dim3(256), 0, s, y, z, norm_w, m, out);
  return hipGetLastError();
}

hipError_t launch_attn_prep_rows(const AttnPrepRowsArgs& a, hipStream_t s) {
  if (!a.qg || !a.k || !a.v || !a.q_gain || !a.k_gain || !a.inv_freq || a.m < 1 || a.pos0 < 0 ||
      a.pos0 + a.m > a.capacity || !a.qr || !a.kcache || !a.vcache)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_attn_prep_rows, dim3(a.m), dim3(768), 0, s, a.qg, a.k, a.v, a.q_gain, a.k_gain,
                     a.inv_freq, a.pos0, a.m, a.qr, a.kcache, a.vcache, a.capacity);
  return hipGetLastError();
}

hipError_t launch_attn_prefill(const uint16_t* qr, const uint16_t* kcache, const uint16_t* vcache, int pos0,
                               int m, int capacity, uint16_t* o, hipStream_t s) {
  // capacity <= 2^22 (the engine's limit) keeps every byte offset within a KV
  // head's rows below 2^31
  if (!qr || !kcache || !vcache || !o || m < 1 || pos0 < 0 || pos0 + m > capacity || capacity > (1 << 22))
    return hipErrorInvalidValue;
  const int tiles = (m + kFaQ - 1) / kFaQ;
  hipLaunchKernelGGL(k_attn_prefill, dim3(8 * ((tiles + 3) / 4)), dim3(512), 0, s, qr, kcache, vcache, pos0, m,
                     capacity, o);
  return hipGetLastError();
}

hipError_t launch_attn_gate_rows(const uint16_t* o, const uint16_t* qg, int m, uint16_t* gated,
                                 hipStream_t s) {
  if (!o || !qg || !gated || m < 1 || m > (1 << 20) - 1) return hipErrorInvalidValue;  // m * 2048 < 2^31
  if (gate_eight(m) && (((uintptr_t)o | (uintptr_t)qg | (uintptr_t)gated) & 15) == 0)
    hipLaunchKernelGGL(k_attn_gate_rows<8>, dim3(m), dim3(256), 0, s, o, qg, m, gated);
  else
    hipLaunchKernelGGL(k_attn_gate_rows<1>, dim3((m * 2048 + 255) / 256), dim3(256), 0, s, o, qg, m, gated);
  return hipGetLastError();
}

}  // namespace es
