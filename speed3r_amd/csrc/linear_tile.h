// One tile of Y = X W^T (X [M, K], W [N, K], both with K contiguous; bf16 / fp16, fp32 accumulation) on the gfx950 matrix
// cores: the part that the kernels for linear layers share.  Four waves, one per SIMD, compute BM tokens x BN channels.
//
//   * v_mfma_f32_16x16x32 with W as the A operand: a lane holds four consecutive channels of one token per 16 x 16 tile.  At
//     these sizes the chip runs at its power limit (1.6 to 1.8 GHz), and this instruction moves half the accumulator
//     bytes per flop of the 32x32x16 one: 8192^3 in 0.73 ms against 0.78.
//   * Each wave owns TT x TC of these tiles, at most 128 x 128 values in all 256 accumulator registers: the fewest LDS
//     reads per product.  One wave per SIMD has nobody to hide behind, so nothing it needs is fetched late: the operands of
//     a half step (32 values of K) are read while the half step before it computes (two register sets), and X and W go
//     global -> LDS by direct transfers two steps (of 64 values of K) ahead, into the buffer whose last reads ended half a
//     step before.  One barrier per step.
//   * The transfers are spread over half a step: the CU's path into LDS takes 64 bytes per cycle, and a queue of them
//     stalls the wave that issues the next one together with its products (0.73 against 0.77 ms in a burst).
//   * A tile's first two steps are requested before the tile in front of it ends: between tiles only the epilogue is
//     left without products.
//   * The products accumulate in place, written out: the builtin has a result register of its own, and where all 256 are
//     accumulators the compiler's copies for it spill.
#pragma once
#include "select_common.h"

namespace s3r {
namespace lin {
using namespace sel;

// 16 bytes per lane from base + voff + soff to dst + 16 lane
__device__ __forceinline__ void to_lds16(const void* base, void* dst, uint32_t voff, uint32_t soff) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}
// 16 bytes to base + off unless that lies at or beyond `bytes`; non-temporal, so that what is written does not push the X and W
// rows of the tiles to come out of the L2 (104 100 x 3072 x 1024: 546 -> 520 us; the projection with its epilogue 722 -> 697).  Issued, and
// counted, whether anything is written or not: a tile's stores are counted on by the next one's first wait (sweep).
__device__ __forceinline__ void store16_if(void* base, uint32_t bytes, uint32_t off, const uint4& v) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(&v), rs, off, 0, 2);
}

// Accumulators in the AGPR half of the register file where they fill it (with two waves per SIMD the compiler would split
// the file in halves for 64 of them).
template <typename E, bool AGPR, bool FIRST = false> __device__ __forceinline__ void mma_acc(typename Mma<E>::V8 a, typename Mma<E>::V8 b, f32x4& c) {
  // (FIRST: an operand all the same, so that a tile's first products take the registers of the ones that follow)
  if constexpr (std::is_same<E, bf16_t>::value) {
    if constexpr (AGPR && FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "+a"(c) : "v"(a), "v"(b));
    else if constexpr (AGPR) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "+v"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  } else {
    if constexpr (AGPR && FIRST) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "+a"(c) : "v"(a), "v"(b));
    else if constexpr (AGPR) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "+v"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
}

// LDS row map: rows of 128 bytes (64 values of K), chunk c of row r at chunk position c ^ swizzle(r)
__device__ __forceinline__ constexpr int row_swizzle(int r) { return (r >> 1) & 7; }

// Work of a workgroup: tiles of an mt x nt grid, dealt out so that the workgroups of one XCD (round robin over workgroup
// numbers) work on neighbouring tiles: groups of kGroup rows of tiles, all columns, so that their X and W rows meet in the L2.
struct TileWalk {
  static constexpr int kGroup = 8;
  int mt, nt, first, count, slots, at;
  __device__ __forceinline__ TileWalk(int mt_, int nt_) : mt(mt_), nt(nt_) {
    const int tiles = mt * nt, xcd = blockIdx.x & 7;
    const int per = tiles >> 3, rem = tiles & 7;
    first = xcd * per + (xcd < rem ? xcd : rem);
    count = per + (xcd < rem ? 1 : 0);
    slots = ((int)gridDim.x >> 3) + (xcd < ((int)gridDim.x & 7) ? 1 : 0);
    at = blockIdx.x >> 3;
  }
  __device__ __forceinline__ void locate(int i, int& m, int& n) const {
    const int vid = first + i, per_group = kGroup * nt;
    const int g = vid / per_group, r = vid - g * per_group;
    const int rows = mt - g * kGroup < kGroup ? mt - g * kGroup : kGroup;
    n = r / rows;
    m = g * kGroup + (r - n * rows);
  }
};

template <typename E, int TT, int TC> struct Tile {
  typedef typename Mma<E>::V8 V8;
  static constexpr int BM = 32 * TT, BN = 32 * TC;  // two waves by two
  static constexpr bool kAgpr = TT * TC == 64;
  static constexpr int NL = TT + TC;                // fragments of a half step; transfers of a step, per wave
  static constexpr int NM = TT * TC;                // products of a half step
  // spacing in sixteenths of a product: reads of the first half step; transfers, and reads, of the second
  static constexpr int kRead1 = 12 * NM / NL, kMove2 = 16 * NM / NL, kRead2 = 16 * (NM - 2) / NL;
  static constexpr int kRead2At = NM / NL > 2 ? 2 : 1;

  int wave, lane, g4, c16, wm, wn;
  int fx, fw;                       // where the wave's first fragment of X, W lies in a buffer
  uint32_t xoff[TT], woff[TC];      // the lane's rows of the requested tile
  const E *bx, *bw;                 // its first rows
  struct Frag8 { V8 x[TT], w[TC]; } P, Q;
  f32x4 acc[TC][TT];

  __device__ __forceinline__ Tile() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    g4 = lane >> 4;
    c16 = lane & 15;
    wm = wave & 1;
    wn = wave >> 1;
    const int at = c16 * 128 + ((g4 ^ row_swizzle(c16)) << 4);
    fx = wm * 16 * TT * 128 + at;
    fw = wn * 16 * TC * 128 + at;
  }
  // requests go to these rows from now on; rows from `xrows` / `wrows` on repeat the last one
  __device__ __forceinline__ void aim(const E* x, int64_t ldx, int xrows, const E* w, int64_t ldw, int wrows) {
    bx = x;
    bw = w;
#pragma unroll
    for (int i = 0; i < TT; i++) {
      const int r = (wave * TT + i) * 8 + (lane >> 3);
      xoff[i] = (uint32_t)(r < xrows ? r : xrows - 1) * (uint32_t)(ldx * 2) + (uint32_t)(((lane & 7) ^ row_swizzle(r)) * 16);
    }
#pragma unroll
    for (int i = 0; i < TC; i++) {
      const int r = (wave * TC + i) * 8 + (lane >> 3);
      woff[i] = (uint32_t)(r < wrows ? r : wrows - 1) * (uint32_t)(ldw * 2) + (uint32_t)(((lane & 7) ^ row_swizzle(r)) * 16);
    }
  }
  template <typename P8> __device__ __forceinline__ void move(P8* lx, P8* lw, int kb, int i) {  // transfer i of the step at byte kb of K
    if (i < TT) to_lds16(bx, lx + (wave * TT + i) * 1024, xoff[i], kb);
    else to_lds16(bw, lw + (wave * TC + i - TT) * 1024, woff[i - TT], kb);
  }
  template <typename P8> __device__ __forceinline__ void read(Frag8& f, P8* lx, P8* lw, int half, int r) {  // fragment r: w0, x0 .., w1 ..
    Frag g;
    if (r >= 1 && r <= TT) {
      g.u = *reinterpret_cast<const uint4*>(lx + (fx ^ (half << 6)) + (r - 1) * 2048);
      f.x[r - 1] = as_v8<E>(g);
    } else {
      const int t = r == 0 ? 0 : r - TT;
      g.u = *reinterpret_cast<const uint4*>(lw + (fw ^ (half << 6)) + t * 2048);
      f.w[t] = as_v8<E>(g);
    }
  }
  // before the first step: both buffers requested, the first one's first half read
  template <typename P8> __device__ __forceinline__ void begin(P8* x0, P8* w0) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (NL & 15) | ((NL >> 4) << 14));  // the first step has landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read_first(x0, w0);
  }
  template <typename P8> __device__ __forceinline__ void read_first(P8* x0, P8* w0) {
#pragma unroll
    for (int r = 0; r < NL; r++) read(P, x0, w0, 0, r);
  }
  // One step on the buffer (lx, lw), whose first half is in P; leaves the first half of the other buffer (ox, ow) in P and
  // the step at kb requested into (lx, lw).  A tile's first step starts its sums (FIRST) instead of adding to cleared ones.
  template <bool FIRST, typename P8> __device__ __forceinline__ void first_half(P8* lx, P8* lw) {
#pragma unroll
    for (int j = 0; j < NM; j++) {
#pragma unroll
      for (int r = 0; r < NL; r++)
        if (r * kRead1 / 16 == j) read(Q, lx, lw, 1, r);
      mma_acc<E, kAgpr, FIRST>(P.w[j / TT], P.x[j % TT], acc[j / TT][j % TT]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the buffer's last reads are in registers and the other buffer's transfers have landed, in every wave, if the wave has issued LEFT or more
  // requests and stores behind those transfers (with fewer the wait would pass while some of them are still under way)
  template <int LEFT = 0> __device__ __forceinline__ void turn() {
    static_assert(LEFT < 64, "what the counter holds");
    __builtin_amdgcn_s_waitcnt(0x0070 | (LEFT & 15) | ((LEFT >> 4) << 14));  // vmcnt(LEFT) lgkmcnt(0)
  }
  template <typename P8> __device__ __forceinline__ void second_half(P8* lx, P8* lw, P8* ox, P8* ow, int kb) {
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NM; j++) {
#pragma unroll
      for (int r = 0; r < NL; r++) {
        if (r * kMove2 / 16 == j) move(lx, lw, kb, r);
        if (r * kRead2 / 16 + kRead2At == j) read(P, ox, ow, 0, r);
      }
      mma_acc<E, kAgpr, false>(Q.w[j / TT], Q.x[j % TT], acc[j / TT][j % TT]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // A tile: its K / 64 steps (an even number), two at a time, `advance` in front of each of them.  STORES: every wave has issued at least so
  // many for the tile before, behind the transfers that the first step waits for, so that these have landed when as many operations are left.
  // None of them may depend on a branch; a wave that has issued fewer, or has no tile before, says `fresh` and waits for all.
  template <int STORES, typename P8, typename F> __device__ __forceinline__ void sweep(P8* x0, P8* w0, P8* x1, P8* w1, int steps, bool fresh, const int& kb, F&& advance) {
    start();
    advance();
    first_half<true>(x0, w0);
    if (fresh) turn<0>();
    else turn<STORES>();
    second_half(x0, w0, x1, w1, kb);
    advance();
    step(x1, w1, x0, w0, kb);
    for (steps -= 2; steps > 0; steps -= 2) {
      advance();
      step(x0, w0, x1, w1, kb);
      advance();
      step(x1, w1, x0, w0, kb);
    }
  }
  template <typename P8> __device__ __forceinline__ void step(P8* lx, P8* lw, P8* ox, P8* ow, int kb) {
    first_half<false>(lx, lw);
    turn<0>();
    second_half(lx, lw, ox, ow, kb);
  }
  __device__ __forceinline__ void start() {  // (whatever the registers hold: a tile's first products do not read it)
#pragma unroll
    for (int c = 0; c < TC; c++)
#pragma unroll
      for (int t = 0; t < TT; t++) {
        if constexpr (kAgpr) asm volatile("" : "=a"(acc[c][t]));
        else asm volatile("" : "=v"(acc[c][t]));
      }
  }
  // Around the products written out the compiler knows of no hazards: the last products are given time before vector
  // instructions read their accumulators.  (The first ones of a tile take no accumulators, and write what has been read.)
  __device__ __forceinline__ void after_products() {
    asm volatile("s_nop 15\n s_nop 15");
    touch();
  }
  __device__ __forceinline__ void touch() {
#pragma unroll
    for (int c = 0; c < TC; c++)
#pragma unroll
      for (int t = 0; t < TT; t++) {
        if constexpr (kAgpr) asm volatile("" : "+a"(acc[c][t]));
        else asm volatile("" : "+v"(acc[c][t]));
      }
  }
};

// Tiles of 256 or of 128.  Time of a round of tiles in steps of the large tile: its K / 64 and 4 for the epilogue; a round
// of the small ones (two per CU) takes 0.61 of that, half a round (one per CU) 0.36: measured at 2 016 to 104 100 rows, 1024 to
// 4096 channels; the choice is the faster one at all of them.
inline bool large_tiles(int64_t M, int N) {
  const int64_t big = ((M + 255) / 256) * ((N + 255) / 256), small = ((M + 127) / 128) * ((N + 127) / 128);
  const double t_big = (double)((big + 255) / 256);
  const double t_small = small <= 256 ? 0.36 : 0.61 * (double)((small + 511) / 512);
  return t_big <= t_small;
}

}  // namespace lin
}  // namespace s3r
