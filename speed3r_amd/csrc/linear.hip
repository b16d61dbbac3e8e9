// Linear layers of the inference paths on the matrix cores: y = x W^T + b, optionally with GELU (exact, by the error
// function) in the epilogue.  bf16 / fp16, matrix-core bound; the tile is linear_tile.h's.
//
// Persistent workgroups.  256 x 256 tiles, one workgroup per CU, where these fill the chip; 128 x 128 tiles, two workgroups
// per CU, where they do not.  us, this / the library's product on the same card (with bias; and with bias and GELU,
// where the library's product is followed by a pass over its output):
//   104 100 x 3072 x 1024     520 / 610     626 / 860
//     8 064 x 4096 x 1024      58 /  57      68 /  87
//     8 064 x 1024 x 4096      55 /  58
//     8 064 x 1024 x 1024      18.5 / 21.3
//     2 016 x 1024 x 1024       9.7 / 10.4 on the device, 9.7 / 19.8 with the host's share
// What bounds the large tile: 81 % of the cycles inside the sweep over K are products (8192^3), at the clock the power limit
// leaves; with K = 1024 the epilogue takes a sixth of a tile.
#include "linear_tile.h"

namespace s3r {
namespace lin {

struct LinearParams {
  const void *x, *w, *bias;
  void* y;
  int64_t M, ldx, ldw, ldy;
  int N, K, mt, nt;
};

// x/2 (1 + erf(x / sqrt 2)).  With t = 1 / (1 + p |x| / sqrt 2) the complementary error function is t times a polynomial
// of degree 4 in t times exp(-x^2 / 2), absolute error 1.5e-7 (Abramowitz and Stegun, 7.1.26); the negative side is taken
// from the complement itself, so that nothing cancels there.  From 16 on the correction is zero: +inf stays itself (and -inf
// gives NaN, as x/2 (1 + erf) does).
__device__ __forceinline__ float gelu(float x) {
  const float a = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(fmaf(a, 0.3275911f * 0.70710678f, 1.f));
  const float e = __builtin_amdgcn_exp2f(x * x * -0.72134752f);
  float q = fmaf(t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
  q = fmaf(t, q, 0.5f * 1.421413741f);
  q = fmaf(t, q, 0.5f * -0.284496736f);
  q = fmaf(t, q, 0.5f * 0.254829592f);
  return fmaf(-fabsf(fminf(x, 16.f)), q * t * e, fmaxf(x, 0.f));
}

template <typename E, int T, bool GELU, int WPS>
__global__ __launch_bounds__(256, WPS) void linear_kernel(LinearParams p) {
  typedef Tile<E, T, T> Tl;
  typedef typename Mma<E>::V2 V2;
  constexpr int BM = Tl::BM, BN = Tl::BN, kStage = 16 * 32 * T;  // kStage: 16 tokens x the wave's channels
  constexpr int PC = 2 * T, RPI = 64 / PC, NS = 16 / RPI;        // 16-byte pieces per row, rows per store, stores per 16 tokens
  __shared__ __attribute__((aligned(1024))) unsigned char lx0[BM * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lx1[BM * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lw0[BN * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lw1[BN * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lst[4 * 2 * kStage];
  TileWalk walk(p.mt, p.nt);
  if (walk.at >= walk.count) return;
  Tl tl;
  int m, n, ask = walk.at, kb = 0;  // ask: the tile that is being requested, kb: at this byte of K
  uint2 nb[T];                      // its bias: channels 4 g4 .. + 3 of each channel tile
  auto aim = [&](int i) {
    int tm, tn;
    walk.locate(i, tm, tn);
    const int64_t r0 = (int64_t)tm * BM;
    const int c0 = tn * BN;
    tl.aim((const E*)p.x + r0 * p.ldx, p.ldx, (int)(p.M - r0 < BM ? p.M - r0 : BM), (const E*)p.w + c0 * p.ldw, p.ldw,
           p.N - c0 < BN ? p.N - c0 : BN);
    if (p.bias != nullptr) {
#pragma unroll
      for (int c = 0; c < T; c++) {
        const int ch = c0 + tl.wn * 16 * T + c * 16 + 4 * tl.g4;
        nb[c] = *reinterpret_cast<const uint2*>((const E*)p.bias + (ch < p.N ? ch : p.N - 4));
      }
    }
  };
  auto advance = [&]() {  // past the last tile its rows are requested again: nothing to tell apart in the loop
    kb += 128;
    if (kb == p.K * 2) {
      kb = 0;
      ask = ask + walk.slots < walk.count ? ask + walk.slots : ask;
      aim(ask);
    }
  };
#pragma unroll
  for (int c = 0; c < T; c++) nb[c] = make_uint2(0, 0);
  walk.locate(walk.at, m, n);
  aim(walk.at);
#pragma unroll
  for (int i = 0; i < Tl::NL; i++) tl.move(lx0, lw0, kb, i);
  // (K = 128: the tile's requests end here, but the aim moves on only after the bias has been taken)
  kb = 128;
#pragma unroll
  for (int i = 0; i < Tl::NL; i++) tl.move(lx1, lw1, kb, i);
  tl.begin(lx0, lw0);
  bool fresh = true;
  for (;;) {
    uint2 cb[T];  // this tile's bias (nb moves on to the next tile's)
#pragma unroll
    for (int c = 0; c < T; c++) cb[c] = nb[c];
    tl.template sweep<T * NS>(lx0, lw0, lx1, lw1, p.K >> 6, fresh, kb, advance);
    fresh = false;
    tl.after_products();

    // A lane holds 4 channels of a token in each tile; 16 tokens at a time go through LDS so that consecutive lanes store
    // consecutive 16-byte pieces of a row (64-byte runs of four lanes sixteen apart: 8 % of the whole kernel at K = 1024).
    const int64_t r0 = (int64_t)m * BM;
    const uint32_t row_bytes = (uint32_t)(p.ldy * 2);
    const uint32_t bytes = (uint32_t)(p.M - r0 < BM ? p.M - r0 : BM) * row_bytes;
    const int pc = tl.lane & (PC - 1), pr = tl.lane / PC;
    const int och = n * BN + tl.wn * 16 * T + pc * 8;
    const uint32_t yo = och < p.N ? (uint32_t)(tl.wm * 16 * T + pr) * row_bytes + (uint32_t)och * 2 : 0x80000000u;
    unsigned char* const mine = lst + tl.wave * (2 * kStage);
    float bias[T][4];  // added last, as the library's product does: the same bits where that does not split K
#pragma unroll
    for (int c = 0; c < T; c++) {
      union { uint2 u; E e[4]; } b;
      b.u = cb[c];
#pragma unroll
      for (int i = 0; i < 4; i++) bias[c][i] = (float)b.e[i];
    }
#pragma unroll
    for (int t = 0; t < T; t++) {
      unsigned char* const buf = mine + (t & 1) * kStage;
#pragma unroll
      for (int c = 0; c < T; c++) {
        union { V2 v[2]; uint2 u; } o;
#pragma unroll
        for (int r = 0; r < 2; r++) {
          float a = tl.acc[c][t][2 * r] + bias[c][2 * r], b = tl.acc[c][t][2 * r + 1] + bias[c][2 * r + 1];
          if constexpr (GELU) {
            a = gelu(a);
            b = gelu(b);
          }
          o.v[r][0] = (E)a;
          o.v[r][1] = (E)b;
        }
        *reinterpret_cast<uint2*>(buf + tl.c16 * (32 * T) + (((c * 2 + (tl.g4 >> 1)) ^ (tl.c16 & (PC - 1))) << 4) + (tl.g4 & 1) * 8) = o.u;
      }
#pragma unroll
      for (int i = 0; i < NS; i++) {
        const int r = i * RPI + pr;
        const uint4 v = *reinterpret_cast<const uint4*>(buf + r * (32 * T) + ((pc ^ (r & (PC - 1))) << 4));
        store16_if((E*)p.y + r0 * p.ldy, bytes, yo + (uint32_t)(t * 16 + i * RPI) * row_bytes, v);
      }
    }
    walk.at += walk.slots;
    if (walk.at >= walk.count) break;
    walk.locate(walk.at, m, n);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // no transfer may still write LDS when the wave ends
}

template <typename E> static void launch_linear(LinearParams& p, bool act, hipStream_t st) {
  const bool large = large_tiles(p.M, p.N);
  const int b = large ? 256 : 128;
  p.mt = (int)((p.M + b - 1) / b);
  p.nt = (p.N + b - 1) / b;
  const int64_t tiles = (int64_t)p.mt * p.nt, most = large ? 256 : 512;
  const dim3 grid((unsigned)(tiles < most ? tiles : most)), blk(256);
  if (large && act) hipLaunchKernelGGL((linear_kernel<E, 8, true, 1>), grid, blk, 0, st, p);
  else if (large) hipLaunchKernelGGL((linear_kernel<E, 8, false, 1>), grid, blk, 0, st, p);
  else if (act) hipLaunchKernelGGL((linear_kernel<E, 4, true, 2>), grid, blk, 0, st, p);
  else hipLaunchKernelGGL((linear_kernel<E, 4, false, 2>), grid, blk, 0, st, p);
}

}  // namespace lin
}  // namespace s3r

using namespace s3r;

extern "C" int s3r_linear(const void* x, const void* w, const void* bias, void* y, int64_t M, int N, int K, int64_t ldx, int64_t ldw,
                          int64_t ldy, int activation, int dtype, void* stream) {
  if (!x || !w || !y) return fail(S3R_ERR_BAD_ARG, "s3r_linear: null pointer");
  if (M <= 0 || N <= 0 || K <= 0) return fail(S3R_ERR_BAD_ARG, "s3r_linear: non-positive size");
  if ((dtype != S3R_BF16 && dtype != S3R_F16) || K % 128 || N % 8 || (activation != S3R_ACT_NONE && activation != S3R_ACT_GELU))
    return fail(S3R_ERR_UNSUPPORTED, "s3r_linear: dtype %d, %d outputs, %d inputs, activation %d (built for 16-bit types, outputs in "
                "steps of 8, inputs in steps of 128, no activation or GELU)", dtype, N, K, activation);
  // a tile's rows are addressed by 32-bit byte offsets from its first one
  if (ldx < K || ldw < K || ldy < N || ldx >= (1 << 21) || ldw >= (1 << 21) || ldy >= (1 << 21))
    return fail(S3R_ERR_BAD_ARG, "s3r_linear: rows overlap or lie 2^21 elements or more apart");
  if (!aligned16(x) || !aligned16(w) || !aligned16(y) || ldx % 8 || ldw % 8 || ldy % 8 || (reinterpret_cast<uintptr_t>(bias) & 7u))
    return fail(S3R_ERR_BAD_ARG, "s3r_linear: x, w, y and their rows must be multiples of 16 bytes, the bias of 8");
  if (((M + 127) / 128) * ((N + 127) / 128) > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "s3r_linear: tensor too large for one launch");
  lin::LinearParams p = {x, w, bias, y, M, ldx, ldw, ldy, N, K, 0, 0};
  const bool act = activation == S3R_ACT_GELU;
  if (dtype == S3R_BF16) lin::launch_linear<bf16_t>(p, act, (hipStream_t)stream);
  else lin::launch_linear<f16_t>(p, act, (hipStream_t)stream);
  return check_launch("s3r_linear");
}
