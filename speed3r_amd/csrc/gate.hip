// Gate of the layer, sigmoid(x W^T + b) with 2 outputs per head (pi3/models/layers/sparse_attention.py:88,127), HBM bound:
// [rows, C] in, [rows, O <= 32] out.
//
// A matrix product with 32 columns leaves a tiled GEMM without parallelism (118 us for the 213 MB of 104 100 rows of 1024
// = 1.8 TB/s, 20 us for 8 064 and 32 256 rows, and the sigmoid as a launch of 4 to 7 us).  41, 9.9 and 20 us here: the weight never moves
// again: the four waves of a workgroup each keep a quarter of W's columns as MFMA operands in registers (64 for C = 1024)
// and go over tiles of 16 rows; the rows come straight into operand layout, the next tile's requested before the four
// partial sums meet in LDS.
#include "select_common.h"

namespace s3r {
namespace gate {
using namespace sel;

template <typename E> __device__ __forceinline__ f32x4 mma16(typename Mma<E>::V8 a, typename Mma<E>::V8 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mma16<bf16_t>(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
template <> __device__ __forceinline__ f32x4 mma16<f16_t>(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// C = 128 * KS.  Rounding points of the two torch modules: the product with its bias to the I/O type, then the sigmoid.
template <typename E, int KS>
__global__ __launch_bounds__(256, 4) void gate_kernel(const E* __restrict__ x, const E* __restrict__ w, const E* __restrict__ bias,
                                                      E* __restrict__ out, int64_t rows, int O, int64_t tiles) {
  typedef typename Mma<E>::V8 V8;
  constexpr int C = 128 * KS;
  __shared__ float part[2][4][8][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = lane & 15, g = lane >> 4;
  const int k0 = wave * 32 * KS + g * 8;  // the lane's eight columns of step ks: k0 + 32 ks ..
  V8 wf[2][KS];  // A operand: lane = output
#pragma unroll
  for (int ot = 0; ot < 2; ot++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      Frag f;
      f.u = make_uint4(0, 0, 0, 0);
      if (16 * ot + t < O) f.u = *reinterpret_cast<const uint4*>(w + (16 * ot + t) * C + k0 + 32 * ks);
      wf[ot][ks] = as_v8<E>(f);
    }
  // this wave finishes outputs o, o + 1 of every row: registers 2 wave, 2 wave + 1 of the accumulators
  const int o = 16 * (wave >> 1) + 4 * g + 2 * (wave & 1);
  const bool keep = o < O;
  const float b0 = bias != nullptr && keep ? (float)bias[o] : 0.f, b1 = bias != nullptr && keep ? (float)bias[o + 1] : 0.f;
  V8 xf[KS];  // B operand: lane = row
  auto fetch = [&](int64_t tile) {
    int64_t row = tile * 16 + t;
    row = row < rows ? row : rows - 1;
    const E* xr = x + row * C + k0;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      Frag f;
      f.u = *reinterpret_cast<const uint4*>(xr + 32 * ks);
      xf[ks] = as_v8<E>(f);
    }
  };
  fetch(blockIdx.x);
  int buf = 0;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x, buf ^= 1) {
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      acc[0] = mma16<E>(wf[0][ks], xf[ks], acc[0]);
      acc[1] = mma16<E>(wf[1][ks], xf[ks], acc[1]);
    }
    if (tile + gridDim.x < tiles) fetch(tile + gridDim.x);
#pragma unroll
    for (int r = 0; r < 8; r++) part[buf][wave][r][lane] = acc[r >> 2][r & 3];
    __syncthreads();  // one per tile: the other buffer is written next, and read last before this barrier
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int wv = 0; wv < 4; wv++) {
      s0 += part[buf][wv][2 * wave][lane];
      s1 += part[buf][wv][2 * wave + 1][lane];
    }
    const int64_t row = tile * 16 + t;
    if (keep && row < rows) {
      union { E e[2]; uint32_t u; } r;
      r.e[0] = (E)(1.f / (1.f + expf(-round_to<E>(s0 + b0))));
      r.e[1] = (E)(1.f / (1.f + expf(-round_to<E>(s1 + b1))));
      *reinterpret_cast<uint32_t*>(out + row * O + o) = r.u;
    }
  }
}

template <typename E>
static void launch(const void* x, const void* w, const void* bias, void* out, int64_t rows, int C, int O, hipStream_t st) {
  const int64_t tiles = (rows + 15) / 16;
  // four workgroups per CU: 128 registers a lane, 16 waves with 8 KB of rows in flight each
  const dim3 grid((unsigned)(tiles < 1024 ? tiles : 1024)), blk(256);
#define S3R_GATE(KS) hipLaunchKernelGGL((gate_kernel<E, KS>), grid, blk, 0, st, (const E*)x, (const E*)w, (const E*)bias, (E*)out, rows, O, tiles)
  switch (C / 128) {
    case 2: S3R_GATE(2); break;
    case 4: S3R_GATE(4); break;
    case 6: S3R_GATE(6); break;
    default: S3R_GATE(8); break;
  }
#undef S3R_GATE
}

}  // namespace gate
}  // namespace s3r

using namespace s3r;

extern "C" int s3r_gate(const void* x, const void* w, const void* bias, void* out, int64_t rows, int C, int O, int dtype, void* stream) {
  if (!x || !w || !out) return fail(S3R_ERR_BAD_ARG, "s3r_gate: null pointer");
  if (rows <= 0 || C <= 0 || O <= 0) return fail(S3R_ERR_BAD_ARG, "s3r_gate: non-positive size");
  if ((dtype != S3R_BF16 && dtype != S3R_F16) || C % 256 || C > 1024 || O > 32 || O % 2)
    return fail(S3R_ERR_UNSUPPORTED, "s3r_gate: dtype %d, %d channels, %d outputs (built for 16-bit types, 256 to 1024 channels in "
                "steps of 256, an even number of outputs up to 32)", dtype, C, O);
  if (!aligned16(x) || !aligned16(w) || (reinterpret_cast<uintptr_t>(out) & 3u))
    return fail(S3R_ERR_BAD_ARG, "s3r_gate: x and w must be multiples of 16 bytes, out of 4");
  if (dtype == S3R_BF16) gate::launch<bf16_t>(x, w, bias, out, rows, C, O, (hipStream_t)stream);
  else gate::launch<f16_t>(x, w, bias, out, rows, C, O, (hipStream_t)stream);
  return check_launch("s3r_gate");
}
