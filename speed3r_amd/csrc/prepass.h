// Pieces shared by the forward and the backward pass over the packed q/k/v projection: argument block, rotation tables
// and LayerNorm parameters staged in LDS, the row transforms.
#pragma once
#include "s3r_common.h"
#include <climits>
#include <type_traits>

namespace s3r {

struct PrepassParams {
  const void *q, *k, *v;        // raw projection, [B,H,N,64] views with common strides
  void *q_out, *k_out;          // contiguous [B,H,N,64]
  void *qc, *kc, *vc;           // contiguous [B,H,Nc,64]
  void *q_raw, *k_raw;          // optional: the block means before norm and rotation
  const void* pos;              // [B,N,2] int32 or int64 (pos64), (y, x) pairs contiguous; nullptr: no rotation
  const void *cos_tab, *sin_tab;  // [P,16] in T
  const float* inv_freq;        // optional [16]: angles of positions >= P; without it such positions are clamped to P - 1
  const void *qn_w, *qn_b, *kn_w, *kn_b;  // LayerNorm(64) parameters (nullptr weights: no norm) in T, or fp32 (ln_f32)
  float eps;
  int pos64, ln_f32, finish;    // finish: qc, kc after norm and rotation
  int lowest;                   // positions below are taken as this: 0, or the lowest there is (own angles below zero too)
  int P, staged_rows;           // rows of the tables; the first staged_rows of them are held in LDS
  int B, H, block;
  int64_t N, sxb, sxh, sxn, spb, spn;
};

// Table rows held in LDS as fp32 (cosine, sine and minus sine: 192 bytes per row).  64 rows = 12 KB: every frame of up
// to 64 patches a side; further rows are read from the caller's tables.  A workgroup copies all of them, so that more
// rows than a call has positions would cost time.  Against up to 165 rows in LDS (as many as four resident workgroups hold
// without the lanes' slots), 100 000 tokens x 16 heads, bf16: 209 us / 206 us at 100 positions a side, 225 / 222 at 164.
constexpr int kStagedRows = 64;
// tables, parameter rows and, with a rotation, the lanes' slots (64 bytes each at most)
inline size_t staged_bytes(int rows, bool rot) { return ((size_t)3 * rows * 16 + 4 * 64) * sizeof(float) + (rot ? 256 * 64 : 0); }

inline PrepassParams prepass_params(const s3r_prepass_args& a) {
  PrepassParams p = {};
  p.q = a.q; p.k = a.k; p.v = a.v; p.q_out = a.q_out; p.k_out = a.k_out; p.qc = a.q_pool; p.kc = a.k_pool; p.vc = a.v_pool;
  p.q_raw = a.q_raw; p.k_raw = a.k_raw; p.pos = a.positions; p.pos64 = a.positions_int64;
  p.cos_tab = a.cos_table; p.sin_tab = a.sin_table; p.inv_freq = a.inv_freq; p.P = a.table_rows;
  p.qn_w = a.q_norm_weight; p.qn_b = a.q_norm_bias; p.kn_w = a.k_norm_weight; p.kn_b = a.k_norm_bias; p.ln_f32 = a.norm_fp32; p.eps = a.eps;
  p.finish = a.finish_pooled; p.lowest = a.inv_freq != nullptr && a.signed_positions ? INT_MIN : 0; p.B = a.B; p.H = a.H; p.N = a.N; p.block = a.block;
  p.sxb = a.stride_b; p.sxh = a.stride_h; p.sxn = a.stride_n; p.spb = a.pos_stride_b; p.spn = a.pos_stride_n;
  return p;
}

int check_prepass(const char* who, PrepassParams& p, int head_dim, int dtype);

// [cos | sin | -sin][staged_rows][16], then q_norm weight, bias, k_norm weight, bias [64] each; a step then reads ready
// operands instead of unpacking 16-bit table and parameter values for every row (a fifth of a step's vector instructions).
template <typename T> __device__ __forceinline__ void stage_tables(const PrepassParams& p, float* staged) {
  constexpr int VEC = 16 / sizeof(T);
  const int rows16 = p.staged_rows * 16;
  for (int i = threadIdx.x * VEC; i < rows16; i += 256 * VEC) {  // table rows are 16 values: whole 16-byte pieces
    const uint4 c = *reinterpret_cast<const uint4*>((const T*)p.cos_tab + i);
    const uint4 s = *reinterpret_cast<const uint4*>((const T*)p.sin_tab + i);
#pragma unroll
    for (int e = 0; e < VEC; e++) {
      const float sv = to_f32(reinterpret_cast<const T*>(&s)[e]);
      staged[i + e] = to_f32(reinterpret_cast<const T*>(&c)[e]);
      staged[rows16 + i + e] = sv;
      staged[2 * rows16 + i + e] = -sv;
    }
  }
  if (p.qn_w != nullptr) {
    const int which = threadIdx.x >> 6, e = threadIdx.x & 63;
    const void* const src = which == 0 ? p.qn_w : which == 1 ? p.qn_b : which == 2 ? p.kn_w : p.kn_b;
    staged[3 * rows16 + threadIdx.x] = src == nullptr ? 0.f : p.ln_f32 ? ((const float*)src)[e] : to_f32(((const T*)src)[e]);
  }
}

__device__ __forceinline__ int load_pos(const PrepassParams& p, int64_t b, int64_t n, int c) {
  const int64_t o = b * p.spb + n * p.spn + c;
  return p.pos64 ? (int)((const int64_t*)p.pos)[o] : ((const int32_t*)p.pos)[o];
}

// which part of a row a lane holds
template <typename T> struct RotLane {
  static constexpr int VEC = 16 / sizeof(T), QL = 16 / VEC;  // QL: lanes per quarter of the head dimension
  int half, second, f0;
  __device__ __forceinline__ explicit RotLane(int lr)
      : half(lr / (2 * QL)),          // 0: y half, 1: x half
        second((lr / QL) & 1),        // which quarter of the half this lane holds
        f0((lr % QL) * VEC) {}        // frequency index of the lane's first value
};

// truncated mean of the block's positions along the lane's coordinate; pos_sum: lane parity 0 adds up y, 1 x
__device__ __forceinline__ int block_position(int pos_sum, float cnt, int half) {
#pragma unroll
  for (int off = 2; off < 64; off <<= 1) pos_sum += __shfl_xor(pos_sum, off);
  return (int)((float)(half ? __builtin_amdgcn_readlane(pos_sum, 1) : __builtin_amdgcn_readlane(pos_sum, 0)) / cnt);
}

template <int VEC> __device__ __forceinline__ void load_row(const float* src, float (&x)[VEC]) {
#pragma unroll
  for (int i = 0; i < VEC; i += 4) *reinterpret_cast<float4*>(&x[i]) = *reinterpret_cast<const float4*>(src + i);
}

// LayerNorm over the 64 values of the row (the lane's VEC of them in x): fp32 statistics, result rounded to T
template <typename T, int VEC> __device__ __forceinline__ void norm_row(const PrepassParams& p, const float* staged, float (&x)[VEC], int ln_row, int lr) {
#pragma clang fp contract(off)
  constexpr int LPR = 64 / VEC;
  const float* lw = staged + 3 * p.staged_rows * 16 + ln_row * 64 + lr * VEC;
  float wgt[VEC], bias[VEC];
  load_row(lw, wgt);
  load_row(lw + 64, bias);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VEC; i++) s += x[i];
  s = group_sum<LPR>(s);
  const float mean = s * (1.0f / 64);
  float var = 0.f;
#pragma unroll
  for (int i = 0; i < VEC; i++) var += (x[i] - mean) * (x[i] - mean);
  var = group_sum<LPR>(var);
  const float rstd = inv_sqrt(var * (1.0f / 64) + p.eps);
#pragma unroll
  for (int i = 0; i < VEC; i++) x[i] = round_keep<T>((x[i] - mean) * rstd * wgt[i] + bias[i]);
}

// Where the lane reads the VEC cosines and sines of its frequencies at position pp: the staged tables or, for positions
// outside of them (rare; below zero too unless they are clamped to it), a slot of its own in LDS that is filled here.  Called by whole waves.  Pointers
// instead of values keep the rare case out of the registers of the common one (with both in registers the pass spills).
struct TablePtr {
  const float *c, *s;
};
template <typename T>
__device__ __forceinline__ TablePtr table_ptr(const PrepassParams& p, float* staged, const RotLane<T>& rl, int pp, bool minus_sine) {
  constexpr int VEC = RotLane<T>::VEC;
  pp = pp < p.lowest ? p.lowest : pp;
  const bool outside = (uint32_t)pp >= (uint32_t)p.staged_rows;
  TablePtr t;
  t.c = staged + (outside ? 0 : pp) * 16 + rl.f0;
  t.s = t.c + (minus_sine ? 2 : 1) * p.staged_rows * 16;
  if (__any(outside)) {
    if (outside) {
      float* const slot = staged + (3 * p.staged_rows * 16 + 4 * 64) + threadIdx.x * (2 * VEC);
      if ((uint32_t)pp < (uint32_t)p.P || p.inv_freq == nullptr) {
        const int64_t row = (int64_t)(pp < p.P ? pp : p.P - 1) * 16 + rl.f0;
        const uint4 c = *reinterpret_cast<const uint4*>((const T*)p.cos_tab + row), sv = *reinterpret_cast<const uint4*>((const T*)p.sin_tab + row);
#pragma unroll
        for (int i = 0; i < VEC; i++) {
          const float s = to_f32(reinterpret_cast<const T*>(&sv)[i]);
          slot[i] = to_f32(reinterpret_cast<const T*>(&c)[i]);
          slot[VEC + i] = minus_sine ? -s : s;
        }
      } else {
#pragma unroll 1
        for (int i = 0; i < VEC; i++) {
          // (each value exists in fp32 before it is rounded to T: the empty asm keeps the compiler from forming a product
          // that is rounded to fp16 at once)
          float angle = (float)pp * p.inv_freq[rl.f0 + i];
          asm volatile("" : "+v"(angle));
          angle = round_to<T>(angle);
          const float s = round_to<T>(sinf(angle));
          slot[i] = round_to<T>(cosf(angle));
          slot[VEC + i] = minus_sine ? -s : s;
        }
      }
      t.c = slot;
      t.s = slot + VEC;
    }
  }
  return t;
}

// Rotation in place: "rotate half" is (-second quarter, first quarter); the lanes of a first quarter take their partner's
// value with a minus sign, which is put on the sine instead (minus_sine = first quarter; rounding is symmetric:
// round(-a * s) = round(a * -s)).  Both products and the sum are rounded to T.
template <typename T, int VEC> __device__ __forceinline__ void rotate_row(float (&x)[VEC], const TablePtr& t) {
#pragma clang fp contract(off)
  float cs[VEC], sn[VEC];
  load_row(t.c, cs);
  load_row(t.s, sn);
#pragma unroll
  for (int i = 0; i < VEC; i++) {
    const float other = lane_xor<RotLane<T>::QL>(x[i]);  // the paired value, one quarter away
    const float a = round_keep<T>(x[i] * cs[i]);
    const float c2 = round_keep<T>(other * sn[i]);
    x[i] = a + c2;
  }
}

}  // namespace s3r
