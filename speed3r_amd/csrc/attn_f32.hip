// fp32 attention on the matrix cores (head_dim 64): the selection branch for blocks of 64, 32 and 16 tokens and the
// compressed branch with its fp32 scores.
//
// Blocks of 64 go to attn_f32_split_kernel from 385 of them on, up to a softmax scale of 2^30 (launch_64); what follows is about attn_f32_kernel.
//
// Bound: the fp32 matrix instructions (v_mfma_f32_16x16x4_f32: 64 FLOP per cycle and SIMD, 157 TFLOP/s; a product of
// 8192 x 8192 matrices by the library reaches 154).  At 8 328 tokens x 16 heads, 16 blocks of 64 (3.5e10 FLOP, 0.23 ms)
// the generic kernel, whose vector FMAs wait for one LDS read per four products, takes 1.36 ms, this one 0.29 ms; at
// 16-token blocks, top-32, 4.8 and 0.22 ms.  The vector instructions of the softmax hardly overlap with these products (they
// share the SIMD's FMA units), so what a probability costs beside its products is what is lost.  Base 2 with one constant
// (scale log2(e)): a fused multiply-add, an exponential and an addition, in place of exp(x) from exp2 with the rounding of
// x log2(e) put back (ten instructions): 342 -> 316 us.  A reference that moves only when a score exceeds it by
// kSlack, in place of the running maximum, whose exchange between lanes every stage waited for: 316 -> 307.  Error against 64 bits
// over 5 scales of the inputs: 0.65e-6 to 2.34e-6 before and after.  Half blocks at the end of a launch (launch_t): 307 ->
// 292.  What is left: 33 us per 1 041 tokens = 86 % of the matrix rate, and 28 us beside them (the first loads, a SIMD's last waves).
//
// One wave owns 16 query rows: S^T = K Q^T puts one query per lane (column c = lane % 16) and four keys of every
// 16-key group (4 g + r, g = lane / 16), so the probabilities are already the B operand of O^T = V^T P^T and never
// leave their registers.  The waves of a query block share its K and V stages in LDS (direct transfers, two buffers,
// one barrier per stage).  Measured at 8 328 tokens: stages of 32 keys 0.335 ms, of 16 keys 0.364; two waves per
// workgroup (a query block in two) 0.366, single waves with stages of their own 0.453; all fragments of a stage read
// ahead of its products: 0.361 (registers).
// K rows (256 bytes) are stored with chunk ^ row, so that the 16 rows of a fragment read lie in different banks; the
// fragment of step s holds head dimensions 4 s + g: the matrix core adds them in the order of a scalar FMA chain over
// the head dimension (the scores come out with the generic kernel's bits).  A V fragment read (lane = chunk of the row)
// serves four products: operand row m of product dg is head dimension 4 m + dg, so that a lane ends up with 16
// consecutive dimensions of its query.
#include "block16.h"
#include "attn_params.h"

namespace s3r {
namespace f32 {
using namespace sel;

constexpr float kLn2 = 0.693147182f, kLn2Lo = -1.90465421e-9f;  // ln 2 = their sum
constexpr int kRow = 256;  // bytes of a K or V row

// Base-2 units by which a score may exceed the row's reference: probabilities and sums scale with 2^kSlack, their
// relative errors do not.
constexpr float kSlack = 4.f;
// ln(l 2^m): the exponent of l joins m, so that the logarithm of what is left is small and the sum is rounded once
__device__ __forceinline__ float log_sum(float m, float l) {
  if (!(l > 0.f)) return -INFINITY;
  const float e = m + (float)__builtin_amdgcn_frexp_expf(l);
  return fmaf(e, kLn2, fmaf(e, kLn2Lo, logf(__builtin_amdgcn_frexp_mantf(l))));
}
// W waves share a workgroup's 16 W query rows and its stages of KS keys.  SELECT: the rows are one query block of 16 W
// tokens, the stages the parts of its listed key blocks; otherwise every key.  SPLIT: workgroups from number `whole` on take half
// a block's rows each; two waves share 16 rows, each takes one half of every stage, and the first adds up what the two have.
template <int W, int KS, int BLK, bool SPLIT>
__global__ __launch_bounds__(64 * W, 4) void attn_f32_kernel(AttnParams p, int ngrp, int total, int whole) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k0[KS * kRow], lds_k1[KS * kRow];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v0[KS * kRow], lds_v1[KS * kRow];
  constexpr bool SELECT = BLK > 0;
  constexpr int SUB = SELECT ? BLK / KS : 1, NG = KS / 16, NI = KS / (4 * W);
  static_assert(!SELECT || (BLK % KS == 0 && BLK % (16 * W) == 0), "a block is a whole number of stages and of workgroups");
  static_assert(!SPLIT || (SELECT && W == 4 && NG == 2), "four waves as two row groups and two halves of a stage");
  static_assert(NI * 4 * W == KS, "every wave moves the same number of 1 KB pieces");

  const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  // each XCD takes a contiguous range of query blocks: neighbours list mostly the same key blocks
  const bool half = SPLIT && (int)blockIdx.x >= whole;  // this workgroup takes half a block's rows
  const int w = half ? blockIdx.x - whole : blockIdx.x, items = half ? 2 * (total - whole) : SPLIT ? whole : total;
  const int xcd = w & 7, per = items >> 3, rem = items & 7;
  const int item = xcd * per + (xcd < rem ? xcd : rem) + (w >> 3);
  const int vid = half ? whole + (item >> 1) : item;
  const int bh = vid / ngrp;
  const int64_t row0 = (int64_t)(vid - bh * ngrp) * (16 * W);
  const int rows_at = half ? (item & 1) * 32 + (wave & 1) * 16 : wave * 16, part = half ? wave >> 1 : 0;
  const int b = bh / p.H;
  const int h = bh - b * p.H;

  const int64_t N = p.Lk;
  const int64_t qrow = row0 + rows_at + c;
  const bool live = qrow < p.Lq;
  const float* qp = (const float*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const float* kp = (const float*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const float* vp = (const float*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;

  // the stages: listed blocks in order (entries < 0 or beyond the sequence skipped), or all keys
  int32_t entry = -1;
  uint64_t mask = 0;
  if constexpr (SELECT) {
    if (lane < p.K) entry = p.idx[(int64_t)b * p.sib + (int64_t)h * p.sih + row0 / BLK * p.sim + lane];
    mask = __ballot(entry >= 0 && (int64_t)entry * BLK < N);
  }
  int64_t start = 0;  // first key of the stage to be requested next; negative: none left
  int sub = 0;
  auto first = [&]() {
    if constexpr (SELECT) start = mask ? (int64_t)__builtin_amdgcn_readlane(entry, __builtin_ctzll(mask)) * BLK : -1;
  };
  auto advance = [&]() {
    if constexpr (SELECT) {
      if (++sub < SUB && start + KS < N) {
        start += KS;
      } else {
        sub = 0;
        mask &= mask - 1;
        first();
      }
    } else {
      start = start + KS < N ? start + KS : -1;
    }
  };

  const uint32_t krow = (uint32_t)p.skn * 4u, vrow = (uint32_t)p.svn * 4u;
  auto request = [&](int64_t s0, unsigned char* kb, unsigned char* vb) {  // rows beyond the sequence re-read its last row
    const int last = (int)((N - s0 < KS ? N - s0 : KS) - 1);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kp + s0 * p.skn), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vp + s0 * p.svn), 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int piece = wave * NI + i;
      const int lrow = piece * 4 + g;
      const int row = lrow < last ? lrow : last;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(kb + piece * 1024), 16,
                                               (uint32_t)row * krow + (uint32_t)((c ^ (lrow & 15)) * 16), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)(vb + piece * 1024), 16,
                                               (uint32_t)row * vrow + (uint32_t)(c * 16), 0, 0, 0);
    }
  };

  float q[16];  // B operand of step s: head dimension 4 s + g of the lane's query
#pragma unroll
  for (int s = 0; s < 16; s++) q[s] = live ? qp[qrow * p.sqm + 4 * s + g] : 0.f;

  const float sl2 = (float)((double)p.scale * 1.4426950408889634);

  f32x4 o[4];
#pragma unroll
  for (int dg = 0; dg < 4; dg++)
#pragma unroll
    for (int r = 0; r < 4; r++) o[dg][r] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;

  auto compute = [&](auto groups, int64_t s0, const unsigned char* kb, const unsigned char* vb) {
    constexpr int NG = decltype(groups)::value, KC = 16 * NG;
    const int nvalid = (int)(N - s0 < KC ? N - s0 : KC);
    f32x4 st[NG];
#pragma unroll
    for (int kg = 0; kg < NG; kg++)
#pragma unroll
      for (int r = 0; r < 4; r++) st[kg][r] = 0.f;
#pragma unroll
    for (int s = 0; s < 16; s++)
#pragma unroll
      for (int kg = 0; kg < NG; kg++) {
        const float a = *reinterpret_cast<const float*>(kb + (kg * 16 + c) * kRow + ((s ^ c) << 4) + g * 4);
        st[kg] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, q[s], st[kg], 0, 0, 0);
      }
    static_assert(NG <= 2, "every group's product is waited for");
    if constexpr (NG == 2) settle_f32(st[0], st[1]);
    else settle_f32(st[0]);
    if constexpr (!SELECT) {
      if (p.scores != nullptr && live) {
        float* srow = p.scores + (((int64_t)b * p.H + h) * p.Lq + qrow) * p.Lk + s0;
#pragma unroll
        for (int kg = 0; kg < NG; kg++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (kg * 16 + 4 * g + r < nvalid) srow[kg * 16 + 4 * g + r] = st[kg][r];
      }
    }
    if (nvalid < KC) {  // (wave-uniform) the ragged end of the sequence
#pragma unroll
      for (int kg = 0; kg < NG; kg++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (kg * 16 + 4 * g + r >= nvalid) st[kg][r] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kg = 0; kg < NG; kg++)
#pragma unroll
      for (int r = 0; r < 4; r++) mx = fmaxf(mx, st[kg][r]);
    if (__any(mx * sl2 > m_i + kSlack)) {  // scale > 0
      mx = xh_max(fmaxf(mx, lane_xor<16>(mx))) * sl2;
      const float m_new = fmaxf(m_i, mx);
      const float alpha = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i - m_new);
      l_i *= alpha;
#pragma unroll
      for (int dg = 0; dg < 4; dg++)
#pragma unroll
        for (int r = 0; r < 4; r++) o[dg][r] *= alpha;
      m_i = m_new;
    }
    const float m_neg = m_i == -INFINITY ? 0.f : -m_i;
#pragma unroll
    for (int kg = 0; kg < NG; kg++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float pv = __builtin_amdgcn_exp2f(fmaf(st[kg][r], sl2, m_neg));
        l_i += pv;
        const float4 vf = *reinterpret_cast<const float4*>(vb + (kg * 16 + 4 * g + r) * kRow + c * 16);
        o[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.x, pv, o[0], 0, 0, 0);
        o[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.y, pv, o[1], 0, 0, 0);
        o[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.z, pv, o[2], 0, 0, 0);
        o[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf.w, pv, o[3], 0, 0, 0);
      }
  };

  // Stage loop, written for both buffer parities.  Each stage: this wave's own transfers have landed (vmcnt 0), the
  // barrier makes everybody's visible and says that the other buffers are no longer read; then the next stage is
  // requested into them and passes under the arithmetic of this one.
  auto ready = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    if constexpr (W > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto sweep = [&](auto groups) __attribute__((always_inline)) {
    const int at = part * (16 * kRow);
    while (true) {
      int64_t cur = start;
      advance();
      ready();
      if (start >= 0) request(start, lds_k1, lds_v1);
      compute(groups, cur + 16 * part, lds_k0 + at, lds_v0 + at);
      if (start < 0) break;
      cur = start;
      advance();
      ready();
      if (start >= 0) request(start, lds_k0, lds_v0);
      compute(groups, cur + 16 * part, lds_k1 + at, lds_v1 + at);
      if (start < 0) break;
    }
  };
  first();
  if (start >= 0) {
    request(start, lds_k0, lds_v0);
    if constexpr (SPLIT) {
      if (half) sweep(std::integral_constant<int, 1>{});
      else sweep(std::integral_constant<int, NG>{});
    } else {
      sweep(std::integral_constant<int, NG>{});
    }
  }
  if constexpr (SPLIT) {
    if (half) {  // the waves of the stages' second halves hand over to those of the first ones
      __syncthreads();
      float* const to = reinterpret_cast<float*>((wave & 1) ? lds_k1 : lds_k0);
      float* const stat = reinterpret_cast<float*>(lds_v0) + (wave & 1) * 128;
      if (part == 1) {
#pragma unroll
        for (int dg = 0; dg < 4; dg++)
#pragma unroll
          for (int r = 0; r < 4; r++) to[(dg * 4 + r) * 64 + lane] = o[dg][r];
        stat[lane] = m_i;
        stat[64 + lane] = l_i;
      }
      __syncthreads();
      if (part == 1) return;
      const float m1 = stat[lane], m_new = fmaxf(m_i, m1);
      const float a0 = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i - m_new), a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - m_new);
      m_i = m_new;
      l_i = l_i * a0 + stat[64 + lane] * a1;
#pragma unroll
      for (int dg = 0; dg < 4; dg++)
#pragma unroll
        for (int r = 0; r < 4; r++) o[dg][r] = o[dg][r] * a0 + to[(dg * 4 + r) * 64 + lane] * a1;
    }
  }

  const float l = xh_sum(l_i + lane_xor<16>(l_i));
  if (live) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if constexpr (SELECT) {
      // The gated merge (rounded as s3r_gated_merge does: each product, then the sum) in place of the output: a pass over it less,
      // 8 328 tokens x 16 heads 357 -> 344 us for the whole path.
      if (p.merge_out != nullptr) {
#pragma clang fp contract(off)
        const float* const gp = (const float*)p.merge_gate + (int64_t)b * p.sgb + (int64_t)h * p.sgh + qrow * p.sgn;
        const float* const oc = (const float*)p.merge_oc + (int64_t)b * p.scb + (int64_t)h * p.sch + (qrow / BLK) * p.scm + 16 * g;
        float* const to = (float*)p.merge_out + (((int64_t)b * p.Lq + qrow) * p.H + h) * 64 + 16 * g;
        const float g0 = gp[0], g1 = gp[1];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float4 c4 = *reinterpret_cast<const float4*>(oc + 4 * r);
          const float x[4] = {c4.x, c4.y, c4.z, c4.w};
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float s = o[e][r] * inv, a0 = g0 * x[e], a1 = g1 * s;
            y[e] = a0 + a1;
          }
          *reinterpret_cast<float4*>(to + 4 * r) = make_float4(y[0], y[1], y[2], y[3]);
        }
        return;
      }
    }
    float* op = (float*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh + qrow * p.som + 16 * g;
#pragma unroll
    for (int r = 0; r < 4; r++)
      *reinterpret_cast<float4*>(op + 4 * r) = make_float4(o[0][r] * inv, o[1][r] * inv, o[2][r] * inv, o[3][r] * inv);
    if (p.lse != nullptr && g == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = log_sum(m_i, l);
  }
}

// ---- blocks of 64 tokens on the 16-bit matrix instructions ---------------------------------------------------------
// Every value as the sum of three bf16 numbers (24 bits) and of the nine products of their parts the six that count: what is left out lies 2^-26
// below a product, the fp32 accumulator's own rounding at 2^-24.  Six bf16 products take 6/16 of the fp32 instruction's time, and unlike that one they
// leave the vector unit to other waves.  The small products of a stage come first, those of P V have a sum of their own, so that
// a stage of 32 keys rounds the output's sum once.
// Error against 64 bits, fp32 instructions / this, 1 041 tokens, 8 blocks, queries of standard deviation 0.3 to 6: 2.9e-7 / 1.4e-7, 4.0e-7 /
// 1.9e-7, 7.8e-7 / 3.4e-7, 9.4e-7 / 4.1e-7 (probabilities and sums are fp32 as there); log-sum-exp of scores up to 180 1.4e-4 / 6.5e-5.  The scores
// are closer to 64 bits than the chain of fp32 products, so not its bits.
// us, fp32 instructions / this, 16 heads, random lists of 16: 1 041 tokens 62.9 / 61.3, 2 600 118 / 82, 8 328 296 / 223, 33 312 1 093 / 846; the
// whole operator at 8 328 tokens of a video 331 / 264.
// Bound: a stage costs a wave 48 products and 220 vector instructions (88 of them the splitting of a sixteenth of the stage's K and V, shared
// by the four waves, 44 that of the probabilities), and with four waves to a SIMD the two units overlap by half: without a third
// of the products 176 us, without the splitting 221.  K and V come through registers, a stage ahead, into one LDS buffer of
// 24 KB (two barriers a stage): with two buffers only three waves fit a SIMD, 235 us.
// Where something does not split (infinities, values from 2^60 on, values of V next to the lower end of the range) the workgroup starts over on
// the fp32 instructions, operands from memory.  Probabilities below 2^-112 of the row's reference keep fewer than 24 bits, those below
// 2^-126 are lost on both paths: 2.9e-6 / 3.4e-6 at 2^-112, 2.9e-6 / 1.6e-5 at 2^-117, 2.9e-6 / 3.2e-4 at 2^-122 (seen where the keys above have values of zero).
__device__ __forceinline__ uint32_t pair_bf16(float a, float b) {  // (by hand: the compiler converts once more for each part it takes out)
  uint32_t o;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(o) : "v"(a), "v"(b));
  return o;
}
// a, b -> three bf16 parts each, the nearest to what the parts before leave: 24 bits and the sign
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pair_bf16(a, b);
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  m = pair_bf16(a, b);
  a -= __uint_as_float(m << 16);
  b -= __uint_as_float(m & 0xffff0000u);
  l = pair_bf16(a, b);
}
// the largest magnitude of eight values (a NaN loses)
__device__ __forceinline__ float largest(const float4& a, const float4& b) {
  float x;
  asm("v_max3_f32 %0, |%1|, |%2|, |%3|\n\tv_max3_f32 %0, %0, |%4|, |%5|\n\tv_max3_f32 %0, %0, |%6|, |%7|\n\tv_max_f32 %0, %0, |%8|"
      : "=&v"(x) : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w));
  return x;
}
// Do three parts hold their products too?  From 2^60 on a score's or an output's partial sums may leave the range (64 products of two values
// below it reach 2^126), and what cancels in a chain of whole products does not in the parts': infinities of either sign, a NaN
// where the chain has a score of -inf.
__device__ __forceinline__ bool bounded(float largest) { return largest < 0x1p60f; }
// At the other end a part that is a subnormal bf16 number (kept by conversion and product) ends at 2^-133: three hold every value from 2^-110 on.
// Values of V: an output column may hold nothing larger, so the smallest of them counts, zeros apart.  Of queries and keys a score loses
// 2^-134 2^60 a product, which the softmax scale does not bring back up to 2^30 (launch_64).
constexpr float kSmallest = 0x1p-110f;
__device__ __forceinline__ float smallest(const float4& a, const float4& b) {  // (zeros count, a NaN does not)
  float x;
  asm("v_min3_f32 %0, |%1|, |%2|, |%3|\n\tv_min3_f32 %0, %0, |%4|, |%5|\n\tv_min3_f32 %0, %0, |%6|, |%7|\n\tv_min_f32 %0, %0, |%8|"
      : "=&v"(x) : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w));
  return x;
}
__device__ __forceinline__ bool too_small(float x) { return x != 0.f && fabsf(x) < kSmallest; }
typedef float Any4 __attribute__((ext_vector_type(4), aligned(4)));
struct Parts {
  u32x4 p[3];
};
__device__ __forceinline__ Parts split8(const float4& a, const float4& b) {
  Parts o;
  uint32_t h, m, l;
  split_pair(a.x, a.y, h, m, l);
  o.p[0][0] = h; o.p[1][0] = m; o.p[2][0] = l;
  split_pair(a.z, a.w, h, m, l);
  o.p[0][1] = h; o.p[1][1] = m; o.p[2][1] = l;
  split_pair(b.x, b.y, h, m, l);
  o.p[0][2] = h; o.p[1][2] = m; o.p[2][2] = l;
  split_pair(b.z, b.w, h, m, l);
  o.p[0][3] = h; o.p[1][3] = m; o.p[2][3] = l;
  return o;
}

__global__ __launch_bounds__(256, 4) void attn_f32_split_kernel(AttnParams p, int ngrp, int total) {
  typedef typename Mma<bf16_t>::V8 V8;
  constexpr int kPlane = 32 * 128, kStageBytes = 6 * kPlane;  // K then V: 32 rows of 64 bf16 values, three planes each
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kStageBytes];
  __shared__ __attribute__((aligned(16))) int wide[2][4];     // per wave: something it staged does not split
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = blockIdx.x, xcd = w & 7, per = total >> 3, rem = total & 7;
  const int vid = xcd * per + (xcd < rem ? xcd : rem) + (w >> 3);
  const int bh = vid / ngrp;
  const int64_t row0 = (int64_t)(vid - bh * ngrp) * 64;
  const int b = bh / p.H, h = bh - b * p.H;
  const int64_t N = p.Lk, qrow = row0 + wave * 16 + c;
  const bool live = qrow < p.Lq;
  const float* const kp = (const float*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const float* const vp = (const float*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;

  int32_t entry = -1;
  if (lane < p.K) entry = p.idx[(int64_t)b * p.sib + (int64_t)h * p.sih + row0 / 64 * p.sim + lane];
  const uint64_t listed = __ballot(entry >= 0 && (int64_t)entry * 64 < N);
  uint64_t mask = listed;
  int64_t start = 0;  // first key of the stage to be loaded next; negative: none left
  auto first = [&]() { start = mask ? (int64_t)__builtin_amdgcn_readlane(entry, __builtin_ctzll(mask)) * 64 : -1; };
  auto advance = [&]() {
    if ((start & 32) == 0 && start + 32 < N) {
      start += 32;
    } else {
      mask &= mask - 1;
      first();
    }
  };
  first();
  // The thread's eight values of a stage's K and V: dimensions 4 chunk .. + 3 and 32 + 4 chunk .. + 3, so that eight lanes load 128 bytes.
  // (Chunk by chunk this is the order of the head dimensions everywhere below: position 8 j + e is dimension 32 (e / 4) + 4 j + e % 4.)
  const int srow = tid >> 3, chunk = tid & 7;
  const uint32_t koff = ((uint32_t)srow * (uint32_t)p.skn + chunk * 4) * 4u, voff = ((uint32_t)srow * (uint32_t)p.svn + chunk * 4) * 4u;
  float4 kr[2], vr[2];
  auto load = [&]() {
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kp + start * p.skn), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vp + start * p.svn), 0, 0x7fffffff, 0x00020000);
    uint32_t ko = koff, vo = voff;
    if (__builtin_expect(start + 32 > N, 0)) {  // rows beyond the sequence re-read its last one
      const uint32_t last = (uint32_t)(N - 1 - start), row = (uint32_t)srow < last ? srow : last;
      ko = (row * (uint32_t)p.skn + chunk * 4) * 4u;
      vo = (row * (uint32_t)p.svn + chunk * 4) * 4u;
      asm volatile("" : "+v"(ko), "+v"(vo));    // (stays inside this branch)
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      kr[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rk, ko, 128 * i, 0));
      vr[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rv, vo, 128 * i, 0));
    }
  };
  if (start >= 0) load();

  const float* const qp = (const float*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh + (live ? qrow : p.Lq - 1) * p.sqm;
  V8 bq[2][3];  // B operands: lane = query, positions 32 ks + 8 g ..
  bool plain = true;
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    // (a row of q may begin at any value: 4-byte alignment)
    const float4 x = __builtin_bit_cast(float4, *reinterpret_cast<const Any4*>(qp + 16 * ks + 4 * g));
    const float4 y = __builtin_bit_cast(float4, *reinterpret_cast<const Any4*>(qp + 32 + 16 * ks + 4 * g));
    plain = plain && bounded(largest(x, y));
    const Parts q = split8(x, y);
#pragma unroll
    for (int i = 0; i < 3; i++) bq[ks][i] = b16x::frag_of<bf16_t>(q.p[i]);
  }

  const float sl2 = (float)((double)p.scale * 1.4426950408889634);
  f32x4 o[4], u[4];  // O^T: lane = query, positions 16 dt + 4 g ..; u: its small products
#pragma unroll
  for (int dt = 0; dt < 4; dt++) o[dt] = u[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m_i = -INFINITY, l_i = 0.f;

  const int r16 = srow & 15;
  const int put = (srow >> 4) * 2048 + r16 * 128 + ((chunk ^ b16x::swz(r16)) << 4);
  const int row_off = c * 128 + ((g ^ b16x::swz(c)) << 4);
  const int tr_row = 4 * g + (c >> 2), tr_off = 3 * kPlane + tr_row * 128 + ((((c & 3) >> 1) ^ b16x::swz(tr_row)) << 4) + (c & 1) * 8;

  // softmax of a stage's scores: probabilities, sums, the reference
  auto softmax = [&](f32x4 (&st)[2], int nvalid, float (&pv)[2][4]) {
    if (nvalid < 32) {  // (wave-uniform) the ragged end of the sequence
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (t * 16 + 4 * g + r >= nvalid) st[t][r] = -INFINITY;
    }
    float mx;
    asm("v_max3_f32 %0, %1, %2, %3\n\tv_max3_f32 %0, %0, %4, %5\n\tv_max3_f32 %0, %0, %6, %7\n\tv_max_f32 %0, %0, %8"
        : "=&v"(mx) : "v"(st[0][0]), "v"(st[0][1]), "v"(st[0][2]), "v"(st[0][3]), "v"(st[1][0]), "v"(st[1][1]), "v"(st[1][2]), "v"(st[1][3]));
    if (__any(mx * sl2 > m_i + kSlack)) {  // scale > 0
      mx = xh_max(fmaxf(mx, lane_xor<16>(mx))) * sl2;
      const float m_new = fmaxf(m_i, mx);
      const float alpha = m_i == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i - m_new);
      l_i *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        o[dt] *= alpha;
        u[dt] *= alpha;
      }
      m_i = m_new;
    }
    const float m_neg = m_i == -INFINITY ? 0.f : -m_i;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        pv[t][r] = __builtin_amdgcn_exp2f(fmaf(st[t][r], sl2, m_neg));
        l_i += pv[t][r];
      }
  };

  bool whole = false;  // some value does not split
  bool fits = plain;
  for (int buf = 0; start >= 0; buf ^= 1) {
    const int nvalid = (int)(N - start < 32 ? N - start : 32);
    {
      fits = fits && bounded(largest(kr[0], kr[1])) && bounded(largest(vr[0], vr[1]));
      if (__any(!(smallest(vr[0], vr[1]) >= kSmallest))) {  // (zeros, mostly)
#pragma unroll
        for (int i = 0; i < 2; i++) fits = fits && !(too_small(vr[i].x) || too_small(vr[i].y) || too_small(vr[i].z) || too_small(vr[i].w));
      }
      if (lane == 0) wide[buf][wave] = 0;
      if (!__all(fits) && lane == 0) wide[buf][wave] = 1;
      const Parts k3 = split8(kr[0], kr[1]), v3 = split8(vr[0], vr[1]);
      __syncthreads();  // the stage before is read
#pragma unroll
      for (int i = 0; i < 3; i++) {
        *reinterpret_cast<u32x4*>(lds + i * kPlane + put) = k3.p[i];
        *reinterpret_cast<u32x4*>(lds + (3 + i) * kPlane + put) = v3.p[i];
      }
    }
    advance();
    if (start >= 0) load();
    __syncthreads();
    const int4 far = *reinterpret_cast<const int4*>(wide[buf]);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(far.x | far.y | far.z | far.w) != 0, 0)) {
      whole = true;
      break;
    }
    constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};  // which parts: the small products first
    f32x4 st[2];
    st[0] = st[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; t++) {
      V8 a[2][3];
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
#pragma unroll
        for (int i = 0; i < 3; i++)
          a[ks][i] = b16x::frag_of<bf16_t>(*reinterpret_cast<const u32x4*>(lds + i * kPlane + t * 2048 + (row_off ^ (ks << 6))));
#pragma unroll
      for (int x = 0; x < 6; x++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) st[t] = b16x::mma16<bf16_t>(a[ks][kA[x]], bq[ks][kB[x]], st[t]);
    }
    settle(st[0], st[1]);
    float pv[2][4];
    softmax(st, nvalid, pv);
    const Parts pr = split8(make_float4(pv[0][0], pv[0][1], pv[0][2], pv[0][3]), make_float4(pv[1][0], pv[1][1], pv[1][2], pv[1][3]));
    V8 pb[3];
#pragma unroll
    for (int i = 0; i < 3; i++) pb[i] = b16x::frag_of<bf16_t>(pr.p[i]);
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
      V8 a[3];
#pragma unroll
      for (int i = 0; i < 3; i++) {
        unsigned char* const at = lds + i * kPlane + (tr_off ^ (dt << 5));
        Frag f;
        f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(at));
        f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(at + 2048));
        a[i] = as_v8<bf16_t>(f);
      }
#pragma unroll
      for (int x = 0; x < 5; x++) u[dt] = b16x::mma16<bf16_t>(a[kA[x]], pb[kB[x]], u[dt]);
      o[dt] = b16x::mma16<bf16_t>(a[0], pb[0], o[dt]);
    }
  }
  if (__builtin_expect(whole, 0)) {  // all of it on the fp32 instructions, operands from memory
    mask = listed;
    first();
    m_i = -INFINITY;
    l_i = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; dt++) o[dt] = u[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int vd = 4 * (c >> 3) + 32 * ((c >> 2) & 1) + (c & 3);  // of position 16 dt + c, less 8 dt
    for (; start >= 0; advance()) {
      f32x4 st[2];
      st[0] = st[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int s = 0; s < 16; s++) {
        const float q = live ? qp[4 * s + g] : 0.f;
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const int64_t row = start + t * 16 + c < N ? start + t * 16 + c : N - 1;
          st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kp[row * p.skn + 4 * s + g], q, st[t], 0, 0, 0);
        }
      }
      settle_f32(st[0], st[1]);
      float pv[2][4];
      softmax(st, (int)(N - start < 32 ? N - start : 32), pv);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int64_t key = start + (i >> 2) * 16 + 4 * g + (i & 3), row = key < N ? key : N - 1;
#pragma unroll
        for (int dt = 0; dt < 4; dt++) o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vp[row * p.svn + 8 * dt + vd], pv[i >> 2][i & 3], o[dt], 0, 0, 0);
      }
    }
  }
  asm volatile("s_nop 7\n\ts_nop 1" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
#pragma unroll
  for (int dt = 0; dt < 4; dt++) o[dt] += u[dt];

  const float l = xh_sum(l_i + lane_xor<16>(l_i));
  const int od = 32 * (g & 1) + 4 * (g >> 1);
  if (live) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if (p.merge_out != nullptr) {  // the gated merge, rounded as s3r_gated_merge does: each product, then the sum
#pragma clang fp contract(off)
      const float* const gp = (const float*)p.merge_gate + (int64_t)b * p.sgb + (int64_t)h * p.sgh + qrow * p.sgn;
      const float* const oc = (const float*)p.merge_oc + (int64_t)b * p.scb + (int64_t)h * p.sch + (qrow / 64) * p.scm + od;
      float* const to = (float*)p.merge_out + (((int64_t)b * p.Lq + qrow) * p.H + h) * 64 + od;
      const float g0 = gp[0], g1 = gp[1];
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        const float4 c4 = *reinterpret_cast<const float4*>(oc + 8 * dt);
        const float x[4] = {c4.x, c4.y, c4.z, c4.w};
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float s = o[dt][e] * inv, a0 = g0 * x[e], a1 = g1 * s;
          y[e] = a0 + a1;
        }
        *reinterpret_cast<float4*>(to + 8 * dt) = make_float4(y[0], y[1], y[2], y[3]);
      }
      return;
    }
    float* const op = (float*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh + qrow * p.som + od;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
      *reinterpret_cast<float4*>(op + 8 * dt) = make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
    if (p.lse != nullptr && g == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = log_sum(m_i, l);
  }
}

template <int W, int KS, int BLK, bool SPLIT = false> static int launch_t(const AttnParams& p, hipStream_t st) {
  const int64_t ngrp = (p.Lq + 16 * W - 1) / (16 * W);
  const int64_t total = ngrp * p.B * p.H;
  // Blocks over a whole number per CU (256) make one CU in a few work a block longer than the others: where they are so
  // few that their halves still fit one to a CU, they go in halves.  16 heads, us without and with: 1 041 tokens (16
  // blocks over) 77 / 62, 1 500 (128 over) 79 / 64; 700 tokens (176 blocks in all, whole) 36.6 / 37.0.
  const int64_t over = total & 255;
  const int64_t whole = SPLIT && over <= 128 ? total - over : total;
  const int64_t grid = whole + 2 * (total - whole);
  if (grid > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention: grid too large");
  hipLaunchKernelGGL((attn_f32_kernel<W, KS, BLK, SPLIT>), dim3((unsigned)grid), dim3(64 * W), 0, st, p, (int)ngrp, (int)total, (int)whole);
  return check_launch("attn_f32_kernel");
}

// Blocks of 64.  Up to 128 of them the fp32 instructions are the faster ones; at 176 to 384, with half blocks in the last round, they are 3 to 11 %
// slower, and stay for their scores' bits, those of a chain of fp32 products; then they take a second whole round.  16 heads, us, fp32 instructions / split values: 333 tokens (96 blocks) 16.2 /
// 19.6, 500 (128) 21.4 / 26.7, 700 (176) 38.8 / 35.0, 1 041 (272) 62.9 / 61.3, 1 500 (384) 66.5 / 63.1, 1 900 (480) 84.8 / 63.8, 2 600 (656) 118 / 82.
static int launch_64(const AttnParams& p, hipStream_t st) {
  const int64_t ngrp = (p.Lq + 63) / 64, total = ngrp * p.B * p.H;
  if (total <= 384 || p.scale > 0x1p30f) return launch_t<4, 32, 64, true>(p, st);
  if (total > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention: grid too large");
  hipLaunchKernelGGL(attn_f32_split_kernel, dim3((unsigned)total), dim3(256), 0, st, p, (int)ngrp, (int)total);
  return check_launch("attn_f32_split_kernel");
}

}  // namespace f32

int launch_attn_f32(const AttnParams& p, bool select, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  if (select) {
    if (p.block == 64) return f32::launch_64(p, st);
    if (p.block == 32) return f32::launch_t<2, 32, 32>(p, st);
    return f32::launch_t<1, 16, 16>(p, st);
  }
  // Every key for every query.  Four waves share the tiles where that still gives every CU a workgroup; below that (131
  // pooled tokens x 16 heads: 48 workgroups) single waves with tiles of their own: 0.022 ms against 0.049 ms for the
  // generic kernel, which has no such split.
  if ((p.Lq + 63) / 64 * p.B * p.H >= 256) return f32::launch_t<4, 32, 0>(p, st);
  return f32::launch_t<1, 16, 0>(p, st);
}

}  // namespace s3r
