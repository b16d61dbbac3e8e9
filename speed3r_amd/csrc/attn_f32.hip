// fp32 attention on the matrix cores (head_dim 64): the selection branch for blocks of 64, 32 and 16 tokens and the
// compressed branch with its fp32 scores.
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
#include "select_common.h"
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

template <int W, int KS, int BLK, bool SPLIT = false> static int launch_t(const AttnParams& p, hipStream_t st) {
  const int64_t ngrp = (p.Lq + 16 * W - 1) / (16 * W);
  const int64_t total = ngrp * p.B * p.H;
  // Blocks over a whole number per CU (256) make one CU in a few work a block longer than the others: where they are so
  // few that their halves still fit one to a CU, they go in halves.  16 heads, us without and with: 1 041 tokens (16
  // blocks over) 77 / 62, 1 500 (128 over) 79 / 64, 4 164 (32) 177 / 163, 8 328 (48) 307 / 292; 2 600 (144 over) 111.8 / 112.9,
  // 700 tokens (176 blocks in all) 36.6 / 37.0.  All blocks in halves: 8 328 tokens 325.
  const int64_t over = total & 255;
  const int64_t whole = SPLIT && over <= 128 ? total - over : total;
  const int64_t grid = whole + 2 * (total - whole);
  if (grid > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention: grid too large");
  hipLaunchKernelGGL((attn_f32_kernel<W, KS, BLK, SPLIT>), dim3((unsigned)grid), dim3(64 * W), 0, st, p, (int)ngrp, (int)total, (int)whole);
  return check_launch("attn_f32_kernel");
}

}  // namespace f32

int launch_attn_f32(const AttnParams& p, bool select, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  if (select) {
    if (p.block == 64) return f32::launch_t<4, 32, 64, true>(p, st);
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
