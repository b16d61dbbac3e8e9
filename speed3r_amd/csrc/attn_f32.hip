// fp32 attention on the matrix cores (head_dim 64): the selection branch for blocks of 64, 32 and 16 tokens and the
// compressed branch with its fp32 scores.
//
// Bound: the fp32 matrix instructions (v_mfma_f32_16x16x4_f32: 64 FLOP per cycle and SIMD, 157 TFLOP/s; a product of
// 8192 x 8192 matrices by the library reaches 154).  At 8 328 tokens x 16 heads, 16 blocks of 64 (3.5e10 FLOP, 0.23 ms)
// the generic kernel, whose vector FMAs wait for one LDS read per four products, takes 1.36 ms, this one 0.34 ms; at
// 16-token blocks, top-32, 4.8 and 0.24 ms.  What is left: 38 us per 1 041 tokens = 73 % of the matrix rate (the vector
// instructions of the softmax do not overlap with it fully) plus 45 us for the last wave of a SIMD.
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

constexpr int kRow = 256;  // bytes of a K or V row

// exp(x) for x <= 0 to about one unit in the last place: exp2 of the product x log2(e), corrected by what its rounding
// left out (without the correction the error grows with |x|).  Arguments below -200 (exp is 0 from -104 on) give 0.
__device__ __forceinline__ float exp_nonpos(float x) {
  constexpr float kHi = 1.44269502f, kLo = 1.92596303e-8f, kLn2 = 0.693147181f;  // log2(e) = kHi + kLo
  x = x < -200.f ? -200.f : x;
  const float t = x * kHi;
  const float e = fmaf(x, kLo, fmaf(x, kHi, -t));
  const float y = __builtin_amdgcn_exp2f(t);
  return fmaf(y, e * kLn2, y);
}

// W waves share a workgroup's 16 W query rows and its stages of KS keys.  SELECT: the rows are one query block of 16 W
// tokens, the stages the parts of its listed key blocks; otherwise every key.
template <int W, int KS, int BLK>
__global__ __launch_bounds__(64 * W, 4) void attn_f32_kernel(AttnParams p, int ngrp, int total) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k0[KS * kRow], lds_k1[KS * kRow];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v0[KS * kRow], lds_v1[KS * kRow];
  constexpr bool SELECT = BLK > 0;
  constexpr int SUB = SELECT ? BLK / KS : 1, NG = KS / 16, NI = KS / (4 * W);
  static_assert(!SELECT || (BLK % KS == 0 && BLK % (16 * W) == 0), "a block is a whole number of stages and of workgroups");
  static_assert(NI * 4 * W == KS, "every wave moves the same number of 1 KB pieces");

  const int wave = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  // each XCD takes a contiguous range of query blocks: neighbours list mostly the same key blocks
  const int w = blockIdx.x;
  const int xcd = w & 7, per = total >> 3, rem = total & 7;
  const int vid = xcd * per + (xcd < rem ? xcd : rem) + (w >> 3);
  const int bh = vid / ngrp;
  const int64_t row0 = (int64_t)(vid - bh * ngrp) * (16 * W);
  const int b = bh / p.H;
  const int h = bh - b * p.H;

  const int64_t N = p.Lk;
  const int64_t qrow = row0 + wave * 16 + c;
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

  f32x4 o[4];
#pragma unroll
  for (int dg = 0; dg < 4; dg++)
#pragma unroll
    for (int r = 0; r < 4; r++) o[dg][r] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;

  auto compute = [&](int64_t s0, const unsigned char* kb, const unsigned char* vb) {
    const int nvalid = (int)(N - s0 < KS ? N - s0 : KS);
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
    if (nvalid < KS) {  // (wave-uniform) the ragged end of the sequence
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
    mx = xh_max(fmaxf(mx, lane_xor<16>(mx))) * p.scale;  // scale > 0: the maximum of the scaled scores
    const float m_new = fmaxf(m_i, mx);
    if (__any(m_new != m_i)) {
      const float alpha = m_i == -INFINITY ? 0.f : exp_nonpos(m_i - m_new);
      l_i *= alpha;
#pragma unroll
      for (int dg = 0; dg < 4; dg++)
#pragma unroll
        for (int r = 0; r < 4; r++) o[dg][r] *= alpha;
    }
    m_i = m_new;
    const float m_neg = m_new == -INFINITY ? 0.f : -m_new;
#pragma unroll
    for (int kg = 0; kg < NG; kg++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float pv = exp_nonpos(fmaf(st[kg][r], p.scale, m_neg));
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
  first();
  if (start >= 0) {
    request(start, lds_k0, lds_v0);
    while (true) {
      int64_t cur = start;
      advance();
      ready();
      if (start >= 0) request(start, lds_k1, lds_v1);
      compute(cur, lds_k0, lds_v0);
      if (start < 0) break;
      cur = start;
      advance();
      ready();
      if (start >= 0) request(start, lds_k0, lds_v0);
      compute(cur, lds_k1, lds_v1);
      if (start < 0) break;
    }
  }

  const float l = xh_sum(l_i + lane_xor<16>(l_i));
  if (live) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    float* op = (float*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh + qrow * p.som + 16 * g;
#pragma unroll
    for (int r = 0; r < 4; r++)
      *reinterpret_cast<float4*>(op + 4 * r) = make_float4(o[0][r] * inv, o[1][r] * inv, o[2][r] * inv, o[3][r] * inv);
    if (p.lse != nullptr && g == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = l > 0.f ? m_i + logf(l) : -INFINITY;
  }
}

template <int W, int KS, int BLK> static int launch_t(const AttnParams& p, hipStream_t st) {
  const int64_t ngrp = (p.Lq + 16 * W - 1) / (16 * W);
  const int64_t total = ngrp * p.B * p.H;
  if (total > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention: grid too large");
  hipLaunchKernelGGL((attn_f32_kernel<W, KS, BLK>), dim3((unsigned)total), dim3(64 * W), 0, st, p, (int)ngrp, (int)total);
  return check_launch("attn_f32_kernel");
}

}  // namespace f32

int launch_attn_f32(const AttnParams& p, bool select, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  if (select) {
    if (p.block == 64) return f32::launch_t<4, 32, 64>(p, st);
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
