// Backward of the selection attention for 16-token blocks (bf16 / fp16 I/O, head_dim 64): same mathematics, inputs and
// outputs as the kernels of attn_bwd.hip (references there), which serve 64-token blocks and the dense branch.
//
// Built from 16 x 16 products (v_mfma_f32_16x16x32 over the head dimension, 16x16x16 or 16x16x32 over the rows): a list entry
// is a whole product, nothing is computed for pairs of blocks that no list names.  (The kernels before these put two listed
// blocks and four query blocks into 32 x 32 products, of which lists that share little fill a quarter.)
//   * bwd16_dq_kernel: two query blocks a wave.  S^T = K Q^T and dP^T = V dO^T put one query per lane (column lane % 16, keys
//     4 (lane / 16) + r), so lse and delta are per-lane scalars and the rounded dS^T is already the B operand of
//     dQ^T += K^T dS^T, whose A operand comes from ds_read_b64_tr_b16.  The wave walks the union of the two lists: a block
//     is fetched and read from LDS once and scored against the query blocks that list it.
//   * bwd16_dkdv_kernel: one key block a wave, two query blocks of its list a step.  S = Q K^T and dP = dO V^T put one key
//     per lane; dV^T += dO^T P, dK^T += Q^T dS.
// Rows go global -> LDS by direct transfers, two steps in flight: a step reads all its operands into registers, requests
// the step after next into the same buffers and computes meanwhile; nothing else is pipelined, the other waves of the
// SIMD fill the gaps.
// Bound: the address unit on the way from the vector cache into the LDS.  Counters, layer features, 2 x 12 096 tokens, 16 heads, top-32,
// dQ / dK/dV: that unit busy 81 / 74 %, vector port 38 / 28 %, matrix cores 26 / 19 %, LDS reads 21 / 23 %, 90 / 83 % of the requests
// served by the L2.
// us, 16 heads, top-32, before / now: layer features, 24 192 tokens: dQ 304 / 141, dK/dV 504 / 234; 4 032 tokens 74 / 34 and
// 115 / 62; video (lists of neighbours that agree), 96 768 tokens: 577 / 467 and 1 317 / 863, 24 192: 160 / 113 and 381 / 229.
#include "block16.h"
#include "attn_bwd.h"

namespace s3r {
namespace bwd16 {
using namespace b16x;

// Row fragments of a pair in two tensors' buffers (x: [block][k-step]): lane = row lane % 16, chunk 4 ks + lane / 16.
// `row` = the lane's byte offset for k-step 0; the k-step flips chunk bit 2.  Reads and wait are one statement: the compiler
// neither adds waits for the transfers in flight nor moves a register whose value has not arrived.
__device__ __forceinline__ void read_rows(uint32_t a, uint32_t b, u32x4 (&x)[2][2], u32x4 (&y)[2][2]) {
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %8 offset:2048\n\tds_read_b128 %3, %9 offset:2048\n\t"
      "ds_read_b128 %4, %10\n\tds_read_b128 %5, %11\n\tds_read_b128 %6, %10 offset:2048\n\tds_read_b128 %7, %11 offset:2048\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(y[0][0]), "=&v"(y[0][1]), "=&v"(y[1][0]), "=&v"(y[1][1])
      : "v"(a), "v"(a ^ 64u), "v"(b), "v"(b ^ 64u)
      : "memory");
}
// Transposed fragments of a pair in two tensors' buffers (t: [dim tile][block]): lane = head dimension 16 dt + lane % 16, rows
// 4 (lane / 16) .. + 3.  The tile flips chunk bits 1 and 2 of the lane's byte offset.
__device__ __forceinline__ void read_cols2(uint32_t a, uint32_t b, u32x2 (&t)[4][2], u32x2 (&s)[4][2]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %1, %16 offset:2048\n\tds_read_b64_tr_b16 %2, %17\n\tds_read_b64_tr_b16 %3, %17 offset:2048\n\t"
      "ds_read_b64_tr_b16 %4, %18\n\tds_read_b64_tr_b16 %5, %18 offset:2048\n\tds_read_b64_tr_b16 %6, %19\n\tds_read_b64_tr_b16 %7, %19 offset:2048\n\t"
      "ds_read_b64_tr_b16 %8, %20\n\tds_read_b64_tr_b16 %9, %20 offset:2048\n\tds_read_b64_tr_b16 %10, %21\n\tds_read_b64_tr_b16 %11, %21 offset:2048\n\t"
      "ds_read_b64_tr_b16 %12, %22\n\tds_read_b64_tr_b16 %13, %22 offset:2048\n\tds_read_b64_tr_b16 %14, %23\n\tds_read_b64_tr_b16 %15, %23 offset:2048\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(t[0][0]), "=&v"(t[0][1]), "=&v"(t[1][0]), "=&v"(t[1][1]), "=&v"(t[2][0]), "=&v"(t[2][1]), "=&v"(t[3][0]), "=&v"(t[3][1]),
        "=&v"(s[0][0]), "=&v"(s[0][1]), "=&v"(s[1][0]), "=&v"(s[1][1]), "=&v"(s[2][0]), "=&v"(s[2][1]), "=&v"(s[3][0]), "=&v"(s[3][1])
      : "v"(a), "v"(a ^ 32u), "v"(a ^ 64u), "v"(a ^ 96u), "v"(b), "v"(b ^ 32u), "v"(b ^ 64u), "v"(b ^ 96u)
      : "memory");
}

// The transfers of a step's two blocks in two tensors of the same rows.  a < 0: no step (the same instructions, nothing is
// fetched, so that the waits are constants); b2 < 0: no second block, the first one again (finite values).
template <typename E, bool WIDE>
__device__ __forceinline__ void fetch_pair(const Rows<E, WIDE>& x, const Rows<E, WIDE>& y, int32_t a, int32_t b2, LdsPtr xb, LdsPtr yb, int lane) {
  int32_t rec, first;
  records(a, rec, first);
  const int32_t second = b2 < 0 ? first : b2;
  if (__builtin_expect(first == x.ragged || second == x.ragged, 0)) {
    x.template fetch<true>(first, rec, xb, lane);
    x.template fetch<true>(second, rec, xb + 2048, lane);
    y.template fetch<true>(first, rec, yb, lane);
    y.template fetch<true>(second, rec, yb + 2048, lane);
  } else {
    x.template fetch<false>(first, rec, xb, lane);
    x.template fetch<false>(second, rec, xb + 2048, lane);
    y.template fetch<false>(first, rec, yb, lane);
    y.template fetch<false>(second, rec, yb + 2048, lane);
  }
}
// No probability for rows (registers 4 (lane / 16) + r of a block) beyond the end, nor for a missing second block
template <typename E, bool WIDE>
__device__ __forceinline__ void mask_scores(f32x4 (&st)[2], const Rows<E, WIDE>& x, int32_t a, int32_t b2, int g) {
  if (__builtin_expect(b2 < 0 || a == x.ragged || b2 == x.ragged, 0)) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int32_t blk = s ? b2 : a;
      const int end = blk < 0 ? -1 : blk == x.ragged ? x.last : 15;
#pragma unroll
      for (int r = 0; r < 4; r++) st[s][r] = 4 * g + r > end ? -INFINITY : st[s][r];
    }
  }
}

// acc[dt][r] of lane (row lane % 16): head dimension 16 dt + 4 (lane / 16) + r
template <typename E> __device__ __forceinline__ void store_rows(const f32x4 (&acc)[4], E* row, int g) {
#pragma unroll
  for (int dt = 0; dt < 4; dt++) {
    union { E e[4]; uint2 u; } o;
#pragma unroll
    for (int r = 0; r < 4; r++) o.e[r] = (E)acc[dt][r];
    *reinterpret_cast<uint2*>(row + 16 * dt + 4 * g) = o.u;
  }
}

constexpr int kVm10 = 0x0F7A, kVm0 = 0x0F70;

// ---- dQ ----------------------------------------------------------------------------------------------------------
// The operands of a block in a slot (K rows, V rows behind them) and two entries of the walk list
__device__ __forceinline__ void read_block(uint32_t row, uint32_t tr, uint32_t now, uint32_t ahead, u32x4 (&k)[2], u32x4 (&v)[2], u32x2 (&t)[4],
                                           u32x2& e_now, u32x2& e_ahead) {
  asm volatile(
      "ds_read_b64 %8, %14\n\tds_read_b64 %9, %15\n\t"
      "ds_read_b128 %0, %10\n\tds_read_b128 %1, %11\n\tds_read_b128 %2, %10 offset:2048\n\tds_read_b128 %3, %11 offset:2048\n\t"
      "ds_read_b64_tr_b16 %4, %12\n\tds_read_b64_tr_b16 %5, %13\n\tds_read_b64_tr_b16 %6, %16\n\tds_read_b64_tr_b16 %7, %17\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0]), "=&v"(k[1]), "=&v"(v[0]), "=&v"(v[1]), "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(e_now), "=&v"(e_ahead)
      : "v"(row), "v"(row ^ 64u), "v"(tr), "v"(tr ^ 32u), "v"(now), "v"(ahead), "v"(tr ^ 64u), "v"(tr ^ 96u)
      : "memory");
}
// Query blocks per wave and blocks in its LDS.  Two and two fit four waves on a SIMD (121 registers, 9 KB each), which hides
// more than longer prefetches or larger unions do.  us, dQ alone, 16 heads, top-32: layer features, 24 192 tokens / 4 032, video,
// 96 768 / 24 192 tokens: four query blocks and four slots 166 / 48 / 438 / 115, four and three 158 / 48 / 434 / 115, two and
// four 164 / 35 / 507 / 130, two and three 151 / 35 / 487 / 120, two and two 141 / 34 / 467 / 113; one wave per query block,
// pairs of list entries: 185 / - / 693 / -.  Before (32 x 32 products on the union of four lists): 304 / 74 / 577 / 160.
constexpr int kSlots = 2, kNQ = 2;

// DELTA: rowsum(dO * O) from O rows loaded beside those of dO, instead of from a kernel that reads both.  dQ, dK and dV with that kernel / this
// way, us, random lists of 32: 8 064 tokens 132.5 / 125.6, 24 192 416 / 402, 96 768 3 112 / 3 075.
template <typename E, bool WIDE, bool DELTA>
__global__ __launch_bounds__(64, 4) void bwd16_dq_kernel(BwdParams p, int nqb, int ngrp, int total) {
  typedef typename Mma<E>::V8 V8;
  typedef typename Mma4<E>::V4 V4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_slots[kSlots * kPair];
  __shared__ __attribute__((aligned(16))) int2 walk[64 * kNQ + kSlots];
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int vid = work_item(blockIdx.x, total);
  // (divisions run on the vector unit; the descriptors below want their results in scalar registers)
  const int bh = __builtin_amdgcn_readfirstlane(vid / ngrp), grp = vid - bh * ngrp;
  const int b = __builtin_amdgcn_readfirstlane(bh / p.H), h = bh - b * p.H;

  // the lists head the longest chain of the start: first in the queue
  const int32_t* lists = p.idx + (int64_t)b * p.sib + (int64_t)h * p.sih + (int64_t)grp * kNQ * p.sim;
  asm volatile("" : "+s"(lists));  // (computed ahead of the lanes' branch: b and h stay in scalar registers)
  int32_t mine[kNQ];
#pragma unroll
  for (int j = 0; j < kNQ; j++) {
    mine[j] = -1;
    if (grp * kNQ + j < nqb && lane < p.K) mine[j] = lists[(int64_t)j * p.sim + lane];
  }
  const int64_t row0 = (int64_t)grp * (16 * kNQ) + c;
  const E* qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh + 8 * g;
  const E* gp = (const E*)p.dout + (int64_t)b * p.sgb + (int64_t)h * p.sgh + 8 * g;
  const int64_t stat = ((int64_t)b * p.H + h) * p.Lq;
  V8 bq[kNQ][2], bg[kNQ][2];  // B operands of the query blocks: lane = query, head dimensions 32 ks + 8 g ..
  float nlse[kNQ], dls[kNQ];
#pragma unroll
  for (int j = 0; j < kNQ; j++) {
    const int64_t row = row0 + 16 * j;
    const bool live = row < p.Lq;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      Frag f, d;
      f.u = d.u = make_uint4(0, 0, 0, 0);
      if (live) {
        f.u = *reinterpret_cast<const uint4*>(qp + row * p.sqm + 32 * ks);
        d.u = *reinterpret_cast<const uint4*>(gp + row * p.sgm + 32 * ks);
      }
      bq[j][ks] = as_v8<E>(f);
      bg[j][ks] = as_v8<E>(d);
    }
    nlse[j] = live ? -p.lse[stat + row] * kLog2e : -INFINITY;
    if constexpr (DELTA) {
      const E* const op = (const E*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh + 8 * g;
      float part[2] = {0.f, 0.f};
      if (live) {
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          const u32x4 ov = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(op + row * p.som + 32 * ks));
          const E* const oe = reinterpret_cast<const E*>(&ov);
#pragma unroll
          for (int e = 0; e < 8; e++) part[ks] = fmaf((float)oe[e], (float)bg[j][ks][e], part[ks]);
        }
      }
      const float t = sum_step<32>(sum_step<16>(part[0] + part[1]));
      if (live && g == 0) p.delta_out[stat + row] = t;
      dls[j] = t * p.scale;
    } else {
      dls[j] = live ? p.delta[stat + row] * p.scale : 0.f;
    }
  }

  bool dup;  // some list names a block more than once (wave-uniform)
  const int n = walk_list<kNQ>(mine, p.Lk, lds_slots, walk, kSlots, lane, dup);

  const Rows<E, WIDE> kr(p.k, (int64_t)b * p.skb + (int64_t)h * p.skh, p.skn, p.Lk, lane);
  const Rows<E, WIDE> vr(p.v, (int64_t)b * p.svb + (int64_t)h * p.svh, p.svn, p.Lk, lane);
  const LdsPtr slots = (LdsPtr)lds_slots;
  const uint32_t row_off = lds_addr(slots) + (uint32_t)(c * 128 + ((g ^ swz(c)) << 4));
  const int tr_row = 4 * g + (c >> 2);
  const uint32_t tr_off = lds_addr(slots) + (uint32_t)(tr_row * 128 + ((((c & 3) >> 1) ^ swz(tr_row)) << 4) + (c & 1) * 8);
  const uint32_t walk_at = lds_addr((LdsPtr)reinterpret_cast<char*>(walk));
  const float scale = p.scale, sl2 = scale * kLog2e;

  f32x4 dq[kNQ][4];
#pragma unroll
  for (int j = 0; j < kNQ; j++)
#pragma unroll
    for (int dt = 0; dt < 4; dt++) dq[j][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  auto request = [&](int32_t blk, int slot) {  // four transfers
    int32_t rec, some;
    records(blk, rec, some);
    const LdsPtr dst = slots + slot * kPair;
    if (__builtin_expect(some == kr.ragged, 0)) {
      kr.template fetch<true>(some, rec, dst, lane);
      vr.template fetch<true>(some, rec, dst + 2048, lane);
    } else {
      kr.template fetch<false>(some, rec, dst, lane);
      vr.template fetch<false>(some, rec, dst + 2048, lane);
    }
  };
#pragma unroll
  for (int s = 0; s < kSlots; s++) request(s < n ? __builtin_amdgcn_readfirstlane(walk[s].x) : -1, s);
  int slot = -1;
  for (int i = 0; i < n; i++) {
    slot = slot + 1 == kSlots ? 0 : slot + 1;
    u32x4 kw[2], vw[2];
    u32x2 kt[4], now, ahead;
    __builtin_amdgcn_s_waitcnt(0x0F70 | (4 * (kSlots - 1)));  // this block's transfers have landed, the next ones' may be in flight
    read_block(row_off + slot * kPair, tr_off + slot * kPair, walk_at + 8u * i, walk_at + 8u * (i + kSlots), kw, vw, kt, now, ahead);
    const int32_t blk = __builtin_amdgcn_readfirstlane((int32_t)now[0]);
    const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)now[1]);
    const bool rare = dup || blk == kr.ragged;
    request(__builtin_amdgcn_readfirstlane((int32_t)ahead[0]), slot);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kNQ; j++) {
      const uint32_t w = (cnt >> (8 * j)) & 0xffu;
      if (w != 0) {
        f32x4 st = {0.f, 0.f, 0.f, 0.f}, dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          st = mma16<E>(frag_of<E>(kw[ks]), bq[j][ks], st);
          dp = mma16<E>(frag_of<E>(vw[ks]), bg[j][ks], dp);
        }
        settle(st, dp);
        float nl = nlse[j];
        if (__builtin_expect(rare, 0)) {
          nl += __builtin_amdgcn_logf((float)w);  // a block listed w times weighs w times
          const int end = blk == kr.ragged ? kr.last : 15;
#pragma unroll
          for (int r = 0; r < 4; r++) st[r] = 4 * g + r > end ? -INFINITY : st[r];
        }
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; r++) e[r] = __builtin_amdgcn_exp2f(fmaf(st[r], sl2, nl)) * fmaf(dp[r], scale, -dls[j]);  // scale * P * (dP - delta)
        const V4 ds = pack4<E>(e);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) dq[j][dt] = Mma4<E>::mma(kt[dt], ds, dq[j][dt]);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(kVm0);
  E* out = (E*)p.dq + (int64_t)b * p.sdqb + (int64_t)h * p.sdqh;
#pragma unroll
  for (int j = 0; j < kNQ; j++) {
    const int64_t row = row0 + 16 * j;
    if (row < p.Lq) store_rows<E>(dq[j], out + row * p.sdqm, g);
  }
}

// ---- dK, dV ------------------------------------------------------------------------------------------------------
// One key block a wave: lists differ in length (layer features: mean 32, one in a thousand 250 and more), and a wave with two
// of them, merged, was slower everywhere but on long videos (24 192 tokens 282 us against 234, 96 768 of a video 839 against
// 863).  One query block a step in half the LDS, four waves a SIMD: 239 and 945.
template <typename E, bool WIDE>
__global__ __launch_bounds__(64, 2) void bwd16_dkdv_kernel(BwdParams p, int nkb, int total) {
  typedef typename Mma<E>::V8 V8;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_q0[kPair], lds_q1[kPair], lds_g0[kPair], lds_g1[kPair];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_s0[512], lds_s1[512];  // 64 lse and 64 delta of a pair (32 queries, twice)
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  // Two passes over the key blocks: those whose lists are long start first.
  const bool long_pass = (int)blockIdx.x < total;
  const int vid = work_item(long_pass ? (int)blockIdx.x : (int)blockIdx.x - total, total);
  // (divisions run on the vector unit; the descriptors below want their results in scalar registers)
  const int bh = __builtin_amdgcn_readfirstlane(vid / nkb), kb = vid - bh * nkb;
  const int b = __builtin_amdgcn_readfirstlane(bh / p.H), h = bh - b * p.H;
  const int32_t* off = p.kq_off + (int64_t)bh * (nkb + 1) + kb;
  const int32_t lo = __builtin_amdgcn_readfirstlane(off[0]);
  const int n = __builtin_amdgcn_readfirstlane(off[1]) - lo;
  if ((n > 4 * p.K) != long_pass) return;
  const int32_t* list = p.kq_list + (int64_t)bh * p.list_stride + lo;
  // list entries 64 at a time, one per lane; the wait is inside, so that no later one is needed
  int32_t held = -1;
  int at = 0;
  auto refill = [&]() {
    held = -1;
    if (at + lane < n) held = list[at + lane];
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(held));
  };
  refill();
  auto next = [&]() -> int32_t {  // -1: none left
    if (at >= n) return -1;
    const int32_t e = __builtin_amdgcn_readlane(held, at & 63);
    at++;
    if ((at & 63) == 0) refill();
    return e;
  };

  const int64_t key = (int64_t)kb * 16 + c;
  const bool live = key < p.Lk;
  const E* kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh + key * p.skn + 8 * g;
  const E* vp = (const E*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh + key * p.svn + 8 * g;
  V8 bk[2], bv[2];  // B operands: lane = key, head dimensions 32 ks + 8 g ..
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    Frag f, d;
    f.u = d.u = make_uint4(0, 0, 0, 0);
    if (live) {
      f.u = *reinterpret_cast<const uint4*>(kp + 32 * ks);
      d.u = *reinterpret_cast<const uint4*>(vp + 32 * ks);
    }
    bk[ks] = as_v8<E>(f);
    bv[ks] = as_v8<E>(d);
  }
  const Rows<E, WIDE> qr(p.q, (int64_t)b * p.sqb + (int64_t)h * p.sqh, p.sqm, p.Lq, lane);
  const Rows<E, WIDE> gr(p.dout, (int64_t)b * p.sgb + (int64_t)h * p.sgh, p.sgm, p.Lq, lane);
  const float* lsep = p.lse + (int64_t)bh * p.Lq;
  const float* dlp = p.delta + (int64_t)bh * p.Lq;
  const uint32_t row_off = (uint32_t)(c * 128 + ((g ^ swz(c)) << 4));
  const int tr_row = 4 * g + (c >> 2);
  const uint32_t tr_off = (uint32_t)(tr_row * 128 + ((((c & 3) >> 1) ^ swz(tr_row)) << 4) + (c & 1) * 8);
  const float scale = p.scale, sl2 = scale * kLog2e;
  constexpr bool LATE_SCALE = std::is_same<E, bf16_t>::value;  // the softmax scale goes onto dK at the end (fp16: onto dS, its range is narrow)

  f32x4 dk[4], dv[4];
#pragma unroll
  for (int dt = 0; dt < 4; dt++) dk[dt] = dv[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  auto request = [&](int32_t a, int32_t b2, LdsPtr qb, LdsPtr gb, LdsPtr sb) {  // ten transfers
    fetch_pair(qr, gr, a, b2, qb, gb, lane);
    // lanes 0..15 and 32..47: rows of the first block, the others of the second
    int32_t rec, first;
    records(a, rec, first);
    const int32_t second = b2 < 0 ? first : b2;
    uint32_t r = (uint32_t)((lane & 16) ? second : first) * 16u + (uint32_t)c;
    r = r < (uint32_t)p.Lq ? r : (uint32_t)p.Lq - 1u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)lsep, 0, rec, 0x00020000), sb, 4, r * 4u, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)dlp, 0, rec, 0x00020000), sb + 256, 4, r * 4u, 0, 0, 0);
  };
  auto step = [&](LdsPtr qb, LdsPtr gb, LdsPtr sb, int32_t& a, int32_t& b2) {
    const int32_t ca = a, cb = b2;
    u32x4 qw[2][2], gw[2][2];
    u32x2 gt[4][2], qt[4][2];
    f32x4 ls[2], dl[2];
    __builtin_amdgcn_s_waitcnt(kVm10);  // this step's transfers have landed, the next step's may be in flight
    read_rows(lds_addr(qb) + row_off, lds_addr(gb) + row_off, qw, gw);
    f32x4 st[2], dp[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
      st[s] = dp[s] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        st[s] = mma16<E>(frag_of<E>(qw[s][ks]), bk[ks], st[s]);
        dp[s] = mma16<E>(frag_of<E>(gw[s][ks]), bv[ks], dp[s]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:64\n\tds_read_b128 %2, %4 offset:256\n\tds_read_b128 %3, %4 offset:320\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(ls[0]), "=&v"(ls[1]), "=&v"(dl[0]), "=&v"(dl[1])
        : "v"(lds_addr(sb) + 16u * (uint32_t)g)
        : "memory");
    read_cols2(lds_addr(gb) + tr_off, lds_addr(qb) + tr_off, gt, qt);
    a = next();
    b2 = next();
    request(a, b2, qb, gb, sb);
    __builtin_amdgcn_sched_barrier(0);
    mask_scores(st, qr, ca, cb, g);
    V8 pr, ds;
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float x = __builtin_amdgcn_exp2f(fmaf(st[s][r], sl2, ls[s][r] * -kLog2e));
        pr[4 * s + r] = (E)x;
        const float d = dp[s][r] - dl[s][r];
        ds[4 * s + r] = (E)(LATE_SCALE ? x * d : x * (d * scale));
      }
    }
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
      dv[dt] = mma16<E>(frag_of<E>(gt[dt][0], gt[dt][1]), pr, dv[dt]);
      dk[dt] = mma16<E>(frag_of<E>(qt[dt][0], qt[dt][1]), ds, dk[dt]);
    }
  };
  int32_t a0 = next(), b0 = next(), a1 = next(), b1 = next();
  request(a0, b0, (LdsPtr)lds_q0, (LdsPtr)lds_g0, (LdsPtr)lds_s0);
  request(a1, b1, (LdsPtr)lds_q1, (LdsPtr)lds_g1, (LdsPtr)lds_s1);
  while (a0 >= 0) {
    step((LdsPtr)lds_q0, (LdsPtr)lds_g0, (LdsPtr)lds_s0, a0, b0);
    if (a1 < 0) break;
    step((LdsPtr)lds_q1, (LdsPtr)lds_g1, (LdsPtr)lds_s1, a1, b1);
  }
  __builtin_amdgcn_s_waitcnt(kVm0);
  if (!live) return;
  if constexpr (LATE_SCALE) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) dk[dt] *= scale;
  }
  store_rows<E>(dk, (E*)p.dk + (int64_t)b * p.sdkb + (int64_t)h * p.sdkh + key * p.sdkn, g);
  store_rows<E>(dv, (E*)p.dv + (int64_t)b * p.sdvb + (int64_t)h * p.sdvh + key * p.sdvn, g);
}

}  // namespace bwd16

int launch_attn_bwd16(const BwdParams& p, int dtype, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  const int64_t nqb = (p.Lq + 15) / 16, nkb = (p.Lk + 15) / 16;
  const int64_t ngrp = (nqb + bwd16::kNQ - 1) / bwd16::kNQ;
  const int64_t total_q = ngrp * p.B * p.H, total_k = nkb * p.B * p.H;
  if (total_q > 0x7fffffffLL || 2 * total_k > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention backward: grid too large");
  auto far = [](int64_t len, int64_t row) { return (len - 1) * row * 2 + 128 > 0xffffffffLL; };
  const bool wide = far(p.Lk, p.skn) || far(p.Lk, p.svn) || far(p.Lq, p.sqm) || far(p.Lq, p.sgm);
#define S3R_BWD16(E, W)                                                                                                                      \
  do {                                                                                                                                       \
    if (p.dq != nullptr && p.o != nullptr)                                                                                                   \
      hipLaunchKernelGGL((bwd16::bwd16_dq_kernel<E, W, true>), dim3((unsigned)total_q), dim3(64), 0, st, p, (int)nqb, (int)ngrp, (int)total_q); \
    else if (p.dq != nullptr)                                                                                                                \
      hipLaunchKernelGGL((bwd16::bwd16_dq_kernel<E, W, false>), dim3((unsigned)total_q), dim3(64), 0, st, p, (int)nqb, (int)ngrp, (int)total_q); \
    if (p.dk != nullptr)                                                                                                                     \
      hipLaunchKernelGGL((bwd16::bwd16_dkdv_kernel<E, W>), dim3((unsigned)(2 * total_k)), dim3(64), 0, st, p, (int)nkb, (int)total_k);        \
  } while (0)
  if (dtype == S3R_BF16) { if (wide) S3R_BWD16(bf16_t, true); else S3R_BWD16(bf16_t, false); }
  else { if (wide) S3R_BWD16(f16_t, true); else S3R_BWD16(f16_t, false); }
#undef S3R_BWD16
  return check_launch("attention backward");
}

}  // namespace s3r
