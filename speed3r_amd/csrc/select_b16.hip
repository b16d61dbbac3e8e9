// Selection-branch attention for 16-token blocks on the gfx950 matrix cores (bf16 / fp16 I/O, head_dim 64):
// the reference layer's own setting, block_size**2 = 16 with 32 blocks per query block
// (pi3/models/layers/sparse_attention.py:73,98,125; kernel topk_blocksparse_attention.py:35-128).
//
// select_b16_kernel: one wave owns NQ consecutive query blocks (1, 2 or 4) of one head and walks the union of their lists, a
// distinct key block a step: its K and V rows are fetched and read from LDS once and scored against the query blocks that
// list it, in 16 x 16 products (S^T = K Q^T with v_mfma_f32_16x16x32, one query per lane and four keys; P rounded to the I/O
// type is the B operand of O^T += V^T P^T with v_mfma_f32_16x16x16, V^T from ds_read_b64_tr_b16).  Nothing is computed for a
// pair of blocks that no list names.  Two steps are in flight: a step reads its operands into registers, requests the block
// after next into the same slot and computes meanwhile; the other waves of the SIMD fill the gaps.  One wave per workgroup
// (unions differ in size, a workgroup holds its slots until its slowest wave ends).
// Bound (counters, 16 heads, top-32, NQ 4): lists that share little (layer features, 2 x 12 096 tokens) the address unit on the way
// from the vector cache into the LDS, busy 73 % (vector port 36 %, matrix cores 22 %); lists of neighbours that agree (video, 266 496
// tokens) the vector port, 67 %, beside it (65 %; matrix cores 40 %).
// NQ, us, 16 heads (the kernel before this one, 32 x 32 products over unions of four lists / 1 / 2 / 4): layer features, top-32,
// 2 016 tokens 40 / 18.5 / 26 / 41, 4 032 42 / 28 / 30.5 / 45, 8 064 63 / 52 / 50 / 58, 16 128 111 / 97 / 86 / 105, 24 192 152 / 136 / 120 /
// 115, 32 256 218 / 198 / 186 / 177, 100 800 824 / 878 / 847 / 830; video (neighbours' lists agree) 4 164 34.5 / 29 / 29.5 / 36, 16 656
// 81 / 95 / 75 / 78, 66 624 top-16 191 / 251 / 184 / 163, 266 496 top-32 1 009 / 1 617 / 1 095 / 902.  Few query blocks need many waves,
// many of them gain from what their lists share: the lines below lie between those sizes.
//
// select_b16_pairs_kernel (S3R_B16_KERNEL=pairs, cross-check): a tile pairs TWO query blocks with ONE list entry of each, rows
// 0-15 of the 32-row tile hold the block the first query block lists at position i, rows 16-31 the block the second one lists
// there; S^T = K Q^T with v_mfma_f32_32x32x16 then has two useful 16x16 quadrants, the other two are masked to probability
// zero; online softmax on the 8 own registers.
// Entries < 0 or starting at or beyond N are skipped, keys beyond N in the ragged last block are masked, a query
// block with no valid entry gives zeros; up to 64 entries per query block.
#include "block16.h"
#include "attn_params.h"
#include <stdlib.h>
#include <string.h>

namespace s3r {
namespace b16 {
using namespace sel;
using b16x::work_item;

constexpr int kHalfBytes = 32 * 128;
constexpr float kLog2e = 1.4426950408889634f;
typedef std::integral_constant<int, 0> H0;
typedef std::integral_constant<int, 1> H1;

template <typename E>
__global__ __launch_bounds__(64, 2) void select_b16_pairs_kernel(AttnParams p, int nqb, int ngrp, int total_wg) {
  typedef typename Mma<E>::V8 V8;
  typedef typename Mma<E>::V2 V2;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k0[kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k1[kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v0[kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v1[kHalfBytes];

  const int lane = threadIdx.x;
  const int hh = lane >> 5;
  const int c = lane & 31;

  const int vid = work_item(blockIdx.x, total_wg);
  const int bh = vid / ngrp;
  const int grp = vid - bh * ngrp;  // group of four query blocks = 64 queries
  const int b = bh / p.H;
  const int h = bh - b * p.H;

  const int64_t N = p.Lq;
  const int64_t q0 = (int64_t)grp * 64;
  const E* qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const E* kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const E* vp = (const E*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  E* op = (E*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh;

  char* k_buf[2] = {reinterpret_cast<char*>(lds_k0), reinterpret_cast<char*>(lds_k1)};
  char* v_buf[2] = {reinterpret_cast<char*>(lds_v0), reinterpret_cast<char*>(lds_v1)};

  // the four index rows of the group, one entry per lane; invalid entries are skipped
  int32_t my_idx[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int qb = grp * 4 + j;
    my_idx[j] = -1;
    if (qb < nqb && lane < p.K) my_idx[j] = __builtin_nontemporal_load(p.idx + ((int64_t)b * p.sib + (int64_t)h * p.sih + (int64_t)qb * p.sim + lane));
    if (my_idx[j] < 0 || (int64_t)my_idx[j] * 16 >= N) my_idx[j] = -1;
  }
  // B operand Q: lane = query row, head_dim chunk hh + 2 ks
  V8 bq[2][4];
#pragma unroll
  for (int qt = 0; qt < 2; qt++) {
    const int64_t row = q0 + qt * 32 + c;
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      Frag f;
      f.u = make_uint4(0, 0, 0, 0);
      if (row < N) f.u = *reinterpret_cast<const uint4*>(qp + row * p.sqm + ks * 16 + hh * 8);
      bq[qt][ks] = as_v8<E>(f);
    }
  }

  f32x16 ot[2][2];  // O^T [dt][qt]
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int qt = 0; qt < 2; qt++)
#pragma unroll
      for (int r = 0; r < 16; r++) ot[dt][qt][r] = 0.f;
  float m_i[2] = {-INFINITY, -INFINITY}, l_i[2] = {0.f, 0.f};
  const float sl2 = p.scale * kLog2e;
  const uint32_t krow = (uint32_t)p.skn * (uint32_t)sizeof(E), vrow = (uint32_t)p.svn * (uint32_t)sizeof(E);

  // per-lane pieces of the transfers and reads
  const int lr = lane >> 3;
  const int i16 = lane & 15;
  const int tr_row = 4 * hh + (i16 >> 2);
  const int tr_chunk = (((lane >> 4) & 1) * 2 + ((i16 & 3) >> 1)) ^ (((tr_row >> 1) & 1) << 2);
  const int tr_off = tr_row * 128 + tr_chunk * 16 + (i16 & 1) * 8;
  const int kr_off = c * 128 + ((hh ^ k_swizzle(c)) << 4);

  // Unit (i, QT): list position i of query blocks 2 QT and 2 QT + 1.  blk[0], blk[1]: their key blocks (-1: skip).
  auto entry = [&](int i, auto qt_tag, int32_t (&blk)[2]) {
    constexpr int QT = decltype(qt_tag)::value;
    blk[0] = __builtin_amdgcn_readlane(my_idx[2 * QT], i);
    blk[1] = __builtin_amdgcn_readlane(my_idx[2 * QT + 1], i);
  };
  auto fetch = [&](int i, auto qt_tag) {  // the unit's K and V half tiles -> buffers QT (skipped blocks re-read block 0)
    constexpr int QT = decltype(qt_tag)::value;
    int32_t blk[2];
    entry(i, qt_tag, blk);
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int64_t start = (int64_t)(blk[s] < 0 ? 0 : blk[s]) * 16;
      const int last = (int)((N - start < 16 ? N - start : 16) - 1);
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kp + start * p.skn), 0, 0x7fffffff, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vp + start * p.svn), 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const int ldsrow = 16 * s + 8 * t + lr;   // row of the 32-row half tile
        int row = 8 * t + lr;                     // row of the 16-token block
        row = row < last ? row : last;
        const uint32_t kc = (uint32_t)(((lane & 7) ^ k_swizzle(ldsrow)) * 16);
        const uint32_t vc = (uint32_t)(((lane & 7) ^ (((ldsrow >> 1) & 1) << 2)) * 16);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(k_buf[QT] + (2 * s + t) * 1024), 16,
                                                 (uint32_t)row * krow + kc, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)(v_buf[QT] + (2 * s + t) * 1024), 16,
                                                 (uint32_t)row * vrow + vc, 0, 0, 0);
      }
    }
  };
  auto compute = [&](int i, auto qt_tag) {
    constexpr int QT = decltype(qt_tag)::value;
    int32_t blk[2];
    entry(i, qt_tag, blk);
    // this lane's query belongs to block `mine` of the pair; only that block's 16 keys count for it
    const int mine = c >> 4;
    const int32_t myblk = mine == 0 ? blk[0] : blk[1];
    const int nkeys = myblk < 0 ? 0 : (int)(N - (int64_t)myblk * 16 < 16 ? N - (int64_t)myblk * 16 : 16);
    V8 ak[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      Frag f;
      f.u = *reinterpret_cast<const uint4*>(k_buf[QT] + (kr_off ^ (ks << 5)));
      ak[ks] = as_v8<E>(f);
    }
    f32x16 st;
#pragma unroll
    for (int r = 0; r < 16; r++) st[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ks++) st = Mma<E>::mma(ak[ks], bq[QT][ks], st);
    // register r holds key row 4hh + 8(r/4) + r%4 of the half tile: rows 0-15 (r < 8) are block 0's keys, 16-31 block
    // 1's.  Only the 8 registers of this lane's own block are scores of its query: they are picked first, and the
    // softmax runs on 8 values instead of 16.
    const uint32_t m0 = mine == 0 ? 0xFFFFFFFFu : 0u;  // bit masks instead of per-value selects on a condition register
    const uint32_t own_sel = mine == 0 ? 0x07060504u : 0x03020100u;  // v_perm_b32 selector: all four bytes of the first / second source
    float su[8];
#pragma unroll
    for (int j = 0; j < 8; j++) su[j] = __uint_as_float(__builtin_amdgcn_perm(__float_as_uint(st[j]), __float_as_uint(st[8 + j]), own_sel));
    if (__any(nkeys < 16)) {  // a ragged last block or a skipped entry somewhere in the wave
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (4 * hh + 8 * (j >> 2) + (j & 3) >= nkeys) su[j] = -INFINITY;
    }
    float mx = su[0];
#pragma unroll
    for (int j = 1; j < 8; j++) mx = fmaxf(mx, su[j]);
    mx = xh_max(mx) * sl2;  // sl2 > 0: the maximum of the scaled scores
    const float m_new = fmaxf(m_i[QT], mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;   // nothing valid so far: every probability is exp2(-inf) = 0
    const float alpha = __builtin_amdgcn_exp2f(m_i[QT] - m_use);  // 0 while m_i is -inf
    if (__any(m_new != m_i[QT])) {
      l_i[QT] *= alpha;
#pragma unroll
      for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) ot[dt][QT][r] *= alpha;
    }
    m_i[QT] = m_new;
    // probabilities of the own block, then the B operand of the PV product: the own block's k-group carries them,
    // the other block's k-group zeros
    union { V8 v; uint32_t w[4]; } pown, pf[2];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      V2 pk;
      pk[0] = (E)__builtin_amdgcn_exp2f(fmaf(su[e], sl2, -m_use));
      pk[1] = (E)__builtin_amdgcn_exp2f(fmaf(su[e + 1], sl2, -m_use));
      pown.v[e] = pk[0];
      pown.v[e + 1] = pk[1];
      l_i[QT] = Mma<E>::dot_ones(pk, l_i[QT]);
    }
#pragma unroll
    for (int wi = 0; wi < 4; wi++) {
      pf[0].w[wi] = pown.w[wi] & m0;
      pf[1].w[wi] = pown.w[wi] & ~m0;
    }
    V8 vfr[2][2];
#pragma unroll
    for (int jj = 0; jj < 2; jj++)
#pragma unroll
      for (int dt = 0; dt < 2; dt++) {
        const char* a0 = v_buf[QT] + (tr_off ^ (dt * 64)) + (jj * 16) * 128;
        Frag f;
        f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a0));
        f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a0 + 8 * 128));
        vfr[jj][dt] = as_v8<E>(f);
      }
#pragma unroll
    for (int jj = 0; jj < 2; jj++)
#pragma unroll
      for (int dt = 0; dt < 2; dt++) ot[dt][QT] = Mma<E>::mma(vfr[jj][dt], pf[jj].v, ot[dt][QT]);
  };

  const int nsteps = p.K;
  if (nsteps > 0) {
    fetch(0, H0{});
    for (int i = 0; i < nsteps; i++) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the reads of buffers 1 (previous step) are done
      fetch(i, H1{});
      __builtin_amdgcn_s_waitcnt(0x0F78);  // vmcnt(8): unit (i, 0) has landed
      compute(i, H0{});
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the reads of buffers 0 are done
      if (i + 1 < nsteps) {
        fetch(i + 1, H0{});
        __builtin_amdgcn_s_waitcnt(0x0F78);  // vmcnt(8): unit (i, 1) has landed
      } else {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      }
      compute(i, H1{});
    }
  }

  // output: as in the 64-token kernels (one exchange with lane ^ 32 per packed word, 16-byte stores).  With merge
  // operands the gated merge runs here (gate pair of the row, the compressed output of the row's 16-token block; the
  // three roundings of the eager expression kept) and the result goes to the [B, N, H*D] tensor.
  const bool merge = p.merge_out != nullptr;
#pragma unroll
  for (int qt = 0; qt < 2; qt++) {
    const float l = xh_sum(l_i[qt]);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int64_t row = q0 + qt * 32 + c;
    const bool live = row < N;
    float g0 = 0.f, g1 = 0.f;
    const E* ocp = nullptr;
    if (merge && live) {
      const E* gp = (const E*)p.merge_gate + (int64_t)b * p.sgb + (int64_t)h * p.sgh + row * p.sgn;
      g0 = (float)gp[0];
      g1 = (float)gp[1];
      ocp = (const E*)p.merge_oc + (int64_t)b * p.scb + (int64_t)h * p.sch + (row >> 4) * p.scm;
    }
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int gp = 0; gp < 2; gp++) {
        union { E e[8]; uint32_t w[4]; uint4 u; } pc;
        union { E e[2]; uint32_t w; } t;
#pragma unroll
        for (int wi = 0; wi < 2; wi++) {
          t.e[0] = (E)(ot[dt][qt][8 * gp + 2 * wi] * inv);
          t.e[1] = (E)(ot[dt][qt][8 * gp + 2 * wi + 1] * inv);
          const uint32_t a = t.w;
          t.e[0] = (E)(ot[dt][qt][8 * gp + 4 + 2 * wi] * inv);
          t.e[1] = (E)(ot[dt][qt][8 * gp + 4 + 2 * wi + 1] * inv);
          const uint32_t bw = t.w;
          const auto r = __builtin_amdgcn_permlane32_swap(a, bw, false, false);
          pc.w[wi] = r[0];
          pc.w[2 + wi] = r[1];
        }
        const int d0 = dt * 32 + 8 * (2 * gp + hh);
        if (live) {
          if (!merge) {
            *reinterpret_cast<uint4*>(op + row * p.som + d0) = pc.u;
          } else {
            union { E e[8]; uint4 u; } oc, res;
            oc.u = *reinterpret_cast<const uint4*>(ocp + d0);
#pragma unroll
            for (int e = 0; e < 8; e++) {
              const float x = round_to<E>(g0 * (float)oc.e[e]);
              const float y = round_to<E>(g1 * (float)pc.e[e]);
              res.e[e] = (E)(x + y);
            }
            *reinterpret_cast<uint4*>((E*)p.merge_out + (((int64_t)b * N + row) * p.H + h) * 64 + d0) = res.u;
          }
        }
      }
    if (live && p.lse != nullptr && hh == 0)
      p.lse[((int64_t)b * p.H + h) * N + row] = l > 0.f ? (m_i[qt] + __builtin_amdgcn_logf(l)) * 0.6931471805599453f : -INFINITY;
  }
}

}  // namespace b16

namespace b16u {
using namespace b16x;

// Blocks in a wave's LDS.  A third one costs a wave per SIMD: 32 256 tokens 186 -> 193 us (NQ 2), 180 -> 199 (NQ 4).
constexpr int kSlots = 2;

// The operands of a block in a slot (K rows, V columns 2 KB behind) and two entries of the walk list
__device__ __forceinline__ void read_block(uint32_t row, uint32_t tr, uint32_t now, uint32_t ahead, u32x4 (&k)[2], u32x2 (&v)[4], u32x2& e_now, u32x2& e_ahead) {
  asm volatile(
      "ds_read_b64 %6, %14\n\tds_read_b64 %7, %15\n\tds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\t"
      "ds_read_b64_tr_b16 %2, %10 offset:2048\n\tds_read_b64_tr_b16 %3, %11 offset:2048\n\tds_read_b64_tr_b16 %4, %12 offset:2048\n\t"
      "ds_read_b64_tr_b16 %5, %13 offset:2048\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(k[0]), "=&v"(k[1]), "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(e_now), "=&v"(e_ahead)
      : "v"(row), "v"(row ^ 64u), "v"(tr), "v"(tr ^ 32u), "v"(tr ^ 64u), "v"(tr ^ 96u), "v"(now), "v"(ahead)
      : "memory");
}

template <typename E, int NQ, bool WIDE>
__global__ __launch_bounds__(64, NQ > 2 ? 3 : 4) void select_b16_kernel(AttnParams p, int nqb, int ngrp, int total) {
  typedef typename Mma<E>::V8 V8;
  typedef typename Mma4<E>::V4 V4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_slots[kSlots * kPair];
  __shared__ __attribute__((aligned(16))) int2 walk[64 * NQ + kSlots];
  const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  const int vid = work_item(blockIdx.x, total);
  // (divisions run on the vector unit; the descriptors below want their results in scalar registers)
  const int bh = __builtin_amdgcn_readfirstlane(vid / ngrp), grp = vid - bh * ngrp;
  const int b = __builtin_amdgcn_readfirstlane(bh / p.H), h = bh - b * p.H;

  // the lists head the longest chain of the start: first in the queue
  const int32_t* lists = p.idx + (int64_t)b * p.sib + (int64_t)h * p.sih + (int64_t)grp * NQ * p.sim;
  asm volatile("" : "+s"(lists));  // (computed ahead of the lanes' branch: b and h stay in scalar registers)
  int32_t mine[NQ];
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    mine[j] = -1;
    if (grp * NQ + j < nqb && lane < p.K) mine[j] = __builtin_nontemporal_load(lists + (int64_t)j * p.sim + lane);
  }
  const int64_t row0 = (int64_t)grp * (16 * NQ) + c;
  const E* qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh + 8 * g;
  V8 bq[NQ][2];  // B operands of the query blocks: lane = query, head dimensions 32 ks + 8 g ..
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    const int64_t row = row0 + 16 * j;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      Frag f;
      f.u = make_uint4(0, 0, 0, 0);
      if (row < p.Lq) f.u = *reinterpret_cast<const uint4*>(qp + row * p.sqm + 32 * ks);
      bq[j][ks] = as_v8<E>(f);
    }
  }
  bool dup;  // some list names a block more than once (wave-uniform)
  const int n = walk_list<NQ>(mine, p.Lq, lds_slots, walk, kSlots, lane, dup);

  const Rows<E, WIDE> kr(p.k, (int64_t)b * p.skb + (int64_t)h * p.skh, p.skn, p.Lq, lane);
  const Rows<E, WIDE> vr(p.v, (int64_t)b * p.svb + (int64_t)h * p.svh, p.svn, p.Lq, lane);
  const LdsPtr slots = (LdsPtr)lds_slots;
  const uint32_t row_off = lds_addr(slots) + (uint32_t)(c * 128 + ((g ^ swz(c)) << 4));
  const int tr_row = 4 * g + (c >> 2);
  const uint32_t tr_off = lds_addr(slots) + (uint32_t)(tr_row * 128 + ((((c & 3) >> 1) ^ swz(tr_row)) << 4) + (c & 1) * 8);
  const uint32_t walk_at = lds_addr((LdsPtr)reinterpret_cast<char*>(walk));
  const float sl2 = p.scale * kLog2e;
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

  f32x4 o[NQ][4];
  float m[NQ], l[NQ];  // reference in base 2 (the same in a query's four lanes), sums of this lane's probabilities
  for (int pass = 0; pass < 2; pass++) {
    const bool exact = pass == 1;  // second walk: running maximum
    uint32_t fresh = (1u << NQ) - 1u;  // query blocks without a reference yet
#pragma unroll
    for (int j = 0; j < NQ; j++) {
      m[j] = -INFINITY;
      l[j] = 0.f;
#pragma unroll
      for (int dt = 0; dt < 4; dt++) o[j][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int s = 0; s < kSlots; s++) request(s < n ? __builtin_amdgcn_readfirstlane(walk[s].x) : -1, s);
    int slot = -1;
    for (int i = 0; i < n; i++) {
      slot = slot + 1 == kSlots ? 0 : slot + 1;
      u32x4 kw[2];
      u32x2 vt[4], now, ahead;
      __builtin_amdgcn_s_waitcnt(0x0F70 | (4 * (kSlots - 1)));  // this block's transfers have landed, the next ones' may be in flight
      read_block(row_off + slot * kPair, tr_off + slot * kPair, walk_at + 8u * i, walk_at + 8u * (i + kSlots), kw, vt, now, ahead);
      const int32_t blk = __builtin_amdgcn_readfirstlane((int32_t)now[0]);
      const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)now[1]);
      const bool rare = dup || exact || blk == kr.ragged;
      request(__builtin_amdgcn_readfirstlane((int32_t)ahead[0]), slot);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NQ; j++) {
        const uint32_t w = (cnt >> (8 * j)) & 0xffu;
        if (w != 0) {
          f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 2; ks++) st = mma16<E>(frag_of<E>(kw[ks]), bq[j][ks], st);
          settle(st);
          float more = -m[j];
          if (__builtin_expect(rare || (fresh & (1u << j)) != 0, 0)) {
            const int end = blk == kr.ragged ? kr.last : 15;
#pragma unroll
            for (int r = 0; r < 4; r++) st[r] = 4 * g + r > end ? -INFINITY : st[r];
            if (exact || (fresh & (1u << j)) != 0) {
              float mx = fmaxf(fmaxf(st[0], st[1]), fmaxf(st[2], st[3]));
              mx = sel::xh_max(fmaxf(mx, lane_xor<16>(mx))) * sl2;  // sl2 > 0: the maximum of the scaled scores
              const float was = m[j];
              m[j] = fmaxf(was, mx);
              if ((fresh & (1u << j)) == 0) {
                const float alpha = __builtin_amdgcn_exp2f(was - (m[j] == -INFINITY ? 0.f : m[j]));  // 0 while there is none
                l[j] *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; dt++) o[j][dt] *= alpha;
              }
              fresh &= ~(1u << j);
            }
            more = (m[j] == -INFINITY ? 0.f : -m[j]) + __builtin_amdgcn_logf((float)w);  // a block listed w times counts w times
          }
          float x[4];
#pragma unroll
          for (int r = 0; r < 4; r++) x[r] = __builtin_amdgcn_exp2f(fmaf(st[r], sl2, more));
          l[j] += (x[0] + x[1]) + (x[2] + x[3]);
          const V4 pr = pack4<E>(x);
#pragma unroll
          for (int dt = 0; dt < 4; dt++) o[j][dt] = Mma4<E>::mma(vt[dt], pr, o[j][dt]);
        }
      }
    }
    // The sums add the unrounded fp32 probabilities (all >= 0): a sum below the bound proves that every probability was below
    // it when it was rounded; fp16 ends at 65504, bf16 has fp32's range (2^100 leaves room for the products).
    const float big = std::is_same<E, f16_t>::value ? 65504.f : 1.2676506e30f;
    bool over = false;
#pragma unroll
    for (int j = 0; j < NQ; j++) over |= !(l[j] < big);
    if (exact || !__any(over)) break;
    // rare: some reference was far too low; start over with the running maximum
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);

  // Output: registers hold head dimensions 16 dt + 4 g + r of query c.  One exchange between neighbouring rows of sixteen lanes
  // per packed word gives a lane eight consecutive ones (tile dt + (g & 1), dimensions 8 (g / 2) ..): 16-byte stores.  With
  // merge operands the gated merge runs here (the roundings of the eager expression) and the result goes to [B, N, H*D].
  const bool merge = p.merge_out != nullptr;
  E* op = (E*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh;
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    const int64_t row = row0 + 16 * j;
    const bool live = row < p.Lq;
    const float sum = sel::xh_sum(l[j] + lane_xor<16>(l[j]));
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    float g0 = 0.f, g1 = 0.f;
    const E* ocp = nullptr;
    if (merge && live) {
      const E* gp = (const E*)p.merge_gate + (int64_t)b * p.sgb + (int64_t)h * p.sgh + row * p.sgn;
      g0 = (float)gp[0];
      g1 = (float)gp[1];
      ocp = (const E*)p.merge_oc + (int64_t)b * p.scb + (int64_t)h * p.sch + (row >> 4) * p.scm;
    }
#pragma unroll
    for (int dp = 0; dp < 2; dp++) {
      float y[2][4];
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) y[t][r] = o[j][2 * dp + t][r] * inv;
      const u32x2 wa = __builtin_bit_cast(u32x2, pack4<E>(y[0])), wb = __builtin_bit_cast(u32x2, pack4<E>(y[1]));
      union { E e[8]; uint32_t w[4]; uint4 u; } pc;
#pragma unroll
      for (int wi = 0; wi < 2; wi++) {
        const auto r = __builtin_amdgcn_permlane16_swap(wa[wi], wb[wi], false, false);
        pc.w[wi] = r[0];
        pc.w[2 + wi] = r[1];
      }
      const int d0 = 16 * (2 * dp + (g & 1)) + 8 * (g >> 1);
      if (live) {
        if (!merge) {
          *reinterpret_cast<uint4*>(op + row * p.som + d0) = pc.u;
        } else {
          union { E e[8]; uint4 u; } oc, res;
          oc.u = *reinterpret_cast<const uint4*>(ocp + d0);
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float x = round_to<E>(g0 * (float)oc.e[e]);
            const float z = round_to<E>(g1 * (float)pc.e[e]);
            res.e[e] = (E)(x + z);
          }
          *reinterpret_cast<uint4*>((E*)p.merge_out + (((int64_t)b * p.Lq + row) * p.H + h) * 64 + d0) = res.u;
        }
      }
    }
    if (live && p.lse != nullptr && g == 0)
      p.lse[((int64_t)b * p.H + h) * p.Lq + row] = sum > 0.f ? (m[j] + __builtin_amdgcn_logf(sum)) * 0.6931471805599453f : -INFINITY;
  }
}

}  // namespace b16u

int launch_select_b16(const AttnParams& p, int dtype, void* stream) {
  const int64_t nqb = (p.Lq + 15) / 16, blocks = nqb * p.B * p.H;
  if (blocks > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "s3r_select_attn: grid too large");
  hipStream_t st = (hipStream_t)stream;
  // S3R_B16_KERNEL=pairs picks the walk over pairs of list entries (kept as a cross-check)
  static const bool pairs = [] {
    const char* e = getenv("S3R_B16_KERNEL");
    return e != nullptr && strcmp(e, "pairs") == 0;
  }();
  // 32-bit byte offsets inside a transfer instruction span 16 rows of a block
  if (16 * p.skn * 2 + 128 > 0xffffffffLL || 16 * p.svn * 2 + 128 > 0xffffffffLL)
    return fail(S3R_ERR_UNSUPPORTED, "s3r_select_attn, 16-token blocks: row stride too large");
  auto far = [&](int64_t row) { return (p.Lq - 1) * row * 2 + 128 > 0xffffffffLL; };
  const bool wide = far(p.skn) || far(p.svn);
#define S3R_B16(E, NQ, W)                                                                                                    \
  do {                                                                                                                       \
    const int64_t ngrp = (nqb + NQ - 1) / NQ, total = ngrp * p.B * p.H;                                                      \
    hipLaunchKernelGGL((b16u::select_b16_kernel<E, NQ, W>), dim3((unsigned)total), dim3(64), 0, st, p, (int)nqb, (int)ngrp, (int)total); \
  } while (0)
#define S3R_B16_TYPE(E)                                                                                                      \
  do {                                                                                                                       \
    if (pairs) {                                                                                                             \
      const int64_t ngrp = (nqb + 3) / 4, total = ngrp * p.B * p.H;                                                          \
      hipLaunchKernelGGL(b16::select_b16_pairs_kernel<E>, dim3((unsigned)total), dim3(64), 0, st, p, (int)nqb, (int)ngrp, (int)total); \
    } else if (wide) {                                                                                                       \
      S3R_B16(E, 4, true);                                                                                                   \
    } else if (blocks <= 5000) { /* (query block, head) pairs */                                                             \
      S3R_B16(E, 1, false);                                                                                                  \
    } else if (blocks <= 20000) {                                                                                            \
      S3R_B16(E, 2, false);                                                                                                  \
    } else {                                                                                                                 \
      S3R_B16(E, 4, false);                                                                                                  \
    }                                                                                                                        \
  } while (0)
  if (dtype == S3R_BF16) S3R_B16_TYPE(bf16_t);
  else S3R_B16_TYPE(f16_t);
#undef S3R_B16_TYPE
#undef S3R_B16
  return check_launch("select_b16_kernel");
}

}  // namespace s3r
