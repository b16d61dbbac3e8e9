// Backward of the two attention operators on the gfx950 matrix cores (bf16 / fp16 I/O, block 64, head_dim 64).
//
// Reference: _topk_blocksparse_attention_bwd with backward_sum_o_do, backward_dkdv, backward_dq
// (pi3/models/sparse_attn/topk_blocksparse_attention.py:132-170,558-712,722-850,907-1038) for the selection
// branch and _flash_attn_backward (pi3/models/sparse_attn/flash_attention_topk.py:204-630) for the compressed
// branch, which is the same computation over ALL key tiles (DENSE below).  With P = exp(scale*S - lse) recomputed
// from the forward's log-sum-exp and delta = rowsum(dO * O):
//   dV = P^T dO          dP = dO V^T          dS = scale * P * (dP - delta)          dQ = dS K          dK = dS^T Q
// P (for dV) and dS (for dQ, dK) are rounded to the I/O dtype before the products, accumulation is fp32
// (reference :683-690, :826-838).
//
// Three kernels:
//   * bwd_delta_kernel: delta[b,h,n] = sum_d o * dO in fp32 (HBM bound), where the dQ kernel does not compute it on its way.
//   * bwd_dq_kernel: one wavefront per 64-row query block, four independent waves per workgroup; walks the block's
//     selected key tiles (or all of them).  Everything is computed transposed, as in the forward kernels:
//     S^T = K Q^T and dP^T = V dO^T put one QUERY per lane, so lse and delta are per-lane scalars;
//     dQ^T += K^T dS^T takes K^T fragments from ds_read_b64_tr_b16.  K and V half tiles (32 keys) go global -> LDS
//     by direct transfers, double buffered (16 KB per wave).  The K half is staged once, in a layout that serves
//     the transposed reads and the row reads (A operand of S^T) without bank conflicts.
//   * bwd_dkdv_kernel: one workgroup of two waves per 64-key block, each wave owns 32 keys (one KEY per lane:
//     S = Q K^T, dP = dO V^T with K, V fragments in registers as B operands) and walks the query blocks that
//     selected the key block (key-centric lists built by the host from the index tensor, reference :423-554).
//     Q and dO half tiles (32 queries) go global -> LDS, shared by the two waves, three half tiles ahead, one barrier
//     per half tile; dV^T += dO^T P and dK^T += Q^T dS read their A operands transposed from the same buffers.
// Query rows beyond Lq have lse = +inf (P = 0), keys beyond Lk are masked (P = 0); rows past the end of a tensor are
// never read (transfers re-read the last valid row).
#include "block16.h"
#include "attn_bwd.h"

namespace s3r {
namespace bwd {
using namespace sel;

constexpr int kHalfBytes = 32 * 128;  // one half tile: 32 rows of 64 two-byte values
constexpr float kLog2e = 1.4426950408889634f;

typedef std::integral_constant<int, 0> H0;
typedef std::integral_constant<int, 1> H1;

// ---- delta ---------------------------------------------------------------------------------------------------
template <typename E>
__global__ __launch_bounds__(256) void bwd_delta_kernel(const E* __restrict__ o, const E* __restrict__ dout, float* __restrict__ delta,
                                                         int H, int64_t N, int64_t rows, int64_t sob, int64_t soh, int64_t son,
                                                         int64_t sdb, int64_t sdh, int64_t sdn) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = gid >> 3;  // 8 lanes of 16 bytes per 64-value row
  const int part = (int)(gid & 7);
  const bool live = row < rows;
  const int64_t rr = live ? row : rows - 1;
  const int64_t n = rr % N, bh = rr / N;
  const int h = (int)(bh % H);
  const int64_t b = bh / H;
  // both tensors are streamed once: non-temporal loads
  const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(o + b * sob + h * soh + n * son + part * 8));
  const u32x4 g = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(dout + b * sdb + h * sdh + n * sdn + part * 8));
  const E* ae = reinterpret_cast<const E*>(&a);
  const E* ge = reinterpret_cast<const E*>(&g);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) s += (float)ae[i] * (float)ge[i];
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) s += __shfl_xor(s, off);
  if (live && part == 0) delta[rr] = s;
}

// ---- dQ ----------------------------------------------------------------------------------------------------------
// One wave per 64-row query block.  The unit of its pipeline is 32 keys x 16 queries, twelve products of 16 x 16; in the phase of unit u
// the wave issues, one per slot,
//     dQ^T of unit u-1 (4),  S^T and dP^T of unit u+1 (8)
// and between them the vector work of unit u, cut into pairs of scores (two fused multiply-adds, two exponentials, two multiplications, one
// conversion over three slots), so that nothing waits for a product or an exponential of its own slot.  The wave's key tile is read in halves of 32 keys:
// row fragments of K and V and transposed fragments of K, each requested from LDS eight products ahead of its first use, into the registers
// that the half before has just left.
//   * dS = P (dP - delta) with the softmax scale inside P: P = exp2(scale log2(e) S - lse log2(e) + log2(scale)), and the accumulator
//     of dP starts at -delta (a tuple per 16 queries that stays in registers): per score one fused multiply-add, one exponential, one
//     multiplication and half a conversion, against two multiply-adds, one exponential, one multiplication and half a conversion before.
//   * 16 x 16 x 32 products: a lane's tuple is four scores, so a unit is small enough to be pipelined in registers (32 x 32 products
//     with both halves of the queries in flight did not fit, and the compiler's order left matrix cores and vector unit taking turns).
//   * DELTA: delta comes from O, whose rows a wave reads beside the dO that it holds in LDS anyway, instead of from a kernel of its own that
//     reads both (171 us at 266 496 tokens).  Two operators with gradients at that size 5 842 / 5 742; dQ, dK and dV of random lists of 16,
//     8 328 tokens 171.5 / 162.4, 104 100 1 906 / 1 876, dense over 1 041 58.5 / 56.5.  One sum of eight values per lane, in the order of that kernel.
// us, before / now: 266 496 tokens x 16 heads, top-16 1 902 / 1 531 (1.1 PFLOP/s: matrix cores and vector unit have the same work, 1 536
// cycles each per tile, and the chip runs below 2 GHz under it), dense over 4 164 tokens 212 / 161.
template <typename E, bool DENSE, bool DELTA>
__global__ __launch_bounds__(256, 2) void bwd_dq_kernel(BwdParams p, int nqb, int nqg, int total_wg) {
  typedef typename Mma<E>::V8 V8;
  typedef typename Mma<E>::V2 V2;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k0[4 * kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k1[4 * kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v0[4 * kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v1[4 * kHalfBytes];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  const int c = lane & 15;

  const int w = blockIdx.x;  // workgroup w -> work item: each XCD walks a contiguous range of query blocks of one head
  const int xcd = w & 7, slot = w >> 3;
  const int per = total_wg >> 3, rem = total_wg & 7;
  const int vid = xcd * per + (xcd < rem ? xcd : rem) + slot;
  const int bh = vid / nqg;
  const int qg = vid - bh * nqg;
  const int b = bh / p.H;
  const int h = bh - b * p.H;
  const int qb = qg * 4 + wave;
  if (qb >= nqb) return;

  const int64_t Lq = p.Lq, Lk = p.Lk;
  const int64_t q0 = (int64_t)qb * 64;
  const E* qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const E* kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const E* vp = (const E*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  const E* gp = (const E*)p.dout + (int64_t)b * p.sgb + (int64_t)h * p.sgh;
  const float* lsep = p.lse + ((int64_t)b * p.H + h) * Lq;
  const float* dlp = p.delta + ((int64_t)b * p.H + h) * Lq;

  // the list first: it heads the longest chain of the start
  int32_t my_idx = -1;
  if constexpr (!DENSE) {
    const int32_t* idx_row = p.idx + (int64_t)b * p.sib + (int64_t)h * p.sih + (int64_t)qb * p.sim;
    if (lane < p.K) my_idx = idx_row[lane];
  }
  float nl[4];    // log2(scale) - lse log2(e)
  f32x4 nd[4];    // -delta, what the products of dP^T start from
  const float log2_scale = __builtin_amdgcn_logf(p.scale);
#pragma unroll
  for (int qt = 0; qt < 4; qt++) {
    const int64_t row = q0 + qt * 16 + c;
    const bool live = row < Lq;
    nl[qt] = live ? fmaf(lsep[row], -kLog2e, log2_scale) : -INFINITY;
    if constexpr (!DELTA) {
      const float m = live ? -dlp[row] : 0.f;
      nd[qt] = (f32x4){m, m, m, m};
    }
  }
  f32x4 dq[4][4];  // dQ^T [qt][dt]: lane = query, registers = head dimensions 16 dt + 4 g ..
#pragma unroll
  for (int qt = 0; qt < 4; qt++)
#pragma unroll
    for (int dt = 0; dt < 4; dt++) dq[qt][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // key tiles of this query block: full ones go through the pipeline, occurrences of the ragged last one come after it
  const int32_t ragged_blk = (Lk & 63) ? (int32_t)(Lk >> 6) : -1;
  uint64_t todo = 0;
  int n_full, n_ragged;
  int dense_next = 0;
  if constexpr (DENSE) {
    n_full = (int)(Lk >> 6);
    n_ragged = (Lk & 63) ? 1 : 0;
  } else {
    const bool valid = my_idx >= 0 && (int64_t)my_idx * 64 < Lk;
    todo = __ballot(valid && my_idx != ragged_blk);
    n_ragged = __popcll(__ballot(valid && my_idx == ragged_blk));
    n_full = __popcll(todo);
  }
  int64_t last_start = 0;
  auto pop_or_last = [&]() -> int64_t {  // first row of the next full tile, or the last one again
    if constexpr (DENSE) {
      last_start = (int64_t)(dense_next < n_full ? dense_next : n_full - 1) * 64;
      dense_next++;
    } else {
      const bool any = todo != 0;
      const int t = any ? __ffsll((unsigned long long)todo) - 1 : 0;
      const int64_t s = (int64_t)__builtin_amdgcn_readlane(my_idx, t) * 64;
      todo &= todo - 1;
      last_start = any ? s : last_start;
    }
    return last_start;
  };

  const float sl2 = p.scale * kLog2e;
  const uint32_t krow = (uint32_t)p.skn * (uint32_t)sizeof(E), vrow = (uint32_t)p.svn * (uint32_t)sizeof(E);
  typedef __attribute__((address_space(3))) void* Lds;
  // every buffer is named through one array: the compiler then knows that a read of one does not wait for transfers into another
  auto k_buf = [&](auto hf) -> char* { return reinterpret_cast<char*>(decltype(hf)::value == 0 ? lds_k0 : lds_k1) + wave * kHalfBytes; };
  auto v_buf = [&](auto hf) -> char* { return reinterpret_cast<char*>(decltype(hf)::value == 0 ? lds_v0 : lds_v1) + wave * kHalfBytes; };
  // transfer i of a half tile moves its rows 8 i .. 8 i + 7 (chunk c of row r at c ^ swz(r), the same for all four)
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ b16x::swz(lane >> 3)) * 16);
  const uint32_t k_voff = (uint32_t)(lane >> 3) * krow + chunk, v_voff = (uint32_t)(lane >> 3) * vrow + chunk;
  auto dma_k = [&](auto hf, auto i_tag, int64_t start) {
    constexpr int HF = decltype(hf)::value, i = decltype(i_tag)::value;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(kp + (start + 32 * HF) * p.skn), 0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (Lds)(k_buf(hf) + i * 1024), 16, k_voff, 8u * i * krow, 0, 0);
  };
  auto dma_v = [&](auto hf, auto i_tag, int64_t start) {
    constexpr int HF = decltype(hf)::value, i = decltype(i_tag)::value;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(vp + (start + 32 * HF) * p.svn), 0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (Lds)(v_buf(hf) + i * 1024), 16, v_voff, 8u * i * vrow, 0, 0);
  };
  const int row_off = c * 128 + ((g ^ b16x::swz(c)) << 4);
  const int tr_row = 4 * g + (c >> 2);
  const int tr_off = tr_row * 128 + ((((c & 3) >> 1) ^ b16x::swz(tr_row)) << 4) + (c & 1) * 8;
  // B operands Q and dO: lane = query 16 qt + c, head dimensions 32 ks + 8 g ..; through the K and V buffers, whose map the transfers and
  // the reads share (rows beyond Lq re-read the last one, never stored).  Loaded in the operands' own pattern, they took the address unit
  // four times as long.
  V8 bq[4][2], bg[4][2];
  {
    const uint32_t qrow = (uint32_t)p.sqm * (uint32_t)sizeof(E), grow = (uint32_t)p.sgm * (uint32_t)sizeof(E);
    const int left = (int)(Lq - q0 < 64 ? Lq - q0 : 64) - 1;
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void*)(qp + q0 * p.sqm), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc((void*)(gp + q0 * p.sgm), 0, 0x7fffffff, 0x00020000);
    u32x4 out[8];  // DELTA: the forward's output, the same chunks of the same rows that the lane's transfers move of dO
    if constexpr (DELTA) {
      const E* const op = (const E*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh;
      const uint32_t orow = (uint32_t)p.som * (uint32_t)sizeof(E);
      const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void*)(op + q0 * p.som), 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int row = 8 * i + (lane >> 3);
        out[i] = __builtin_amdgcn_raw_buffer_load_b128(ro, (uint32_t)(row < left ? row : left) * orow + chunk, 0, 2 /* nt: read once */);
      }
    }
    static_for<2>([&](auto hf) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        int row = 32 * decltype(hf)::value + 8 * i + (lane >> 3);
        row = row < left ? row : left;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (Lds)(k_buf(hf) + i * 1024), 16, (uint32_t)row * qrow + chunk, 0, 0, 2 /* nt: read once */);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (Lds)(v_buf(hf) + i * 1024), 16, (uint32_t)row * grow + chunk, 0, 0, 2);
      }
    });
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    static_for<4>([&](auto qt_tag) {
      constexpr int QT = decltype(qt_tag)::value;
      typedef std::integral_constant<int, (QT >> 1)> HF;
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        Frag f, d;
        f.u = *reinterpret_cast<const uint4*>(k_buf(HF{}) + (QT & 1) * 2048 + (row_off ^ (ks << 6)));
        d.u = *reinterpret_cast<const uint4*>(v_buf(HF{}) + (QT & 1) * 2048 + (row_off ^ (ks << 6)));
        bq[QT][ks] = as_v8<E>(f);
        bg[QT][ks] = as_v8<E>(d);
      }
    });
    if constexpr (DELTA) {
      float s = 0.f;  // of row 8 (lane % 8) + lane / 8
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const u32x4 gv = *reinterpret_cast<const u32x4*>((i < 4 ? v_buf(H0{}) : v_buf(H1{})) + (i & 3) * 1024 + lane * 16);
        const E* const oe = reinterpret_cast<const E*>(&out[i]);
        const E* const ge = reinterpret_cast<const E*>(&gv);
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) t = fmaf((float)oe[e], (float)ge[e], t);
        t = group_sum<8>(t);
        s = (lane & 7) == i ? t : s;
      }
      const int64_t row = q0 + 8 * (lane & 7) + (lane >> 3);
      if (row < Lq) p.delta_out[((int64_t)b * p.H + h) * Lq + row] = s;
#pragma unroll
      for (int qt = 0; qt < 4; qt++) {
        const float m = -__int_as_float(__builtin_amdgcn_ds_bpermute(((c & 7) * 8 + 2 * qt + (c >> 3)) * 4, __float_as_int(s)));
        nd[qt] = (f32x4){m, m, m, m};
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): read before the first tile is requested
    asm volatile("" ::: "memory");
  }
  V8 ak[2][2], av[2][2];  // row fragments [16 keys][ks]
  V8 kt[4];               // K^T [dt]: head dimension 16 dt + c, keys 4 g .. of either 16
  auto read_rows16 = [&](const char* half, V8 (&dst)[2][2]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        Frag f;
        f.u = *reinterpret_cast<const uint4*>(half + t * 2048 + (row_off ^ (ks << 6)));
        dst[t][ks] = as_v8<E>(f);
      }
  };
  auto read_kt = [&](const char* half) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
      const char* a = half + (tr_off ^ (dt << 5));
      Frag f;
      f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a));
      f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a + 2048));
      kt[dt] = as_v8<E>(f);
    }
  };
  f32x4 st[2][2], dp[2][2];  // S^T and dP^T [parity of the unit][16 keys]
  V8 ds;                     // dS^T of the unit before
  auto score = [&](auto i_tag, auto qt_tag) {  // product i of 8 of the scores of 16 queries
    constexpr int i = decltype(i_tag)::value, QT = decltype(qt_tag)::value, t = i & 1, ks = (i >> 1) & 1, B = QT & 1;
    if constexpr (i < 4) st[B][t] = b16x::mma16<E>(ak[t][ks], bq[QT][ks], ks ? st[B][t] : (f32x4){0.f, 0.f, 0.f, 0.f});
    else dp[B][t] = b16x::mma16<E>(av[t][ks], bg[QT][ks], ks ? dp[B][t] : nd[QT]);
  };
  auto pair_of = [&](float a, float b2) -> uint32_t {
    V2 v;
    v[0] = (E)a;
    v[1] = (E)b2;
    return __builtin_bit_cast(uint32_t, v);
  };
  // Phase of unit (half HF of the tile, queries 16 QT ..).  Transfers: V of the next tile's half HF while QT = 0 (V's last reads of the buffer
  // went into registers a unit ago), K of it while QT = 1 (behind the products that took kt), in this order, so that eight transfers are
  // younger than what is read from the other half's buffers while QT = 2 and 3.
  auto phase = [&](auto hf, auto qt_tag, int64_t next) {
    constexpr int HF = decltype(hf)::value, QT = decltype(qt_tag)::value, B = QT & 1;
    typedef std::integral_constant<int, HF ^ 1> HO;
    typedef std::integral_constant<int, (QT + 1) & 3> NQ;
    constexpr int PQ = (QT + 3) & 3;
    float x0 = 0.f, x1 = 0.f, e0 = 0.f, e1 = 0.f;
    u32x4 dn;
    static_for<12>([&](auto j_tag) {
      constexpr int j = decltype(j_tag)::value;
      if constexpr (QT == 0 && j == 4) read_kt(k_buf(hf));
      if constexpr (QT == 0 && j >= 6 && j < 10) dma_v(hf, std::integral_constant<int, (j - 6) & 3>{}, next);
      if constexpr (QT == 1 && j >= 4 && j < 8) dma_k(hf, std::integral_constant<int, j & 3>{}, next);
      if constexpr (QT == 2 && j == 8) {
        __builtin_amdgcn_s_waitcnt(0x0F78);  // vmcnt(8): the other half of K and of V have landed
        read_rows16(k_buf(HO{}), ak);
      }
      if constexpr (QT == 3 && j == 0) read_rows16(v_buf(HO{}), av);
      if constexpr (j < 4) dq[PQ][j] = b16x::mma16<E>(kt[j], ds, dq[PQ][j]);
      else score(std::integral_constant<int, (j + 8) % 12>{}, NQ{});
      {
        constexpr int pr = j / 3, s = j % 3, t = pr >> 1, r = 2 * (pr & 1);
        if constexpr (s == 0) {
          x0 = fmaf(st[B][t][r], sl2, nl[QT]);
          x1 = fmaf(st[B][t][r + 1], sl2, nl[QT]);
          e0 = __builtin_amdgcn_exp2f(x0);
          asm volatile("" ::"v"(x1), "v"(e0));
        } else if constexpr (s == 1) {
          e1 = __builtin_amdgcn_exp2f(x1);
          e0 *= dp[B][t][r];
          asm volatile("" ::"v"(e0), "v"(e1));
        } else {
          e1 *= dp[B][t][r + 1];
          uint32_t wd = pair_of(e0, e1);
          asm volatile("" ::"v"(wd));
          dn[pr] = wd;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    ds = b16x::frag_of<E>(dn);
  };
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 3> I3;

  if (n_full > 0) {
    int64_t cur = pop_or_last(), next = pop_or_last();
    static_for<4>([&](auto i) { dma_v(H0{}, i, cur); });
    static_for<4>([&](auto i) { dma_k(H0{}, i, cur); });
    static_for<4>([&](auto i) { dma_v(H1{}, i, cur); });
    static_for<4>([&](auto i) { dma_k(H1{}, i, cur); });
    __builtin_amdgcn_s_waitcnt(0x0F78);  // vmcnt(8): half 0
    read_rows16(k_buf(H0{}), ak);
    read_rows16(v_buf(H0{}), av);
    static_for<8>([&](auto i) { score(i, H0{}); });
    const u32x4 zero = {0, 0, 0, 0};
    ds = b16x::frag_of<E>(zero);  // nothing for the first phase to add
#pragma unroll
    for (int dt = 0; dt < 4; dt++) kt[dt] = b16x::frag_of<E>(zero);
    for (int i = n_full; i > 0; i--) {  // past the last tile its rows are requested and scored again, for nothing
      phase(H0{}, H0{}, next);
      phase(H0{}, H1{}, next);
      phase(H0{}, I2{}, next);
      phase(H0{}, I3{}, next);
      phase(H1{}, H0{}, next);
      phase(H1{}, H1{}, next);
      phase(H1{}, I2{}, next);
      phase(H1{}, I3{}, next);
      next = pop_or_last();
    }
#pragma unroll
    for (int dt = 0; dt < 4; dt++) dq[3][dt] = b16x::mma16<E>(kt[dt], ds, dq[3][dt]);
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0): no transfer is on its way, nothing is read any more
  }
  for (; n_ragged > 0; n_ragged--) {  // the ragged last tile: rows beyond Lk re-read the last one and carry no probability
    const int64_t start = (int64_t)ragged_blk * 64;
    const int nvalid = (int)(Lk - start);
    static_for<2>([&](auto hf) {
      constexpr int HF = decltype(hf)::value;
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kp + start * p.skn), 0, 0x7fffffff, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vp + start * p.svn), 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        int row = 32 * HF + 8 * i + (lane >> 3);
        row = row < nvalid ? row : nvalid - 1;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (Lds)(k_buf(hf) + i * 1024), 16, (uint32_t)row * krow + chunk, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (Lds)(v_buf(hf) + i * 1024), 16, (uint32_t)row * vrow + chunk, 0, 0, 0);
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      read_rows16(k_buf(hf), ak);
      read_rows16(v_buf(hf), av);
      read_kt(k_buf(hf));
      static_for<4>([&](auto qt_tag) {
        constexpr int QT = decltype(qt_tag)::value, B = QT & 1;
        static_for<8>([&](auto i) { score(i, qt_tag); });
        u32x4 dn;
#pragma unroll
        for (int pr = 0; pr < 4; pr++) {
          const int t = pr >> 1, r = 2 * (pr & 1), key = 32 * HF + 16 * t + 4 * g + r;
          const float p0 = __builtin_amdgcn_exp2f(fmaf(st[B][t][r], sl2, nl[QT])), p1 = __builtin_amdgcn_exp2f(fmaf(st[B][t][r + 1], sl2, nl[QT]));
          dn[pr] = pair_of((key < nvalid ? p0 : 0.f) * dp[B][t][r], (key + 1 < nvalid ? p1 : 0.f) * dp[B][t][r + 1]);
        }
        ds = b16x::frag_of<E>(dn);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) dq[QT][dt] = b16x::mma16<E>(kt[dt], ds, dq[QT][dt]);
      });
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): read before the next occurrence's transfers
    });
  }

  E* dqp = (E*)p.dq + (int64_t)b * p.sdqb + (int64_t)h * p.sdqh;
#pragma unroll
  for (int qt = 0; qt < 4; qt++) {
    const int64_t row = q0 + qt * 16 + c;
    if (row < Lq) {
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        const u32x2 o = {pair_of(dq[qt][dt][0], dq[qt][dt][1]), pair_of(dq[qt][dt][2], dq[qt][dt][3])};
        *reinterpret_cast<u32x2*>(dqp + row * p.sdqm + 16 * dt + 4 * g) = o;
      }
    }
  }
}

// ---- dK, dV ------------------------------------------------------------------------------------------------------
// A workgroup of two waves per 64-key block, 32 keys a wave: K and V of its keys as B operands (32 registers), dK^T and dV^T (64) and the
// fragments of 32 queries (64).  The unit of the pipeline is 32 queries x 16 keys: S and dP (8 products of 16 x 16 x 32), P and dS of
// eight scores a lane, dV^T and dK^T (8).  In the phase of unit u a wave issues, one product per slot,
//     dV^T and dK^T of unit u-1,  S and dP of unit u+1
// and between them the vector work of unit u, a pair of scores over four slots.  Fragments are requested from LDS twelve products ahead,
// into the registers that the half tile before has just left.  Tiles of 64 queries go global -> LDS once for both waves (each moves half of
// every half tile), three half tiles ahead, with one barrier per half tile: behind it both waves' parts of the next half tile have landed
// and nobody reads the one before this any more, whose buffers are then requested again.
// The per-query terms ride in the accumulators: S starts at -lse / scale, so P = exp2(scale log2(e) S), and dP at -delta, so dS / scale =
// P dP; bf16 puts the scale onto dK once at the end, fp16, with its narrow range, onto every dS.
// us, before (32 x 32 products, two tiles, the scores of a tile's first half and the products of its second one with nothing beside them) /
// now: 266 496 tokens x 16 heads, top-16 2 532 / 2 336, dense over 8 192 x 16 537 / 472, 4 164 x 16 208 / 188.  Dense it runs at 1.17 PFLOP/s, the rate of
// a large library product (the chip's power: on zeros the same instructions take 384); with lists a workgroup's start and end, 1.1 GB each
// of K and V, Q and dO, dK and dV, take 0.4 ms beside it.  Tried: one wave a SIMD with 64 keys (half the LDS reads, but a lone wave issues a vector
// instruction every eight cycles, two of them one every four: 2 478).
template <typename E, bool DENSE>
__global__ __launch_bounds__(128, 2) void bwd_dkdv_kernel(BwdParams p, int nkb, int nqb_all, int total) {
  typedef typename Mma<E>::V8 V8;
  typedef typename Mma<E>::V2 V2;
  typedef __attribute__((address_space(3))) void* Lds;
  // half tiles [tile parity][half]; separate arrays: a read of one does not wait for transfers into another
  __shared__ __attribute__((aligned(1024))) unsigned char lds_q00[kHalfBytes], lds_q01[kHalfBytes], lds_q10[kHalfBytes], lds_q11[kHalfBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_g00[kHalfBytes], lds_g01[kHalfBytes], lds_g10[kHalfBytes], lds_g11[kHalfBytes];
  __shared__ __attribute__((aligned(256))) float lds_s[2][64];  // per wave, of a half tile: [0, 32) -lse / scale, [32, 64) -delta

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  const int c = lane & 15;

  // With lists the grid has two passes over the key blocks: the first (workgroups [0, total)) takes the blocks whose
  // lists are long, the second the others, so the longest lists of a skewed index tensor start first instead of
  // wherever their key block falls in the launch order.
  const bool long_pass = DENSE || (int)blockIdx.x < total;
  const int vid = b16x::work_item((int)blockIdx.x < total ? (int)blockIdx.x : (int)blockIdx.x - total, total);
  const int bh = __builtin_amdgcn_readfirstlane(vid / nkb);
  const int kb = __builtin_amdgcn_readfirstlane(vid - bh * nkb);
  const int b = __builtin_amdgcn_readfirstlane(bh / p.H);
  const int h = bh - b * p.H;

  const int64_t Lq = p.Lq, Lk = p.Lk;
  // query blocks that attend to this key block
  int n;
  const int32_t* list = nullptr;
  if constexpr (DENSE) {
    n = nqb_all;
  } else {
    const int32_t* off = p.kq_off + ((int64_t)b * p.H + h) * (nkb + 1);
    const int32_t lo = off[kb], hi = off[kb + 1];
    n = __builtin_amdgcn_readfirstlane(hi - lo);
    if ((n > 4 * p.K) != long_pass) return;
    list = p.kq_list + ((int64_t)b * p.H + h) * p.list_stride + lo;
  }
  const E* qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const E* kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const E* vp = (const E*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  const E* gp = (const E*)p.dout + (int64_t)b * p.sgb + (int64_t)h * p.sgh;
  const int64_t key0 = (int64_t)kb * 64 + wave * 32 + c;
  E* dkp = (E*)p.dk + (int64_t)b * p.sdkb + (int64_t)h * p.sdkh + 4 * g;
  E* dvp = (E*)p.dv + (int64_t)b * p.sdvb + (int64_t)h * p.sdvh + 4 * g;
  if (n == 0) {  // nobody attends to these keys
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const int64_t key = key0 + 16 * kt;
      if (key < Lk) {
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
          *reinterpret_cast<u32x2*>(dkp + key * p.sdkn + 16 * dt) = (u32x2){0, 0};
          *reinterpret_cast<u32x2*>(dvp + key * p.sdvn + 16 * dt) = (u32x2){0, 0};
        }
      }
    }
    return;
  }
  const float* const stat = (lane < 32 ? p.lse : p.delta) + ((int64_t)b * p.H + h) * Lq;

  // List entries come 64 at a time (lane l holds entry base + l), so the latency of the list read is paid once per
  // 64 tiles and not in front of every tile's transfers.
  int32_t held = -1;
  int base = -64;
  auto block_of = [&](int i) -> int32_t {
    if constexpr (DENSE) return i;
    if (i >= base + 64) {
      base = i & ~63;
      held = base + lane < n ? list[base + lane] : -1;
      asm volatile("" : "+v"(held));  // (waited for here: behind the branch every tile would wait)
    }
    return __builtin_amdgcn_readlane(held, i - base);
  };

  const float scale = p.scale;
  const float sl2 = scale * kLog2e;
  const float factor = lane < 32 ? -1.0f / scale : -1.0f;
  constexpr bool LATE_SCALE = std::is_same<E, bf16_t>::value;  // the softmax scale goes onto dK at the end
  const uint32_t qrow = (uint32_t)p.sqm * (uint32_t)sizeof(E), grow = (uint32_t)p.sgm * (uint32_t)sizeof(E);
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ b16x::swz(lane >> 3)) * 16);
  const uint32_t q_voff = (uint32_t)(lane >> 3) * qrow + chunk, g_voff = (uint32_t)(lane >> 3) * grow + chunk;
  const int row_off = c * 128 + ((g ^ b16x::swz(c)) << 4);
  const int tr_row = 4 * g + (c >> 2);
  const int tr_off = tr_row * 128 + ((((c & 3) >> 1) ^ b16x::swz(tr_row)) << 4) + (c & 1) * 8;
  auto q_buf = [&](auto par, auto hf) -> char* {
    if constexpr (decltype(par)::value == 0) return reinterpret_cast<char*>(decltype(hf)::value == 0 ? lds_q00 : lds_q01);
    else return reinterpret_cast<char*>(decltype(hf)::value == 0 ? lds_q10 : lds_q11);
  };
  auto g_buf = [&](auto par, auto hf) -> char* {
    if constexpr (decltype(par)::value == 0) return reinterpret_cast<char*>(decltype(hf)::value == 0 ? lds_g00 : lds_g01);
    else return reinterpret_cast<char*>(decltype(hf)::value == 0 ? lds_g10 : lds_g11);
  };

  // A half tile's requests: of a wave four transfers (number i of 0, 1 of Q, 2, 3 of dO: rows 8 (2 wave + i % 2) .. + 7) and one load of lse
  // or delta per lane.  The tile that ends the tensor early issues the same four without records, which fetch nothing, and then transfers whose
  // rows beyond the end re-read the last one: the waits count the requests behind the one they need, and more of them only wait for more.
  float staged[2][2];  // lse or delta as loaded [tile parity][half]
  int end[2][2];       // (scalar) last row of its tile
  int last[2];         // (scalar) last row of the tile that is being requested
  int64_t first[2];    // (scalar) its first row
  const int32_t ragged_blk = (Lq & 63) ? (int32_t)(Lq >> 6) : -1;
  auto aim = [&](auto par, int32_t blk) {
    constexpr int PAR = decltype(par)::value;
    first[PAR] = (int64_t)blk * 64;
    last[PAR] = blk == ragged_blk ? (int)(Lq & 63) - 1 : 63;
  };
  auto request = [&](auto par, auto hf, auto i_tag) {
    constexpr int PAR = decltype(par)::value, HF = decltype(hf)::value, i = decltype(i_tag)::value;
    const uint32_t part = (uint32_t)(2 * wave + (i & 1)), r = 32 * HF + 8 * part;
    int32_t rec, some;
    b16x::records(last[PAR] - 63, rec, some);
    if constexpr (i < 2) {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(qp + first[PAR] * p.sqm), 0, rec, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (Lds)(q_buf(par, hf) + part * 1024), 16, q_voff, r * qrow, 0, 0);
    } else {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(gp + first[PAR] * p.sgm), 0, rec, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (Lds)(g_buf(par, hf) + part * 1024), 16, g_voff, r * grow, 0, 0);
    }
    if constexpr (i == 3) {
      if (__builtin_expect(last[PAR] < 63, 0)) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): behind the ones that fetch nothing
        const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void*)(qp + first[PAR] * p.sqm), 0, 0x7fffffff, 0x00020000);
        const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc((void*)(gp + first[PAR] * p.sgm), 0, 0x7fffffff, 0x00020000);
#pragma unroll
        for (int k = 0; k < 2; k++) {
          int row = 32 * HF + 8 * (2 * wave + k) + (lane >> 3);
          row = row < last[PAR] ? row : last[PAR];
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (Lds)(q_buf(par, hf) + (2 * wave + k) * 1024), 16, (uint32_t)row * qrow + chunk, 0, 0, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (Lds)(g_buf(par, hf) + (2 * wave + k) * 1024), 16, (uint32_t)row * grow + chunk, 0, 0, 0);
        }
      }
      end[PAR][HF] = last[PAR];
      const int row = 32 * HF + (lane & 31);
      staged[PAR][HF] = (stat + first[PAR])[row < last[PAR] ? row : last[PAR]];
    }
  };
  auto request_all = [&](auto par, auto hf) { static_for<4>([&](auto i) { request(par, hf, i); }); };
  // The loaded value is first touched when its half tile's transfers have been waited for (the counter is in order).
  auto publish = [&](auto par, auto hf) {
    constexpr int PAR = decltype(par)::value, HF = decltype(hf)::value;
    const bool live = 32 * HF + (lane & 31) <= end[PAR][HF];  // query rows beyond Lq: no probability
    lds_s[wave][lane] = live ? staged[PAR][HF] * factor : lane < 32 ? -INFINITY : 0.f;
  };
  V8 aq[2][2], ag[2][2];   // row fragments of Q, dO [16 queries][ks]: A operands of S, dP
  V8 qt[4], gt[4];         // Q^T, dO^T [dt]: head dimension 16 dt + c, queries 4 g .. of either 16
  f32x4 lse4[2], delta4[2];  // what S and dP start from [16 queries]
  auto read_rows16 = [&](const char* half, V8 (&dst)[2][2]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        Frag f;
        f.u = *reinterpret_cast<const uint4*>(half + t * 2048 + (row_off ^ (ks << 6)));
        dst[t][ks] = as_v8<E>(f);
      }
  };
  auto read_cols = [&](const char* half, V8 (&dst)[4]) {
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
      const char* a = half + (tr_off ^ (dt << 5));
      Frag f;
      f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a));
      f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a + 2048));
      dst[dt] = as_v8<E>(f);
    }
  };
  auto read_terms = [&](f32x4 (&dst)[2], int at) {
#pragma unroll
    for (int t = 0; t < 2; t++) dst[t] = *reinterpret_cast<const f32x4*>(&lds_s[wave][at + 16 * t + 4 * g]);
  };
  V8 bk[2][2], bv[2][2];     // K, V as B operands: lane = key 16 kt + c, head dimensions 32 ks + 8 g ..
  f32x4 st[2][2], dp[2][2];  // S, dP [parity of the unit][16 queries]
  f32x4 dk[2][4], dv[2][4];  // dK^T, dV^T [kt][dt]: lane = key, registers = head dimensions 16 dt + 4 g ..
  V8 pf, ds;                 // P, dS of the unit before
  auto score = [&](auto i_tag, auto kt_tag) {  // product i of 8 of the scores of 16 keys
    constexpr int i = decltype(i_tag)::value, KT = decltype(kt_tag)::value, t = i & 1, ks = (i >> 1) & 1, B = KT & 1;
    if constexpr (i < 4) st[B][t] = b16x::mma16<E>(aq[t][ks], bk[KT][ks], ks ? st[B][t] : lse4[t]);
    else dp[B][t] = b16x::mma16<E>(ag[t][ks], bv[KT][ks], ks ? dp[B][t] : delta4[t]);
  };
  auto pair_of = [&](float x, float y) -> uint32_t {
    V2 v;
    v[0] = (E)x;
    v[1] = (E)y;
    return __builtin_bit_cast(uint32_t, v);
  };
  // the requests of a half tile have landed in both waves, LEFT of this wave's being younger; nobody reads the half tile two before any more
  auto meet = [&](auto left) {
    constexpr int LEFT = decltype(left)::value;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70 | LEFT);  // vmcnt(LEFT)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Phase of unit (half HF of the tile, keys 16 KT ..).  KT = 0: transposed fragments of this half tile behind the last products of the one
  // before; then the barrier and row fragments of the next one, and requests of the half tile three further on into the buffers of the
  // one before this.
  auto phase = [&](auto par, auto hf, auto kt_tag) {
    constexpr int PAR = decltype(par)::value, HF = decltype(hf)::value, KT = decltype(kt_tag)::value, B = KT;
    typedef std::integral_constant<int, HF == 0 ? PAR : PAR ^ 1> NPar;  // the next half tile
    typedef std::integral_constant<int, HF ^ 1> NHf;
    typedef std::integral_constant<int, HF == 0 ? PAR ^ 1 : PAR> LPar;  // the half tile before, and the one three further on
    typedef std::integral_constant<int, KT ^ 1> NK;
    constexpr int PK = KT ^ 1;
    float x1 = 0.f, e0 = 0.f, e1 = 0.f, d0 = 0.f, d1 = 0.f;
    u32x4 pn, dn;
    static_for<16>([&](auto j_tag) {
      constexpr int j = decltype(j_tag)::value;
      if constexpr (KT == 0 && j == 4) read_cols(g_buf(par, hf), gt);
      if constexpr (KT == 0 && j == 8) read_cols(q_buf(par, hf), qt);
      if constexpr (KT == 0 && j == 12) {
        meet(std::integral_constant<int, 5>{});
        publish(NPar{}, NHf{});
        read_terms(lse4, 0);
        read_rows16(q_buf(NPar{}, NHf{}), aq);
      }
      if constexpr (KT == 1 && j == 0) {
        read_terms(delta4, 32);
        read_rows16(g_buf(NPar{}, NHf{}), ag);
      }
      if constexpr (KT == 1 && j >= 4 && j < 8) request(LPar{}, NHf{}, std::integral_constant<int, j & 3>{});
      if constexpr (j < 4) dv[PK][j] = b16x::mma16<E>(gt[j], pf, dv[PK][j]);
      else if constexpr (j < 8) dk[PK][j - 4] = b16x::mma16<E>(qt[j - 4], ds, dk[PK][j - 4]);
      else score(std::integral_constant<int, j & 7>{}, NK{});
      {
        constexpr int pr = j >> 2, s = j & 3, t = pr >> 1, r = 2 * (pr & 1);
        if constexpr (s == 0) {
          e0 = __builtin_amdgcn_exp2f(st[B][t][r] * sl2);
          x1 = st[B][t][r + 1] * sl2;
          asm volatile("" ::"v"(e0), "v"(x1));
        } else if constexpr (s == 1) {
          e1 = __builtin_amdgcn_exp2f(x1);
          d0 = LATE_SCALE ? e0 * dp[B][t][r] : e0 * (dp[B][t][r] * scale);
          asm volatile("" ::"v"(e1), "v"(d0));
        } else if constexpr (s == 2) {
          d1 = LATE_SCALE ? e1 * dp[B][t][r + 1] : e1 * (dp[B][t][r + 1] * scale);
          uint32_t wd = pair_of(e0, e1);
          asm volatile("" ::"v"(wd), "v"(d1));
          pn[pr] = wd;
        } else {
          uint32_t wd = pair_of(d0, d1);
          asm volatile("" ::"v"(wd));
          dn[pr] = wd;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    pf = b16x::frag_of<E>(pn);
    ds = b16x::frag_of<E>(dn);
  };

  // K and V of the wave's keys, on their way through the buffers of the second tile (rows beyond Lk re-read the last one, never stored)
  {
    const uint32_t krow = (uint32_t)p.skn * (uint32_t)sizeof(E), vrow = (uint32_t)p.svn * (uint32_t)sizeof(E);
    const int64_t k0 = (int64_t)kb * 64;
    const int left = (int)(Lk - k0 < 64 ? Lk - k0 : 64) - 1;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)(kp + k0 * p.skn), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)(vp + k0 * p.svn), 0, 0x7fffffff, 0x00020000);
    char* const kl = wave == 0 ? q_buf(H1{}, H0{}) : q_buf(H1{}, H1{});
    char* const vl = wave == 0 ? g_buf(H1{}, H0{}) : g_buf(H1{}, H1{});
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int row = 32 * wave + 8 * i + (lane >> 3);
      row = row < left ? row : left;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (Lds)(kl + i * 1024), 16, (uint32_t)row * krow + chunk, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (Lds)(vl + i * 1024), 16, (uint32_t)row * vrow + chunk, 0, 0, 0);
    }
  }
  int next = 0;
  auto next_block = [&]() -> int32_t {  // past the end the last one again
    const int i = next < n ? next : n - 1;
    next++;
    return block_of(i);
  };
  aim(H0{}, next_block());
  request_all(H0{}, H0{});
  request_all(H0{}, H1{});
  aim(H1{}, next_block());
  __builtin_amdgcn_s_waitcnt(0x0F7A);  // vmcnt(10): K and V
  if (wave == 0) {
    read_rows16(q_buf(H1{}, H0{}), bk);
    read_rows16(g_buf(H1{}, H0{}), bv);
  } else {
    read_rows16(q_buf(H1{}, H1{}), bk);
    read_rows16(g_buf(H1{}, H1{}), bv);
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  meet(std::integral_constant<int, 5>{});  // the first half tile; both waves have read K and V
  request_all(H1{}, H0{});
  publish(H0{}, H0{});
  read_terms(lse4, 0);
  read_terms(delta4, 32);
  read_rows16(q_buf(H0{}, H0{}), aq);
  read_rows16(g_buf(H0{}, H0{}), ag);
  static_for<8>([&](auto i) { score(i, H0{}); });
  const u32x4 zero = {0, 0, 0, 0};  // nothing for the first phase to add
  pf = ds = b16x::frag_of<E>(zero);
#pragma unroll
  for (int dt = 0; dt < 4; dt++) qt[dt] = gt[dt] = b16x::frag_of<E>(zero);
#pragma unroll
  for (int kt = 0; kt < 2; kt++)
#pragma unroll
    for (int dt = 0; dt < 4; dt++) dk[kt][dt] = dv[kt][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto tile = [&](auto par) {  // the tile behind it comes into the other parity's buffers, its second half while this one's first is worked on
    phase(par, H0{}, H0{});
    phase(par, H0{}, H1{});
    aim(par, next_block());
    phase(par, H1{}, H0{});
    phase(par, H1{}, H1{});
  };
  for (int left = n >> 1; left > 0; left--) {
    tile(H0{});
    tile(H1{});
  }
  if (n & 1) tile(H0{});
#pragma unroll
  for (int dt = 0; dt < 4; dt++) {
    dv[1][dt] = b16x::mma16<E>(gt[dt], pf, dv[1][dt]);
    dk[1][dt] = b16x::mma16<E>(qt[dt], ds, dk[1][dt]);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): no transfer may still write LDS when the wave ends
  const float after = LATE_SCALE ? scale : 1.f;
#pragma unroll
  for (int kt = 0; kt < 2; kt++) {
    const int64_t key = key0 + 16 * kt;
    if (key < Lk) {
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        const f32x4 a = dk[kt][dt], d = dv[kt][dt];
        const u32x2 ko = {pair_of(a[0] * after, a[1] * after), pair_of(a[2] * after, a[3] * after)};
        const u32x2 vo = {pair_of(d[0], d[1]), pair_of(d[2], d[3])};
        *reinterpret_cast<u32x2*>(dkp + key * p.sdkn + 16 * dt) = ko;
        *reinterpret_cast<u32x2*>(dvp + key * p.sdvn + 16 * dt) = vo;
      }
    }
  }
}

}  // namespace bwd

int launch_attn_bwd(const BwdParams& p, int dtype, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  const bool dense = p.idx == nullptr, own = p.o != nullptr;
  if (!dense && p.block == 16) return launch_attn_bwd16(p, dtype, stream);
  const int64_t nqb = (p.Lq + 63) / 64, nkb = (p.Lk + 63) / 64;
  const int64_t nqg = (nqb + 3) / 4;
  const int64_t total_q = nqg * p.B * p.H, total_k = nkb * p.B * p.H;
  if (total_q > 0x7fffffffLL || total_k > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention backward: grid too large");
  if (!dense && 2 * total_k > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "attention backward: grid too large");
  dim3 gq((unsigned)total_q), bq(256), gk((unsigned)(dense ? total_k : 2 * total_k)), bk(128);
#define S3R_BWD_LAUNCH(E)                                                                                                       \
  do {                                                                                                                          \
    if (p.dq != nullptr) {                                                                                                      \
      if (dense && own) hipLaunchKernelGGL((bwd::bwd_dq_kernel<E, true, true>), gq, bq, 0, st, p, (int)nqb, (int)nqg, (int)total_q);   \
      else if (dense) hipLaunchKernelGGL((bwd::bwd_dq_kernel<E, true, false>), gq, bq, 0, st, p, (int)nqb, (int)nqg, (int)total_q);    \
      else if (own) hipLaunchKernelGGL((bwd::bwd_dq_kernel<E, false, true>), gq, bq, 0, st, p, (int)nqb, (int)nqg, (int)total_q);      \
      else hipLaunchKernelGGL((bwd::bwd_dq_kernel<E, false, false>), gq, bq, 0, st, p, (int)nqb, (int)nqg, (int)total_q);              \
    }                                                                                                                           \
    if (p.dk != nullptr) {                                                                                                      \
      if (dense) hipLaunchKernelGGL((bwd::bwd_dkdv_kernel<E, true>), gk, bk, 0, st, p, (int)nkb, (int)nqb, (int)total_k);   \
      else hipLaunchKernelGGL((bwd::bwd_dkdv_kernel<E, false>), gk, bk, 0, st, p, (int)nkb, (int)nqb, (int)total_k);        \
    }                                                                                                                           \
  } while (0)
  if (dtype == S3R_BF16) S3R_BWD_LAUNCH(bf16_t);
  else S3R_BWD_LAUNCH(f16_t);
#undef S3R_BWD_LAUNCH
  return check_launch("attention backward");
}

int launch_bwd_delta(const void* o, const void* dout, float* delta, int B, int H, int64_t N, int64_t sob, int64_t soh, int64_t son,
                     int64_t sdb, int64_t sdh, int64_t sdn, int dtype, void* stream) {
  const int64_t rows = (int64_t)B * H * N;
  const int64_t blocks = (rows * 8 + 255) / 256;
  if (blocks > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "s3r_attn_bwd_delta: tensor too large for one launch");
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)blocks), blk(256);
  if (dtype == S3R_BF16)
    hipLaunchKernelGGL(bwd::bwd_delta_kernel<bf16_t>, grid, blk, 0, st, (const bf16_t*)o, (const bf16_t*)dout, delta, H, N, rows, sob, soh, son, sdb, sdh, sdn);
  else
    hipLaunchKernelGGL(bwd::bwd_delta_kernel<f16_t>, grid, blk, 0, st, (const f16_t*)o, (const f16_t*)dout, delta, H, N, rows, sob, soh, son, sdb, sdh, sdn);
  return check_launch("bwd_delta_kernel");
}

}  // namespace s3r
