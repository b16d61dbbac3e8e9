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
//   * bwd_delta_kernel: delta[b,h,n] = sum_d o * dO in fp32 (HBM bound).
//   * bwd_dq_kernel: one wavefront per 64-row query block, four independent waves per workgroup; walks the block's
//     selected key tiles (or all of them).  Everything is computed transposed, as in the forward kernels:
//     S^T = K Q^T and dP^T = V dO^T put one QUERY per lane, so lse and delta are per-lane scalars;
//     dQ^T += K^T dS^T takes K^T fragments from ds_read_b64_tr_b16.  K and V half tiles (32 keys) go global -> LDS
//     by direct transfers, double buffered (16 KB per wave).  The K half is staged once, in a layout that serves
//     the transposed reads and the row reads (A operand of S^T) without bank conflicts.
//   * bwd_dkdv_kernel: one workgroup of two waves per 64-key block, each wave owns 32 keys (one KEY per lane:
//     S = Q K^T, dP = dO V^T with K, V fragments in registers as B operands) and walks the query blocks that
//     selected the key block (key-centric lists built by the host from the index tensor, reference :423-554).
//     Q and dO tiles (64 queries) and the matching lse / delta values go global -> LDS, shared by the two waves,
//     double buffered (the next tile's transfers fly during a whole tile of work), one barrier per tile;
//     dV^T += dO^T P and dK^T += Q^T dS read their A operands transposed from the same buffers.
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

// ---- shared pieces of the two MFMA kernels -----------------------------------------------------------------------
// Transfer of rows [8*i0*.., ...) of a 32-row half tile: instruction i moves rows 8i .. 8i+7 (16 bytes per lane).
// LDS chunk (row, c') holds head_dim chunk c' ^ k_swizzle(row) in every tile: 16-byte row reads and
// ds_read_b64_tr_b16 reads both run without bank conflicts with it.  (VSW marks the tiles that are also read
// transposed; the map is the same.)  Rows are clamped to `last` (relative to `base`'s row 0).
template <typename E, bool VSW>
__device__ __forceinline__ void dma_rows(const E* base, uint32_t rowbytes, int first_row, int last, char* lds_half, int lane, int i_begin, int i_end) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x00020000);
  const int lr = lane >> 3;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (i >= i_begin && i < i_end) {
      const int ldsrow = 8 * i + lr;
      int row = first_row + ldsrow;
      row = row < last ? row : last;
      const int chunk = (lane & 7) ^ k_swizzle(ldsrow);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(lds_half + i * 1024), 16,
                                               (uint32_t)row * rowbytes + (uint32_t)(chunk * 16), 0, 0, 0);
    }
  }
}

// A operand from row reads of a half tile: lane = row c, k-step ks: head_dim chunk 2ks + hh.
template <typename E, bool VSW>
__device__ __forceinline__ void read_rows(const char* half, int c, int hh, typename Mma<E>::V8 (&dst)[4]) {
  const int sw = k_swizzle(c);
#pragma unroll
  for (int ks = 0; ks < 4; ks++) {
    Frag f;
    f.u = *reinterpret_cast<const uint4*>(half + c * 128 + (((2 * ks + hh) ^ sw) << 4));
    dst[ks] = as_v8<E>(f);
  }
}

template <typename E, bool VSW>
__device__ __forceinline__ typename Mma<E>::V8 read_row_frag(const char* half, int c, int hh, int ks) {
  const int sw = k_swizzle(c);
  Frag f;
  f.u = *reinterpret_cast<const uint4*>(half + c * 128 + (((2 * ks + hh) ^ sw) << 4));
  return as_v8<E>(f);
}

// A operand X^T from transposed reads of a half tile staged with VSW: fragment [jj][dt] holds, for head_dim row
// dt*32 + c, the 8 rows 16jj + {4hh..4hh+3, 8+4hh..8+4hh+3} of the half: the order in which a 32x32 accumulator
// with one column per lane hands over its registers 8jj .. 8jj+7.
template <typename E>
__device__ __forceinline__ void read_transposed(const char* half, int tr_off, typename Mma<E>::V8 (&dst)[2][2]) {
#pragma unroll
  for (int jj = 0; jj < 2; jj++)
#pragma unroll
    for (int dt = 0; dt < 2; dt++) {
      const char* a0 = half + (tr_off ^ (dt * 64)) + (jj * 16) * 128;
      const char* a8 = half + (tr_off ^ (dt * 64) ^ (k_swizzle(8) << 4)) + (jj * 16 + 8) * 128;  // rows 8 further down: chunk map ^ k_swizzle(8)
      Frag f;
      f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a0));
      f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a8));
      dst[jj][dt] = as_v8<E>(f);
    }
}

template <typename E>
__device__ __forceinline__ typename Mma<E>::V8 read_transposed_frag(const char* half, int tr_off, int jj, int dt) {
  const char* a0 = half + (tr_off ^ (dt * 64)) + (jj * 16) * 128;
  const char* a8 = half + (tr_off ^ (dt * 64) ^ (k_swizzle(8) << 4)) + (jj * 16 + 8) * 128;
  Frag f;
  f.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a0));
  f.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(a8));
  return as_v8<E>(f);
}

__device__ __forceinline__ int tr_offset(int lane) {
  const int hh = lane >> 5;
  const int i16 = lane & 15;
  const int tr_row = 4 * hh + (i16 >> 2);
  const int tr_chunk = (((lane >> 4) & 1) * 2 + ((i16 & 3) >> 1)) ^ k_swizzle(tr_row);
  return tr_row * 128 + tr_chunk * 16 + (i16 & 1) * 8;
}

// Store of a transposed 64 x 64 accumulator pair acc[dt] (lane = row of the output, registers = head_dim values
// dt*32 + 8*(r/4) + 4*hh + r%4): one exchange with lane ^ 32 per packed word gives every lane 8 consecutive values.
template <typename E>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[2], E* rowptr, bool live, int hh) {
#pragma unroll
  for (int dt = 0; dt < 2; dt++)
#pragma unroll
    for (int gp = 0; gp < 2; gp++) {
      union { E e[8]; uint32_t w[4]; uint4 u; } pc;
      union { E e[2]; uint32_t w; } t;
#pragma unroll
      for (int wi = 0; wi < 2; wi++) {
        t.e[0] = (E)acc[dt][8 * gp + 2 * wi];
        t.e[1] = (E)acc[dt][8 * gp + 2 * wi + 1];
        const uint32_t a = t.w;
        t.e[0] = (E)acc[dt][8 * gp + 4 + 2 * wi];
        t.e[1] = (E)acc[dt][8 * gp + 4 + 2 * wi + 1];
        const uint32_t bw = t.w;
        const auto r = __builtin_amdgcn_permlane32_swap(a, bw, false, false);
        pc.w[wi] = r[0];
        pc.w[2 + wi] = r[1];
      }
      if (live) *reinterpret_cast<uint4*>(rowptr + dt * 32 + 8 * (2 * gp + hh)) = pc.u;
    }
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
// us, before / now: 266 496 tokens x 16 heads, top-16 1 902 / 1 531 (1.1 PFLOP/s: matrix cores and vector unit have the same work, 1 536
// cycles each per tile, and the chip runs below 2 GHz under it), dense over 4 164 tokens 212 / 161.
template <typename E, bool DENSE>
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
  // B operands Q and dO: lane = query 16 qt + c, head dimensions 32 ks + 8 g ..
  V8 bq[4][2], bg[4][2];
  float nl[4];    // log2(scale) - lse log2(e)
  f32x4 nd[4];    // -delta, what the products of dP^T start from
  const float log2_scale = __builtin_amdgcn_logf(p.scale);
#pragma unroll
  for (int qt = 0; qt < 4; qt++) {
    const int64_t row = q0 + qt * 16 + c;
    const bool live = row < Lq;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      Frag f, d;
      f.u = make_uint4(0, 0, 0, 0);
      d.u = make_uint4(0, 0, 0, 0);
      if (live) {
        f.u = *reinterpret_cast<const uint4*>(qp + row * p.sqm + ks * 32 + g * 8);
        d.u = *reinterpret_cast<const uint4*>(gp + row * p.sgm + ks * 32 + g * 8);
      }
      bq[qt][ks] = as_v8<E>(f);
      bg[qt][ks] = as_v8<E>(d);
    }
    nl[qt] = live ? fmaf(lsep[row], -kLog2e, log2_scale) : -INFINITY;
    const float m = live ? -dlp[row] : 0.f;
    nd[qt] = (f32x4){m, m, m, m};
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
          asm volatile("" : "+v"(st[B][t]));
          x0 = fmaf(st[B][t][r], sl2, nl[QT]);
          x1 = fmaf(st[B][t][r + 1], sl2, nl[QT]);
          e0 = __builtin_amdgcn_exp2f(x0);
          asm volatile("" : "+v"(x1), "+v"(e0));
        } else if constexpr (s == 1) {
          e1 = __builtin_amdgcn_exp2f(x1);
          e0 *= dp[B][t][r];
          asm volatile("" : "+v"(e0), "+v"(e1));
        } else {
          e1 *= dp[B][t][r + 1];
          uint32_t wd = pair_of(e0, e1);
          asm volatile("" : "+v"(wd));
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
template <typename E, bool DENSE>
__global__ __launch_bounds__(128, 2) void bwd_dkdv_kernel(BwdParams p, int nkb, int nqb_all, int total_wg) {
  typedef typename Mma<E>::V8 V8;
  constexpr int kTileBytes = 2 * kHalfBytes;  // a 64-row query tile
  __shared__ __attribute__((aligned(1024))) unsigned char lds_q0[kTileBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_q1[kTileBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_g0[kTileBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_g1[kTileBytes];
  // per-query scalars of a tile: [0,64) lse, [64,128) delta
  constexpr int kDeltaAt = 64;
  __shared__ __attribute__((aligned(256))) float lds_s0[128];
  __shared__ __attribute__((aligned(256))) float lds_s1[128];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int hh = lane >> 5;
  const int c = lane & 31;

  // With lists the grid has two passes over the key blocks: the first (workgroups [0, total_wg)) takes the blocks whose
  // lists are long, the second the others, so the longest lists of a skewed index tensor start first instead of
  // wherever their key block falls in the launch order.
  const bool long_pass = DENSE || (int)blockIdx.x < total_wg;
  const int w = (int)blockIdx.x < total_wg ? (int)blockIdx.x : (int)blockIdx.x - total_wg;
  const int xcd = w & 7, slot = w >> 3;
  const int per = total_wg >> 3, rem = total_wg & 7;
  const int vid = xcd * per + (xcd < rem ? xcd : rem) + slot;
  const int bh = vid / nkb;
  const int kb = vid - bh * nkb;
  const int b = bh / p.H;
  const int h = bh - b * p.H;

  const int64_t Lq = p.Lq, Lk = p.Lk;
  if constexpr (!DENSE) {
    const int32_t* off = p.kq_off + ((int64_t)b * p.H + h) * (nkb + 1);
    int len = off[kb + 1] - off[kb];
    len = __builtin_amdgcn_readfirstlane(len);
    if ((len > 4 * p.K) != long_pass) return;
  }
  const E* qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const E* kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const E* vp = (const E*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  const E* gp = (const E*)p.dout + (int64_t)b * p.sgb + (int64_t)h * p.sgh;
  const float* lsep = p.lse + ((int64_t)b * p.H + h) * Lq;
  const float* dlp = p.delta + ((int64_t)b * p.H + h) * Lq;

  // B operands K and V of this wave's 32 keys (lane = key, head_dim chunk hh + 2 ks)
  const int64_t key = (int64_t)kb * 64 + wave * 32 + c;
  V8 bk[4], bv[4];
  f32x16 dkt[2], dvt[2];  // dK^T, dV^T [dt]: lane = key, registers = head_dim
  auto load_keys = [&]() {
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      Frag f, g;
      f.u = make_uint4(0, 0, 0, 0);
      g.u = make_uint4(0, 0, 0, 0);
      if (key < Lk) {
        f.u = *reinterpret_cast<const uint4*>(kp + key * p.skn + ks * 16 + hh * 8);
        g.u = *reinterpret_cast<const uint4*>(vp + key * p.svn + ks * 16 + hh * 8);
      }
      bk[ks] = as_v8<E>(f);
      bv[ks] = as_v8<E>(g);
    }
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) { dkt[dt][r] = 0.f; dvt[dt][r] = 0.f; }
  };
  load_keys();

  // query blocks that attend to this key block
  int n_lists;
  const int32_t* list = nullptr;
  if constexpr (DENSE) {
    n_lists = nqb_all;
  } else {
    const int32_t* off = p.kq_off + ((int64_t)b * p.H + h) * (nkb + 1);
    const int32_t lo = off[kb], hi = off[kb + 1];
    n_lists = hi - lo;
    list = p.kq_list + ((int64_t)b * p.H + h) * p.list_stride + lo;
  }
  // List entries come 64 at a time (lane l holds entry base + l), so the latency of the list read is paid once per
  // 64 tiles and not in front of every tile's transfers.  The lists are walked front to back.
  int32_t held_a = -1;
  int base_a = -64;
  auto entry = [&](const int32_t* lst, int len, int32_t& held, int& base, int i) -> int32_t {
    if (i >= base + 64) {
      base = i & ~63;
      held = base + lane < len ? lst[base + lane] : -1;
    }
    return __builtin_amdgcn_readlane(held, i - base);
  };
  auto block_of = [&](int i) -> int64_t {
    if constexpr (DENSE) {
      return (int64_t)i;
    } else {
      return (int64_t)entry(list, n_lists, held_a, base_a, i);
    }
  };

  const float scale = p.scale;
  const float sl2 = scale * kLog2e;
  // The per-query terms ride in the accumulators instead of in the vector slots.  The accumulator of S starts at
  // -lse / scale, so P = exp2(scale * log2(e) * accumulator); the accumulator of dP starts at -delta, so
  // dS / scale = P * accumulator.  No slot then begins with an LDS read of per-query values in front of the arithmetic
  // that needs them: the start values come with four ds_read_b128 per accumulator ahead of the half's products (those of
  // the second half's dP a quarter per slot, next to the fragments of its products).  bf16 also puts the softmax scale
  // onto dK once at the end (the rounding of dS to the I/O type is relative and does not care for the factor): per score
  // a multiplication, an exponential and a multiplication instead of two fused multiply-adds, an exponential and a
  // multiplication; fp16, with its narrow range, scales every dS.  bf16, 266 496 tokens, top-16: 2.88 -> 2.79 (delta) ->
  // 2.62 ms (lse).
  const float inv_scale = 1.0f / scale;
  constexpr bool FOLD = true;  // (kept as a switch: the other form reads lse and delta from LDS inside the vector slots)
  constexpr bool LATE_SCALE = std::is_same<E, bf16_t>::value;  // the softmax scale goes onto dK at the end
  const uint32_t qrow = (uint32_t)p.sqm * (uint32_t)sizeof(E), grow = (uint32_t)p.sgm * (uint32_t)sizeof(E);
  const int tr_off = tr_offset(lane);
  // (one per parity of the instruction inside its half tile: the chunk map of rows 8..15 differs from that of rows 0..7)
  const uint32_t q_voff[2] = {(uint32_t)(lane >> 3) * qrow + (uint32_t)(((lane & 7) ^ k_swizzle(lane >> 3)) * 16),
                              (uint32_t)(lane >> 3) * qrow + (uint32_t)(((lane & 7) ^ k_swizzle((lane >> 3) + 8)) * 16)};
  const uint32_t g_voff[2] = {(uint32_t)(lane >> 3) * grow + (uint32_t)(((lane & 7) ^ k_swizzle(lane >> 3)) * 16),
                              (uint32_t)(lane >> 3) * grow + (uint32_t)(((lane & 7) ^ k_swizzle((lane >> 3) + 8)) * 16)};

  float staged = 0.f;          // this lane's lse or delta value of the tile in flight, as loaded (wave 0 lse, wave 1 delta)
  bool staged_inf = false;     // rows past the end of the tensor publish lse = +inf
  int staged_buf = -1;         // (wave-uniform) the buffer it goes to; -1: nothing staged
  // One query tile (64 rows of Q and dO, 64 lse and delta values) -> buffer BUF; each wave moves half of every
  // operand (instructions 2*wave, 2*wave+1 of both 32-row halves), wave 0 the lse values, wave 1 delta.
  auto fetch = [&](int64_t qblk, auto bufc) {
    constexpr int BUF = decltype(bufc)::value;
    char* qb = reinterpret_cast<char*>(BUF == 0 ? lds_q0 : lds_q1);
    char* gb = reinterpret_cast<char*>(BUF == 0 ? lds_g0 : lds_g1);
    const int64_t start = qblk * 64;
    const int last = (int)((Lq - start < 64 ? Lq - start : 64) - 1);
    if (last >= 63) {
      // (wave-uniform) a full tile: per-lane offsets (row lane/8 and its chunk) that do not depend on the tile, the
      // instruction's rows ride in the scalar offset
      const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void*)(qp + start * p.sqm), 0, 0x7fffffff, 0x00020000);
      const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc((void*)(gp + start * p.sgm), 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int hf = 0; hf < 2; hf++)
#pragma unroll
        for (int ii = 0; ii < 2; ii++) {
          const int i = 2 * wave + ii;
          const uint32_t rows = (uint32_t)(32 * hf + 8 * i);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (__attribute__((address_space(3))) void*)(qb + hf * kHalfBytes + i * 1024), 16,
                                                   q_voff[ii], rows * qrow, 0, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (__attribute__((address_space(3))) void*)(gb + hf * kHalfBytes + i * 1024), 16,
                                                   g_voff[ii], rows * grow, 0, 0);
        }
    } else {
#pragma unroll
      for (int hf = 0; hf < 2; hf++) {
        dma_rows<E, true>(qp + start * p.sqm, qrow, 32 * hf, last, qb + hf * kHalfBytes, lane, 2 * wave, 2 * wave + 2);
        dma_rows<E, true>(gp + start * p.sgm, grow, 32 * hf, last, gb + hf * kHalfBytes, lane, 2 * wave, 2 * wave + 2);
      }
    }
    // per-query scalars pass through a register and are stored to LDS by `publish` before the barrier that opens
    // the tile
    const int r = lane < last ? lane : last;
    staged = ((wave == 0 ? lsep : dlp) + start)[r];
    staged_inf = wave == 0 && lane > last;  // query rows beyond Lq: lse = +inf, no probability
    staged_buf = BUF;
  };
  // The loaded value is first touched here, a whole tile of work after its load: any arithmetic on it inside `fetch`
  // would make the wave wait for the load there, and with it (the counter is in order) for the tile transfers issued
  // just before, which is the tile that should be in flight during the current tile's work.
  auto publish = [&]() {
    if (staged_buf < 0) return;
    float* const sb = staged_buf == 0 ? lds_s0 : lds_s1;
    // scaled once here (lse to base 2, delta by the softmax scale) instead of once per score
    if constexpr (FOLD) sb[64 * wave + lane] = staged_inf ? -INFINITY : wave == 0 ? -staged * inv_scale : -staged;
    else sb[64 * wave + lane] = staged_inf ? INFINITY : staged * (wave == 0 ? kLog2e : scale);
    staged_buf = -1;
  };
  // One tile in three stages per 32-query half (A = row reads + S, dP; B = P and dS from the per-query scalars; C =
  // transposed reads + dV^T, dK^T) with every instruction placed by hand, as in the forward kernel.  The vector work of
  // a 32-query half (16 scores per lane: P, dS, their roundings) is cut into eight slots of two scores; each slot also
  // issues one matrix product of another stage: the scores of half 1 run under the vector work of half 0, the dV / dK
  // products of half 0 under the vector work of half 1.  Only the scores of half 0 and the products of half 1 have no
  // vector work to hide behind.  Query rows beyond Lq need no masks: their lse is +inf.
  auto tile64 = [&](auto bufc) {
    constexpr int BUF = decltype(bufc)::value;
    const char* qb = reinterpret_cast<const char*>(BUF == 0 ? lds_q0 : lds_q1);
    const char* gb = reinterpret_cast<const char*>(BUF == 0 ? lds_g0 : lds_g1);
    const float* sb = BUF == 0 ? lds_s0 : lds_s1;
    f32x16 sc[2], dpv[2];   // S and dP of the two halves
    V8 pbv[2][2], dbv[2][2];  // P and dS as B operands [half][jj]
    V8 aq[4], ag[4];          // row fragments of Q, dO (A operands of the scores)
    V8 gt[2][2], qt[2][2];    // transposed fragments of dO, Q (A operands of dV^T, dK^T)
    auto mma_a = [&](auto hf_tag, auto i_tag) {  // product i of 8 of a half's scores: 0-3 S, 4-7 dP
      constexpr int HF = decltype(hf_tag)::value, i = decltype(i_tag)::value, ks = i & 3;
      f32x16 z;
#pragma unroll
      for (int r = 0; r < 16; r++) z[r] = 0.f;
      if constexpr (i < 4) sc[HF] = Mma<E>::mma(aq[ks], bk[ks], ks == 0 && !FOLD ? z : sc[HF]);
      else dpv[HF] = Mma<E>::mma(ag[ks], bv[ks], ks == 0 && !FOLD ? z : dpv[HF]);
    };
    // FOLD: the accumulator of a half's dP starts at minus delta of its queries (registers 4g .. 4g+3 hold the queries
    // 4hh + 8g .. + 3 of the half)
    auto lse_init = [&](auto hf_tag) {
      constexpr int HF = decltype(hf_tag)::value;
      if constexpr (FOLD) {
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
          const float4 l4 = *reinterpret_cast<const float4*>(sb + 32 * HF + 4 * hh + 8 * g4);
          sc[HF][4 * g4] = l4.x;
          sc[HF][4 * g4 + 1] = l4.y;
          sc[HF][4 * g4 + 2] = l4.z;
          sc[HF][4 * g4 + 3] = l4.w;
        }
      }
    };
    auto delta_init_piece = [&](auto hf_tag, auto g_tag) {  // registers 4g .. 4g+3 of the half's dP accumulator
      constexpr int HF = decltype(hf_tag)::value, g4 = decltype(g_tag)::value;
      if constexpr (FOLD) {
        const float4 d4 = *reinterpret_cast<const float4*>(sb + kDeltaAt + 32 * HF + 4 * hh + 8 * g4);
        dpv[HF][4 * g4] = d4.x;
        dpv[HF][4 * g4 + 1] = d4.y;
        dpv[HF][4 * g4 + 2] = d4.z;
        dpv[HF][4 * g4 + 3] = d4.w;
      }
    };
    auto delta_init = [&](auto hf_tag) {
      lse_init(hf_tag);
      static_for<4>([&](auto g_tag) { delta_init_piece(hf_tag, g_tag); });
    };
    auto mma_c = [&](auto hf_tag, auto i_tag) {  // product i of 8 of a half's dV^T / dK^T updates
      constexpr int HF = decltype(hf_tag)::value, i = decltype(i_tag)::value, jj = (i >> 1) & 1, dt = i & 1;
      if constexpr (i < 4) dvt[dt] = Mma<E>::mma(gt[jj][dt], pbv[HF][jj], dvt[dt]);
      else dkt[dt] = Mma<E>::mma(qt[jj][dt], dbv[HF][jj], dkt[dt]);
    };
    auto vec = [&](auto hf_tag, auto j_tag) {  // scores 2j, 2j+1 of the half: P, dS, both rounded
      constexpr int HF = decltype(hf_tag)::value, j = decltype(j_tag)::value, r = 2 * j;
      // queries 4hh + 8(j/2) + 2(j%2) + {0, 1} of the half
      f32x16& sh = sc[HF];
      f32x16& dh = dpv[HF];
      float p0, p1, e0, e1;
      if constexpr (FOLD) {
        p0 = __builtin_amdgcn_exp2f(sh[r] * sl2);
        p1 = __builtin_amdgcn_exp2f(sh[r + 1] * sl2);
        e0 = LATE_SCALE ? p0 * dh[r] : p0 * (dh[r] * scale);
        e1 = LATE_SCALE ? p1 * dh[r + 1] : p1 * (dh[r + 1] * scale);
      } else {
        const float2 l2 = *reinterpret_cast<const float2*>(sb + 32 * HF + 4 * hh + 8 * (j >> 1) + 2 * (j & 1));
        p0 = __builtin_amdgcn_exp2f(fmaf(sh[r], sl2, -l2.x));
        p1 = __builtin_amdgcn_exp2f(fmaf(sh[r + 1], sl2, -l2.y));
        const float2 d2 = *reinterpret_cast<const float2*>(sb + kDeltaAt + 32 * HF + 4 * hh + 8 * (j >> 1) + 2 * (j & 1));
        e0 = p0 * fmaf(dh[r], scale, -d2.x);
        e1 = p1 * fmaf(dh[r + 1], scale, -d2.y);
      }
      V8& pv = pbv[HF][r >> 3];
      V8& dv = dbv[HF][r >> 3];
      pv[r & 7] = (E)p0;
      pv[(r & 7) + 1] = (E)p1;
      dv[r & 7] = (E)e0;
      dv[(r & 7) + 1] = (E)e1;
    };
    read_rows<E, true>(qb, c, hh, aq);
    read_rows<E, true>(gb, c, hh, ag);
    delta_init(H0{});
    static_for<8>([&](auto i_tag) { mma_a(H0{}, i_tag); });
    __builtin_amdgcn_sched_barrier(0);
    // the fragments of a region's second four products are requested four slots ahead, one per slot, so that at most
    // five fragments are in registers at a time
    read_rows<E, true>(qb + kHalfBytes, c, hh, aq);
    lse_init(H1{});
    static_for<8>([&](auto j_tag) {
      constexpr int j = decltype(j_tag)::value;
      if constexpr (j < 4) ag[j] = read_row_frag<E, true>(gb + kHalfBytes, c, hh, j);
      if constexpr (j < 4) delta_init_piece(H1{}, j_tag);  // (a quarter per slot: needed from the fifth product on)
      mma_a(H1{}, j_tag);
      vec(H0{}, j_tag);
      __builtin_amdgcn_sched_barrier(0);
    });
    read_transposed<E>(gb, tr_off, gt);
    static_for<8>([&](auto j_tag) {
      constexpr int j = decltype(j_tag)::value;
      if constexpr (j < 4) qt[(j >> 1) & 1][j & 1] = read_transposed_frag<E>(qb, tr_off, (j >> 1) & 1, j & 1);
      mma_c(H0{}, j_tag);
      vec(H1{}, j_tag);
      __builtin_amdgcn_sched_barrier(0);
    });
    read_transposed<E>(gb + kHalfBytes, tr_off, gt);
    read_transposed<E>(qb + kHalfBytes, tr_off, qt);
    static_for<8>([&](auto i_tag) { mma_c(H1{}, i_tag); });
  };
  // this wave's part of the tile has landed, its reads of the other buffer are done; after the barrier both hold
  // for both waves
  auto sync = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    publish();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
  };

  auto walk = [&]() {  // all tiles of the current list, double buffered
    if (n_lists > 0) {
      int64_t cur = block_of(0);
      fetch(cur, H0{});
      for (int t = 0; t < n_lists; t += 2) {
        sync();
        const bool more1 = t + 1 < n_lists;
        const int64_t nxt1 = more1 ? block_of(t + 1) : cur;
        if (more1) fetch(nxt1, H1{});
        tile64(H0{});
        if (!more1) break;
        sync();
        const bool more2 = t + 2 < n_lists;
        cur = more2 ? block_of(t + 2) : nxt1;
        if (more2) fetch(cur, H0{});
        tile64(H1{});
      }
    }
  };
  E* dkp = (E*)p.dk + (int64_t)b * p.sdkb + (int64_t)h * p.sdkh;
  E* dvp = (E*)p.dv + (int64_t)b * p.sdvb + (int64_t)h * p.sdvh;
  walk();
  if constexpr (LATE_SCALE) {
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) dkt[dt][r] *= scale;
  }
  store_rows<E>(dkt, dkp + key * p.sdkn, key < Lk, hh);
  store_rows<E>(dvt, dvp + key * p.sdvn, key < Lk, hh);
}

}  // namespace bwd

int launch_attn_bwd(const BwdParams& p, int dtype, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  const bool dense = p.idx == nullptr;
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
      if (dense) hipLaunchKernelGGL((bwd::bwd_dq_kernel<E, true>), gq, bq, 0, st, p, (int)nqb, (int)nqg, (int)total_q);     \
      else hipLaunchKernelGGL((bwd::bwd_dq_kernel<E, false>), gq, bq, 0, st, p, (int)nqb, (int)nqg, (int)total_q);          \
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
