// One pass over the layer's packed q/k/v projection (head_dim 64), HBM bound: every token row of q and k is read once,
// normalised (LayerNorm over the head dimension), rotated (2-D rotary embedding) and written contiguous for the
// attention kernels, and in the same pass the RAW rows of q, k and v are summed into the block means of the compressed
// branch, which are then normalised and rotated at the block's mean position while they are still in registers.  v
// itself is not rewritten: the attention kernels read it in place through its strides.
//
// Replaces, in pi3/models/layers/sparse_attention.py, the pooling of the raw projection (:97-99), q_norm / k_norm, the
// casts and rope of the pooled tokens at their mean positions (:103-110), the three .contiguous() copies and the same
// chain on the full tokens (:115-124): there each of q and k is read three times (pooling, norm, rope) and written
// twice; here 3*N*C elements are read and 2*N*C written.
//
// One wavefront per (batch, head, block).  A lane owns 16 bytes of a row (8 bf16 / 4 fp32 values), 8 (16) lanes own a
// row, the wave covers 8 (4) token rows per step; row statistics are xor-shuffle folds over the lanes of a row, the
// rotation partner (element +-16 inside a half) lives two (four) lanes away.  Rounding points are those of the
// separate kernels (s3r_pool_mean, s3r_norm_rope), and the order of the additions is the pooling kernel's, so all
// results are the same bits as theirs.
#include "prepass.h"

namespace s3r {

// A wave works on one wave-wide step (8 or 4 token rows of q, k and v) while the rows of the next one are on their
// way, and q's temporaries are dead before k's are born: the kernel lives on many resident waves (at most 128
// registers, four per SIMD), not on deep batches per wave -- with two steps computed together the register file held
// half as many waves and the pass took 2.4 times as long.
// ROWS: the full-token q and k are wanted; POOL: the block means are.
template <typename T, bool NORM, bool ROT, bool ROWS, bool POOL>
__global__ __launch_bounds__(256, 4) void qkv_prepass_kernel(PrepassParams p, int64_t Nc, int64_t total) {
#pragma clang fp contract(off)
  constexpr int D = 64;
  constexpr int VEC = 16 / sizeof(T);
  constexpr int LPR = D / VEC;       // lanes per row
  constexpr int RPW = 64 / LPR;      // rows per wave-wide step
  extern __shared__ __align__(16) float staged[];
  const int lane = threadIdx.x & 63;
  const int64_t w_own = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t w = w_own < total ? w_own : total - 1;  // (a wave past the end leaves after the workgroup's barrier)
  // heads fastest: the waves that run side by side read neighbouring 128-byte pieces of the same token rows of the
  // packed projection (one head each), not rows 3*H*128 bytes apart
  const int h = (int)(w % p.H);
  const int64_t bj = w / p.H;
  const int64_t j = bj % Nc;
  const int64_t b = bj / Nc;
  const int r0 = lane / LPR;
  const int lr = lane - r0 * LPR;
  const int64_t t0 = j * p.block;
  const int nvalid = (int)((p.N - t0 < p.block) ? (p.N - t0) : p.block);
  const int64_t in_off = b * p.sxb + h * p.sxh + lr * VEC;
  T* const qo = (T*)p.q_out + ((b * p.H + h) * p.N) * D + lr * VEC;
  T* const ko = (T*)p.k_out + ((b * p.H + h) * p.N) * D + lr * VEC;
  const RotLane<T> rl(lr);

  // The block's positions, fetched with two coalesced loads per 64 tokens (lane l holds values l and 64 + l of the
  // (y, x) pairs) and handed out by shuffles: the table rows of a step then need no load of their own position first.
  int pos_lo = 0, pos_hi = 0;
  int pos_sum = 0;  // lane parity 0: y, 1: x
  auto fetch_positions = [&](int first) {  // tokens first .. first + 63 of the block
    const int ta = first + (lane >> 1), tb = first + 32 + (lane >> 1);
    pos_lo = load_pos(p, b, t0 + (ta < nvalid ? ta : nvalid - 1), lane & 1);
    pos_hi = load_pos(p, b, t0 + (tb < nvalid ? tb : nvalid - 1), lane & 1);
    if constexpr (POOL) pos_sum += (ta < nvalid ? pos_lo : 0) + (tb < nvalid ? pos_hi : 0);
  };

  float aq[VEC], ak[VEC], av[VEC];
#pragma unroll
  for (int i = 0; i < VEC; i++) aq[i] = ak[i] = av[i] = 0.f;

  // the rows of a step (q, k and v: three 16-byte loads per lane) are requested one step ahead
  u32x4 nq, nk, nv = {0, 0, 0, 0};
  auto request = [&](int rbase) {
    const int rr = rbase + r0;
    const int64_t off = in_off + (t0 + (rr < nvalid ? rr : nvalid - 1)) * p.sxn;
    nq = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.q + off));
    nk = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.k + off));
    if constexpr (POOL) nv = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.v + off));
  };
  u32x4 first[ROWS ? 1 : 12];  // block means alone: the rows of the first four steps
  if constexpr (ROWS) {
    request(0);
  } else {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int rr = u * RPW + r0;
      const int64_t off = in_off + (t0 + (rr < nvalid ? rr : nvalid - 1)) * p.sxn;
      if (u * RPW < nvalid) {
        first[3 * u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.q + off));
        first[3 * u + 1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.k + off));
        first[3 * u + 2] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.v + off));
      }
    }
    if constexpr (ROT) {
      for (int t = 0; t < nvalid; t += 64) fetch_positions(t);
    }
  }
  // the first rows are on their way while the workgroup stages its tables
  if constexpr (NORM || ROT) {
    stage_tables<T>(p, staged);
    __syncthreads();
  }
  if (w_own >= total) return;
  // one wave-wide step; WHOLE: all its rows are inside the block (no row to keep out of the sums and the stores)
  auto step = [&](int rbase, auto whole_tag) {
    constexpr bool WHOLE = decltype(whole_tag)::value;
    const int rr = rbase + r0;
    const bool keep = WHOLE || rr < nvalid;
    const int rcl = keep ? rr : nvalid - 1;  // rows beyond the block shadow its last row (not added, not stored)
    if (ROT && (rbase & 63) == 0) fetch_positions(rbase);
    const u32x4 lq = nq, lk = nk, lv = nv;
    if (rbase + RPW < nvalid) request(rbase + RPW);
    int pp = 0;
    if constexpr (ROT && ROWS) {
      const int slot = 2 * (rcl & 63) + rl.half;  // index of (token, y or x) among the fetched 128
      const int from_lo = __shfl(pos_lo, slot & 63), from_hi = __shfl(pos_hi, slot & 63);
      pp = slot < 64 ? from_lo : from_hi;
    }
    TablePtr tab = {};
    if constexpr (ROT && ROWS) tab = table_ptr<T>(p, staged, rl, pp, !rl.second);
    if constexpr (POOL) {
#pragma unroll
      for (int i = 0; i < VEC; i++) av[i] += keep ? to_f32(reinterpret_cast<const T*>(&lv)[i]) : 0.f;
    }
    auto one = [&](const u32x4& raw, float (&acc)[VEC], int ln_row, T* dst) {
      float x[VEC];
#pragma unroll
      for (int i = 0; i < VEC; i++) x[i] = to_f32(reinterpret_cast<const T*>(&raw)[i]);
      if constexpr (POOL) {
#pragma unroll
        for (int i = 0; i < VEC; i++) acc[i] += keep ? x[i] : 0.f;
      }
      if constexpr (ROWS) {
        if constexpr (NORM) norm_row<T>(p, staged, x, ln_row, lr);
        if constexpr (ROT) rotate_row<T>(x, tab);
        if (keep) {
          uint4 o;
#pragma unroll
          for (int i = 0; i < VEC; i++) reinterpret_cast<T*>(&o)[i] = from_f32<T>(x[i]);
          // non-temporal like the loads: nothing of this pass is read again before the attention kernels (0.50 against
          // 0.55 ms at 266 496 tokens x 16 heads)
          store16_nt(dst + (t0 + rr) * D, o);
        }
      }
    };
    one(lq, aq, 0, qo);
    __builtin_amdgcn_sched_barrier(0);  // q's temporaries are dead before k's are born
    one(lk, ak, 2, ko);
  };
  if constexpr (!ROWS) {  // the sums alone: four steps' rows in flight
    for (int rbase = 0; rbase < nvalid; rbase += 4 * RPW) {
      if (rbase > 0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int rr = rbase + u * RPW + r0;
          const int64_t off = in_off + (t0 + (rr < nvalid ? rr : nvalid - 1)) * p.sxn;
          if (rbase + u * RPW < nvalid) {
            first[3 * u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.q + off));
            first[3 * u + 1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.k + off));
            first[3 * u + 2] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.v + off));
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (rbase + u * RPW + r0 < nvalid) {
#pragma unroll
          for (int i = 0; i < VEC; i++) {
            aq[i] += to_f32(reinterpret_cast<const T*>(&first[3 * u])[i]);
            ak[i] += to_f32(reinterpret_cast<const T*>(&first[3 * u + 1])[i]);
            av[i] += to_f32(reinterpret_cast<const T*>(&first[3 * u + 2])[i]);
          }
        }
      }
    }
  }
  for (int rbase = 0; ROWS && rbase < nvalid; rbase += RPW) {  // wave-uniform trip count: the position shuffles span the wave
    if (rbase + RPW <= nvalid) step(rbase, std::true_type{});
    else step(rbase, std::false_type{});
  }
  if constexpr (POOL) {
    // Block means: fold the row groups, divide by the number of valid tokens.  The row groups share the rest of the work:
    // even ones go on with q, odd ones with k (one pass of norm and rotation for both; with 16-token blocks this tail is
    // as long as the block's two steps), the third stores v.
    const bool odd = (r0 & 1) != 0;
    float x[VEC];
#pragma unroll
    for (int i = 0; i < VEC; i++) {
      const float mine = odd ? ak[i] : aq[i], other = odd ? aq[i] : ak[i];
      if constexpr (LPR == 8) {
        x[i] = mine + lane_xor<8>(other);
        av[i] = sum_step<8>(av[i]);
        x[i] = sum_step<32>(sum_step<16>(x[i]));
      } else {
        x[i] = mine + lane_xor<16>(other);
        av[i] = sum_step<16>(av[i]);
        x[i] = sum_step<32>(x[i]);
      }
      av[i] = LPR == 8 ? sum_step<32>(sum_step<16>(av[i])) : sum_step<32>(av[i]);
    }
    const float cnt = (float)nvalid;
    if ((nvalid & (nvalid - 1)) == 0) {  // (wave-uniform) a power of two: its reciprocal is exact and the product the quotient
      const float inv = 1.0f / cnt;
#pragma unroll
      for (int i = 0; i < VEC; i++) {
        x[i] = round_to<T>(x[i] * inv);
        av[i] = round_to<T>(av[i] * inv);
      }
    } else {
#pragma unroll
      for (int i = 0; i < VEC; i++) {
        x[i] = round_to<T>(x[i] / cnt);
        av[i] = round_to<T>(av[i] / cnt);
      }
    }
    const int64_t o = ((b * p.H + h) * Nc + j) * D + lr * VEC;
    auto put = [&](void* dst, const float (&y)[VEC]) {
      uint4 r;
#pragma unroll
      for (int i = 0; i < VEC; i++) reinterpret_cast<T*>(&r)[i] = from_f32<T>(y[i]);
      *reinterpret_cast<uint4*>((T*)dst + o) = r;
    };
    if (r0 == 2) put(p.vc, av);
    void* const raw = odd ? p.k_raw : p.q_raw;
    if (r0 < 2 && raw != nullptr) put(raw, x);
    if (p.finish) {  // the means as tokens of the compressed branch: norm, rotation at the truncated mean position
      if constexpr (NORM) norm_row<T>(p, staged, x, odd ? 2 : 0, lr);
      if constexpr (ROT) {
        const int pc = block_position(pos_sum, cnt, rl.half);
        rotate_row<T>(x, table_ptr<T>(p, staged, rl, pc, !rl.second));
      }
    }
    if (r0 < 2) put(odd ? p.kc : p.qc, x);
  }
}

template <typename T, bool NORM, bool ROT>
static void launch_prepass_t(const PrepassParams& p, bool rows, bool pool, hipStream_t st) {
  const int64_t Nc = (p.N + p.block - 1) / p.block;
  const int64_t total = (int64_t)p.B * p.H * Nc;
  dim3 grid((unsigned)((total + 3) / 4)), blk(256);
  const unsigned lds = NORM || ROT ? (unsigned)staged_bytes(p.staged_rows, ROT) : 0u;
  if (rows && pool) hipLaunchKernelGGL((qkv_prepass_kernel<T, NORM, ROT, true, true>), grid, blk, lds, st, p, Nc, total);
  else if (rows) hipLaunchKernelGGL((qkv_prepass_kernel<T, NORM, ROT, true, false>), grid, blk, lds, st, p, Nc, total);
  else hipLaunchKernelGGL((qkv_prepass_kernel<T, NORM, ROT, false, true>), grid, blk, lds, st, p, Nc, total);
}

template <typename T> static void launch_prepass(const PrepassParams& p, bool rows, bool pool, hipStream_t st) {
  const bool norm = p.qn_w != nullptr, rot = p.pos != nullptr;
  if (norm && rot) launch_prepass_t<T, true, true>(p, rows, pool, st);
  else if (norm) launch_prepass_t<T, true, false>(p, rows, pool, st);
  else if (rot) launch_prepass_t<T, false, true>(p, rows, pool, st);
  else launch_prepass_t<T, false, false>(p, rows, pool, st);
}

// the checks that the forward and the backward pass over the projection share
int check_prepass(const char* who, PrepassParams& p, int D, int dtype) {
  if (!p.q || !p.k || !p.v) return fail(S3R_ERR_BAD_ARG, "%s: null pointer", who);
  if (p.B <= 0 || p.H <= 0 || p.N <= 0 || p.block <= 0) return fail(S3R_ERR_BAD_ARG, "%s: non-positive size", who);
  if (dtype != S3R_F32 && dtype != S3R_BF16 && dtype != S3R_F16) return fail(S3R_ERR_UNSUPPORTED, "%s: dtype %d", who, dtype);
  if (D != 64) return fail(S3R_ERR_UNSUPPORTED, "%s: head_dim %d (built for 64)", who, D);
  if (p.pos != nullptr && (!p.cos_tab || !p.sin_tab || p.P <= 0)) return fail(S3R_ERR_BAD_ARG, "%s: positions without tables", who);
  if ((p.qn_w == nullptr) != (p.kn_w == nullptr)) return fail(S3R_ERR_BAD_ARG, "%s: q and k are normalised together or not at all", who);
  const int es = elt_size(dtype);
  const void* ptrs[] = {p.q, p.k, p.v, p.q_out, p.k_out, p.qc, p.kc, p.vc, p.q_raw, p.k_raw, p.cos_tab, p.sin_tab, p.qn_w, p.qn_b, p.kn_w, p.kn_b};
  for (const void* ptr : ptrs)
    if (ptr != nullptr && !aligned16(ptr)) return fail(S3R_ERR_BAD_ARG, "%s: pointers must be multiples of 16 bytes", who);
  if ((p.sxb * es) % 16 || (p.sxh * es) % 16 || (p.sxn * es) % 16) return fail(S3R_ERR_BAD_ARG, "%s: strides must be multiples of 16 bytes", who);
  const int64_t total = (int64_t)p.B * p.H * ((p.N + p.block - 1) / p.block);
  if ((total + 3) / 4 > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "%s: tensor too large for one launch", who);
  p.staged_rows = p.pos == nullptr ? 0 : p.P < kStagedRows ? p.P : kStagedRows;
  return S3R_OK;
}

}  // namespace s3r

using namespace s3r;

static int run_prepass(const char* who, PrepassParams& p, int D, int dtype, void* stream) {
  const bool rows = p.q_out != nullptr, pool = p.qc != nullptr;
  if ((!rows && !pool) || rows != (p.k_out != nullptr) || pool != (p.kc != nullptr) || pool != (p.vc != nullptr))
    return fail(S3R_ERR_BAD_ARG, "%s: null pointer", who);
  const int rc = check_prepass(who, p, D, dtype);
  if (rc != S3R_OK) return rc;
  if (!rows) p.staged_rows = 0;  // one table row per block: read where it is needed instead of copying the tables
  if (dtype == S3R_F32) launch_prepass<float>(p, rows, pool, (hipStream_t)stream);
  else if (dtype == S3R_BF16) launch_prepass<bf16_t>(p, rows, pool, (hipStream_t)stream);
  else launch_prepass<f16_t>(p, rows, pool, (hipStream_t)stream);
  return check_launch(who);
}

extern "C" int s3r_qkv_prepass(const void* q, const void* k, const void* v, void* q_out, void* k_out, void* qc, void* kc, void* vc,
                               const int32_t* pos, const void* cos_tab, const void* sin_tab, int P, const void* qn_w,
                               const void* qn_b, const void* kn_w, const void* kn_b, float eps, int B, int H, int64_t N, int D,
                               int block, int64_t sxb, int64_t sxh, int64_t sxn, int64_t spb, int64_t spn, int dtype, void* stream) {
  if (!q || !k || !v || !q_out || !k_out || !qc || !kc || !vc) return fail(S3R_ERR_BAD_ARG, "s3r_qkv_prepass: null pointer");
  PrepassParams p = {};
  p.q = q; p.k = k; p.v = v; p.q_out = q_out; p.k_out = k_out; p.qc = qc; p.kc = kc; p.vc = vc;
  p.pos = pos; p.cos_tab = cos_tab; p.sin_tab = sin_tab; p.P = P;
  p.qn_w = qn_w; p.qn_b = qn_b; p.kn_w = kn_w; p.kn_b = kn_b; p.eps = eps;
  p.B = B; p.H = H; p.N = N; p.block = block; p.sxb = sxb; p.sxh = sxh; p.sxn = sxn; p.spb = spb; p.spn = spn;
  return run_prepass("s3r_qkv_prepass", p, D, dtype, stream);
}

extern "C" int s3r_layer_prepass(const s3r_prepass_args* a, void* stream) {
  if (!a) return fail(S3R_ERR_BAD_ARG, "s3r_layer_prepass: null pointer");
  PrepassParams p = prepass_params(*a);
  return run_prepass("s3r_layer_prepass", p, a->head_dim, a->dtype, stream);
}
