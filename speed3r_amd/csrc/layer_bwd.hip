// Backward of what surrounds the two attention operators in the layer (head_dim 64, bf16 / fp16), both HBM bound:
//   gated merge  (pi3/models/layers/sparse_attention.py:127-136)  -> s3r_gated_merge_bwd
//   block means, qk-norm and rotary embedding of the packed projection (:97-110,115-124)  -> s3r_layer_prepass_bwd
// Differentiated by autograd these expressions are some 250 launches over fp32 and 16-bit copies of every tensor (5.5 of
// the 7.8 ms of a training step of one layer at 24 192 tokens); here each tensor is read and written once, sums are fp32
// and each gradient is rounded once.  At that size: merge 33 us = 4.5 TB/s, projection 94 us = 4.2 TB/s (a large copy on this card: 4.8).
#include "prepass.h"

namespace s3r {

// Lane layout of both kernels as in the forward pass: a wave owns one (batch, head, block), a lane 16 bytes of a row, 8
// lanes a row, 8 rows per step; heads fastest, so that neighbouring waves touch neighbouring 128-byte pieces of the
// [B,N,H*64] tensors.

// out[b,n,h*64+d] = g0 * oc[b,h,n/block,d] + g1 * os[b,h,n,d]:
//   d_os = g1 * dout, d_oc = sum over the block of g0 * dout, d_g0 = <dout, oc>, d_g1 = <dout, os>,
// and the row sums <d_oc, oc>, <d_os, os> ("delta") that both attention backwards start from, of the rounded gradients.
template <typename T>
__global__ __launch_bounds__(256) void merge_bwd_kernel(const T* __restrict__ dout, const T* __restrict__ oc, const T* __restrict__ os,
                                                        const T* __restrict__ gate, T* __restrict__ d_oc, T* __restrict__ d_os,
                                                        T* __restrict__ d_gate, float* __restrict__ delta_c, float* __restrict__ delta_s,
                                                        int H, int64_t N, int block, int64_t Nc, int64_t total, int64_t sgb, int64_t sgh, int64_t sgn) {
  constexpr int D = 64, VEC = 8, LPR = 8, RPW = 8;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= total) return;
  const int lane = threadIdx.x & 63, r0 = lane >> 3, lr = lane & 7;
  const int h = (int)(w % H);
  const int64_t bj = w / H, j = bj % Nc, b = bj / Nc, bh = b * H + h;
  const int64_t t0 = j * block;
  const int nvalid = (int)((N - t0 < block) ? (N - t0) : block);
  float c[VEC], acc[VEC];
  const uint4 rc = *reinterpret_cast<const uint4*>(oc + (bh * Nc + j) * D + lr * VEC);
#pragma unroll
  for (int i = 0; i < VEC; i++) {
    c[i] = to_f32(reinterpret_cast<const T*>(&rc)[i]);
    acc[i] = 0.f;
  }
  const T* const gp = gate + b * sgb + h * sgh;
  for (int r = r0; r - r0 < nvalid; r += RPW) {
    const bool keep = r < nvalid;
    const int64_t n = t0 + (keep ? r : nvalid - 1);
    const u32x4 ro = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(os + (bh * N + n) * D + lr * VEC));
    const u32x4 rd = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(dout + ((b * N + n) * H + h) * D + lr * VEC));
    const float g0 = to_f32(gp[n * sgn]), g1 = to_f32(gp[n * sgn + 1]);
    float s0 = 0.f, s1 = 0.f, ds = 0.f;
    uint4 out;
#pragma unroll
    for (int i = 0; i < VEC; i++) {
      const float d = to_f32(reinterpret_cast<const T*>(&rd)[i]), o = to_f32(reinterpret_cast<const T*>(&ro)[i]);
      s0 += d * c[i];
      s1 += d * o;
      acc[i] += keep ? g0 * d : 0.f;
      const float e = round_to<T>(g1 * d);
      reinterpret_cast<T*>(&out)[i] = from_f32<T>(e);
      ds += e * o;
    }
    s0 = group_sum<LPR>(s0);
    s1 = group_sum<LPR>(s1);
    ds = group_sum<LPR>(ds);
    if (keep) {
      *reinterpret_cast<uint4*>(d_os + (bh * N + n) * D + lr * VEC) = out;
      if (lr == 0) {
        T* const dg = d_gate + ((b * N + n) * H + h) * 2;
        dg[0] = from_f32<T>(s0);
        dg[1] = from_f32<T>(s1);
        delta_s[bh * N + n] = ds;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < VEC; i++) acc[i] = across_groups<LPR>(acc[i]);
  uint4 out;
  float dc = 0.f;
#pragma unroll
  for (int i = 0; i < VEC; i++) {
    const float e = round_to<T>(acc[i]);
    reinterpret_cast<T*>(&out)[i] = from_f32<T>(e);
    dc += e * c[i];
  }
  dc = group_sum<LPR>(dc);
  if (r0 == 0) *reinterpret_cast<uint4*>(d_oc + (bh * Nc + j) * D + lr * VEC) = out;
  if (lane == 0) delta_c[bh * Nc + j] = dc;
}

struct PrepassGrads {
  const void *dq, *dk, *dv;     // contiguous [B,H,N,64]: gradients of the rotated q and k, of v
  const void *dqc, *dkc, *dvc;  // contiguous [B,H,Nc,64]: of the finished block means
  void* dx[3];                  // gradients of the raw q, k, v: views with the projection's strides
  float* partial;               // [workgroups, 256]: sums for q_norm weight, bias, k_norm weight, bias
};

// Gradient of a rotated row with respect to the row before the rotation: its transpose (the minus sign is on the sine of
// the second quarter).
template <typename T, int VEC> __device__ __forceinline__ void rotate_row_bwd(float (&d)[VEC], const TablePtr& t) {
  float cs[VEC], sn[VEC];
  load_row(t.c, cs);
  load_row(t.s, sn);
#pragma unroll
  for (int i = 0; i < VEC; i++) {
    const float other = lane_xor<RotLane<T>::QL>(d[i]);
    d[i] = d[i] * cs[i] + other * sn[i];
  }
}

// Gradient of LayerNorm: d (in: of the normalised row, out: of the raw row x); the parameters' sums where `count`.
template <int VEC>
__device__ __forceinline__ void norm_row_bwd(const PrepassParams& p, const float* staged, const float (&x)[VEC], float (&d)[VEC], int ln_row, int lr,
                                             float (&dw)[VEC], float (&db)[VEC], bool count) {
  constexpr int LPR = 64 / VEC;
  const float* lw = staged + 3 * p.staged_rows * 16 + ln_row * 64 + lr * VEC;
  float s = 0.f, var = 0.f, m1 = 0.f, m2 = 0.f;
#pragma unroll
  for (int i = 0; i < VEC; i++) s += x[i];
  const float mean = group_sum<LPR>(s) * (1.0f / 64);
#pragma unroll
  for (int i = 0; i < VEC; i++) var += (x[i] - mean) * (x[i] - mean);
  const float rstd = inv_sqrt(group_sum<LPR>(var) * (1.0f / 64) + p.eps);
#pragma unroll
  for (int i = 0; i < VEC; i++) {
    const float xh = (x[i] - mean) * rstd;
    dw[i] += count ? d[i] * xh : 0.f;
    db[i] += count ? d[i] : 0.f;
    d[i] *= lw[i];
    m1 += d[i];
    m2 += d[i] * xh;
  }
  m1 = group_sum<LPR>(m1) * (1.0f / 64);
  m2 = group_sum<LPR>(m2) * (1.0f / 64);
#pragma unroll
  for (int i = 0; i < VEC; i++) d[i] = rstd * (d[i] - m1 - (x[i] - mean) * rstd * m2);
}

// Workgroups stay for several blocks (the parameter sums live in registers until the end); block <= 64.
template <typename T, bool NORM, bool ROT>
__global__ __launch_bounds__(256, 3) void prepass_bwd_kernel(PrepassParams p, PrepassGrads g, int64_t Nc, int64_t total) {
  constexpr int D = 64, VEC = 8, LPR = 8, RPW = 8;
  extern __shared__ __align__(16) float staged[];
  const int lane = threadIdx.x & 63, r0 = lane >> 3, lr = lane & 7;
  stage_tables<T>(p, staged);
  __syncthreads();
  const RotLane<T> rl(lr);
  float sums[4][VEC];  // q_norm weight, bias, k_norm weight, bias
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int i = 0; i < VEC; i++) sums[k][i] = 0.f;

  for (int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); w < total; w += (int64_t)gridDim.x * 4) {
    const int h = (int)(w % p.H);
    const int64_t bj = w / p.H, j = bj % Nc, b = bj / Nc, bh = b * p.H + h;
    const int64_t t0 = j * p.block;
    const int nvalid = (int)((p.N - t0 < p.block) ? (p.N - t0) : p.block);
    const float inv_cnt = 1.f / (float)nvalid;
    int pos_lo = 0, pos_hi = 0;
    TablePtr tab = {};
    if constexpr (ROT) {
      const int ta = lane >> 1, tb = 32 + (lane >> 1);
      pos_lo = load_pos(p, b, t0 + (ta < nvalid ? ta : nvalid - 1), lane & 1);
      pos_hi = load_pos(p, b, t0 + (tb < nvalid ? tb : nvalid - 1), lane & 1);
      const int pc = block_position((ta < nvalid ? pos_lo : 0) + (tb < nvalid ? pos_hi : 0), (float)nvalid, rl.half);
      tab = table_ptr<T>(p, staged, rl, pc, rl.second);
    }
    // what every token of the block gets through its mean (all row groups compute it, the first one counts)
    float mean_grad[3][VEC];
    const int64_t co = (bh * Nc + j) * D + lr * VEC;
    auto load8 = [](const void* base, int64_t o, float (&x)[VEC]) {
      const uint4 r = *reinterpret_cast<const uint4*>((const T*)base + o);
#pragma unroll
      for (int i = 0; i < VEC; i++) x[i] = to_f32(reinterpret_cast<const T*>(&r)[i]);
    };
    load8(g.dqc, co, mean_grad[0]);
    load8(g.dkc, co, mean_grad[1]);
    load8(g.dvc, co, mean_grad[2]);
    if constexpr (ROT) {
      rotate_row_bwd<T>(mean_grad[0], tab);
      rotate_row_bwd<T>(mean_grad[1], tab);
    }
    if constexpr (NORM) {
      float x[VEC];
      load8(p.q_raw, co, x);
      norm_row_bwd(p, staged, x, mean_grad[0], 0, lr, sums[0], sums[1], r0 == 0);
      load8(p.k_raw, co, x);
      norm_row_bwd(p, staged, x, mean_grad[1], 2, lr, sums[2], sums[3], r0 == 0);
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int i = 0; i < VEC; i++) mean_grad[k][i] *= inv_cnt;

    for (int rbase = 0; rbase < nvalid; rbase += RPW) {
      const int rr = rbase + r0;
      const bool keep = rr < nvalid;
      const int rcl = keep ? rr : nvalid - 1;
      const int64_t xo = b * p.sxb + h * p.sxh + (t0 + rcl) * p.sxn + lr * VEC;
      const int64_t go = (bh * p.N + t0 + rcl) * D + lr * VEC;
      if constexpr (ROT) {
        const int slot = 2 * rcl + rl.half;
        const int from_lo = __shfl(pos_lo, slot & 63), from_hi = __shfl(pos_hi, slot & 63);
        const int pp = slot < 64 ? from_lo : from_hi;
        tab = table_ptr<T>(p, staged, rl, pp, rl.second);
      }
      u32x4 rx[2], rd[3];
      if constexpr (NORM) {
        rx[0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.q + xo));
        rx[1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)p.k + xo));
      }
      rd[0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)g.dq + go));
      rd[1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)g.dk + go));
      rd[2] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const T*)g.dv + go));
#pragma unroll
      for (int k = 0; k < 3; k++) {
        float d[VEC];
#pragma unroll
        for (int i = 0; i < VEC; i++) d[i] = to_f32(reinterpret_cast<const T*>(&rd[k])[i]);
        if (k < 2) {
          if constexpr (ROT) rotate_row_bwd<T>(d, tab);
          if constexpr (NORM) {
            float x[VEC];
#pragma unroll
            for (int i = 0; i < VEC; i++) x[i] = to_f32(reinterpret_cast<const T*>(&rx[k < 2 ? k : 0])[i]);
            norm_row_bwd(p, staged, x, d, 2 * k, lr, sums[k < 2 ? 2 * k : 0], sums[k < 2 ? 2 * k + 1 : 1], keep);
          }
        }
        uint4 o;
#pragma unroll
        for (int i = 0; i < VEC; i++) reinterpret_cast<T*>(&o)[i] = from_f32<T>(d[i] + mean_grad[k][i]);
        if (keep) *reinterpret_cast<uint4*>((T*)g.dx[k] + xo) = o;
      }
    }
  }
  if constexpr (NORM) {
    // parameter sums: over the row groups of a wave, then over the four waves through LDS (the tables are done with)
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int i = 0; i < VEC; i++) sums[k][i] = across_groups<LPR>(sums[k][i]);
    __syncthreads();
    if (r0 == 0) {
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int i = 0; i < VEC; i++) staged[(threadIdx.x >> 6) * 256 + k * 64 + lr * VEC + i] = sums[k][i];
    }
    __syncthreads();
    const int t = threadIdx.x;
    g.partial[(int64_t)blockIdx.x * 256 + t] = (staged[t] + staged[256 + t]) + (staged[512 + t] + staged[768 + t]);
  }
}

// column sums of partial [rows, 256] -> out [256]; 64 columns and 16 rows at a time per workgroup
__global__ __launch_bounds__(1024) void column_sum_kernel(const float* __restrict__ partial, float* __restrict__ out, int rows) {
  __shared__ float part[16][64];
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6, col = blockIdx.x * 64 + c;
  float s = 0.f;
#pragma unroll 8
  for (int r = r0; r < rows; r += 16) s += partial[(int64_t)r * 256 + col];
  part[r0][c] = s;
  __syncthreads();
  if (r0 == 0) {
#pragma unroll
    for (int k = 1; k < 16; k++) s += part[k][c];
    out[col] = s;
  }
}

template <typename T>
static void launch_prepass_bwd(const PrepassParams& p, const PrepassGrads& g, float* sums, int groups, int64_t Nc, int64_t total, hipStream_t st) {
  const bool norm = p.qn_w != nullptr, rot = p.pos != nullptr;
  size_t lds = staged_bytes(p.staged_rows, rot);
  if (lds < 1024 * sizeof(float)) lds = 1024 * sizeof(float);  // the four waves' parameter sums
  dim3 grid((unsigned)groups), blk(256);
  if (norm && rot) hipLaunchKernelGGL((prepass_bwd_kernel<T, true, true>), grid, blk, (unsigned)lds, st, p, g, Nc, total);
  else if (norm) hipLaunchKernelGGL((prepass_bwd_kernel<T, true, false>), grid, blk, (unsigned)lds, st, p, g, Nc, total);
  else if (rot) hipLaunchKernelGGL((prepass_bwd_kernel<T, false, true>), grid, blk, (unsigned)lds, st, p, g, Nc, total);
  else hipLaunchKernelGGL((prepass_bwd_kernel<T, false, false>), grid, blk, (unsigned)lds, st, p, g, Nc, total);
  if (norm) hipLaunchKernelGGL(column_sum_kernel, dim3(4), dim3(1024), 0, st, g.partial, sums, groups);
}

}  // namespace s3r

using namespace s3r;

extern "C" int s3r_gated_merge_bwd(const void* dout, const void* o_cmp, const void* o_sel, const void* gate, void* d_o_cmp, void* d_o_sel,
                                   void* d_gate, float* delta_cmp, float* delta_sel, int B, int H, int64_t N, int D, int block,
                                   int64_t sgb, int64_t sgh, int64_t sgn, int dtype, void* stream) {
  if (!dout || !o_cmp || !o_sel || !gate || !d_o_cmp || !d_o_sel || !d_gate || !delta_cmp || !delta_sel)
    return fail(S3R_ERR_BAD_ARG, "s3r_gated_merge_bwd: null pointer");
  if (B <= 0 || H <= 0 || N <= 0 || block <= 0) return fail(S3R_ERR_BAD_ARG, "s3r_gated_merge_bwd: non-positive size");
  if ((dtype != S3R_BF16 && dtype != S3R_F16) || D != 64) return fail(S3R_ERR_UNSUPPORTED, "s3r_gated_merge_bwd: built for bf16/fp16, head_dim 64");
  const void* ptrs[] = {dout, o_cmp, o_sel, d_o_cmp, d_o_sel};
  for (const void* ptr : ptrs)
    if (!aligned16(ptr)) return fail(S3R_ERR_BAD_ARG, "s3r_gated_merge_bwd: pointers must be multiples of 16 bytes");
  const int64_t Nc = (N + block - 1) / block, total = (int64_t)B * H * Nc;
  if ((total + 3) / 4 > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "s3r_gated_merge_bwd: tensor too large for one launch");
  dim3 grid((unsigned)((total + 3) / 4)), blk(256);
  hipStream_t st = (hipStream_t)stream;
#define S3R_MERGE_BWD(T)                                                                                                                      \
  hipLaunchKernelGGL(merge_bwd_kernel<T>, grid, blk, 0, st, (const T*)dout, (const T*)o_cmp, (const T*)o_sel, (const T*)gate, (T*)d_o_cmp,     \
                     (T*)d_o_sel, (T*)d_gate, delta_cmp, delta_sel, H, N, block, Nc, total, sgb, sgh, sgn)
  if (dtype == S3R_BF16) S3R_MERGE_BWD(bf16_t);
  else S3R_MERGE_BWD(f16_t);
#undef S3R_MERGE_BWD
  return check_launch("s3r_gated_merge_bwd");
}

extern "C" int s3r_layer_prepass_bwd(const s3r_prepass_args* a, const void* dq, const void* dk, const void* dv, const void* dqc, const void* dkc,
                                     const void* dvc, void* dx_q, void* dx_k, void* dx_v, float* norm_grads, float* workspace, int workspace_rows,
                                     void* stream) {
  if (!a || !dq || !dk || !dv || !dqc || !dkc || !dvc || !dx_q || !dx_k || !dx_v) return fail(S3R_ERR_BAD_ARG, "s3r_layer_prepass_bwd: null pointer");
  PrepassParams p = prepass_params(*a);
  if (a->dtype != S3R_BF16 && a->dtype != S3R_F16) return fail(S3R_ERR_UNSUPPORTED, "s3r_layer_prepass_bwd: built for bf16/fp16");
  const int rc = check_prepass("s3r_layer_prepass_bwd", p, a->head_dim, a->dtype);
  if (rc != S3R_OK) return rc;
  if (p.block > 64) return fail(S3R_ERR_UNSUPPORTED, "s3r_layer_prepass_bwd: block %d > 64", p.block);
  if (p.qn_w != nullptr && (!p.q_raw || !p.k_raw || !norm_grads || !workspace || workspace_rows <= 0))
    return fail(S3R_ERR_BAD_ARG, "s3r_layer_prepass_bwd: the norm's gradient needs the raw block means, its result and a workspace");
  const void* ptrs[] = {dq, dk, dv, dqc, dkc, dvc, dx_q, dx_k, dx_v};
  for (const void* ptr : ptrs)
    if (!aligned16(ptr)) return fail(S3R_ERR_BAD_ARG, "s3r_layer_prepass_bwd: pointers must be multiples of 16 bytes");
  const int64_t Nc = (p.N + p.block - 1) / p.block, total = (int64_t)p.B * p.H * Nc;
  // three workgroups per CU hold their parameter sums over several blocks; without a norm there is nothing to hold
  int64_t groups = (total + 3) / 4;
  if (p.qn_w != nullptr && groups > workspace_rows) groups = workspace_rows;
  const PrepassGrads g = {dq, dk, dv, dqc, dkc, dvc, {dx_q, dx_k, dx_v}, workspace};
  if (a->dtype == S3R_BF16) launch_prepass_bwd<bf16_t>(p, g, norm_grads, (int)groups, Nc, total, (hipStream_t)stream);
  else launch_prepass_bwd<f16_t>(p, g, norm_grads, (int)groups, Nc, total, (hipStream_t)stream);
  return check_launch("s3r_layer_prepass_bwd");
}
