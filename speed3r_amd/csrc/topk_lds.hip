// Compressed branch for up to 1216 pooled keys (flash_attention_topk.py:101-157): exact top-k block indices, and in the same launch, by
// workgroups of their own, the attention output (attend below).  The scores of
// 16 query rows against all keys stay in LDS, and a row is selected by one wave that sees all of it.
//
// The two-sweep kernel (compressed_mfma.hip) meets at a barrier per 64 keys and folds queues of survivors into register lists;
// with few tiles its chains of barriers, LDS round trips and folds are all there is (1 041 keys, 33 tiles of 32, 16 heads, top-32, alone
// on the chip: 61 us, 3 % of the matrix rate).  Here:
//   * Scores: S^T = K Q^T with v_mfma_f32_32x32x16 as there, same operands in the same order, so the scores are the same bits.  A
//     workgroup has 16 rows, so half of the 32 query columns repeat the other half: the products are a fiftieth of the work.  The
//     eight waves share the key tiles; all of a wave's keys, up to five tiles, are on their way at once and go through the columns of
//     LDS that the scores will fill into operand order (each is used once per workgroup).
//   * Selection: a wave reads a row, 4 neighbouring columns per lane and 256-column piece, into registers.  The K-th largest of
//     256 group maxima (a lane's four columns modulo 4: neighbours in different groups, since large scores come in runs; the lanes
//     turned from piece to piece, since they come at one place of every frame of a still scene) is a
//     lower bound of the row's K-th largest score; the search for it looks at the upper 24 bits of the sortable pattern only (its result may only be lower).  Scores at or above it, K to 1.4 K of them as a
//     rule, are gathered in the row's own LDS space, one per lane, and ranked by counting: lane l compares its key with every
//     other one.  No chain of exchanges, no sort.
//   * More than 64 candidates (a looser bound, equal scores): the bound is raised by halving the range of patterns, and of columns
//     with one pattern, until 64 or fewer are left.  1 041 keys, top-32: 36 us as a rule, 65 where all scores are equal (two-sweep
//     kernel 61 / 84); still scenes of 64 blocks a frame, 1 024 and 1 216 keys 27 and 37 (58 and 65; without turned lanes 37 and 51).
// Order, fillers and NaN as in the two-sweep kernel: descending (sortable score, lowest column first), NaN never chosen, Lk - 1
// in slots that nothing fills.
//
// us alone on the chip, two-sweep kernel / this, 16 heads, as many rows as keys: 126 keys, top-32 16 / 8; 504, top-32 40 / 13; 1 041,
// top-16 46 / 34; 1 200, top-32 66 / 38.  Bound: the vector instructions of the selection, about 700 per row at 1 041 keys.  The instances
// of three to five pieces spill 15 to 32 scalar registers to lanes of vector registers, the others none.
//
// Up to kMostKeys keys two workgroups fit a CU (78 KB each; up to 512 keys three, by registers too).  With more keys one does, and the two phases have nobody to hide
// behind: 2 016 keys, top-32, 95 / 112.  With more than kMostGroups workgroups the two-sweep kernel, which shares its key tiles
// among more rows, is no longer bound by latency: 24 heads of 1 041 47 / 48, 32 of them 53 / 58, 48 of 756 44 / 46.  Up to
// top-8 its folds are short, and it is as good from fewer keys on (whole operator, us, top-8: 537 keys 182 / 172, 1 009 287 /
// 286, 1 201 336 / 344; top-4: 537 145 / 142, 814 191 / 192, 1 009 225 / 230; top-1: 537 136 / 119, 814 156 / 163).
#include "block16.h"
#include "attn_params.h"

namespace s3r {
namespace tkl {
using namespace sel;

constexpr int kRows = 16, kWaves = 8;
constexpr int kAttnRows = 16 * kWaves;  // query rows of an attention workgroup

// The attention itself, by workgroups of their own in front of the others' grid: 16 query rows a wave, 64 keys and their values at a
// time through LDS (`lds`: 16 KB), the next step's requested while it computes; 16 x 16 products as in the kernels for 16-token
// blocks, scaled fp32 scores, running maximum (exchanged between the lanes only in steps that raise it).  As a launch of its own (the
// selection kernel's dense sweep) a chain of waits with the chip idle around it; here it runs beside the selection.  Attention and
// indices, us, two launches / one (the indices alone): 16 heads, top-32, 126 pooled tokens 15.0 / 8.0 (7.9), 504 22.6 / 16.9 (12.9), 756
// 32.1 / 25.3 (20.8), 1 200 52.4 / 46.0 (38.1); top-8 393 20.8 / 13.3; 2 heads 1 200 26.4 / 22.7; 2 x 16 heads 756 45.4 / 44.2.  Bound: the
// vector instructions that it adds to the selection's.  Two or four waves to a row's keys, for shorter chains: 504 18.9, 1 041 51 against
// 40.  Error of the output against 64 bits, bf16, scores of standard deviation 0.25 to 9, 126 to 1 041 tokens: 1.6e-3 to 2.4e-3 (before
// 1.6e-3 to 3.7e-3: queries scaled in bf16), with the log-sum-exp before 1.7e-3 to 2.4e-3; fp16 2.1e-4 to 3.0e-4 (2.1e-4 to 5.2e-4).
template <typename E> __device__ __forceinline__ void attend(const AttnParams& p, int vid, int groups, unsigned char* lds) {
  using namespace b16x;
  typedef typename Mma<E>::V8 V8;
  typedef typename Mma4<E>::V4 V4;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int bh = vid / groups, b = bh / p.H, h = bh - b * p.H;
  const int row = (vid - bh * groups) * kAttnRows + wave * 16 + c, Lk = (int)p.Lk;
  const bool live = row < (int)p.Lq;
  const E* const qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh + (int64_t)(live ? row : (int)p.Lq - 1) * p.sqm + 8 * g;
  V8 bq[2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) bq[ks] = frag_of<E>(*reinterpret_cast<const u32x4*>(qp + 32 * ks));
  const E* const kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh + (tid & 7) * 8;
  const E* const vp = (const E*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh + (tid & 7) * 8;
  u32x4 kv, vv;  // this thread's piece of the next step
  auto fetch = [&](int first) {
    const int at = first + (tid >> 3), key = at < Lk ? at : Lk - 1;
    kv = *reinterpret_cast<const u32x4*>(kp + (int64_t)key * p.skn);
    vv = *reinterpret_cast<const u32x4*>(vp + (int64_t)key * p.svn);
    if (at >= Lk) vv = (u32x4){0, 0, 0, 0};  // (0 times what the last row holds may be NaN)
  };
  const int r16 = (tid >> 3) & 15;
  unsigned char* const put = lds + (tid >> 7) * 2048 + r16 * 128 + (((tid & 7) ^ swz(r16)) << 4);
  const int row_off = c * 128 + ((g ^ swz(c)) << 4);
  const int tr_row = 4 * g + (c >> 2), tr_off = 8192 + tr_row * 128 + ((((c & 3) >> 1) ^ swz(tr_row)) << 4) + (c & 1) * 8;
  const float sl2 = p.scale * kLog2e;
  float m = -INFINITY, l = 0.f;  // reference in base 2 (the same in a query's four lanes), sum of this lane's probabilities
  f32x4 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; dt++) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  fetch(0);
  for (int first = 0; first < Lk; first += 64) {
    *reinterpret_cast<u32x4*>(put) = kv;
    *reinterpret_cast<u32x4*>(put + 8192) = vv;
    if (first + 64 < Lk) fetch(first + 64);
    __syncthreads();
    f32x4 st[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      st[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
      st[t] = mma16<E>(frag_of<E>(*reinterpret_cast<const u32x4*>(lds + row_off + t * 2048)), bq[0], st[t]);
      st[t] = mma16<E>(frag_of<E>(*reinterpret_cast<const u32x4*>(lds + (row_off ^ 64) + t * 2048)), bq[1], st[t]);
    }
    settle(st);
    if (first + 64 > Lk) {
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) st[t][r] = first + 16 * t + 4 * g + r < Lk ? st[t][r] : -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; t++) mx = fmaxf(mx, fmaxf(fmaxf(st[t][0], st[t][1]), fmaxf(st[t][2], st[t][3])));
    mx *= sl2;            // sl2 > 0: the maximum of the scaled scores
    if (__any(mx > m)) {  // (the first step: unless all of its scores are -inf)
      mx = fmaxf(m, xh_max(fmaxf(mx, lane_xor<16>(mx))));
      const float alpha = __builtin_amdgcn_exp2f(m - (mx == -INFINITY ? 0.f : mx));  // 0 while there is none
      m = mx;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; dt++) o[dt] *= alpha;
    }
    const float use = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      float x[4];
#pragma unroll
      for (int r = 0; r < 4; r++) x[r] = __builtin_amdgcn_exp2f(fmaf(st[t][r], sl2, -use));
      l += (x[0] + x[1]) + (x[2] + x[3]);
      const V4 pr = pack4<E>(x);
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        const s16x4 vt = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(lds + t * 2048 + (tr_off ^ (32 * dt))));
        o[dt] = Mma4<E>::mma(__builtin_bit_cast(u32x2, vt), pr, o[dt]);
      }
    }
    __syncthreads();  // the step's rows are read
  }
  const float sum = xh_sum(l + lane_xor<16>(l));
  const float inv = sum == 0.f ? 0.f : 1.f / sum;
  E* const op = (E*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh + (int64_t)row * p.som;
#pragma unroll
  for (int dp = 0; dp < 2; dp++) {  // (the exchange and the stores of the kernels for 16-token blocks)
    float y[2][4];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) y[t][r] = o[2 * dp + t][r] * inv;
    const u32x2 wa = __builtin_bit_cast(u32x2, pack4<E>(y[0])), wb = __builtin_bit_cast(u32x2, pack4<E>(y[1]));
    union { uint32_t w[4]; uint4 u; } pc;
#pragma unroll
    for (int wi = 0; wi < 2; wi++) {
      const auto r = __builtin_amdgcn_permlane16_swap(wa[wi], wb[wi], false, false);
      pc.w[wi] = r[0];
      pc.w[2 + wi] = r[1];
    }
    if (live) *reinterpret_cast<uint4*>(op + 16 * (2 * dp + (g & 1)) + 8 * (g >> 1)) = pc.u;
  }
  if (live && p.lse != nullptr && g == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + row] = (m + __builtin_amdgcn_logf(sum)) * 0.6931471805599453f;
}

__device__ __forceinline__ float sortable_to_float(uint32_t k) {  // the inverse of sortable_key
  return __uint_as_float(k ^ ((k & 0x80000000u) ? 0x80000000u : 0xFFFFFFFFu));
}

template <typename E, int NC>  // NC: pieces of 256 columns
__global__ __launch_bounds__(64 * kWaves, NC <= 2 ? 6 : 4) void topk_lds_kernel(AttnParams p, int groups, int total, int attn_groups, int attn_total, int attn_wgs) {
  typedef typename Mma<E>::V8 V8;
  // rows of the scores, 4 mod 64 values apart: what 16 lanes on 16 rows touch lies in different banks
  constexpr int stride = (NC == 5 ? (int)kMostKeys : 256 * NC) + 4;
  __shared__ __attribute__((aligned(1024))) float sc[kRows * stride];
  static_assert(sizeof(sc) >= 16384, "a step of the attention");
  // the workgroups of a head run on one XCD, whose L2 then holds its keys (attn_wgs is a multiple of 8)
  const int xcd = blockIdx.x & 7;
  auto item = [&](int w, int all) { return xcd * (all >> 3) + (xcd < (all & 7) ? xcd : (all & 7)) + (w >> 3); };
  if ((int)blockIdx.x < attn_wgs) {
    if ((int)(blockIdx.x >> 3) < (attn_total >> 3) + (xcd < (attn_total & 7) ? 1 : 0))
      attend<E>(p, item(blockIdx.x, attn_total), attn_groups, reinterpret_cast<unsigned char*>(sc));
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int hh = lane >> 5, c = lane & 31;
  const int vid = item((int)blockIdx.x - attn_wgs, total);
  const int bh = vid / groups, g = vid - bh * groups;
  const int b = bh / p.H, h = bh - b * p.H;
  const int Lk = (int)p.Lk, q0 = g * kRows;
  const int rows = (int)p.Lq - q0 < kRows ? (int)p.Lq - q0 : kRows;
  const E* const kp = (const E*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;

  // ---- scores ----
  {
    const int qr = (c & 15) < rows ? (c & 15) : rows - 1;
    const E* const qp = (const E*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh + (int64_t)(q0 + qr) * p.sqm + hh * 8;
    Frag qf[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) qf[ks].u = *reinterpret_cast<const uint4*>(qp + ks * 16);
    const int tiles = (Lk + 31) >> 5;
    // The keys come with lane-linear loads, all of a wave's tiles on their way at once (lane = key takes the address unit 64
    // cycles per instruction instead of 18), and go through LDS into operand order: 16 keys of 128 bytes fit the columns that a
    // tile's scores will take, so a tile's keys use its own columns and the wave's next ones.
    const int lr = lane >> 3, lc = lane & 7;
    u32x4 kv[NC][4];
#pragma unroll
    for (int u = 0; u < NC; u++)
      if (wave + u * kWaves < tiles) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int key = (wave + u * kWaves) * 32 + 8 * i + lr;
          kv[u][i] = *reinterpret_cast<const u32x4*>(kp + (int64_t)(key < Lk ? key : Lk - 1) * p.skn + lc * 8);
        }
      }
    constexpr int held = (stride - 4) >> 5;  // tiles that the score rows have columns for
#pragma unroll
    for (int u = 0; u < NC; u++) {
      const int t = wave + u * kWaves;
      if (t < tiles) {
        char* const own = reinterpret_cast<char*>(sc + t * 32);
        char* const put = own + lr * stride * 4 + lc * 16;
        const char* const get = own + (c & 15) * stride * 4 + hh * 16;
        u32x4 kf[4];
        *reinterpret_cast<u32x4*>(put) = kv[u][0];
        *reinterpret_cast<u32x4*>(put + 8 * stride * 4) = kv[u][1];
        if (t + kWaves < held) {
          *reinterpret_cast<u32x4*>(put + kWaves * 128) = kv[u][2];
          *reinterpret_cast<u32x4*>(put + kWaves * 128 + 8 * stride * 4) = kv[u][3];
#pragma unroll
          for (int ks = 0; ks < 4; ks++) kf[ks] = *reinterpret_cast<const u32x4*>(get + (c < 16 ? 0 : kWaves * 128) + ks * 32);
        } else {  // the wave's last tile: its own columns twice
          u32x4 lo[4];
#pragma unroll
          for (int ks = 0; ks < 4; ks++) lo[ks] = *reinterpret_cast<const u32x4*>(get + ks * 32);
          *reinterpret_cast<u32x4*>(put) = kv[u][2];
          *reinterpret_cast<u32x4*>(put + 8 * stride * 4) = kv[u][3];
#pragma unroll
          for (int ks = 0; ks < 4; ks++) {
            const u32x4 hi = *reinterpret_cast<const u32x4*>(get + ks * 32);
            kf[ks] = c < 16 ? lo[ks] : hi;
          }
        }
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) acc = Mma<E>::mma(__builtin_bit_cast(V8, kf[ks]), as_v8<E>(qf[ks]), acc);
        settle(acc);
        if (c < kRows) {
          float* const dst = sc + c * stride + t * 32 + 4 * hh;  // rows 8 j + 4 hh + i of the tile
#pragma unroll
          for (int j = 0; j < 4; j++) *reinterpret_cast<float4*>(dst + 8 * j) = make_float4(acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]);
        }
      }
    }
  }
  __syncthreads();

  // ---- selection ----
  const int K = p.K;
  // A lane's columns in piece i: turned against the other pieces, so that places 256 columns apart (or one place of several frames)
  // lie in different lanes' groups
  auto first_col = [&](int i) { return i * 256 + ((lane + (i * (i + 9) >> 1)) & 63) * 4; };
  constexpr int G = 4;               // groups of scores per lane: neighbouring columns in different ones
  constexpr int R = kRows / kWaves;  // rows of a wave, side by side: each hides the other's waits
  float v[R][NC][4];
  float* row[R];
  uint32_t t[R];
  uint32_t gk[R][G];  // largest score of a group, sortable
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int q = wave * R + r;
    row[r] = sc + (q < rows ? q : rows - 1) * stride;  // (rows behind the last one repeat it and store nothing)
    float mx[G];
#pragma unroll
    for (int e = 0; e < G; e++) mx[e] = -INFINITY;
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int col = first_col(i);
      const float4 x = *reinterpret_cast<const float4*>(row[r] + (col < Lk ? col : 0));
      v[r][i][0] = x.x; v[r][i][1] = x.y; v[r][i][2] = x.z; v[r][i][3] = x.w;
      if (i * 256 + 256 > Lk) {  // beyond the keys: NaN, which no comparison lets pass
#pragma unroll
        for (int e = 0; e < 4; e++) v[r][i][e] = col + e < Lk ? v[r][i][e] : __uint_as_float(0x7fc00000u);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) mx[e % G] = fmaxf(mx[e % G], v[r][i][e]);  // (passes over NaN)
    }
#pragma unroll
    for (int e = 0; e < G; e++) gk[r][e] = sortable_key(mx[e]);
    t[r] = 0;
  }
#pragma unroll
  for (int bit = 31; bit >= 8; bit--)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const uint32_t cand = t[r] | (1u << bit);
      int cnt = 0;
#pragma unroll
      for (int e = 0; e < G; e++) cnt += (int)__popcll(__ballot(gk[r][e] >= cand));
      t[r] = cnt >= K ? cand : t[r];
    }
  // lanes' counts -> what the lanes below have; the sum of all
  auto prefix = [](int& own, int& all) {
    int s = own;  // inclusive sum over the lanes below: rows of 16, then across them
#define S3R_STEP(ctrl, rows_on) s += __builtin_amdgcn_update_dpp(0, s, ctrl, rows_on, 0xF, false)
    S3R_STEP(0x111, 0xF);  // row_shr:1
    S3R_STEP(0x112, 0xF);  // row_shr:2
    S3R_STEP(0x114, 0xF);  // row_shr:4
    S3R_STEP(0x118, 0xF);  // row_shr:8
    S3R_STEP(0x142, 0xA);  // row_bcast:15 into rows 1 and 3
    S3R_STEP(0x143, 0xC);  // row_bcast:31 into rows 2 and 3
#undef S3R_STEP
    all = __builtin_amdgcn_readlane(s, 63);
    own = s - own;
  };
  // candidates, packed to the front of the row's space (its scores are in registers): pattern and column
  float bound[R];
  int mine[R], n[R];  // where a lane's first one goes; the number of all
#pragma unroll
  for (int r = 0; r < R; r++) {
    bound[r] = t[r] <= 0x007FFFFFu ? -INFINITY : sortable_to_float(t[r]);  // (below the pattern of -inf lie NaNs)
    mine[r] = 0;
#pragma unroll
    for (int i = 0; i < NC; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) mine[r] += v[r][i][e] >= bound[r] ? 1 : 0;
    prefix(mine[r], n[r]);
  }
#pragma unroll
  for (int r = 0; r < R; r++)
    if (n[r] <= 64 && wave * R + r < rows) {
      uint2* at = reinterpret_cast<uint2*>(row[r]) + mine[r];
#pragma unroll
      for (int i = 0; i < NC; i++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (v[r][i][e] >= bound[r]) *at++ = make_uint2(__float_as_uint(v[r][i][e]), (uint32_t)(first_col(i) + e));
    } else if (wave * R + r < rows) {
      // More than fit the lanes: large scores share groups (256 columns apart, or four frames of 64 blocks: the same place in a still
      // scene), or many are equal.  Halve the range of patterns until K to 64 lie at or above its lower end, or it is one
      // pattern; of its columns then the range of those that are needed.
      uint32_t x[NC][4];  // sortable patterns; NaN below all
#pragma unroll
      for (int i = 0; i < NC; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) x[i][e] = v[r][i][e] >= bound[r] ? sortable_key(v[r][i][e]) : 0;
      uint32_t most = 0;
#pragma unroll
      for (int e = 0; e < G; e++) most = max(most, gk[r][e]);
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) most = max(most, (uint32_t)__shfl_xor((int)most, off));
      most = __builtin_amdgcn_readfirstlane(most);
      uint32_t lo = bound[r] == -INFINITY ? 0x007FFFFFu : t[r], hi = most + 1;  // as many at or above as n, none
      int cols = Lk, cnt = n[r];  // columns below `cols` of those with the pattern `lo`
      auto count = [&](auto takes) {
        int c = 0, all;
#pragma unroll
        for (int i = 0; i < NC; i++)
#pragma unroll
          for (int e = 0; e < 4; e++) c += takes(x[i][e], first_col(i) + e) ? 1 : 0;
        prefix(c, all);
        mine[r] = c;
        return all;
      };
      while (cnt > 64 && hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        const int c = count([&](uint32_t k, int) { return k >= mid; });
        if (c >= K) { lo = mid; cnt = c; }
        else hi = mid;
      }
      if (cnt > 64) {
        int below = 0;  // too few columns
        while (cols - below > 1) {
          const int mid = below + (cols - below) / 2;
          const int c = count([&](uint32_t k, int col) { return k > lo || (k == lo && col < mid); });
          if (c >= K) cols = mid;
          else below = mid;
        }
      }
      n[r] = count([&](uint32_t k, int col) { return k > lo || (k == lo && col < cols); });
      uint2* at = reinterpret_cast<uint2*>(row[r]) + mine[r];
#pragma unroll
      for (int i = 0; i < NC; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int col = first_col(i) + e;
          if (x[i][e] > lo || (x[i][e] == lo && col < cols)) *at++ = make_uint2(__float_as_uint(sortable_to_float(x[i][e])), (uint32_t)col);
        }
    }
  uint64_t key[R];
  uint32_t col[R];
#pragma unroll
  for (int r = 0; r < R; r++) {  // one candidate per lane, as a key, back to where the others read it
    const uint2 x = reinterpret_cast<const uint2*>(row[r])[lane < n[r] ? lane : 0];
    col[r] = x.y;
    key[r] = lane < n[r] ? ((uint64_t)sortable_key(__uint_as_float(x.x)) << 32) | ((uint32_t)(Lk - 1) - x.y) : 0;
  }
#pragma unroll
  for (int r = 0; r < R; r++)
    if (wave * R + r < rows) reinterpret_cast<uint64_t*>(row[r])[lane] = key[r];
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (wave * R + r >= rows) break;
    int32_t* const out = p.topk_idx + ((int64_t)bh * p.Lq + q0 + wave * R + r) * K;
    int rank = 0;
    for (int j = 0; j < n[r]; j += 8) {  // (keys behind the last one are 0: above nothing)
      const ulonglong2* const o = reinterpret_cast<const ulonglong2*>(row[r]) + j / 2;
      ulonglong2 w[4];
#pragma unroll
      for (int u = 0; u < 4; u++) w[u] = o[u];
#pragma unroll
      for (int u = 0; u < 4; u++) rank += (w[u].x > key[r] ? 1 : 0) + (w[u].y > key[r] ? 1 : 0);
    }
    if (lane < n[r] && rank < K) out[rank] = (int32_t)col[r];
    if (lane >= n[r] && lane < K) out[lane] = Lk - 1;
  }
}

template <typename E> static int launch(const AttnParams& p, hipStream_t st) {
  const int64_t groups = (p.Lq + kRows - 1) / kRows, total = groups * p.B * p.H;
  const int64_t attn_groups = p.o != nullptr ? (p.Lq + kAttnRows - 1) / kAttnRows : 0, attn = attn_groups * p.B * p.H, attn_wgs = (attn + 7) / 8 * 8;
#define S3R_TKL(NC)                                                                                                                         \
  hipLaunchKernelGGL((topk_lds_kernel<E, NC>), dim3((unsigned)(attn_wgs + total)), dim3(64 * kWaves), 0, st, p, (int)groups, (int)total, \
                     (int)attn_groups, (int)attn, (int)attn_wgs)
  if (p.Lk <= 256) S3R_TKL(1);
  else if (p.Lk <= 512) S3R_TKL(2);
  else if (p.Lk <= 768) S3R_TKL(3);
  else if (p.Lk <= 1024) S3R_TKL(4);
  else S3R_TKL(5);
#undef S3R_TKL
  return check_launch("topk_lds_kernel");
}

}  // namespace tkl

constexpr int64_t kMostGroups = 1536;

// Few keys and a short list: the two-sweep kernel's folds are fewer than the steps of the search here.  16 heads, as many rows as keys,
// two-sweep / this: top-1 16 keys 4.7 / 6.7, 96 6.9 / 7.1, 126 7.4 / 7.2; top-4 16 5.1 / 6.8, 64 6.2 / 7.0, 65 8.1 / 7.1; top-8 64 6.6 /
// 7.0, 65 8.4 / 7.2; top-16 16 6.1 / 7.0, 33 7.0 / 7.2, 48 8.0 / 7.3; top-32 32 9.5 / 7.3.
static bool short_lists(int64_t BH, int64_t Lq, int64_t Lk, int K) {
  return Lk > (K <= 2 ? 96 : K <= 8 ? 64 : K <= 16 ? 40 : 0) && Lk <= (K <= 4 ? 640 : K <= 8 ? 1024 : kMostKeys) &&
         (Lq + tkl::kRows - 1) / tkl::kRows * BH <= kMostGroups;
}

bool topk_lds_pays(const AttnParams& p) { return short_lists((int64_t)p.B * p.H, p.Lq, p.Lk, p.K); }

int launch_topk_lds(const AttnParams& p, int dtype, void* stream) {
  return dtype == S3R_BF16 ? tkl::launch<bf16_t>(p, (hipStream_t)stream) : tkl::launch<f16_t>(p, (hipStream_t)stream);
}

}  // namespace s3r

extern "C" int s3r_topk_in_lds(int64_t batch_heads, int64_t Lq, int64_t Lk, int K) {
  return batch_heads > 0 && Lq > 0 && Lk > 0 && K > 0 && batch_heads <= s3r::kMostGroups && Lq <= (1 << 20) && s3r::short_lists(batch_heads, Lq, Lk, K);
}
