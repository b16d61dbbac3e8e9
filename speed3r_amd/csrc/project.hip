// The layers' q/k/v projection with everything that follows it row by row: q, k, v = x W^T + b, LayerNorm over the head
// dimension and 2-D rotary embedding of q and k, block means of the raw q, k, v (pi3/models/layers/sparse_attention.py:93-110,
// 115-124), in one kernel, and a short one for norm and rotation of the means.  bf16 / fp16, head_dim 64.
//
// The product followed by the pass over its output (qkv_prepass.hip) writes the projection once and reads it once more:
// at 104 100 tokens x 16 heads 1.28 GB of the 1.7 GB that the two move.  Here a tile of the product is finished in registers.
// The accumulator layout suits it: a lane holds 4 consecutive channels of one token in each of the head's
// four 16 x 16 tiles, so the row sums of the norm take two exchanges per 16 values, the rotation partner (16 channels away)
// sits in the same lane, and 16 tokens' sums for the means are one reduction over 16 lanes.
// The layer's gate, sigmoid(x W^T + b) with 2 outputs per head (sparse_attention.py:88,127), is 32 more columns: thin tiles for the
// workgroups that the last round of tiles leaves idle.
// us, library product + pass / this: 104 100 tokens (64-token blocks) 610 + 207 / 697, 32 256 (16-token blocks) 165 + 81 / 222,
// 8 x 1 008 without means 57 + 20 / 57, 2 016 (16-token blocks) 21 + 23 / 28.
//
// Rounding points: the projection to the I/O type (what norm and means are computed from); then fp32 to the end, one rounding
// (the pass rounds after the norm and after each product of the rotation as well).  The means keep the pass's points.
//
// Bound: the matrix cores inside the sweep over K; behind it about 280 vector instructions per 16 tokens and head of q or k
// with one wave per SIMD, 30 % of the time of a 256 x 256 tile at K = 1024.  The registers are full: the 256-wide instances spill 112 to 120
// scalar registers to lanes of vector registers with means, 62 to 72 without, and none to 4 vector registers to memory; the 128-wide
// ones 42 to 66 scalar ones, fp16 with 64-token means 2 vector ones.  Tried without gain: fp32 tables in LDS instead of
// packed pairs (16 instructions less, 4 % slower), both heads of a wave in one pass, 128 x 128 tiles throughout (809 against 742).
#include "linear_tile.h"
#include "prepass.h"

namespace s3r {
namespace lin {

struct ProjectParams {
  const void *x, *w, *bias;
  int64_t ldx, ldw;
  int M, N, K, C, H, Nc, mt, nt;  // M = B N rows
  void *q, *k, *v, *qc, *kc, *vc;
  const void* pos;
  int64_t spb, spn;
  int pos64, P, staged_rows, ln_f32;
  const void *cos_tab, *sin_tab;
  const float* inv_freq;
  const void* ln[4];  // q norm weight, bias, k norm weight, bias
  float eps;
  const void *gate_w, *gate_b;  // optional: gate_out [M, O] = sigmoid(x gate_w^T + gate_b)
  void* gate_out;
  int O;
};

// (cos, sin) pairs of the I/O type, 16 frequencies per position; chunk of 4 frequencies c of row r at c ^ ((r >> 2) & 3), so
// that 16 lanes on consecutive positions read from 64 different banks
__device__ __forceinline__ int table_at(int row, int chunk) { return row * 16 + ((chunk ^ ((row >> 2) & 3)) << 2); }

template <typename E> __device__ __forceinline__ void unpack_pair(uint32_t u, float& c, float& s);
template <> __device__ __forceinline__ void unpack_pair<bf16_t>(uint32_t u, float& c, float& s) {
  c = __uint_as_float(u << 16);
  s = __uint_as_float(u & 0xffff0000u);
}
template <> __device__ __forceinline__ void unpack_pair<f16_t>(uint32_t u, float& c, float& s) {
  c = (float)__builtin_bit_cast(f16_t, (unsigned short)u);
  s = (float)__builtin_bit_cast(f16_t, (unsigned short)(u >> 16));
}
template <typename E> __device__ __forceinline__ uint32_t pack_pair(E c, E s) {
  return (uint32_t)__builtin_bit_cast(unsigned short, c) | ((uint32_t)__builtin_bit_cast(unsigned short, s) << 16);
}
// the pair of frequency f at a position outside of the staged rows: from the caller's tables, beyond them by its own angle
template <typename E> __device__ __forceinline__ uint32_t far_pair(const ProjectParams& p, int pp, int f) {
  if (pp < p.P || p.inv_freq == nullptr) {
    const int64_t at = (int64_t)(pp < p.P ? pp : p.P - 1) * 16 + f;
    return pack_pair<E>(((const E*)p.cos_tab)[at], ((const E*)p.sin_tab)[at]);
  }
  float angle = (float)pp * p.inv_freq[f];  // (in fp32 before it is rounded, see table_ptr)
  asm volatile("" : "+v"(angle));
  angle = round_to<E>(angle);
  return pack_pair<E>((E)cosf(angle), (E)sinf(angle));
}

template <typename E, int T, bool NORM, int POOL, int WPS>
__global__ __launch_bounds__(256, WPS) void project_kernel(ProjectParams p) {
  typedef Tile<E, T, T> Tl;
  typedef typename Mma<E>::V2 V2;
  constexpr int BM = Tl::BM, BN = Tl::BN, HD = T / 4, NS = 2;  // HD: heads of a wave, NS: stores per head and 16 tokens
  constexpr int WROWS = 16 * T;                        // its tokens
  constexpr int BLOCKS = POOL ? WROWS / (POOL ? POOL : 1) : 0, SETS = (BLOCKS + 3) / 4;
  __shared__ __attribute__((aligned(1024))) unsigned char lx0[BM * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lx1[BM * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lw0[BN * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lw1[BN * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char lst[4 * 2048];  // per wave 16 rows on their way out
  __shared__ __attribute__((aligned(16))) uint32_t ltab[kStagedRows * 16];
  __shared__ __attribute__((aligned(16))) float lln[NORM ? 256 : 4];
  __shared__ int2 lpos[2][BM];  // (y, x) of a tile's tokens: this tile's, and the next one's
  __shared__ __attribute__((aligned(16))) int lfar[2][4];  // per wave: a position it handed out lies outside of the staged rows
  __shared__ __attribute__((aligned(16))) E lbias[2][BN];  // the bias of its channels
  TileWalk walk(p.mt, p.nt);
  const int tid = threadIdx.x;
  if (walk.at < walk.count) {
  Tl tl;
  for (int i = tid; i < p.staged_rows * 16; i += 256)
    ltab[table_at(i >> 4, (i & 15) >> 2) + (i & 3)] = pack_pair<E>(((const E*)p.cos_tab)[i], ((const E*)p.sin_tab)[i]);
  if constexpr (NORM) {
    const void* const src = p.ln[tid >> 6];
    lln[tid] = src == nullptr ? 0.f : p.ln_f32 ? ((const float*)src)[tid & 63] : (float)((const E*)src)[tid & 63];
  }

  int m, n, ask = walk.at, kb = 0, par = 0;
  E nbias = (E)0.f;
  int2 npos = make_int2(0, 0);  // the requested tile's bias at channel `tid` and position of token `tid`
  auto aim = [&](int i) {
    int tm, tn;
    walk.locate(i, tm, tn);
    const int r0 = tm * BM, c0 = tn * BN;
    const int rows = p.M - r0 < BM ? p.M - r0 : BM;
    tl.aim((const E*)p.x + r0 * p.ldx, p.ldx, rows, (const E*)p.w + c0 * p.ldw, p.ldw, 3 * p.C - c0 < BN ? 3 * p.C - c0 : BN);
    if (p.bias != nullptr && tid < BN) nbias = ((const E*)p.bias)[c0 + tid < 3 * p.C ? c0 + tid : 3 * p.C - 1];
    if (tid < BM) {
      const int b0 = r0 / p.N, at = r0 - b0 * p.N + (tid < rows ? tid : rows - 1);
      const int64_t o = at < p.N ? b0 * p.spb + at * p.spn : (b0 + 1) * p.spb + (at - p.N) * p.spn;
      if (p.pos64) npos = make_int2((int)((const int64_t*)p.pos)[o], (int)((const int64_t*)p.pos)[o + 1]);
      else npos = make_int2(((const int32_t*)p.pos)[o], ((const int32_t*)p.pos)[o + 1]);
    }
  };
  // A step behind the aim, whose loads that step has waited for; a barrier lies between this and every use.
  auto hand_out = [&](int to) {
    if (tid < BN) lbias[to][tid] = nbias;
    if (tid < BM) lpos[to][tid] = npos;
    const bool out = tid < BM && (npos.x >= p.staged_rows || npos.y >= p.staged_rows);
    if (tl.lane == 0) lfar[to][tl.wave] = 0;
    if (__any(out) && tl.lane == 0) lfar[to][tl.wave] = 1;
  };
  auto advance = [&]() {  // past the last tile its rows are requested again: nothing to tell apart in the loop
    kb += 128;
    if (kb == p.K * 2) {
      kb = 0;
      ask = ask + walk.slots < walk.count ? ask + walk.slots : ask;
      aim(ask);
    } else if (kb == 128) {
      hand_out(par ^ 1);
    }
  };
  walk.locate(walk.at, m, n);
  aim(walk.at);
  hand_out(0);
#pragma unroll
  for (int i = 0; i < Tl::NL; i++) tl.move(lx0, lw0, kb, i);
  kb = 128;
#pragma unroll
  for (int i = 0; i < Tl::NL; i++) tl.move(lx1, lw1, kb, i);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the tables, and what has been handed out
  tl.begin(lx0, lw0);
  bool fresh = true;
  for (;; par ^= 1) {
    tl.template sweep<T * HD * NS>(lx0, lw0, lx1, lw1, p.K >> 6, fresh, kb, advance);
    tl.after_products();

    // ---- epilogue ----
    const int r0 = m * BM, rows = p.M - r0 < BM ? p.M - r0 : BM;
    const int b0 = r0 / p.N, n0 = r0 - b0 * p.N, cross = p.N - n0;  // rows from `cross` on belong to the next sequence
    const int ch = n * BN + tl.wn * 16 * T;
    const int which = ch / p.C;                                     // 0: q, 1: k, 2: v
    const int head = (ch - which * p.C) >> 6;
    auto finish = [&](auto turn_tag) {
      constexpr bool TURN = decltype(turn_tag)::value;  // q and k: norm and rotation
      E* const out = (E*)(which == 0 ? p.q : which == 1 ? p.k : p.v) + ((int64_t)(b0 * p.H + head) * p.N + n0) * 64;
      const uint32_t jump = (uint32_t)(p.H - 1) * (uint32_t)p.N * 128u;
      // (opaque: the addresses below would otherwise be computed once, in front of all tiles, and spilled)
      int lane = threadIdx.x & 63;
      asm volatile("" : "+v"(lane));
      const int wr = tl.wm * WROWS, c16 = lane & 15, g4 = lane >> 4;
      auto row_offset = [&](int row) { return (uint32_t)row * 128u + (row >= cross ? jump : 0u); };
      const int2* const pos = &lpos[par][wr];
      // Rare: some token of the tile lies outside of the staged rows.  The pairs of all the wave's tokens then go through memory: 32
      // pairs of four bytes are a row's 128, and they take the rows that the results of its last head overwrite, group by group, each
      // after its pairs have been read.
      bool far = false;
      char* const scratch = reinterpret_cast<char*>(out + (int64_t)(HD - 1) * p.N * 64);
      uint32_t at[T];  // where a token's pairs lie in the table (y, x)
      if constexpr (TURN) {
        const int4 f = *reinterpret_cast<const int4*>(lfar[par]);
        far = __builtin_amdgcn_readfirstlane(f.x | f.y | f.z | f.w) != 0;
#pragma unroll
        for (int t = 0; t < T; t++) {
          const int2 pp = pos[t * 16 + c16];
          at[t] = (uint32_t)table_at(pp.x < 0 ? 0 : pp.x & (kStagedRows - 1), g4) | (uint32_t)table_at(pp.y < 0 ? 0 : pp.y & (kStagedRows - 1), g4) << 16;
        }
        if (far) {
#pragma unroll 1
          for (int t = 0; t < T; t++) {
            const int row = wr + t * 16 + c16;
            const int2 pp = pos[t * 16 + c16];
            if (row < rows) {
              uint32_t* const dst = reinterpret_cast<uint32_t*>(scratch + row_offset(row)) + 4 * g4;
#pragma unroll 1
              for (int i = 0; i < 8; i++) {
                const int c = i < 4 ? pp.x : pp.y;
                dst[(i & 3) + (i < 4 ? 0 : 16)] = far_pair<E>(p, c < 0 ? 0 : c, 4 * g4 + (i & 3));
              }
            }
          }
          __builtin_amdgcn_s_waitcnt(0x0F70);  // written before they are read back (by this wave only)
        }
      }
      auto load_pairs = [&](int t, u32x4 (&pr)[2]) {
        if (far) {
          int row = wr + t * 16 + c16;
          row = row < rows ? row : rows - 1;
          const char* const src = scratch + row_offset(row) + 16 * g4;
          pr[0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src));
          pr[1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + 64));
          asm volatile("" : "+v"(pr[0]), "+v"(pr[1]));  // (waited for here: behind the branch the other path would wait too)
        } else {
          pr[0] = *reinterpret_cast<const u32x4*>(ltab + (at[t] & 0xffffu));
          pr[1] = *reinterpret_cast<const u32x4*>(ltab + (at[t] >> 16));
        }
      };
      // norm of a token's row: 16 of its values here, the others in the lanes c16 + 16 k
      auto normalise = [&](float (&x)[4][4], const float (&w)[4][4], const float (&b)[4][4]) {
        auto fold = [](float s) { return sum_step<32>(sum_step<16>(s)); };
        float s[4] = {0.f, 0.f, 0.f, 0.f}, q[4] = {0.f, 0.f, 0.f, 0.f};  // four chains: a lone wave waits for each link of one
#pragma unroll
        for (int i = 0; i < 16; i++) s[i & 3] += x[i >> 2][i & 3];
        const float mean = fold((s[0] + s[1]) + (s[2] + s[3])) * (1.0f / 64);
#pragma unroll
        for (int i = 0; i < 16; i++) {
          x[i >> 2][i & 3] -= mean;
          q[i & 3] = fmaf(x[i >> 2][i & 3], x[i >> 2][i & 3], q[i & 3]);
        }
        const float rstd = inv_sqrt(fold((q[0] + q[1]) + (q[2] + q[3])) * (1.0f / 64) + p.eps);
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (int i = 0; i < 4; i++) x[c][i] = fmaf(x[c][i] * rstd, w[c][i], b[c][i]);
      };
      float lw[4][4], lb[4][4];
      if constexpr (NORM && TURN) {
        const float* const src = lln + (which == 1 ? 128 : 0) + 4 * g4;
#pragma unroll
        for (int c = 0; c < 4; c++) {
          load_row(src + c * 16, lw[c]);
          load_row(src + 64 + c * 16, lb[c]);
        }
      }
      unsigned char* const mine = lst + tl.wave * 2048;
#pragma unroll
      for (int h = 0; h < HD; h++) {
        float bias[4][4];  // added last, as the library's product does: the same bits where that does not split K
#pragma unroll
        for (int c = 0; c < 4; c++) {
          union { uint2 u; E e[4]; } b;
          b.u = *reinterpret_cast<const uint2*>(&lbias[par][tl.wn * 16 * T + (4 * h + c) * 16 + 4 * g4]);
#pragma unroll
          for (int i = 0; i < 4; i++) bias[c][i] = (float)b.e[i];
        }
        E* const dst = out + (int64_t)h * p.N * 64;
        float ps[4][4], pv[SETS ? SETS : 1][4];
#pragma unroll
        for (int s = 0; s < (SETS ? SETS : 1); s++)
#pragma unroll
          for (int i = 0; i < 4; i++) pv[s][i] = 0.f;
        u32x4 pr[2];
        uint4 st[NS];  // the group before, on its way out
        auto put = [&](int t) {
#pragma unroll
          for (int i = 0; i < NS; i++) {
            const int row = wr + t * 16 + i * 8 + (lane >> 3);
            store16_if(dst, 0x80000000u, row < rows ? row_offset(row) + (lane & 7) * 16 : 0x80000000u, st[i]);
          }
        };
        if constexpr (TURN) load_pairs(0, pr);
#pragma unroll
        for (int t = 0; t < T; t++) {
          float cs[2][4], sn[2][4];  // y, x
          if constexpr (TURN) {
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
              for (int i = 0; i < 4; i++) unpack_pair<E>(pr[c][i], cs[c][i], sn[c][i]);
            if (t + 1 < T) load_pairs(t + 1, pr);
          }
          float x[4][4];
#pragma unroll
          for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) x[c][i] = round_keep<E>(tl.acc[4 * h + c][t][i] + bias[c][i]);
          if constexpr (POOL != 0) {
            if (wr + t * 16 + 16 > rows) {  // rows behind the last one repeat it: not in the sums
              asm volatile("");             // (a branch, not 16 selects for every tile)
              const bool live = wr + t * 16 + c16 < rows;
#pragma unroll
              for (int c = 0; c < 4; c++)
#pragma unroll
                for (int i = 0; i < 4; i++) x[c][i] = live ? x[c][i] : 0.f;
            }
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
              for (int i = 0; i < 4; i++) ps[c][i] = POOL == 16 || t % 4 == 0 ? x[c][i] : ps[c][i] + x[c][i];
            if (POOL == 16 || t % 4 == 3) {
              // Sums over the 16 lanes of a group, halving what a lane holds: behind the first two exchanges lane c16 has the
              // four channels of tile c16 / 4, behind the last two all of a quad the whole sum.  Four blocks share the lanes.
              constexpr int per = POOL == 16 ? 1 : 4;
              const int blk = t / per;
              float r[2][4], z[4];
#pragma unroll
              for (int c = 0; c < 2; c++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                  const bool up = (c16 & 8) != 0;
                  const float keep = up ? ps[c + 2][i] : ps[c][i], give = up ? ps[c][i] : ps[c + 2][i];
                  r[c][i] = keep + lane_xor<8>(give);
                }
#pragma unroll
              for (int i = 0; i < 4; i++) {
                const bool up = (c16 & 4) != 0;
                const float keep = up ? r[1][i] : r[0][i], give = up ? r[0][i] : r[1][i];
                const int gi = __float_as_int(give);
                z[i] = keep + __int_as_float(__builtin_amdgcn_update_dpp(gi, gi, 0x141, 0xF, 0xF, false));  // row_half_mirror
                z[i] = sum_step<2>(sum_step<1>(z[i]));
                pv[blk / 4][i] = (c16 & 3) == blk % 4 ? z[i] : pv[blk / 4][i];
              }
            }
          }
          if constexpr (TURN) {
            if constexpr (NORM) normalise(x, lw, lb);
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
              for (int i = 0; i < 4; i++) {
                const float a = x[2 * c][i], b = x[2 * c + 1][i];
                x[2 * c][i] = fmaf(-b, sn[c][i], a * cs[c][i]);
                x[2 * c + 1][i] = fmaf(a, sn[c][i], b * cs[c][i]);
              }
          }
#pragma unroll
          for (int c = 0; c < 4; c++) {
            union { V2 v[2]; uint2 u; } o;
            o.v[0][0] = (E)x[c][0]; o.v[0][1] = (E)x[c][1];
            o.v[1][0] = (E)x[c][2]; o.v[1][1] = (E)x[c][3];
            *reinterpret_cast<uint2*>(mine + c16 * 128 + (((c * 2 + (g4 >> 1)) ^ row_swizzle(c16)) << 4) + (g4 & 1) * 8) = o.u;
          }
          // a group is stored behind the work on the next one, when its rows have come back from LDS
          if (t > 0) put(t - 1);
#pragma unroll
          for (int i = 0; i < NS; i++) {
            const int r = i * 8 + (lane >> 3);
            st[i] = *reinterpret_cast<const uint4*>(mine + r * 128 + (((lane & 7) ^ row_swizzle(r)) << 4));
          }
          __builtin_amdgcn_sched_barrier(0);  // a group's temporaries are dead before the next one's are born
        }
        put(T - 1);
        if constexpr (POOL != 0) {
#pragma unroll
          for (int s = 0; s < SETS; s++) {
            // lane (c16, g4): channels 16 (c16 / 4) + 4 g4 .. + 3 of block 4 s + c16 % 4
            const int blk = 4 * s + (c16 & 3), first = wr + blk * POOL;
            if (blk < BLOCKS && first < rows) {
              const bool over = first >= cross;
              const int to = (n0 + first - (over ? p.N : 0)) / POOL;
              E* const mean = (E*)(which == 0 ? p.qc : which == 1 ? p.kc : p.vc) +
                              ((int64_t)((b0 + over) * p.H + head + h) * p.Nc + to) * 64 + (c16 >> 2) * 16 + 4 * g4;
              const int left = rows - first;
              union { E e[4]; uint2 u; } o;
              if (left >= POOL) {  // (the same quotient: a power of two)
#pragma unroll
                for (int i = 0; i < 4; i++) o.e[i] = (E)(pv[s][i] * (1.0f / POOL));
              } else {
#pragma unroll
                for (int i = 0; i < 4; i++) o.e[i] = (E)(pv[s][i] / (float)left);
              }
              *reinterpret_cast<uint2*>(mean) = o.u;
            }
          }
        }
      }
    };
    if (which < 2) finish(std::true_type{});
    else if (which == 2) finish(std::false_type{});
    fresh = which > 2;  // (a wave beyond the last column has stored nothing)
    walk.at += walk.slots;
    if (walk.at >= walk.count) break;
    walk.locate(walk.at, m, n);
    tl.read_first(lx0, lw0);  // (the last step has read it too: 64 registers that the epilogue needs more)
  }
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // no transfer may still write LDS when the wave ends
  if (p.gate_out == nullptr) return;

  // ---- the gate: tiles of BM tokens x 32 outputs, for the workgroups that have one tile less than others (gate_rides) ----
  typedef Tile<E, T, 1> Gt;
  const int xcd = blockIdx.x & 7;
  const int from = (int)((int64_t)p.mt * xcd / 8), thin = (int)((int64_t)p.mt * (xcd + 1) / 8) - from;
  const int full = walk.count % walk.slots, idle = walk.slots - full;
  Gt gt;
  for (int i = (int)(blockIdx.x >> 3) - full; i >= 0 && i < thin; i += idle) {
    const int r0 = (from + i) * BM, rows = p.M - r0 < BM ? p.M - r0 : BM;
    __syncthreads();  // every wave is done with the LDS buffers
    gt.aim((const E*)p.x + r0 * p.ldx, p.ldx, rows, (const E*)p.gate_w, p.K, p.O);
#pragma unroll
    for (int t = 0; t < Gt::NL; t++) gt.move(lx0, lw0, 0, t);
#pragma unroll
    for (int t = 0; t < Gt::NL; t++) gt.move(lx1, lw1, 128, t);
    gt.begin(lx0, lw0);
    const int last = p.K * 2 - 128;
    int at = 128;
    gt.template sweep<0>(lx0, lw0, lx1, lw1, p.K >> 6, true, at, [&]() { at = at + 128 < last ? at + 128 : last; });  // (beyond the end the last step is requested again)
    gt.after_products();
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the requests beyond the end have landed
    const int o = gt.wn * 16 + 4 * gt.g4;
    if (o < p.O) {
      float bias[4];
#pragma unroll
      for (int e = 0; e < 4; e++) bias[e] = p.gate_b != nullptr ? (float)((const E*)p.gate_b)[o + e] : 0.f;
#pragma unroll
      for (int t = 0; t < T; t++) {
        const int row = gt.wm * WROWS + t * 16 + gt.c16;
        union { E e[4]; uint2 u; } g;  // rounding points of the two modules: the product with its bias, then the sigmoid
#pragma unroll
        for (int e = 0; e < 4; e++) g.e[e] = (E)(1.f / (1.f + expf(-round_to<E>(gt.acc[0][t][e] + bias[e]))));
        if (row < rows) *reinterpret_cast<uint2*>((E*)p.gate_out + (int64_t)(r0 + row) * p.O + o) = g.u;
      }
    }
  }
}


// Norm and rotation of the block means in place, at the truncated mean positions of their blocks: 8 lanes a row, 8 rows a wave,
// q and k; the pass's functions and rounding points.  The selection ranks products of these: other roundings are other
// choices.  (Inside the tiles' epilogue these chains of exchanges had one wave per SIMD to themselves: 65 of 725 us at 104 100
// tokens, where this takes 5.)
template <typename E> __global__ __launch_bounds__(256, 4) void finish_means_kernel(PrepassParams p, int64_t Nc, int64_t groups) {
  extern __shared__ __align__(16) float staged[];
  const int lane = threadIdx.x & 63, lr = lane & 7;
  const int64_t w_own = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), w = w_own < 2 * groups ? w_own : 0;
  const bool of_k = w >= groups;
  const int64_t per = (Nc + 7) / 8, at = of_k ? w - groups : w, bh = at / per, b = bh / p.H;
  const int64_t j = (at - bh * per) * 8 + (lane >> 3), jc = j < Nc ? j : Nc - 1;
  const int64_t t0 = jc * p.block;
  const int n = (int)(p.N - t0 < p.block ? p.N - t0 : p.block);
  E* const row = (E*)(of_k ? p.kc : p.qc) + (bh * Nc + jc) * 64 + lr * 8;
  const u32x4 raw = *reinterpret_cast<const u32x4*>(row);
  int sy = 0, sx = 0;
#pragma unroll
  for (int u = 0; u < 8; u++) {  // blocks of 16 or 64 tokens
    if (8 * u < p.block) {
      const int t = 8 * u + lr < n ? 8 * u + lr : n - 1;
      const int y = load_pos(p, b, t0 + t, 0), x = load_pos(p, b, t0 + t, 1);
      sy += 8 * u + lr < n ? y : 0;
      sx += 8 * u + lr < n ? x : 0;
    }
  }
  stage_tables<E>(p, staged);
  __syncthreads();
  if (w_own >= 2 * groups) return;
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) {
    sy += __shfl_xor(sy, off);
    sx += __shfl_xor(sx, off);
  }
  const RotLane<E> rl(lr);
  const int pp = (int)((float)(rl.half ? sx : sy) / (float)n);
  float x[8];
#pragma unroll
  for (int i = 0; i < 8; i++) x[i] = to_f32(reinterpret_cast<const E*>(&raw)[i]);
  norm_row<E>(p, staged, x, of_k ? 2 : 0, lr);
  rotate_row<E>(x, table_ptr<E>(p, staged, rl, pp, !rl.second));
  uint4 o;
#pragma unroll
  for (int i = 0; i < 8; i++) reinterpret_cast<E*>(&o)[i] = from_f32<E>(x[i]);
  if (j < Nc) *reinterpret_cast<uint4*>(row) = o;
}

template <typename E> static void launch_finish(const s3r_prepass_args& a, int64_t Nc, hipStream_t st) {
  PrepassParams p = prepass_params(a);
  p.staged_rows = 0;  // a row or two per lane: read where they are
  const int64_t groups = (int64_t)p.B * p.H * ((Nc + 7) / 8);
  hipLaunchKernelGGL((finish_means_kernel<E>), dim3((unsigned)((2 * groups + 3) / 4)), dim3(256), (unsigned)staged_bytes(0, true), st, p, Nc, groups);
}

// a wave of the large tile holds two heads: both of q, of k or of v
static bool large_project(int64_t M, int C) { return C % 128 == 0 && large_tiles(M, 3 * C); }

// Whether the gate costs nothing beside the projection: every XCD has two workgroups without a tile in the last round for each three
// of its thin tiles.  One takes half the time of a tile (short steps: it waits for its rows at each); more of them, or any on
// workgroups with a tile of their own, prolong the kernel, while the gate's own kernel can run beside the index kernel
// (layer, us, apart / here: 25 212 tokens 379 / 358, 2 016 131 / 124; 104 100, two per workgroup, 1 547 / 1 555, 32 256, four, 665 / 690).
static bool gate_rides(int64_t M, int C) {
  const bool large = large_project(M, C);
  const int b = large ? 256 : 128, most = large ? 256 : 512;
  const int64_t mt = (M + b - 1) / b, tiles = mt * ((3 * C + b - 1) / b);
  if (tiles + mt <= most) return true;  // (as many workgroups as tiles of both kinds)
  for (int xcd = 0; xcd < 8; xcd++) {
    const int64_t count = tiles / 8 + (xcd < tiles % 8 ? 1 : 0), thin = mt * (xcd + 1) / 8 - mt * xcd / 8;
    if (2 * thin > 3 * (most / 8 - count % (most / 8))) return false;
  }
  return true;
}

template <typename E, bool NORM, int POOL> static void launch_project(ProjectParams& p, hipStream_t st) {
  const bool large = large_project(p.M, p.C);
  const int b = large ? 256 : 128;
  p.mt = (p.M + b - 1) / b;
  p.nt = (3 * p.C + b - 1) / b;
  const int64_t tiles = (int64_t)p.mt * p.nt + (p.gate_out != nullptr ? p.mt : 0), most = large ? 256 : 512;
  // (gate: every XCD, which has its share of the thin tiles, needs a workgroup)
  const dim3 grid((unsigned)(tiles >= most ? most : p.gate_out != nullptr && tiles < 8 ? 8 : tiles)), blk(256);
  if (large) hipLaunchKernelGGL((project_kernel<E, 8, NORM, POOL, 1>), grid, blk, 0, st, p);
  else hipLaunchKernelGGL((project_kernel<E, 4, NORM, POOL, 2>), grid, blk, 0, st, p);
}

template <typename E> static void launch_project(ProjectParams& p, int pool, hipStream_t st) {
  if (p.ln[0] == nullptr) launch_project<E, false, 0>(p, st);
  else if (pool == 0) launch_project<E, true, 0>(p, st);
  else if (pool == 16) launch_project<E, true, 16>(p, st);
  else launch_project<E, true, 64>(p, st);
}

}  // namespace lin
}  // namespace s3r

using namespace s3r;

extern "C" int s3r_qkv_project_gate_rides(int64_t rows, int H) { return rows > 0 && H > 0 && H <= (1 << 20) / 192 && rows <= (1 << 30) && lin::gate_rides(rows, 64 * H); }

extern "C" int s3r_qkv_project(const void* x, const void* w, const void* bias, int64_t ldx, int64_t ldw, void* v_out, const s3r_prepass_args* a,
                               const void* gate_w, const void* gate_bias, void* gate_out, int gate_outputs, void* stream) {
  if (!a || !x || !w || !v_out || !a->q_out || !a->k_out || !a->positions || !a->cos_table || !a->sin_table)
    return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: null pointer");
  if (a->B <= 0 || a->H <= 0 || a->N <= 0 || a->table_rows <= 0) return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: non-positive size");
  const bool pool = a->q_pool != nullptr;
  if (pool != (a->k_pool != nullptr) || pool != (a->v_pool != nullptr) || (a->q_norm_weight == nullptr) != (a->k_norm_weight == nullptr))
    return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: means of q, k and v together or not at all, norms of q and k likewise");
  const int64_t M = (int64_t)a->B * a->N;
  const int C = 64 * a->H;
  if ((a->dtype != S3R_BF16 && a->dtype != S3R_F16) || a->head_dim != 64 || C % 128 || C > (1 << 20) / 3 || M > (1 << 30))
    return fail(S3R_ERR_UNSUPPORTED, "s3r_qkv_project: dtype %d, head_dim %d, %d heads, %lld rows (built for 16-bit types, head_dim 64, an even "
                "number of heads)", a->dtype, a->head_dim, a->H, (long long)M);
  if (a->inv_freq != nullptr && a->signed_positions)
    return fail(S3R_ERR_UNSUPPORTED, "s3r_qkv_project: angles of their own for positions below zero (built for positions that are clamped to zero)");
  // a tile of rows reaches into one more sequence at most; its rows are addressed by 32-bit byte offsets
  if (a->B > 1 && (a->N < 256 || (int64_t)a->H * a->N * 128 > 0x70000000LL))
    return fail(S3R_ERR_UNSUPPORTED, "s3r_qkv_project: %d sequences of %lld tokens (built for 256 tokens or more each)", a->B, (long long)a->N);
  if (pool && ((a->block != 16 && a->block != 64) || a->q_norm_weight == nullptr || !a->finish_pooled || a->q_raw != nullptr ||
               a->k_raw != nullptr || (a->B > 1 && a->N % a->block)))
    return fail(S3R_ERR_UNSUPPORTED, "s3r_qkv_project: means over blocks of %d (built for final means with norms, blocks of 16 or 64 tokens "
                "that end with each sequence of a batch)", a->block);
  if (ldx < C || ldw < C || ldx >= (1 << 21) || ldw >= (1 << 21))
    return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: rows overlap or lie 2^21 elements or more apart");
  const void* ptrs[] = {x, w, a->q_out, a->k_out, v_out, a->q_pool, a->k_pool, a->v_pool, a->cos_table, a->sin_table};
  for (const void* ptr : ptrs)
    if (!aligned16(ptr)) return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: pointers must be multiples of 16 bytes");
  if (ldx % 8 || ldw % 8 || (reinterpret_cast<uintptr_t>(bias) & 7u))
    return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: rows must be multiples of 16 bytes, the bias of 8");
  if (gate_out != nullptr) {
    if (!gate_w) return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: null pointer");
    if (gate_outputs <= 0 || gate_outputs > 32 || gate_outputs % 4)
      return fail(S3R_ERR_UNSUPPORTED, "s3r_qkv_project: %d gate outputs (built for a multiple of 4 up to 32)", gate_outputs);
    if (!aligned16(gate_w) || (reinterpret_cast<uintptr_t>(gate_out) & 7u))
      return fail(S3R_ERR_BAD_ARG, "s3r_qkv_project: the gate's weight must be a multiple of 16 bytes, its output of 8");
  }
  lin::ProjectParams p = {};
  p.gate_w = gate_w; p.gate_b = gate_bias; p.gate_out = gate_out; p.O = gate_outputs;
  p.x = x; p.w = w; p.bias = bias; p.ldx = ldx; p.ldw = ldw;
  p.M = (int)M; p.N = (int)a->N; p.K = C; p.C = C; p.H = a->H; p.Nc = pool ? (int)((a->N + a->block - 1) / a->block) : 0;
  p.q = a->q_out; p.k = a->k_out; p.v = v_out; p.qc = a->q_pool; p.kc = a->k_pool; p.vc = a->v_pool;
  p.pos = a->positions; p.pos64 = a->positions_int64; p.spb = a->pos_stride_b; p.spn = a->pos_stride_n;
  p.cos_tab = a->cos_table; p.sin_tab = a->sin_table; p.inv_freq = a->inv_freq; p.P = a->table_rows;
  p.staged_rows = p.P < kStagedRows ? p.P : kStagedRows;
  p.ln[0] = a->q_norm_weight; p.ln[1] = a->q_norm_bias; p.ln[2] = a->k_norm_weight; p.ln[3] = a->k_norm_bias;
  p.ln_f32 = a->norm_fp32; p.eps = a->eps;
  if (a->dtype == S3R_BF16) lin::launch_project<bf16_t>(p, pool ? a->block : 0, (hipStream_t)stream);
  else lin::launch_project<f16_t>(p, pool ? a->block : 0, (hipStream_t)stream);
  const int rc = check_launch("s3r_qkv_project");
  if (rc != S3R_OK || !pool) return rc;
  if (a->dtype == S3R_BF16) lin::launch_finish<bf16_t>(*a, p.Nc, (hipStream_t)stream);
  else lin::launch_finish<f16_t>(*a, p.Nc, (hipStream_t)stream);
  return check_launch("s3r_qkv_project (means)");
}
