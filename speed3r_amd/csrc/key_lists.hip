// Key-centric lists of the selection branch's index tensor, for the dK/dV kernel of the backward.
//
// Reference: count_query_fixedlen and reorder_topk_idx_fixedlen with the stable argsort between them
// (pi3/models/sparse_attn/topk_blocksparse_attention.py:423-554).  For every (b, h) and key block j the list
// holds the ids of the query blocks whose index row names j, one entry per occurrence, ascending; off[j] .. off[j+1]
// delimit it.  Entries of idx that are < 0 or >= nkb appear in no list.
//
// Up to kHeadEntries index entries per head, with one exception at the launch (count, scan and fill in one kernel, then sort): workgroup (p, head) reads all of the head's
// entries and owns the key blocks lo .. hi: it counts theirs in LDS and, in a register, the entries of the blocks below, which gives the
// start of its first list without a word from the others; then it reads the entries again and writes those of its blocks.  us, five kernels
// without their sorts / this: 2 x 16 heads of 756 rows of 32 46 / 16, 16 heads of 4 164 rows of 16 43 / 26; with the sorts 2 x 16 x 756 x 32 60 / 30,
// 16 x 4 096 x 32 90 / 75, 16 x 16 000 x 8 139 / 95.  Bound: the passes over the entries, eight loads in flight a thread.
// More entries: five small kernels.  No workspace besides the two outputs either way:
//   zero     off[*] = 0
//   count    histogram of the index entries, block j counted at off[j + 2] (pre-aggregated per workgroup in LDS)
//   scan     inclusive prefix sum per (b, h): off[j + 1] = first position of block j's list
//   fill     every entry takes a position with an atomic increment of off[j + 1], which thereby ends up at the END of
//            block j's list = the start of block j+1's: exactly the offsets array, off[0] = 0 included
//   sort     the atomic order is arbitrary, so each list is then sorted ascending, which makes the result unique
//            (equal ids are indistinguishable): lists of up to 512 entries by one wavefront in registers (rank by
//            counting up to 64, a bitonic network beyond), longer ones by one workgroup with Batcher's merge exchange, in LDS (up to 8192 entries) or
//            in place in global memory.
#include "s3r_common.h"

namespace s3r {
namespace kl {

constexpr int kLdsCap = 8192;

__global__ __launch_bounds__(256) void zero_kernel(int32_t* __restrict__ off, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) off[i] = 0;
}

// count and fill share one kernel body.  Neighbouring query blocks name mostly the same key blocks, and atomics on
// one address serialise in memory, so a workgroup first gathers its 1024 index entries in an LDS hash table (key
// block -> occurrences), every entry taking its rank among the workgroup's occurrences of its key block with an LDS
// atomic; one global atomic per DISTINCT key block then adds the count (count pass: at off[j + 2]) or reserves the
// positions (fill pass: at off[j + 1]), and in the fill pass every entry writes its query block at base + rank.
// A workgroup stays inside one (b, h): grid.y = B*H, grid.x = chunks of 1024 entries.
constexpr int kHashSlots = 2048;

template <bool FILL>
__global__ __launch_bounds__(1024) void gather_kernel(const int32_t* __restrict__ idx, int32_t* __restrict__ off, int32_t* __restrict__ list, int H,
                                                      int64_t nqb, int K, int64_t nkb, int64_t sib, int64_t sih, int64_t sim, int64_t list_stride) {
  __shared__ int32_t keys[kHashSlots];
  __shared__ int32_t cnt[kHashSlots];
  __shared__ int32_t base[kHashSlots];
  const int t = threadIdx.x;
  for (int i = t; i < kHashSlots; i += 1024) {
    keys[i] = -1;
    cnt[i] = 0;
  }
  __syncthreads();
  const int64_t bh = blockIdx.y;
  const int64_t hh = bh % H, bb = bh / H;
  const int64_t e = (int64_t)blockIdx.x * 1024 + t;  // entry within this (b, h)
  int32_t j = -1, m = 0;
  if (e < nqb * K) {
    m = (int32_t)(e / K);
    j = idx[bb * sib + hh * sih + (int64_t)m * sim + (e - (int64_t)m * K)];
    if (j < 0 || j >= nkb) j = -1;
  }
  int slot = 0, rank = 0;
  if (j >= 0) {
    slot = (int)(((uint32_t)j * 2654435761u) >> 21);  // 11 bits
    while (true) {
      const int32_t old = atomicCAS(&keys[slot], -1, j);
      if (old == -1 || old == j) break;
      slot = (slot + 1) & (kHashSlots - 1);  // at most 1024 keys in 2048 slots: a free slot exists
    }
    rank = atomicAdd(&cnt[slot], 1);
  }
  __syncthreads();
  for (int i = t; i < kHashSlots; i += 1024) {
    const int32_t kj = keys[i];
    if (kj >= 0) {
      if (FILL) base[i] = atomicAdd(off + bh * (nkb + 1) + kj + 1, cnt[i]);
      else if ((int64_t)kj + 2 <= nkb) atomicAdd(off + bh * (nkb + 1) + kj + 2, cnt[i]);  // the last block's count is not needed
    }
  }
  if (FILL) {
    __syncthreads();
    if (j >= 0) list[bh * list_stride + base[slot] + rank] = m;
  }
}

constexpr int64_t kHeadEntries = 1 << 17;
constexpr int kMostSpan = 1 << 14;  // key blocks of a workgroup

__global__ __launch_bounds__(1024) void head_lists_kernel(const int32_t* __restrict__ idx, int32_t* __restrict__ off, int32_t* __restrict__ list,
                                                           int H, int nqb, int K, int nkb, int span, int64_t sib, int64_t sih,
                                                           int64_t sim, int64_t list_stride) {
  extern __shared__ int32_t cnt[];  // of the workgroup's key blocks; later where the next entry of each goes
  __shared__ int32_t part[1024], below_of[16];
  const int t = threadIdx.x, lo = blockIdx.x * span, hi = lo + span < nkb ? lo + span : nkb;
  if (lo >= nkb) return;
  const int64_t bh = blockIdx.y, hh = bh % H, bb = bh / H;
  const int32_t* const rows = idx + bb * sib + hh * sih;
  for (int i = t; i < hi - lo; i += 1024) cnt[i] = 0;
  __syncthreads();
  // a thread stays in one column: 1024 / K rows at a time
  const int step = 1024 / K, first = t / K;
  const int32_t* const own = rows + (int64_t)first * sim + (t - first * K);
  const int end = first < step ? nqb : 0;
  int below = 0;
  auto walk = [&](auto take) {  // eight entries on their way at once
    const int32_t* from = own;
    for (int m = first; m < end; m += 8 * step) {
      int32_t j[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        j[u] = m + u * step < end ? *from : -1;
        from += step * sim;
      }
#pragma unroll
      for (int u = 0; u < 8; u++) take(m + u * step, j[u]);
    }
  };
  walk([&](int, int32_t j) {
    below += j >= 0 && j < lo ? 1 : 0;
    if (j >= lo && j < hi) atomicAdd(&cnt[j - lo], 1);
  });
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) below += __shfl_xor(below, d);
  if ((t & 63) == 0) below_of[t >> 6] = below;
  __syncthreads();
  const int per = (hi - lo + 1023) / 1024, b0 = t * per, b1 = b0 + per < hi - lo ? b0 + per : hi - lo;
  int32_t sum = 0;
  for (int i = b0; i < b1; i++) sum += cnt[i];
  part[t] = sum;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {  // Hillis-Steele over the 1024 partial sums
    const int32_t v = t >= d ? part[t - d] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int32_t at = t > 0 ? part[t - 1] : 0;
#pragma unroll
  for (int w = 0; w < 16; w++) at += below_of[w];
  int32_t* const starts = off + bh * (nkb + 1);
  for (int i = b0; i < b1; i++) {
    const int32_t n = cnt[i];
    cnt[i] = starts[lo + i] = at;
    at += n;
  }
  if (hi == nkb && b0 < b1 && b1 == hi - lo) starts[nkb] = at;
  __syncthreads();
  walk([&](int m, int32_t j) {
    if (j >= lo && j < hi) list[bh * list_stride + atomicAdd(&cnt[j - lo], 1)] = m;
  });
}

// one workgroup of 1024 per (b, h): in-place inclusive scan of n values
__global__ __launch_bounds__(1024) void scan_kernel(int32_t* __restrict__ off, int64_t n) {
  __shared__ int32_t part[1024];
  int32_t* a = off + (int64_t)blockIdx.x * n;
  const int t = threadIdx.x;
  const int64_t per = (n + 1023) / 1024;
  const int64_t lo = t * per, hi = lo + per < n ? lo + per : n;
  int32_t s = 0;
  for (int64_t i = lo; i < hi; i++) s += a[i];
  part[t] = s;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {  // Hillis-Steele over the 1024 partial sums
    const int32_t v = t >= d ? part[t - d] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int32_t run = t > 0 ? part[t - 1] : 0;
  for (int64_t i = lo; i < hi; i++) {
    run += a[i];
    a[i] = run;
  }
}

// lists of 2 .. 64 entries: one wavefront, one entry per lane; rank of an entry = entries below it + equal entries at lower
// positions.  Every entry is in a register before the first one is written back.
__device__ __forceinline__ void wave_rank_sort(int32_t* a, int n, int lane) {
  const int32_t x = lane < n ? a[lane] : 0x7fffffff;
  int rank = 0;
  for (int i = 0; i < n; i++) {
    const int32_t xi = __builtin_amdgcn_readlane(x, i);
    rank += (xi < x || (xi == x && i < lane)) ? 1 : 0;
  }
  if (lane < n) a[rank] = x;
}

// lists of up to 64*M entries: one wavefront, M entries per lane (entry 64 r + lane in register r), a bitonic network filled up
// with values above all.  A rank count takes n * M comparisons per lane, 65 000 cycles at 512 entries, and the launch lasted as
// long as its longest list; the network takes 45 exchanges of 8 registers.  All lists, 16 heads, us, ranks / networks: 266 496 tokens in 64-token blocks,
// top-16 53 / 22; two sequences of 12 096 in 16-token blocks, top-32 41 / 17.
template <int M>
__device__ __forceinline__ void wave_bitonic_sort(int32_t* a, int n, int lane) {
  int32_t x[M];
#pragma unroll
  for (int r = 0; r < M; r++) x[r] = 64 * r + lane < n ? a[64 * r + lane] : 0x7fffffff;
#pragma unroll
  for (int size = 2; size <= 64 * M; size <<= 1)
#pragma unroll
    for (int step = size >> 1; step > 0; step >>= 1) {
      if (step >= 64) {  // between two registers of a lane
#pragma unroll
        for (int r = 0; r < M; r++) {
          const int s = r ^ (step >> 6);
          if (s > r) {
            const bool up = ((64 * r) & size) == 0;
            const int32_t lo = min(x[r], x[s]), hi = max(x[r], x[s]);
            x[r] = up ? lo : hi;
            x[s] = up ? hi : lo;
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < M; r++) {
          const int32_t y = __shfl_xor(x[r], step);
          const bool up = ((64 * r + lane) & size) == 0, low = (lane & step) == 0;
          x[r] = up == low ? min(x[r], y) : max(x[r], y);
        }
      }
    }
#pragma unroll
  for (int r = 0; r < M; r++)
    if (64 * r + lane < n) a[64 * r + lane] = x[r];
}

constexpr int kWaveSortCap = 512;

__global__ __launch_bounds__(256) void sort_short_kernel(int32_t* __restrict__ list, const int32_t* __restrict__ off, int64_t nkb,
                                                         int64_t list_stride, int64_t nseg) {
  const int64_t seg = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (seg >= nseg) return;
  const int64_t bh = seg / nkb, j = seg - bh * nkb;
  const int32_t lo = off[bh * (nkb + 1) + j], hi = off[bh * (nkb + 1) + j + 1];
  const int n = __builtin_amdgcn_readfirstlane(hi - lo);
  if (n < 2 || n > kWaveSortCap) return;
  int32_t* a = list + bh * list_stride + lo;
  if (n <= 64) wave_rank_sort(a, n, lane);
  else if (n <= 128) wave_bitonic_sort<2>(a, n, lane);
  else if (n <= 256) wave_bitonic_sort<4>(a, n, lane);
  else wave_bitonic_sort<8>(a, n, lane);
}

// Batcher's merge exchange (Knuth, TAOCP 3, algorithm 5.2.2M) on n entries, any n: per stage (p, k) the comparators
// (a, a + k) with (a - k mod p) mod 2k < k and a, a+k in the same block of 2p are disjoint; 256 threads share them.
template <typename P>
__device__ __forceinline__ void merge_exchange(P a, int n) {
  for (int lp = 0; (1 << lp) < n; lp++)  // p = 2^lp
    for (int lk = lp; lk >= 0; lk--) {   // k = 2^lk
      const int k = 1 << lk;
      const int kp = lk == lp ? 0 : k;  // k mod p
      for (int i = threadIdx.x; i < n - k; i += 256) {
        const int r = i - kp;
        if (r >= 0 && (r & (2 * k - 1)) < k && (i >> (lp + 1)) == ((i + k) >> (lp + 1))) {
          const int32_t u = a[i], v = a[i + k];
          if (u > v) {
            a[i] = v;
            a[i + k] = u;
          }
        }
      }
      __syncthreads();
    }
}

// lists beyond the wave sort: workgroup w looks at lists w, w + G, w + 2G, ... (long lists come in runs of
// neighbouring key blocks; the stride spreads a run over many workgroups) and sorts the long ones
__global__ __launch_bounds__(256) void sort_long_kernel(int32_t* __restrict__ list, const int32_t* __restrict__ off, int64_t nkb,
                                                        int64_t list_stride, int64_t nseg) {
  __shared__ int32_t stage[kLdsCap];
  __shared__ int64_t found[256];
  __shared__ int nfound;
  const int64_t G = gridDim.x;
  for (int64_t base = blockIdx.x; base < nseg; base += 256 * G) {
    if (threadIdx.x == 0) nfound = 0;
    __syncthreads();
    const int64_t seg = base + (int64_t)threadIdx.x * G;
    if (seg < nseg) {
      const int64_t bh = seg / nkb, j = seg - bh * nkb;
      if (off[bh * (nkb + 1) + j + 1] - off[bh * (nkb + 1) + j] > kWaveSortCap) found[atomicAdd(&nfound, 1)] = seg;
    }
    __syncthreads();
    const int nf = nfound;
    for (int f = 0; f < nf; f++) {
      const int64_t sg = found[f];
      const int64_t bh = sg / nkb, j = sg - bh * nkb;
      const int32_t lo = off[bh * (nkb + 1) + j];
      const int n = off[bh * (nkb + 1) + j + 1] - lo;
      int32_t* a = list + bh * list_stride + lo;
      if (n <= kLdsCap) {
        for (int i = threadIdx.x; i < n; i += 256) stage[i] = a[i];
        __syncthreads();
        merge_exchange(stage, n);
        for (int i = threadIdx.x; i < n; i += 256) a[i] = stage[i];
        __syncthreads();
      } else {
        merge_exchange(a, n);  // in place in global memory: __syncthreads orders the workgroup's accesses
      }
    }
    __syncthreads();
  }
}

}  // namespace kl

int launch_key_block_lists(const int32_t* idx, int32_t* kq_list, int32_t* kq_off, int B, int H, int64_t nqb, int K, int64_t nkb,
                           int64_t sib, int64_t sih, int64_t sim, int64_t list_stride, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  const int64_t bh = (int64_t)B * H;
  const int64_t noff = bh * (nkb + 1), total = bh * nqb * K, nseg = bh * nkb;
  const int64_t g_off = (noff + 255) / 256, g_ent = (total + 255) / 256, g_short = (nseg * 64 + 255) / 256;
  if (g_off > 0x7fffffffLL || g_ent > 0x7fffffffLL || g_short > 0x7fffffffLL || bh > 65535)
    return fail(S3R_ERR_UNSUPPORTED, "s3r_key_block_lists: tensor too large for one launch");
  // workgroups for every CU once; each reads all of a head's entries
  const int64_t parts = bh >= 256 ? 1 : 256 / bh < nkb ? 256 / bh : nkb, span = (nkb + parts - 1) / parts;
  // One head alone: all 256 workgroups read all of its entries, and with many of them the five kernels are as good while the scan is short
  // and the lists too (us, five kernels / one, entries x key blocks: 98 304 x 8 192 32.6 / 32.7, 131 072 x 4 096 39.9 / 39.6, x 6 144 36.2 / 39.3,
  // x 8 192 35.4 / 39.4, x 9 216 43.3 / 40.1; two heads of 131 072 x 8 192 48.3 / 43.1).
  const bool crowded = bh == 1 && nqb * K > 98304 && nkb > 4096 && nkb <= 8192;
  if (nqb * K <= kl::kHeadEntries && K <= 1024 && span <= kl::kMostSpan && !crowded) {
    hipLaunchKernelGGL(kl::head_lists_kernel, dim3((unsigned)parts, (unsigned)bh), dim3(1024), (unsigned)(span * 4), st, idx, kq_off, kq_list, H,
                       (int)nqb, K, (int)nkb, (int)span, sib, sih, sim, list_stride);
  } else {
    hipLaunchKernelGGL(kl::zero_kernel, dim3((unsigned)g_off), dim3(256), 0, st, kq_off, noff);
    const dim3 g_gather((unsigned)((nqb * K + 1023) / 1024), (unsigned)bh);
    hipLaunchKernelGGL(kl::gather_kernel<false>, g_gather, dim3(1024), 0, st, idx, kq_off, kq_list, H, nqb, K, nkb, sib, sih, sim, list_stride);
    hipLaunchKernelGGL(kl::scan_kernel, dim3((unsigned)bh), dim3(1024), 0, st, kq_off, nkb + 1);
    hipLaunchKernelGGL(kl::gather_kernel<true>, g_gather, dim3(1024), 0, st, idx, kq_off, kq_list, H, nqb, K, nkb, sib, sih, sim, list_stride);
  }
  hipLaunchKernelGGL(kl::sort_short_kernel, dim3((unsigned)g_short), dim3(256), 0, st, kq_list, kq_off, nkb, list_stride, nseg);
  const int64_t g_long = nseg < 4096 ? nseg : 4096;
  hipLaunchKernelGGL(kl::sort_long_kernel, dim3((unsigned)g_long), dim3(256), 0, st, kq_list, kq_off, nkb, list_stride, nseg);
  return check_launch("s3r_key_block_lists");
}

}  // namespace s3r
