// Weight gradients of linear layers on the matrix cores: dW = dY^T X over many tokens (dY [M, N], X [M, C], bf16 / fp16; sums and
// partial sums in fp32).
//
// Few outputs, a long contraction: 3072 x 1024 are 48 tiles of 256 x 256 for 256 CUs, and a library product that does not split
// the tokens leaves the chip idle.  Here each tile's tokens are dealt out over enough workgroups to fill the chip once; their
// partial tiles meet in a workspace and a second kernel adds them.  The sums of dY over the tokens (the bias's gradient) take one
// more product by ones in 64: the tiles that share dY's columns share them out.  bf16, us, the library's product and its sum of
// dY / here: 24 192 tokens 3072 x 1024 246 + 41 / 137 (1.11 PFLOP/s), 1024 x 1024 181 + 29 / 63, 32 x 1024 79 + 10 / 28; 8 192
// tokens 85 + 26 / 62 and 53 + 20 / 38; 50 000 tokens 3072 x 1024 418 + 74 / 267.  The last rows, fewer than 128, come as a
// pair of steps filled up with zeros (added by the second kernel one by one, 64 of them made 24 000 tokens 160 us instead of 125).  Bound by the matrix cores' power where tiles
// are many, by the way of the partial tiles where they are few (64 MB each way for 1024 x 1024).
//
// The tile is linear_tile.h's (four waves of 128 x 128 values in all accumulator registers, operands a half step ahead, transfers
// two steps ahead, one barrier per step), but both operands have their contraction index across rows: a step is 64 tokens x 256
// channels of each, rows of 512 bytes, and ds_read_b64_tr_b16 hands a lane four tokens of one channel.  A transposed read
// touches 4 rows x 32 bytes per 16 lanes; unit u of 32 bytes of row r sits at u ^ unit_swizzle(r), so that the eight rows of a
// pass lie in different banks.
#include "linear_tile.h"

namespace s3r {
namespace lin {

struct WgradParams {
  const void *dy, *x;
  void *dw, *db;  // db: the sums of dY over the tokens, or null
  float* ws;      // [splits][N][C], then with db [splits][N]
  int64_t M, lddy, ldx;
  int N, C, nt, ct, splits;
  int64_t units;  // pairs of steps, 128 tokens each, the last one perhaps fewer
};

__device__ __forceinline__ constexpr int unit_swizzle(int row) { return (row & 3) | (((row >> 3) & 1) << 2); }

__device__ __forceinline__ s16x4 read_tr(const void* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)p);
}

// 16 bytes per lane from base + off to dst + 16 lane; zeros where `off` is not below `bytes`
__device__ __forceinline__ void rows_to_lds(const char* base, int bytes, void* dst, uint32_t off) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes > 0 ? bytes : 0, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, 0);
}

template <typename E> struct TokenTile {
  typedef typename Mma<E>::V8 V8;
  static constexpr int T = 8, NM = 64;
  int wave, lane;
  uint32_t xoff[T], yoff[T];   // the lane's pieces of a step's rows
  uint32_t fx[T], fy[T];       // where the wave's tiles lie in a buffer's first rows
  const char *bx, *by;
  int sx, sy;                  // bytes from step to step
  int nx, ny;                  // bytes of the range's rows: what lies beyond is read as zeros
  struct Frag8 { V8 x[T], y[T], b; } P, Q;
  uint32_t fb;                 // the tile of dY whose sums this wave takes (b)
  V8 ones;
  f32x4 sums;                  // lane: out-channel lane % 16, four times
  f32x4 acc[T][T];             // [out][in]: lane: in-channels 4 (lane / 16) .. + 3 of out-channel lane % 16

  __device__ __forceinline__ void init(const E* x, int64_t ldx, int xcols, const E* dy, int64_t ldy, int ycols, int rows, int sum_tile) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    bx = reinterpret_cast<const char*>(x);
    by = reinterpret_cast<const char*>(dy);
    sx = (int)(ldx * 128);
    sy = (int)(ldy * 128);
    nx = rows * (int)(ldx * 2);
    ny = rows * (int)(ldy * 2);
#pragma unroll
    for (int i = 0; i < T; i++) {
      const int row = 16 * wave + 2 * i + (lane >> 5);
      const int chunk = ((((lane & 31) >> 1) ^ unit_swizzle(row)) << 1) | (lane & 1);  // columns beyond the last repeat its piece
      xoff[i] = (uint32_t)row * (uint32_t)(ldx * 2) + (uint32_t)(chunk * 8 < xcols ? chunk : xcols / 8 - 1) * 16u;
      yoff[i] = (uint32_t)row * (uint32_t)(ldy * 2) + (uint32_t)(chunk * 8 < ycols ? chunk : ycols / 8 - 1) * 16u;
    }
    const int g4 = lane >> 4, i16 = lane & 15;
    const int row = 8 * g4 + (i16 >> 2), f = unit_swizzle(row);
#pragma unroll
    for (int c = 0; c < T; c++) {
      const int at = row * 512 + (i16 & 3) * 8;
      fx[c] = at + (((wave & 1) * T + (c ^ f)) << 5);
      fy[c] = at + (((wave >> 1) * T + (c ^ f)) << 5);
    }
    fb = row * 512 + (i16 & 3) * 8 + (((wave >> 1) * T + ((sum_tile & 7) ^ f)) << 5);
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = (E)1.f;
    sums = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  template <typename P8> __device__ __forceinline__ void move(P8* lx, P8* ly, uint32_t step, int i) {
    const int px = (int)step * sx, py = (int)step * sy;
    if (i < T) rows_to_lds(bx + px, nx - px, lx + (16 * wave + 2 * i) * 512, xoff[i]);
    else rows_to_lds(by + py, ny - py, ly + (16 * wave + 2 * (i - T)) * 512, yoff[i - T]);
  }
  template <typename P8> __device__ __forceinline__ void read(Frag8& f, P8* lx, P8* ly, int half, int r) {  // fragment r: y0, x0 .., y1 ..
    union { s16x4 s[2]; V8 v; } g;
    const bool of_x = r >= 1 && r <= T, of_b = r == 2 * T;
    const int t = of_b ? 0 : of_x ? r - 1 : r == 0 ? 0 : r - T;
    P8* const a = of_b ? ly + fb : of_x ? lx + fx[t] : ly + fy[t];
    g.s[0] = read_tr(a + half * 32 * 512);
    g.s[1] = read_tr(a + half * 32 * 512 + 4 * 512);
    if (of_b) f.b = g.v;
    else if (of_x) f.x[t] = g.v;
    else f.y[t] = g.v;
  }
  template <typename P8> __device__ __forceinline__ void step(P8* lx, P8* ly, P8* ox, P8* oy, uint32_t next) {
#pragma unroll
    for (int j = 0; j < NM; j++) {
      if (j % 3 == 0 && j / 3 <= 2 * T) read(Q, lx, ly, 1, j / 3);
      mma_acc<E, true>(P.x[j % T], P.y[j / T], acc[j / T][j % T]);
      if (j == NM - 1) mma_acc<E, false>(ones, P.b, sums);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0), as in linear_tile.h
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NM; j++) {
      if (j % 4 == 0) move(lx, ly, next, j / 4);
      if (j % 4 == 2) read(P, ox, oy, 0, j / 4);
      if (j == NM - 1) read(P, ox, oy, 0, 2 * T);
      mma_acc<E, true>(Q.x[j % T], Q.y[j / T], acc[j / T][j % T]);
      if (j == NM - 1) mma_acc<E, false>(ones, Q.b, sums);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __device__ __forceinline__ void touch() {
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int b = 0; b < T; b++) asm volatile("" : "+a"(acc[a][b]));
  }
};

template <typename E> __global__ __launch_bounds__(256, 1) void wgrad_kernel(WgradParams p) {
  typedef TokenTile<E> Tl;
  __shared__ __attribute__((aligned(1024))) unsigned char lx0[64 * 512];
  __shared__ __attribute__((aligned(1024))) unsigned char lx1[64 * 512];
  __shared__ __attribute__((aligned(1024))) unsigned char ly0[64 * 512];
  __shared__ __attribute__((aligned(1024))) unsigned char ly1[64 * 512];
  // the tiles of one range of tokens side by side on an XCD: they share its rows
  const int tiles = p.nt * p.ct, total = tiles * p.splits;
  const int xcd = blockIdx.x & 7, per = total >> 3, rem = total & 7;
  const int vid = xcd * per + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int s = vid / tiles, tile = vid - s * tiles;
  const int nb = tile / p.ct, cb = tile - nb * p.ct, n0 = nb * 256, c0 = cb * 256;
  const int sum_tile = 2 * cb + (threadIdx.x >> 6 & 1);  // the tiles of one row of tiles share the sums of its dY
  const int64_t u0 = p.units * s / p.splits, u1 = p.units * (s + 1) / p.splits;
  Tl tl;
  tl.init((const E*)p.x + u0 * 128 * p.ldx + c0, p.ldx, p.C - c0 < 256 ? p.C - c0 : 256, (const E*)p.dy + u0 * 128 * p.lddy + n0, p.lddy,
          p.N - n0 < 256 ? p.N - n0 : 256, (int)(u1 * 128 < p.M ? (u1 - u0) * 128 : p.M - u0 * 128), __builtin_amdgcn_readfirstlane(sum_tile));
  const uint32_t steps = (uint32_t)(u1 - u0) * 2;
  if (steps == 0) return;  // (never: as many splits as units at most)
#pragma unroll
  for (int i = 0; i < 16; i++) tl.move(lx0, ly0, 0, i);
#pragma unroll
  for (int i = 0; i < 16; i++) tl.move(lx1, ly1, 1, i);
  __builtin_amdgcn_s_waitcnt(0x0F70 | (1 << 14));  // vmcnt(16): the first step has landed
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r <= 16; r++) tl.read(tl.P, lx0, ly0, 0, r);
#pragma unroll
  for (int a = 0; a < 8; a++)
#pragma unroll
    for (int b = 0; b < 8; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) tl.acc[a][b][i] = 0.f;
  tl.touch();
  asm volatile("s_nop 7");
  uint32_t t = 0;
  do {  // (beyond the end the last step is requested again)
    tl.step(lx0, ly0, lx1, ly1, t + 2 < steps ? t + 2 : steps - 1);
    tl.step(lx1, ly1, lx0, ly0, t + 3 < steps ? t + 3 : steps - 1);
    t += 2;
  } while (t < steps);
  asm volatile("s_nop 15\n s_nop 15");
  tl.touch();
  asm volatile("" : "+v"(tl.sums));
  float* const ws = p.ws + (int64_t)s * p.N * p.C;
  const int n = n0 + (tl.wave >> 1) * 128 + (tl.lane & 15), c = c0 + (tl.wave & 1) * 128 + 4 * (tl.lane >> 4);
#pragma unroll
  for (int a = 0; a < 8; a++)
#pragma unroll
    for (int b = 0; b < 8; b++)
      if (n + 16 * a < p.N && c + 16 * b < p.C) *reinterpret_cast<f32x4*>(ws + (int64_t)(n + 16 * a) * p.C + c + 16 * b) = tl.acc[a][b];
  if (p.db && sum_tile < 8 && tl.lane < 16) {
    const int o = n0 + (tl.wave >> 1) * 128 + 16 * sum_tile + tl.lane;
    if (o < p.N) p.ws[(int64_t)p.splits * p.N * p.C + (int64_t)s * p.N + o] = tl.sums[0];
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // no transfer may still write LDS when the wave ends
}

// dW = sum of the partial tiles, db = sum of the partial sums: HBM bound.  PARTS threads share an output's partial values (every
// PARTS-th range each) and meet in LDS: with few outputs a thread alone with up to 64 dependent waits is all there is
// (24 192 tokens, 32 x 1024 with their bias, 64 ranges: 18.5 us with one thread per output, 5.2 with eight; 1024 x 1024 16.2 / 12.4).
template <typename E, int PARTS> __global__ __launch_bounds__(256) void wgrad_sum_kernel(WgradParams p) {
  constexpr int kOut = 256 / PARTS;  // threads that hold an output (four weights, or one bias)
  __shared__ f32x4 part[PARTS > 1 ? 256 : 1];
  const int at = threadIdx.x % kOut, g = threadIdx.x / kOut;
  const int64_t quads = (int64_t)p.N * p.C / 4, o = (int64_t)blockIdx.x * kOut + at, n = o - quads;
  const bool weight = o < quads, sum = !weight && p.db != nullptr && n < p.N;  // behind the weights: the biases
  f32x4 a = {0.f, 0.f, 0.f, 0.f};
  if (weight) {
#pragma unroll 8
    for (int s = g; s < p.splits; s += PARTS) a += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.ws + (int64_t)s * p.N * p.C + o * 4));
  } else if (sum) {
#pragma unroll 8
    for (int s = g; s < p.splits; s += PARTS) a[0] += p.ws[(int64_t)p.splits * p.N * p.C + (int64_t)s * p.N + n];
  }
  if constexpr (PARTS > 1) {
    part[threadIdx.x] = a;
    __syncthreads();
    if (g != 0) return;
#pragma unroll
    for (int k = 1; k < PARTS; k++) a += part[k * kOut + at];
  }
  if (weight) {
    union { E e[4]; uint2 u; } out;
#pragma unroll
    for (int k = 0; k < 4; k++) out.e[k] = (E)a[k];
    *reinterpret_cast<uint2*>((E*)p.dw + o * 4) = out.u;
  } else if (sum) {
    ((E*)p.db)[n] = (E)a[0];
  }
}

// Ranges of tokens: the fewest microseconds of rounds of workgroups (1.5 a step of 64 tokens, 6 to fill the pipeline and write a
// partial tile) and of the partial tiles' way through memory, and a range's rows inside 32-bit byte offsets.
static int wgrad_splits(int64_t M, int N, int C, int64_t ld) {
  const int64_t tiles = (int64_t)((N + 255) / 256) * ((C + 255) / 256), units = (M + 127) / 128;
  int best = 1;
  double least = 1e30;
  for (int64_t s = 1; s <= 64 && s <= units; s++) {
    const int64_t mine = (units + s - 1) / s;
    if (mine * 128 * ld * 2 >= 0x7f000000LL) continue;
    const double t = (double)((tiles * s + 255) / 256) * (3.0 * (double)mine + 6.0) + (double)s * N * C * 2e-6;
    if (t < least) { least = t; best = (int)s; }
  }
  return best;
}

}  // namespace lin
}  // namespace s3r

using namespace s3r;

extern "C" int64_t s3r_linear_wgrad_workspace(int64_t M, int N, int C, int64_t lddy, int64_t ldx) {
  if (M <= 0 || N <= 0 || C <= 0) return 0;
  return (int64_t)lin::wgrad_splits(M, N, C, lddy > ldx ? lddy : ldx) * N * (C + 1);
}

extern "C" int s3r_linear_wgrad(const void* dy, const void* x, void* dw, void* db, float* workspace, int64_t M, int N, int C, int64_t lddy,
                                int64_t ldx, int dtype, void* stream) {
  if (!dy || !x || !dw || !workspace) return fail(S3R_ERR_BAD_ARG, "s3r_linear_wgrad: null pointer");
  if (M <= 0 || N <= 0 || C <= 0) return fail(S3R_ERR_BAD_ARG, "s3r_linear_wgrad: non-positive size");
  if ((dtype != S3R_BF16 && dtype != S3R_F16) || N % 8 || C % 8 || N > (1 << 20) || C > (1 << 20) || (db && C <= 768))
    return fail(S3R_ERR_UNSUPPORTED, "s3r_linear_wgrad: dtype %d, %d outputs, %d inputs (built for 16-bit types, both in steps of 8; sums of dY with more than 768 inputs)", dtype, N, C);
  if (lddy < N || ldx < C || lddy >= (1 << 21) || ldx >= (1 << 21))
    return fail(S3R_ERR_BAD_ARG, "s3r_linear_wgrad: rows overlap or lie 2^21 elements or more apart");
  const int64_t ld = lddy > ldx ? lddy : ldx;
  if (M > 64 * (0x7f000000LL / (2 * ld) - 128)) return fail(S3R_ERR_UNSUPPORTED, "s3r_linear_wgrad: 64 ranges of %lld rows are not enough", (long long)M);
  if (!aligned16(dy) || !aligned16(x) || !aligned16(dw) || !aligned16(workspace) || lddy % 8 || ldx % 8)
    return fail(S3R_ERR_BAD_ARG, "s3r_linear_wgrad: pointers and rows must be multiples of 16 bytes");
  lin::WgradParams p = {dy, x, dw, db, workspace, M, lddy, ldx, N, C, (N + 255) / 256, (C + 255) / 256, 0, (M + 127) / 128};
  p.splits = lin::wgrad_splits(M, N, C, ld);
  const int64_t wgs = (int64_t)p.nt * p.ct * p.splits, outs = (int64_t)N * C / 4 + N;
  const int parts = outs >= 65536 ? 1 : 8;  // a thread per output fills the chip
  const int64_t sums = (outs * parts + 255) / 256;
  if (wgs > 0x7fffffffLL || sums > 0x7fffffffLL) return fail(S3R_ERR_UNSUPPORTED, "s3r_linear_wgrad: tensor too large for one launch");
  hipStream_t st = (hipStream_t)stream;
  if (dtype == S3R_BF16) hipLaunchKernelGGL((lin::wgrad_kernel<bf16_t>), dim3((unsigned)wgs), dim3(256), 0, st, p);
  else hipLaunchKernelGGL((lin::wgrad_kernel<f16_t>), dim3((unsigned)wgs), dim3(256), 0, st, p);
  const int rc = check_launch("wgrad_kernel");
  if (rc != S3R_OK) return rc;
#define S3R_SUM(PARTS) \
  if (dtype == S3R_BF16) hipLaunchKernelGGL((lin::wgrad_sum_kernel<bf16_t, PARTS>), dim3((unsigned)sums), dim3(256), 0, st, p); \
  else hipLaunchKernelGGL((lin::wgrad_sum_kernel<f16_t, PARTS>), dim3((unsigned)sums), dim3(256), 0, st, p)
  if (parts == 1) { S3R_SUM(1); } else { S3R_SUM(8); }
#undef S3R_SUM
  return check_launch("wgrad_sum_kernel");
}
