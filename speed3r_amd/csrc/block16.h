// Pieces shared by the kernels for 16-token blocks that are built from 16 x 16 products: matrix instructions, the LDS map of a
// block, its direct transfers.
#pragma once
#include "select_common.h"

namespace s3r {
namespace b16x {
using sel::Frag;
using sel::as_v8;
using sel::Mma;
using sel::settle;

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kPair = 32 * 128;  // bytes of two 16-row blocks

template <typename E> __device__ __forceinline__ f32x4 mma16(typename Mma<E>::V8 a, typename Mma<E>::V8 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mma16<bf16_t>(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
template <> __device__ __forceinline__ f32x4 mma16<f16_t>(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// 16 x 16 x 16: four values of K per lane, rows 4 (lane / 16) .. + 3
template <typename E> struct Mma4;
template <> struct Mma4<bf16_t> {
  typedef bf16x4 V4;
  static __device__ __forceinline__ f32x4 mma(u32x2 a, V4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
  }
};
template <> struct Mma4<f16_t> {
  typedef f16x4 V4;
  static __device__ __forceinline__ f32x4 mma(u32x2 a, V4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), b, c, 0, 0, 0);
  }
};

template <typename E> __device__ __forceinline__ typename Mma4<E>::V4 pack4(const float (&x)[4]) {  // (pair by pair: packed conversions)
  typename Mma<E>::V2 lo, hi;
  lo[0] = (E)x[0];
  lo[1] = (E)x[1];
  hi[0] = (E)x[2];
  hi[1] = (E)x[3];
  const u32x2 w = {__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
  return __builtin_bit_cast(typename Mma4<E>::V4, w);
}

// LDS map of a 16-row block (rows of 128 bytes, 64 banks of 4 bytes: a row's parity picks the bank half): chunk c of row r
// sits at c ^ swz(r).  Row reads (ds_read_b128, lane = row lane % 16, chunk lane / 16) are served in groups of the lanes
// 0-3, 12-15, 20-27, of 4-11, 16-19, 28-31 and so on: rows 0-3 and 12-15 of one chunk with rows 4-11 of the next.
// Transposed reads take rows 0-7 or 8-15 and two neighbouring chunks together.  Row bit 1 -> chunk bit 1, bit 2 -> bit 2
// is free of conflicts for both (with bit 3 -> bit 0 on top every row read took eight cycles instead of four).
__device__ __forceinline__ constexpr int swz(int r) { return r & 6; }

template <typename E> __device__ __forceinline__ typename Mma<E>::V8 frag_of(u32x4 w) {
  Frag f;
  f.u = make_uint4(w[0], w[1], w[2], w[3]);
  return as_v8<E>(f);
}
template <typename E> __device__ __forceinline__ typename Mma<E>::V8 frag_of(u32x2 lo, u32x2 hi) {
  Frag f;
  f.u = make_uint4(lo[0], lo[1], hi[0], hi[1]);
  return as_v8<E>(f);
}
typedef __attribute__((address_space(3))) char* LdsPtr;
__device__ __forceinline__ uint32_t lds_addr(LdsPtr p) { return (uint32_t)(uintptr_t)p; }

// Direct transfers of 16-row blocks of one tensor.  WIDE: the tensor's last row lies 4 GiB or more behind its first one; the
// descriptor is then based at the block, otherwise at the tensor with the block's offset in the 32-bit scalar offset.
template <typename E, bool WIDE> struct Rows {
  const E* base;
  int64_t stride;           // elements
  uint32_t bytes;           // of a row stride
  uint32_t off0, off8;      // this lane's offset in the transfer of rows 0..7 and of rows 8..15
  int32_t ragged;           // the block that ends the tensor early (-2: none) ...
  int last;                 // ... and its last row
  __device__ __forceinline__ Rows(const void* p, int64_t at, int64_t row, int64_t len, int lane)
      : base((const E*)p + at), stride(row), bytes((uint32_t)row * (uint32_t)sizeof(E)) {
    const int r = lane >> 3;
    off0 = (uint32_t)r * bytes + (uint32_t)(((lane & 7) ^ swz(r)) * 16);
    off8 = (uint32_t)r * bytes + (uint32_t)(((lane & 7) ^ swz(r + 8)) * 16);
    ragged = (len & 15) ? (int32_t)(len >> 4) : -2;
    last = (int)(len & 15) - 1;
  }
  // the block's 2 KB -> dst.  rec: -1, or 0 for a descriptor without records: nothing is fetched.  TAIL: the block may be the
  // one that ends early, rows beyond the end re-read the last one
  template <bool TAIL> __device__ __forceinline__ void fetch(int32_t blk, int32_t rec, LdsPtr dst, int lane) const {
    const E* from = WIDE ? base + (int64_t)blk * 16 * stride : base;
    const uint32_t so = WIDE ? 0u : (uint32_t)blk * 16u * bytes;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)from, 0, rec, 0x00020000);
    if constexpr (TAIL) {
      const int end = blk == ragged ? last : 15, r = lane >> 3;
      const uint32_t o0 = (uint32_t)(r < end ? r : end) * bytes + (uint32_t)(((lane & 7) ^ swz(r)) * 16);
      const uint32_t o8 = (uint32_t)(r + 8 < end ? r + 8 : end) * bytes + (uint32_t)(((lane & 7) ^ swz(r + 8)) * 16);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, o0, so, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst + 1024, 16, o8, so, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, off0, so, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst + 1024, 16, off8, so + 8u * bytes, 0, 0);
    }
  }
};
// scalar instructions by hand: the compiler's own select of 0 and -1 lands in a vector register, and the descriptor with it.
// rec = -1 (no limit) for a block, 0 for none; some = the block, or 0
__device__ __forceinline__ void records(int32_t a, int32_t& rec, int32_t& some) {
  asm("s_ashr_i32 %0, %2, 31\n\ts_not_b32 %0, %0\n\ts_and_b32 %1, %2, %0" : "=&s"(rec), "=&s"(some) : "s"(a) : "scc");
}
// XCD-aware work item of a workgroup: each XCD walks a contiguous range of blocks of one head
__device__ __forceinline__ int work_item(int w, int total) {
  const int xcd = w & 7, slot = w >> 3;
  const int per = total >> 3, rem = total & 7;
  return xcd * per + (xcd < rem ? xcd : rem) + slot;
}

// The distinct blocks of NQ lists (mine[j]: entry `lane` of list j; entries < 0 or at or beyond `len` rows are dropped), each with
// a count byte per list (how often list j names it), compacted into walk[0 .. n) with `ends` end marks behind them.  From a
// hash table of 512 slots in `table` (4 KB of LDS that no transfer touches before this returns): every lane inserts its
// entry of list j with a compare-and-swap on the key (linear probing, at most 256 distinct blocks) and adds 1 << 8j to the
// slot's count; the occupied slots are compacted eight per lane, positions from ballots.  One wave.  Returns n.
template <int NQ>
__device__ __forceinline__ int walk_list(const int32_t (&mine)[NQ], int64_t len, unsigned char* table, int2* walk, int ends, int lane, bool& dup) {
  int n = 0;
  int32_t* const hkey = reinterpret_cast<int32_t*>(table);
  uint32_t* const hcnt = reinterpret_cast<uint32_t*>(table + 2048);
  reinterpret_cast<int4*>(hkey)[lane] = reinterpret_cast<int4*>(hkey)[lane + 64] = make_int4(-1, -1, -1, -1);
  reinterpret_cast<int4*>(hcnt)[lane] = reinterpret_cast<int4*>(hcnt)[lane + 64] = make_int4(0, 0, 0, 0);
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    const int32_t e = mine[j];
    bool active = e >= 0 && (int64_t)e * 16 < len;
    uint32_t slot = ((uint32_t)e * 0x9E3779B1u) >> 23;
    while (active) {
      const int32_t old = atomicCAS(hkey + slot, -1, e);
      if (old == -1 || old == e) {
        atomicAdd(hcnt + slot, 1u << (8 * j));
        active = false;
      } else {
        slot = (slot + 1) & 511u;
      }
    }
  }
  const int4 k0 = reinterpret_cast<const int4*>(hkey)[2 * lane], k1 = reinterpret_cast<const int4*>(hkey)[2 * lane + 1];
  const int4 c0 = reinterpret_cast<const int4*>(hcnt)[2 * lane], c1 = reinterpret_cast<const int4*>(hcnt)[2 * lane + 1];
  const int32_t ks8[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
  const int32_t cs8[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  uint32_t pos = 0, bits = 0;  // occupied slots of the lanes below; all count bits
#pragma unroll
  for (int s8 = 0; s8 < 8; s8++) {
    const uint64_t m = __ballot(ks8[s8] >= 0);
    pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, pos));
    n += __popcll(m);
    bits |= (uint32_t)cs8[s8];
  }
#pragma unroll
  for (int s8 = 0; s8 < 8; s8++)
    if (ks8[s8] >= 0) walk[pos++] = make_int2(ks8[s8], cs8[s8]);
  if (lane < ends) walk[n + lane] = make_int2(-1, 0);  // what the last steps look ahead at
  dup = __any((bits & 0xfefefefeu) != 0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the table is read and the list written before the first transfer
  asm volatile("" ::: "memory");
  return n;
}

}  // namespace b16x
}  // namespace s3r
