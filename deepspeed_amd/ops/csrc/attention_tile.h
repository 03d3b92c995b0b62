// What the attention kernels share: products of 32 x 32 x 16, their results as
// operands of the next product, and tiles of rows in LDS (attention.hip says why
// they are as they are).

#pragma once

#include <hip/hip_runtime.h>

#pragma clang diagnostic ignored "-Winline-asm"     // m0 among the clobbers

namespace attn {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16 mfma(s16x8 a, s16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
      __builtin_bit_cast(b16x8, a), __builtin_bit_cast(b16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ s16x4 tr_read(const short* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)p);
}

__device__ __forceinline__ int pack2(float a, float b) {
  return __builtin_bit_cast(
      int, __builtin_convertvector((f32x2{a, b}), b16x2));
}

// 16 bytes a lane to LDS, lane after lane from `lds` on; `arrive` waits for
// them. Not the builtin: behind that the compiler waits for all loads before it
// reads LDS, the next tile's among them.
__device__ __forceinline__ int lds_at(const void* p) {
  return (int)(uintptr_t)(__attribute__((address_space(3))) char*)p;
}
__device__ __forceinline__ void load_lds(const void* p, int lds) {
  asm volatile("s_mov_b32 m0, %1\n\t"
               "s_nop 0\n\t"
               "global_load_lds_dwordx4 %0, off"
               :: "v"(p), "s"(__builtin_amdgcn_readfirstlane(lds))
               : "memory", "m0");
}
// The same from a base for all lanes and an offset in bytes: half the registers.
template <int BYTES>
__device__ __forceinline__ void load_lds(const void* base, unsigned off,
                                         int lds) {
  static_assert(BYTES == 16 || BYTES == 4, "");
  const unsigned lo =
      __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)base);
  const unsigned hi =
      __builtin_amdgcn_readfirstlane((unsigned)((uintptr_t)base >> 32));
  const void* p = (const void*)(((uintptr_t)hi << 32) | lo);
  lds = __builtin_amdgcn_readfirstlane(lds);
  if (BYTES == 16)
    asm volatile("s_mov_b32 m0, %2\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %0, %1"
                 :: "v"(off), "s"(p), "s"(lds) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dword %0, %1"
                 :: "v"(off), "s"(p), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void arrive() {   // own loads, then everybody's
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Registers 8 s .. 8 s + 7 of a result as the next product's B operand.
__device__ __forceinline__ s16x8 operand(const f32x16& p, int s) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  const i32x4 v = {pack2(p[8 * s], p[8 * s + 1]),
                   pack2(p[8 * s + 2], p[8 * s + 3]),
                   pack2(p[8 * s + 4], p[8 * s + 5]),
                   pack2(p[8 * s + 6], p[8 * s + 7])};
  return __builtin_bit_cast(s16x8, v);
}

// Tile of rows of D bf16 in LDS. Within a row the swizzle is an exclusive or,
// so the addresses of one lane's reads differ by one from a first one.
template <int D>
struct Tile {
  static constexpr int CH = D / 8;                  // chunks of a row
  static constexpr int SC = D == 64 ? 8 : 16;       // places of a row
  static constexpr int RB = SC * 16;                // bytes of a row
  static __device__ __forceinline__ int turn(int row) {
    return D == 64 ? (row >> 1) & 7 : row & 15;
  }
  // A operand: rows row0 + col, contracted k = 16 kk + 8 half + j
  static __device__ __forceinline__ int rows_at(int lane) {
    const int col = lane & 31;
    return col * RB + (((lane >> 5) ^ turn(col)) << 4);
  }
  static __device__ __forceinline__ s16x8 rows(const short* t, int row0,
                                               int kk, int at) {
    return *(const s16x8*)((const char*)t + row0 * RB + (at ^ (kk * 32)));
  }
  // A operand of the transpose: rows are the coordinates 32 db + col,
  // contracted the tile's rows row0 + 8 (j >> 2) + 4 half + (j & 3), row0 a
  // multiple of 16
  static __device__ __forceinline__ int cols_at(int lane) {
    const int sub = lane & 15, r = 4 * (lane >> 5) + (sub >> 2);
    const int c = 2 * ((lane >> 4) & 1) + ((sub & 3) >> 1);
    return r * RB + ((c ^ turn(r)) << 4) + (sub & 1) * 8;
  }
  static __device__ __forceinline__ s16x8 cols(const short* t, int row0,
                                               int db, int at) {
    const char* p = (const char*)t + row0 * RB;
    const int lo = at ^ (db * 64), hi = lo ^ (RB / 2);   // row + 8
    const s16x4 a = tr_read((const short*)(p + lo));
    const s16x4 b = tr_read((const short*)(p + 8 * RB + hi));
    return s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  }
  // N rows of src (of which `left` are there: the last is repeated) straight
  // into LDS: the destination of a direct load is linear, so the swizzle goes
  // into the source. TPB threads; places past a row's chunks (D = 96) repeat.
  template <int N, int TPB>
  static __device__ __forceinline__ void fetch(const short* src, int stride,
                                               int left, short* t, int tid) {
#pragma unroll
    for (int i = 0; i < N * SC / TPB; ++i) {
      const int j = tid + i * TPB;
      const int row = j / SC;
      int c = (j % SC) ^ turn(row);
      if (CH < SC) c = min(c, CH - 1);
      const unsigned off = (unsigned)min(row, left - 1) * stride + c * 8;
      load_lds<16>(src, 2u * off, lds_at(t) + ((tid & ~63) + i * TPB) * 16);
    }
  }
};

}  // namespace attn
