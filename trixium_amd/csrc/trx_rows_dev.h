// Decoding of stored ternary rows for the matrix cores: a lane turns the codes of one row's half group
// (64 columns) into eight dwords of nibbles, through a table in LDS. Shared by the float GEMM
// (trx_gemm.hip) and the exact engine matvec (trx_gemv_rows.hip).
#pragma once

#include "trx_internal.h"

namespace trx {

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));

// Code byte -> its weights as nibbles: a trit5 byte's five (digit 0 first), a 2-bit byte's four (twice).
// FP4: E2M1, where 0 is 0, 1 is 2, 2 is 4 and the sign is bit 3; otherwise the codes themselves. Every
// entry is stored once per LDS bank, so the 64 lanes' random bytes never conflict (one copy: 3.3
// times the cycles).
constexpr int kLut = 256 * 32;
template <int KIND, bool FP4, int THREADS>
__device__ __forceinline__ void fill_lut(uint32_t* lut) {
  constexpr int PER = THREADS / 256;                  // threads per entry
  auto nib = [](int c) { return !FP4 ? (uint32_t)c : c == 0 ? 0xAu : c == 1 ? 0u : c == 2 ? 2u : 4u; };
  const int b = threadIdx.x / PER, part = threadIdx.x % PER;
  uint32_t v = 0;
  if (KIND == TRX_KIND_TERNARY5) {
    int r = b;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      v |= nib(r % 3) << (4 * k);
      r /= 3;
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) v |= nib((b >> (2 * k)) & 3) << (4 * k);
    v |= v << 16;
  }
  uint4* d = (uint4*)(lut + 32 * b) + part * (8 / PER);
#pragma unroll
  for (int i = 0; i < 8 / PER; ++i) d[i] = make_uint4(v, v, v, v);
}

// The codes of one row's half group: 16 bytes from a dword boundary, and the group's scale.
struct Codes {
  i32x4_t c;
  uint32_t sc;
};

template <int KIND>
struct RowReader {
  __amdgpu_buffer_rsrc_t rw;
  uint32_t rbase, code_off;
  int h;
  bool valid;
  template <class P>
  __device__ __forceinline__ void init(const P& p, int r, int half) {
    valid = r < p.M;
    rw = make_rsrc(p.W, p.w_bytes);
    rbase = (uint32_t)(valid ? r : 0) * (uint32_t)p.row_bytes;
    code_off = (uint32_t)p.code_off;
    h = half;
  }
  __device__ __forceinline__ uint32_t offset(int g) const {
    return code_off + (KIND == TRX_KIND_TERNARY5 ? 26u * (uint32_t)g + 13u * (uint32_t)h
                                                 : 32u * (uint32_t)g + 16u * (uint32_t)h);
  }
  __device__ __forceinline__ void load(Codes& r, int g) const {
    r.c = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, rbase + (offset(g) & ~3u), 0, 0));
    r.sc = __builtin_amdgcn_raw_buffer_load_b16(rw, rbase + 2u * (uint32_t)g, 0, 0);
  }
  // load() of a group that is the same for the wave: its product stays scalar (as one multiply-add with
  // the row's offset it keeps a 64-bit register pair).
  __device__ __forceinline__ void load_uniform(Codes& r, int g) const {
    uint32_t at = (KIND == TRX_KIND_TERNARY5 ? 26u : 32u) * (uint32_t)g;
    asm("" : "+s"(at));
    r.c = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, rbase + ((offset(0) + at) & ~3u), 0, 0));
    r.sc = __builtin_amdgcn_raw_buffer_load_b16(rw, rbase + 2u * (uint32_t)g, 0, 0);
  }
  // The 64 weights of the half group as nibbles, in the columns' order (trit5: half 1 takes columns 65 ..
  // 127 and then 64, whose code shares a byte with half 0's), in parts that a caller can
  // spread over its other work: begin, look<0 .. 5> (the table reads of byte runs); low() and
  // high() give the first and the second 32.
  struct Half {
    uint32_t d[4], p[KIND == TRX_KIND_TERNARY5 ? 13 : 16];
  };
  __device__ __forceinline__ void begin(const Codes& r, int g, Half& v) const {
    if (KIND == TRX_KIND_TERNARY5) {
      const uint32_t sh = offset(g) & 3u;
      v.d[0] = __builtin_amdgcn_alignbyte(r.c[1], r.c[0], sh);
      v.d[1] = __builtin_amdgcn_alignbyte(r.c[2], r.c[1], sh);
      v.d[2] = __builtin_amdgcn_alignbyte(r.c[3], r.c[2], sh);
      v.d[3] = __builtin_amdgcn_alignbyte(0, r.c[3], sh);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v.d[i] = (uint32_t)r.c[i];
    }
  }
  template <int PART>
  __device__ __forceinline__ void look(Half& v, const uint32_t* t) const {
    constexpr int lo5[7] = {0, 2, 4, 6, 7, 10, 13}, lo2[7] = {0, 2, 4, 6, 8, 12, 16};
    constexpr int a = KIND == TRX_KIND_TERNARY5 ? lo5[PART] : lo2[PART];
    constexpr int b = KIND == TRX_KIND_TERNARY5 ? lo5[PART + 1] : lo2[PART + 1];
#pragma unroll
    for (int i = a; i < b; ++i) v.p[i] = t[((v.d[i >> 2] >> (8 * (i & 3))) & 0xFFu) * 32u];
  }
  __device__ __forceinline__ i32x4_t low(const Half& v) const {
    const uint32_t* p = v.p;
    if (KIND == TRX_KIND_TERNARY5)
      return i32x4_t{(int)(p[0] | p[1] << 20), (int)(p[1] >> 12 | p[2] << 8 | p[3] << 28), (int)(p[3] >> 4 | p[4] << 16),
                     (int)(p[4] >> 16 | p[5] << 4 | p[6] << 24)};
    return i32x4_t{(int)two(p[0], p[1]), (int)two(p[2], p[3]), (int)two(p[4], p[5]), (int)two(p[6], p[7])};
  }
  __device__ __forceinline__ i32x4_t high(const Half& v) const {
    const uint32_t* p = v.p;
    if (KIND == TRX_KIND_TERNARY5) {
      // Half 0's last byte ends with column 64, which half 1 takes after its own 63.
      const auto sw = __builtin_amdgcn_permlane32_swap(p[12], p[12], false, false);
      const uint32_t end = p[11] >> 4 | p[12] << 16;
      return i32x4_t{(int)(p[6] >> 8 | p[7] << 12), (int)(p[8] | p[9] << 20), (int)(p[9] >> 12 | p[10] << 8 | p[11] << 28),
                     (int)(h ? (end & 0x0FFFFFFFu) | (sw[0] >> 16) << 28 : end)};
    }
    return i32x4_t{(int)two(p[8], p[9]), (int)two(p[10], p[11]), (int)two(p[12], p[13]), (int)two(p[14], p[15])};
  }
  // Two 2-bit bytes' nibbles in one dword (a table entry holds its four nibbles twice).
  __device__ __forceinline__ static uint32_t two(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
  __device__ __forceinline__ void decode(const Codes& r, int g, const uint32_t* lut, uint32_t (&D)[8]) const {
    const uint32_t* t = lut + (threadIdx.x & 31);
    Half v;
    begin(r, g, v);
    look<0>(v, t);
    look<1>(v, t);
    look<2>(v, t);
    look<3>(v, t);
    look<4>(v, t);
    look<5>(v, t);
    const i32x4_t a = low(v), b = high(v);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      D[i] = (uint32_t)a[i];
      D[4 + i] = (uint32_t)b[i];
    }
  }
};

}  // namespace trx
