// The ternary GEMM of several positions on the matrix cores: y[r] = W xhat_r.
//
// x enters as five planes of digits in fp6 (E2M3), W's trits as fp4 (E2M1), so that the products run on
// v_mfma_scale_f32_32x32x64_f8f6f4 at its fp6/fp4 rate, four times fp16's:
//   x = 2^u (d0 + d1/2^5 + d2/2^10 + d3/2^15 + d4/2^21), every digit a whole number of the format's eighths
// with one exponent u per position and 32 columns (the largest |x| in [16, 32) * 2^u). E2M3 holds
// whole eighths up to 2, every second one up to 4 and every fourth up to 7.5, and E2M1 holds -1, 0, 1 (and 2,
// the 2-bit code 3); the plane's power of two is the instruction's block scale, and its fp32 accumulation of
// such products is exact while a sum fits 24 bits. A value of the block's highest octave leaves up to four
// units of the next digit, any other two. So the last digit, a bit further down, holds the others to 2^(u - 21)
// (2^-25 of the block's leading power) and the highest octave's, whose last digit ends at 7.5 where 8 is due,
// to 2^(u - 19) (2^-23 of its own). Over normed, SwiGLU and attention inputs that is a smaller error than a
// pair of fp16 values has (root mean square 2.2e-8 against 4.5e-8 for normal x; the last digit at 2^20 and the
// largest |x| in [8, 16) * 2^u: 6.6e-8). A group's sum is then multiplied by the group's fp16 scale and added in fp32.
// Measured on all CUs (operands in registers, random data): 6.1 PFLOP/s for fp6 x fp4, 3.4 for
// int8, 1.57 for fp16; with the planes that each needs for x to about 24 bits (5, 3, 2) that is 1.23,
// 1.14 and 0.79 PFLOP/s, and the int8 planes' sums would need five vector operations per element
// and group where these need one.

#include "trx_internal.h"
#include "trx_prefill.h"
#include "trx_rows_dev.h"

#include <utility>

namespace trx {

typedef int i32x12_t __attribute__((ext_vector_type(12)));
typedef unsigned int u32x6_t __attribute__((ext_vector_type(6)));
typedef float f32x32_t __attribute__((ext_vector_type(32)));

// Digit planes ----------------------------------------------------------------------------------
//
// The matrix instruction's operand order: a step takes 64 columns of a 128-column group, lane half
// h of it 32 of them, position 32 pt + j in lane j. Half h holds the group's columns 64 h .. 64 h +
// 63, step s its 32 from 32 s on (trit5: half 1 takes columns 65 .. 127 and then 64, whose code
// shares a byte with half 0's). A position tile's step is 256 P bytes for its P <= 32 positions:
// eight runs [h][j] of 16-byte pieces that hold a lane's 32 dwords in order, six of each plane (the
// lowest digit's first), then the block's scales and the fp32 sum of the 32 columns' x^2. Four bytes a
// column in all, read by 16-byte loads only (per byte, the vector cache is a quarter slower on 8- and
// 12-byte ones).
constexpr int kPlanes = 5;
constexpr int kUMin = -85;             // smallest u: below it values lose bits under 2^-106
// The block scales hold the planes 2^16 down and the weights' scales 2^16 up, so that no group's sum
// of finite values overflows.
constexpr int kScaleByte = 109 - 16;
// Plane c's power of two above plane 0's.
constexpr uint32_t plane_up(int c) { return c ? 5 * c + 1 : 0; }
constexpr float kScaleUp = 65536.f;
// Wide blocks. Five digits hold what lies far below a block's largest value to few bits of its own, which
// shows where a row's weights on the larger values are 0 (a model's massive channels). A block is wide, and its
// values take part one by one (Wide), if some lie seven octaves or more below the largest and behind at least
// four empty octaves, the empty ones times these values 28 or more (four octaves and seven values, seven and
// four, fourteen and two), or if twelve, an octave counted for two at most, lie ten octaves or more below.
// Values 128 times their neighbours do that; of the blocks of normal, product and SwiGLU inputs, also with
// channels 20 times larger, fewer than 1e-6 do (their smallest values lie apart by chance).
// A wide block holds its values in 30 bits each, the sign, 6 bits of exponent and all of the fraction: value e in
// the low bits of dword e, the last two in the 30 dwords' high pairs of bits. Exponents 32 to 62 count from the
// largest value's (62) down, 1 to 31 from the largest of those below (31); 0 is 0 or less than 2^-31 of that. In
// place of the scales stand a bit that marks the block, the octaves down to the others, the two largest values'
// exponents and scale 0 (the digits' part of the products, of these bits, drowns: below 2^-58 of the
// largest value). Blocks below 2^-40 stay as they are: their digits leave out 2^-65.
constexpr int kWideTop = 127 - 40;

// A lane packs one position's 32 columns with the hardware's fp6 conversions (digit by digit in floats it
// would take ~35 vector operations a column). Bound by memory on long prompts: 2048 x 12288 in 40 us,
// 5 TB/s.
template <bool VEC>
__global__ __launch_bounds__(256) void planes_kernel(PlanesParams p) {
  const int lane = threadIdx.x & 63, h = lane >> 5, j = lane & 31;
  const int st = blockIdx.x * 4 + (threadIdx.x >> 6), pt = blockIdx.y;
  const int P = min(32, p.R - 32 * pt);
  if (st >= p.K / 64 || j >= P) return;
  const int s = st & 1, c0 = 64 * (st & ~1) + 64 * h + 32 * s;
  const float* xr = p.x + (size_t)(32 * pt + j) * p.ldx + c0;
  const float* gr = p.norm_w ? p.norm_w + c0 : nullptr;
  float v[33];
  if (VEC) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float4 a = ((const float4*)xr)[i];
      v[4 * i] = a.x;
      v[4 * i + 1] = a.y;
      v[4 * i + 2] = a.z;
      v[4 * i + 3] = a.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i] = xr[i];
  }
  const bool turned = p.turned && h;
  const int ce = turned ? (s ? -32 : 32) : 0;          // the column that ends a turned block
  v[32] = xr[ce];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 32; ++i) ss += v[i] * v[i];
  if (gr) {
    if (VEC) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float4 a = ((const float4*)gr)[i];
        v[4 * i] *= a.x;
        v[4 * i + 1] *= a.y;
        v[4 * i + 2] *= a.z;
        v[4 * i + 3] *= a.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 32; ++i) v[i] *= gr[i];
    }
    v[32] *= gr[ce];
  }
  // The block's values, even ones in a, odd ones in b (the conversion interleaves its two sources).
  f32x16_t a, b;
  uint32_t top = 0;                                   // the largest magnitude's bits
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    a[i] = turned ? v[2 * i + 1] : v[2 * i];
    b[i] = turned ? v[2 * i + 2] : v[2 * i + 1];
    top = max(top, max(__float_as_uint(a[i]) & 0x7FFFFFFFu, __float_as_uint(b[i]) & 0x7FFFFFFFu));
  }
  const bool finite = top < 0x7F800000u;
  // The octaves, from the largest value's (bit 0) down, that hold a value and those that hold more; the last
  // bit stands for all from there on, and 0.
  const int et = (int)(top >> 23);
  uint32_t seen = 0, more = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int E = (int)(__float_as_uint(i & 1 ? b[i >> 1] : a[i >> 1]) >> 23 & 0xFFu);
    const uint32_t bit = 1u << (max(E, et - 31) & 31);
    more |= seen & bit;
    seen |= bit;
  }
  auto from_top = [&](uint32_t v) { return __builtin_bitreverse32(__builtin_amdgcn_alignbit(v, v, et + 1)); };
  seen = from_top(seen);
  more = from_top(more);
  int n = 0;                                          // the last's values without the zeros
  if ((int)seen < 0) {
    asm volatile("" : "+v"(a), "+v"(b));              // or the 32 exponents stay in registers from above
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int E = (int)(__float_as_uint(i & 1 ? b[i >> 1] : a[i >> 1]) >> 23 & 0xFFu);
      n += E > 0 && E <= et - 31;
    }
    seen = (seen & 0x7FFFFFFFu) | (n > 0 ? 0x80000000u : 0u);
  }
  auto count = [&](uint32_t mask) { return __popc(seen & mask & 0x7FFFFFFFu) + __popc(more & mask & 0x7FFFFFFFu) + n; };
  const uint32_t z = ~seen & ~seen >> 1 & ~seen >> 2 & ~seen >> 3 & 0x0FFFFFFFu;    // four empty ones from here
  const int from = z ? __builtin_ctz(z) : 0;
  const uint32_t low = z ? ~0u << (from + 3) << 1 : 0u;
  const int first = __builtin_ctz((seen & low) | 0x80000000u), gap = first - from;
  int others = low ? count(low) : 0;
  if (first >= 7 && others > 1 && others * gap < 28) {               // how many they are
    asm volatile("" : "+v"(a), "+v"(b));
    others = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int E = (int)(__float_as_uint(i & 1 ? b[i >> 1] : a[i >> 1]) >> 23 & 0xFFu);
      others += E > 0 && E <= et - first;
    }
  }
  const bool apart = first >= 7 && others * gap >= 28;
  const bool wide = finite && et >= kWideTop && (apart || count(~0u << 10) >= 12);
  uint8_t* out = p.xp + (size_t)32 * pt * p.K * 4 + (size_t)st * 256 * P;
  uint4* o = (uint4*)out + h * P + j;
  uint32_t dw[32];
  if (!wide) {
    const int u = max(et - 131, kUMin);               // 2^(E - 127 - 4) from an exponent field E
#pragma unroll
    for (int d = 0; d < kPlanes; ++d) {
      const int c = kPlanes - 1 - d;
      const float sc = __uint_as_float((uint32_t)(u + 3 - 21 + (int)plane_up(c) + 127) << 23);
      const u32x6_t q = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(a, b, sc);
      // The sources stay live past the conversion: it reads them while it writes its result, and the
      // compiler may otherwise give both the same registers.
      asm volatile("" ::"v"(a), "v"(b));
      if (d + 1 < kPlanes) {
        const f32x32_t back = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(q, sc);
        asm volatile("" ::"v"(q));
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          a[i] -= back[2 * i];
          b[i] -= back[2 * i + 1];
        }
      }
#pragma unroll
      for (int i = 0; i < 6; ++i) dw[6 * c + i] = q[i];
    }
    // Byte 0: the block scale of the lowest plane (plane c's is plane_up(c) above); 0xFF, the format's NaN, where
    // a value is not finite.
    dw[30] = finite ? (uint32_t)(u + kScaleByte) : 0xFFu;
  } else {
    uint32_t next = 0;                                // the largest 31 octaves down or more
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const uint32_t m = __float_as_uint(i & 1 ? b[i >> 1] : a[i >> 1]) & 0x7FFFFFFFu;
      next = max(next, (int)(m >> 23) <= et - 31 ? m : 0u);
    }
    const uint32_t eb = next >> 23;
    auto code = [&](float x) {
      const uint32_t v = __float_as_uint(x), m = v & 0x7FFFFFFFu, E = m >> 23;
      const uint32_t at = (int)E > et - 31 ? E + 62 - (uint32_t)et : E && E + 31 > eb ? E + 31 - eb : 0u;
      return (at ? at << 23 | (m & 0x7FFFFFu) : 0u) | (v >> 31) << 29;
    };
    const uint32_t c30 = code(a[15]), c31 = code(b[15]);
#pragma unroll
    for (int i = 0; i < 30; ++i)
      dw[i] = code(i & 1 ? b[i >> 1] : a[i >> 1]) | (i < 15 ? c30 >> (2 * i) : c31 >> (2 * (i - 15))) << 30;
    dw[30] = 0x80000000u | (apart ? (uint32_t)first : 31u) << 24 | eb << 16 | (uint32_t)et << 8;
  }
  dw[31] = __float_as_uint(ss);
#pragma unroll
  for (int i = 0; i < 8; ++i) o[2 * P * i] = make_uint4(dw[4 * i], dw[4 * i + 1], dw[4 * i + 2], dw[4 * i + 3]);
}

int launch_planes(const PlanesParams& p, hipStream_t s) {
  TRX_CHECK(p.R >= 1 && p.K >= kGroup && p.K % kGroup == 0 && p.ldx >= p.K, TRX_E_INVALID,
            "prefill input: R=%d K=%d", p.R, p.K);
  const bool vec = p.ldx % 4 == 0 && ((uintptr_t)p.x & 15) == 0 && ((uintptr_t)p.norm_w & 15) == 0;
  const dim3 grid(cdiv(p.K / 64, 4), cdiv(p.R, 32));
  if (vec) hipLaunchKernelGGL(planes_kernel<true>, grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL(planes_kernel<false>, grid, dim3(256), 0, s, p);
  TRX_LAUNCHED();
  return TRX_OK;
}

// Weights ---------------------------------------------------------------------------------------

// A group's scale, 0 for a row past the end.
template <int KIND>
__device__ __forceinline__ float row_scale(const RowReader<KIND>& row, const Codes& r) {
  const float v = (float)__builtin_bit_cast(_Float16, (uint16_t)r.sc);
  return row.valid ? v * kScaleUp : 0.f;
}

// A step's digit planes of one position tile in registers: planes 0 and 1, 2 and 3, and 4 with the
// block scales (dword 6) and the sum of squares (dword 7).
struct Planes {
  i32x12_t c01, c23;
  i32x8_t c4;
  template <int C>
  __device__ __forceinline__ i32x8_t get() const {
    if constexpr (C == 0) return __builtin_shufflevector(c01, c01, 0, 1, 2, 3, 4, 5, -1, -1);
    else if constexpr (C == 1) return __builtin_shufflevector(c01, c01, 6, 7, 8, 9, 10, 11, -1, -1);
    else if constexpr (C == 2) return __builtin_shufflevector(c23, c23, 0, 1, 2, 3, 4, 5, -1, -1);
    else if constexpr (C == 3) return __builtin_shufflevector(c23, c23, 6, 7, 8, 9, 10, 11, -1, -1);
    else return c4;
  }
  __device__ __forceinline__ uint32_t scales() const { return (uint32_t)c4[6]; }
  __device__ __forceinline__ float ss() const { return __int_as_float(c4[7]); }
};

struct PlaneReader {
  __amdgpu_buffer_rsrc_t r;
  uint32_t v;                          // this lane's offset in a run of pieces
  uint32_t P;
  int st0;
  // Steps st0 .. st1 - 1: below 4 GiB of them (the offsets' range).
  __device__ __forceinline__ void init(const GemmParams& p, int pt, int lane, int st0_, int st1) {
    P = (uint32_t)min(32, p.R - 32 * pt);
    st0 = st0_;
    const uint32_t j = min((uint32_t)(lane & 31), P - 1), h = (uint32_t)(lane >> 5);
    r = make_rsrc(p.xp + ((size_t)32 * pt * p.K * 4 + (size_t)256 * P * st0), 256u * P * (uint32_t)(st1 - st0));
    v = 16u * (h * P + j);
  }
  __device__ __forceinline__ uint32_t base(int st) const { return 256u * P * (uint32_t)(st - st0); }
  __device__ __forceinline__ i32x4_t piece(uint32_t base, uint32_t q) const {
    return __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, v, base + 32u * P * q, 0));
  }
  __device__ __forceinline__ i32x12_t pair(uint32_t base, uint32_t q) const {
    const i32x4_t a = piece(base, q), b = piece(base, q + 1), c = piece(base, q + 2);
    return i32x12_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3], c[0], c[1], c[2], c[3]};
  }
  __device__ __forceinline__ i32x8_t last(uint32_t base) const {
    const i32x4_t a = piece(base, 6), b = piece(base, 7);
    return i32x8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  }
  __device__ __forceinline__ Planes load(int st) const {
    const uint32_t b = base(st);
    Planes q;
    q.c01 = pair(b, 0);
    q.c23 = pair(b, 3);
    q.c4 = last(b);
    return q;
  }
};

// acc += plane C of the step's positions times one tile of weights.
template <int C>
__device__ __forceinline__ f32x16_t mx(const Planes& q, const i32x4_t& w, const f32x16_t& acc) {
  const i32x8_t B = {w[0], w[1], w[2], w[3], 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(q.get<C>(), B, acc, 2, 4, 0, (int)(q.scales() + plane_up(C)), 0,
                                                          0x7F7F7F7F);
}

// One plane times NB tiles of weights (independent accumulators), from zero where FIRST.
template <int C, bool FIRST, int NB>
__device__ __forceinline__ void mx_plane(const Planes& q, const i32x4_t (&w)[NB], f32x16_t (&t)[NB]) {
  const f32x16_t zero = {};
#pragma unroll
  for (int b = 0; b < NB; ++b) t[b] = mx<C>(q, w[b], FIRST ? zero : t[b]);
}
// Keeps the products before it and the loads after it in place: the compiler otherwise moves every
// load of a loop to its end, where its latency is waited out.
template <int NB>
__device__ __forceinline__ void pin(f32x16_t (&t)[NB]) {
#pragma unroll
  for (int i = 0; i < NB; ++i) asm volatile("" : "+v"(t[i]) : : "memory");
}
template <bool FIRST, int NB>
__device__ __forceinline__ void mx_step(const Planes& q, const i32x4_t (&w)[NB], f32x16_t (&t)[NB]) {
  mx_plane<0, FIRST, NB>(q, w, t);
  mx_plane<1, false, NB>(q, w, t);
  mx_plane<2, false, NB>(q, w, t);
  mx_plane<3, false, NB>(q, w, t);
  mx_plane<4, false, NB>(q, w, t);
}

// Weight row of lane j of 32-row tile `tile`: rows in order, or for SwiGLU gate rows f (even tiles)
// and the matching up rows F + f (odd tiles), f = 32 (tile / 2) + j. M for a row past the end.
template <int EPI>
__device__ __forceinline__ int tile_row(int tile, int j, int M) {
  if (EPI == GM_SWIGLU) {
    const int F = M / 2, f = 32 * (tile >> 1) + j;
    return f < F ? ((tile & 1) ? F + f : f) : M;
  }
  return min(32 * tile + j, M);
}

// A step's wide blocks, digit by digit, from the highest on until less is left than 2^-25 of the others' leading
// power (where they lie 31 octaves down or are no cluster of their own: nothing); a lane without one gives zeros.
struct Wide {
  f32x16_t a, b;
  int e, stop;                         // exponent fields: the next digit's unit, the least that takes one
  __device__ __forceinline__ void init(const Planes& q) {
    const uint32_t s = q.scales();
    const bool on = (int)s < 0;
    const uint32_t et = on ? s >> 8 & 0xFFu : 127u, eb = on ? s >> 16 & 0xFFu : 0u;
    uint32_t dw[30], c30 = 0, c31 = 0;
#pragma unroll
    for (int i = 0; i < 30; ++i) dw[i] = on ? (uint32_t)(i < 12 ? q.c01[i % 12] : i < 24 ? q.c23[i % 12] : q.c4[i % 6]) : 0u;
#pragma unroll
    for (int i = 0; i < 15; ++i) {
      c30 |= dw[i] >> 30 << (2 * i);
      c31 |= dw[15 + i] >> 30 << (2 * i);
    }
    auto value = [&](uint32_t c) {
      const uint32_t m = c & 0x1FFFFFFFu, from = m >= 32u << 23 ? et - 62u : eb - 31u;
      return __uint_as_float((m ? m + (from << 23) : 0u) | (c & 0x20000000u) << 2);
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      a[i] = value(i < 15 ? dw[2 * i] : c30);
      b[i] = value(i < 15 ? dw[2 * i + 1] : c31);
    }
    e = (int)et - 1;
    stop = max(on && (s >> 24 & 31u) < 31u ? (int)et - (int)(s >> 24 & 31u) - 25 : 0, 20);
  }
  // The next digit and its block scale; whether any lane has more.
  __device__ __forceinline__ bool next(u32x6_t& c, int& scale) {
    const float sc = __uint_as_float((uint32_t)e << 23);
    scale = e - 16;
    c = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(a, b, sc);
    asm volatile("" ::"v"(a), "v"(b));                // see planes_kernel
    const f32x32_t back = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(c, sc);
    asm volatile("" ::"v"(c));
    float left = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      a[i] -= back[2 * i];
      b[i] -= back[2 * i + 1];
      left = fmaxf(fmaxf(left, fabsf(a[i])), fabsf(b[i]));
    }
    // Down to the largest that is left, past empty octaves; below 2^-107 nothing is.
    const int el = (int)(__float_as_uint(left) >> 23);
    const bool more = el >= stop;
    e = more ? min(e - 5, el - 1) : 17;
    return __any(more);
  }
};
__device__ __forceinline__ f32x16_t mx_digits(const u32x6_t& c, int scale, const i32x4_t& w, const f32x16_t& acc) {
  const i32x8_t A = {(int)c[0], (int)c[1], (int)c[2], (int)c[3], (int)c[4], (int)c[5], 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, i32x8_t{w[0], w[1], w[2], w[3], 0, 0, 0, 0}, acc, 2, 4, 0, scale,
                                                         0, 0x7F7F7F7F);
}

// Block b of nx weight tiles x ny position tiles. Blocks go to the 8 XCDs in turn; each XCD takes
// one run of an order that walks panels of 8 weight tiles position by position, so that the blocks
// which share an L2 at a time share their weights and their positions.
__device__ __forceinline__ void tile_of_block(int b, int nx, int ny, int& x, int& y) {
  const int total = nx * ny, q = total / 8, rem = total % 8, xcd = b % 8, k = b / 8;
  const int L = xcd < rem ? xcd * (q + 1) + k : rem * (q + 1) + (xcd - rem) * q + k;
  const int full = nx / 8 * 8;
  if (L < full * ny) {
    const int panel = L / (8 * ny), r = L - panel * 8 * ny;
    x = 8 * panel + r % 8;
    y = r / 8;
  } else {
    const int w = nx - full, r = L - full * ny;
    x = full + r % w;
    y = r / w;
  }
}

constexpr int kGmThreads = 512;

// f with 0, 1, .. as compile-time constants.
template <class F, int... I>
__device__ __forceinline__ void in_turn(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}

// Large products: a block takes 128 positions x 256 weight rows, four waves of one position tile
// each, one wave a SIMD, so that a wave has 512 registers: eight accumulator tiles, the sums of two pairs
// of tiles and two groups of its positions' planes, which it loads straight into registers a group
// ahead of their use (the operand order makes each load contiguous). Each wave decodes two of the block's
// weight tiles per group into LDS for all, two buffers, one barrier a group.
// A wave alone issues a vector operation every 6 cycles beside the matrix unit's 32-cycle products,
// so all other work (the last pair's sums into the accumulators, the next group's decode, the loads)
// is laid out between the products: slots of two products and about ten operations, ten a pair of tiles.
// What vector operations touch (sums, accumulators) fills the 256 registers that they reach; planes and
// weights lie in the others, which only products and loads reach.
// Eight waves of four tiles each, at two waves a SIMD, read every plane twice as often and had no room for a
// group ahead. 2048 positions, planes included: 24576 x 4096 with SwiGLU 503 us (520), 4096 x 12288 with the
// residual 300 (333); 1024 of 34816 x 5120 491 (521). Per group and round 2.1 to 2.5 us, against 1.75 for the
// products alone at the power-limited clock (a last digit of one bit more draws more power: 489 -> 500 us and
// 471 -> 480, measured in turn with the digits as they were).
template <int KIND, int EPI>
__global__ __launch_bounds__(256, 1) void gemm_kernel(GemmParams p) {
  constexpr int NT = 8, ND = NT / 4, NP = NT / 2;     // weight tiles, of them a wave decodes, pairs
  static_assert(NP % 2 == 0, "the pairs take turns with two sets of registers");
  __shared__ __align__(16) uint32_t lut[kLut];
  __shared__ __align__(16) i32x4_t bs[2][NT][2][64];
  __shared__ float wsc[2][32 * NT];
  __shared__ float rsx[128];
  __shared__ unsigned long long wide_of[4];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, j = lane & 31;
  int bx, by;
  tile_of_block(blockIdx.x, p.nx, p.ny, bx, by);
  const int G = p.K / kGroup, npt = (p.R + 31) / 32;
  const int pt = min(4 * by + w, npt - 1);            // a tile past the last repeats it, unstored
  const bool live = 4 * by + w < npt;

  RowReader<KIND> row[ND];
  Codes codes[ND], next[ND];                          // the next group's, and the one after
  PlaneReader pl;
  pl.init(p, pt, lane, 0, 2 * G);
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    row[d].init(p, tile_row<EPI>(NT * bx + 4 * d + w, j, p.M), h);
    row[d].load(codes[d], 0);
  }
  Planes qa0 = pl.load(0), qa1 = pl.load(1), qb0, qb1;
  fill_lut<KIND, true, 256>(lut);
  __syncthreads();
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    uint32_t D[8];
    row[d].decode(codes[d], 0, lut, D);
    bs[0][4 * d + w][0][lane] = i32x4_t{(int)D[0], (int)D[1], (int)D[2], (int)D[3]};
    bs[0][4 * d + w][1][lane] = i32x4_t{(int)D[4], (int)D[5], (int)D[6], (int)D[7]};
    wsc[0][32 * (4 * d + w) + j] = row_scale<KIND>(row[d], codes[d]);
    row[d].load(codes[d], min(1, G - 1));
    row[d].load(next[d], min(2, G - 1));
  }
  __syncthreads();
  f32x16_t acc[NT] = {}, t[2][2] = {};
  i32x4_t wt[2][2][2];                                // [pair's parity][step][tile]
  float sc[2][2] = {}, ss = 0.f;
  unsigned long long wide = 0;                        // groups with wide blocks, 64 apart
  wt[0][0][0] = bs[0][0][0][lane];
  wt[0][0][1] = bs[0][1][0][lane];
  wt[0][1][0] = bs[0][0][1][lane];
  wt[0][1][1] = bs[0][1][1][lane];
  const uint32_t* lt = lut + (lane & 31);
  typename RowReader<KIND>::Half hv;
  // One slot: S of the group's 10 NP, the C-th of pair I, on planes q0, q1; the next group's go to n0, n1.
  auto slot = [&](auto SC, int g, Planes& q0, Planes& q1, Planes& n0, Planes& n1) __attribute__((always_inline)) {
    constexpr int S = decltype(SC)::value, I = S / 10, C = S % 10, ST = C / 5, T = I & 1, L = (I + NP - 1) % NP;
    const int buf = g & 1, gn = min(g + 1, G - 1);
    const f32x16_t zero = {};
    Planes& q = ST ? q1 : q0;
    if constexpr (I == 0 && C % 5 == 0) asm volatile("" : "+a"(q.c01));
    if constexpr (I == 0 && C % 5 == 2) asm volatile("" : "+a"(q.c23));
    if constexpr (I == 0 && C % 5 == 4) asm volatile("" : "+a"(q.c4));
    t[T][0] = mx<C % 5>(q, wt[T][ST][0], C ? t[T][0] : zero);
    t[T][1] = mx<C % 5>(q, wt[T][ST][1], C ? t[T][1] : zero);
    asm volatile("" : "+v"(t[T][0]), "+v"(t[T][1]) : : "memory");
    if constexpr (S == 4 || S == 9) {
      wide |= (unsigned long long)(__any((int)q.scales() < 0) ? 1u : 0u) << (g & 63);
      ss += q.ss();
      asm volatile("" : "+a"(ss));
    }
    // The last pair's sums, four a slot.
    if constexpr (C >= 1 && C <= 8) {
      constexpr int k = (C - 1) / 4, e0 = 4 * ((C - 1) % 4);
#pragma unroll
      for (int e = e0; e < e0 + 4; ++e) acc[2 * L + k][e] = fmaf(t[T ^ 1][k][e], sc[T ^ 1][k], acc[2 * L + k][e]);
      asm volatile("" : "+v"(acc[2 * L + k]));
    }
    // The next group's planes, in six parts, a step's scales first.
    if constexpr (S % 3 == 0 && S < 18) {
      constexpr int k = S / 3;
      Planes& n = k < 3 ? n0 : n1;
      const uint32_t b = pl.base(2 * gn + k / 3);
      if constexpr (k % 3 == 0) n.c4 = pl.last(b);
      else if constexpr (k % 3 == 1) n.c01 = pl.pair(b, 0);
      else n.c23 = pl.pair(b, 3);
    }
    // The next pair's weights: the next group's for the last pair, behind the barrier.
    if constexpr (I == NP - 1) {
      if constexpr (C == 4) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if constexpr (C == 4 || C == 6) {
        wt[T ^ 1][(C - 4) / 2][0] = bs[buf ^ 1][0][(C - 4) / 2][lane];
        wt[T ^ 1][(C - 4) / 2][1] = bs[buf ^ 1][1][(C - 4) / 2][lane];
      }
    } else if constexpr (C == 2 || C == 4) {
      wt[T ^ 1][(C - 2) / 2][0] = bs[buf][2 * I + 2][(C - 2) / 2][lane];
      wt[T ^ 1][(C - 2) / 2][1] = bs[buf][2 * I + 3][(C - 2) / 2][lane];
    }
    if constexpr (C == 3) {
      sc[T][0] = wsc[buf][32 * (2 * I) + j];
      sc[T][1] = wsc[buf][32 * (2 * I + 1) + j];
    }
    // The next group's decode: a tile over two pairs.
    constexpr int d = I / 2, o = S % 20;
    if constexpr (o == 0) row[d].begin(codes[d], gn, hv);
    if constexpr (o <= 3) row[d].template look<o <= 3 ? o : 0>(hv, lt);
    if constexpr (o == 6) bs[buf ^ 1][4 * d + w][0][lane] = row[d].low(hv);
    if constexpr (o == 7 || o == 8) row[d].template look<o == 7 ? 4 : 5>(hv, lt);
    if constexpr (o == 9) wsc[buf ^ 1][32 * (4 * d + w) + j] = row_scale<KIND>(row[d], codes[d]);
    if constexpr (o == 12) {
      bs[buf ^ 1][4 * d + w][1][lane] = row[d].high(hv);
      codes[d] = next[d];
      asm volatile("" : "+a"(row[d].rbase), "+a"(row[d].h));          // or its sums with the offsets spill
      row[d].load_uniform(next[d], min(g + 3, G - 1));
    }
  };
  auto group = [&](int g, Planes& q0, Planes& q1, Planes& n0, Planes& n1) __attribute__((always_inline)) {
    in_turn([&](auto S) __attribute__((always_inline)) { slot(S, g, q0, q1, n0, n1); },
            std::make_integer_sequence<int, 10 * NP>());
  };
  for (int g = 0; g < G; g += 2) {
    group(g, qa0, qa1, qb0, qb1);
    if (g + 1 == G) break;
    group(g + 1, qb0, qb1, qa0, qa1);
  }
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[NT - 2 + k][e] = fmaf(t[1][k][e], sc[1][k], acc[NT - 2 + k][e]);

  // The groups in which any wave met a wide block once more: the weights decoded by all as above, the products
  // by the waves that hold one, a digit of x for all tiles at a time under the next digit's conversion. About
  // 6 us a group and block: 24576 x 4096, 2048 positions, takes 514 us without wide blocks, 549, 650 and 1079
  // with one, four and sixteen channels 1000 times the others at every position (a pass for each tile, its
  // loads one by one: 843, 1144 and 2469; two fp16 planes, with or without: 750).
  if (!live) wide = 0;
  if (lane == 0) wide_of[w] = wide;
  __syncthreads();
  const unsigned long long some = wide_of[0] | wide_of[1] | wide_of[2] | wide_of[3];
  if (some) {
    // The sums leave the vector registers for this, or the main loop's own registers are spilt to make room.
#pragma unroll
    for (int b = 0; b < NT; ++b) asm volatile("" : "+a"(acc[b]));
    auto next_wide = [&](int g) {
      while (g < G && !(some >> (g & 63) & 1)) ++g;
      return g;
    };
    int g = next_wide(0);
#pragma unroll
    for (int d = 0; d < ND; ++d) row[d].load(codes[d], min(g, G - 1));
    while (g < G) {
      const int gn = next_wide(g + 1);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        uint32_t D[8];
        row[d].decode(codes[d], g, lut, D);
        bs[0][4 * d + w][0][lane] = i32x4_t{(int)D[0], (int)D[1], (int)D[2], (int)D[3]};
        bs[0][4 * d + w][1][lane] = i32x4_t{(int)D[4], (int)D[5], (int)D[6], (int)D[7]};
        wsc[0][32 * (4 * d + w) + j] = row_scale<KIND>(row[d], codes[d]);
        row[d].load(codes[d], min(gn, G - 1));
      }
      __syncthreads();
      if (wide >> (g & 63) & 1) {
        f32x16_t s[NT] = {};
#pragma nounroll
        for (int st = 0; st < 2; ++st) {
          const Planes q = pl.load(2 * g + st);
          if (!__any((int)q.scales() < 0)) continue;
          i32x4_t wd[NT];
#pragma unroll
          for (int b = 0; b < NT; ++b) wd[b] = bs[0][b][st][lane];
          Wide x;
          x.init(q);
          bool more = true;
#pragma nounroll
          while (more) {
            u32x6_t c;
            int scale;
            more = x.next(c, scale);
#pragma unroll
            for (int b = 0; b < NT; ++b) s[b] = mx_digits(c, scale, wd[b], s[b]);
          }
        }
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          const float v = wsc[0][32 * b + j];
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[b][e] = fmaf(s[b][e], v, acc[b][e]);
        }
      }
      __syncthreads();
      g = gn;
    }
  }

  // Accumulator e of lane l holds position i = 8 (e / 4) + 4 (l / 32) + e % 4, weight row l % 32.
  ss += __shfl_xor(ss, 32, 64);
  if (h == 0) rsx[32 * w + j] = p.norm ? 1.0f / sqrtf(ss / (float)p.K + p.eps) : 1.f;
  __syncthreads();
  if (!live) return;
  // Four positions' residuals are read before the first is used: one at a time each waits for memory
  // (128 of them, 30 us a block).
#pragma unroll
  for (int e0 = 0; e0 < 16; e0 += 4) {
    const int i0 = 2 * e0 + 4 * h, r0 = 32 * pt + i0;
    float old[4][NT] = {};
    if (EPI == GM_RESID) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          const int m = 32 * (NT * bx + b) + j;
          if (r0 + k < p.R && m < p.M) old[k][b] = p.y[(size_t)(r0 + k) * p.ldy + m];
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float rs = rsx[32 * w + i0 + k];
      float* yr = p.y + (size_t)(r0 + k) * p.ldy;
#pragma unroll
      for (int b = 0; b < NT; b += EPI == GM_SWIGLU ? 2 : 1) {
        const int m = EPI == GM_SWIGLU ? 32 * ((NT * bx + b) >> 1) + j : 32 * (NT * bx + b) + j;
        if (r0 + k >= p.R || m >= (EPI == GM_SWIGLU ? p.M / 2 : p.M)) continue;
        const float v = acc[b][e0 + k] * rs;
        if constexpr (EPI == GM_SWIGLU) yr[m] = silu(v) * (acc[b + 1][e0 + k] * rs);
        else if (EPI == GM_RESID) yr[m] = old[k][b] + v;
        else yr[m] = v;
      }
    }
  }
}

// Products whose grid of large tiles would leave the chip idle: a block takes 32 positions x 32 NB
// weight rows and its eight waves split K, each decoding its own groups' weights in registers; the
// waves' sums are added through LDS in wave order. Bound by vector issue (each wave decodes for
// itself) and, on the shortest prompts, by latency: 24 positions of 6144 x 4096 15.0 us with the
// planes (69.5 in 24 large fp16 tiles), 509 of 2048 x 6144 40 us (119).
template <int KIND, int EPI, int NB>
__global__ __launch_bounds__(kGmThreads, 1) void gemm_split_kernel(GemmParams p) {
  constexpr int PT = NB < 2 ? 1 : 2;                  // tiles reduced at a time
  constexpr int kRed = 8 * PT * 1024;
  __shared__ __align__(16) uint32_t sm[kRed > kLut ? kRed : kLut];
  __shared__ float ssx[8][32];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, j = lane & 31;
  int bx, pt;
  tile_of_block(blockIdx.x, p.nx, p.ny, bx, pt);
  const int G = p.K / kGroup, g0 = G * w / 8, g1 = G * (w + 1) / 8;
  RowReader<KIND> row[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) row[b].init(p, tile_row<EPI>(NB * bx + b, j, p.M), h);
  PlaneReader pl;
  const int gf = min(g0, G - 1);
  pl.init(p, pt, lane, 2 * gf, 2 * max(g1, gf + 1));
  Codes codes[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) row[b].load(codes[b], gf);
  Planes q0 = pl.load(2 * gf), q1 = pl.load(2 * gf + 1);
  fill_lut<KIND, true, kGmThreads>(sm);
  __syncthreads();
  f32x16_t acc[NB] = {};
  float ss = 0.f;
  unsigned long long wide = 0;                        // groups with wide blocks, 64 apart
  for (int g = g0; g < g1; ++g) {
    i32x4_t b0[NB], b1[NB];
    float sc[NB];
    const int gn = min(g + 1, g1 - 1);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      uint32_t D[8];
      row[b].decode(codes[b], g, sm, D);
      b0[b] = i32x4_t{(int)D[0], (int)D[1], (int)D[2], (int)D[3]};
      b1[b] = i32x4_t{(int)D[4], (int)D[5], (int)D[6], (int)D[7]};
      sc[b] = row_scale<KIND>(row[b], codes[b]);
      asm volatile("" : "+v"(b0[b]), "+v"(b1[b]) : : "memory");
      row[b].load(codes[b], gn);
    }
    wide |= (unsigned long long)(__any((int)(q0.scales() | q1.scales()) < 0) ? 1u : 0u) << ((g - g0) & 63);
    f32x16_t t[NB];
    ss += q0.ss();
    mx_step<true, NB>(q0, b0, t);
    pin(t);
    q0 = pl.load(2 * gn);
    ss += q1.ss();
    mx_step<false, NB>(q1, b1, t);
    pin(t);
    q1 = pl.load(2 * gn + 1);
    asm volatile("" : : : "memory");
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[b][e] = fmaf(t[b][e], sc[b], acc[b][e]);
  }
  if (wide) {
    constexpr int TB = NB < 2 ? 1 : 2;                // tiles at a time (registers)
    for (int g = g0; g < g1; ++g) {
      if (!(wide >> ((g - g0) & 63) & 1)) continue;
#pragma unroll
      for (int t0 = 0; t0 < NB; t0 += TB) {
        i32x4_t b0[TB], b1[TB];
        float sc[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) {
          row[t0 + b].load(codes[b], g);
          uint32_t D[8];
          row[t0 + b].decode(codes[b], g, sm, D);
          b0[b] = i32x4_t{(int)D[0], (int)D[1], (int)D[2], (int)D[3]};
          b1[b] = i32x4_t{(int)D[4], (int)D[5], (int)D[6], (int)D[7]};
          sc[b] = row_scale<KIND>(row[t0 + b], codes[b]);
        }
        f32x16_t s[TB] = {};
#pragma nounroll
        for (int st = 0; st < 2; ++st) {
          const Planes q = pl.load(2 * g + st);
          if (!__any((int)q.scales() < 0)) continue;
          Wide x;
          x.init(q);
          bool more = true;
#pragma nounroll
          while (more) {
            u32x6_t c;
            int scale;
            more = x.next(c, scale);
#pragma unroll
            for (int b = 0; b < TB; ++b) s[b] = mx_digits(c, scale, st ? b1[b] : b0[b], s[b]);
          }
        }
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[t0 + b][e] = fmaf(s[b][e], sc[b], acc[t0 + b][e]);
      }
    }
  }
  ss += __shfl_xor(ss, 32, 64);
  if (h == 0) ssx[w][j] = ss;
  float4* red = (float4*)sm;                          // [wave][tile][e / 4][lane]
#pragma unroll
  for (int b0 = 0; b0 < NB; b0 += PT) {
    __syncthreads();                                  // the table's or the last pass's reads are done
#pragma unroll
    for (int b = 0; b < PT; ++b)
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4)
        red[((w * PT + b) * 4 + e4) * 64 + lane] = make_float4(acc[b0 + b][4 * e4], acc[b0 + b][4 * e4 + 1],
                                                               acc[b0 + b][4 * e4 + 2], acc[b0 + b][4 * e4 + 3]);
    __syncthreads();
    constexpr int per = EPI == GM_SWIGLU ? 1 : PT;    // output tiles of the pass
    if (w >= 4 * per) continue;
    const int tb = w >> 2, e4 = w & 3;
    float4 v[2];
#pragma unroll
    for (int u = 0; u < (EPI == GM_SWIGLU ? 2 : 1); ++u) {
      v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      const int b = EPI == GM_SWIGLU ? u : tb;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float4 a = red[((k * PT + b) * 4 + e4) * 64 + lane];
        v[u] = make_float4(v[u].x + a.x, v[u].y + a.y, v[u].z + a.z, v[u].w + a.w);
      }
    }
    const int tile = NB * bx + b0 + tb;
    const int m = EPI == GM_SWIGLU ? 32 * (tile >> 1) + j : 32 * tile + j;
    const float a0[4] = {v[0].x, v[0].y, v[0].z, v[0].w}, a1[4] = {v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = 8 * e4 + 4 * h + k, r = 32 * pt + i;
      if (r >= p.R || m >= (EPI == GM_SWIGLU ? p.M / 2 : p.M)) continue;
      float rs = 1.f;
      if (p.norm) {
        float tot = 0.f;
#pragma unroll
        for (int z = 0; z < 8; ++z) tot += ssx[z][i];
        rs = 1.0f / sqrtf(tot / (float)p.K + p.eps);
      }
      float* y = p.y + (size_t)r * p.ldy + m;
      if (EPI == GM_SWIGLU) *y = silu(a0[k] * rs) * (a1[k] * rs);
      else if (EPI == GM_RESID) *y += a0[k] * rs;
      else *y = a0[k] * rs;
    }
  }
}

template <int KIND, int EPI>
static void gemm_ternary_kind(GemmParams& p, int nb, hipStream_t s) {
  const int tiles = EPI == GM_SWIGLU ? 2 * cdiv(p.M / 2, 32) : cdiv(p.M, 32);
  if (nb == 0) {
    p.nx = cdiv(tiles, 8);
    p.ny = cdiv(p.R, 128);
    hipLaunchKernelGGL((gemm_kernel<KIND, EPI>), dim3(p.nx * p.ny), dim3(256), 0, s, p);
    return;
  }
  p.nx = cdiv(tiles, nb);
  p.ny = cdiv(p.R, 32);
  const dim3 grid(p.nx * p.ny);
  if (nb == 4) {
    hipLaunchKernelGGL((gemm_split_kernel<KIND, EPI, 4>), grid, dim3(kGmThreads), 0, s, p);
  } else if (nb == 2) {
    hipLaunchKernelGGL((gemm_split_kernel<KIND, EPI, 2>), grid, dim3(kGmThreads), 0, s, p);
  } else if constexpr (EPI != GM_SWIGLU) {             // SwiGLU takes a gate tile and its up tile
    hipLaunchKernelGGL((gemm_split_kernel<KIND, EPI, 1>), grid, dim3(kGmThreads), 0, s, p);
  }
}

template <int KIND>
static void gemm_ternary_epi(GemmParams& p, int nb, hipStream_t s) {
  if (p.epi == GM_SWIGLU) gemm_ternary_kind<KIND, GM_SWIGLU>(p, nb, s);
  else if (p.epi == GM_RESID) gemm_ternary_kind<KIND, GM_RESID>(p, nb, s);
  else gemm_ternary_kind<KIND, GM_STORE>(p, nb, s);
}

int launch_gemm_ternary(const GemmParams& params, hipStream_t s) {
  GemmParams p = params;
  TRX_CHECK(p.kind == TRX_KIND_TERNARY || p.kind == TRX_KIND_TERNARY5, TRX_E_INVALID,
            "prefill GEMM: weight kind %d unsupported", p.kind);
  TRX_CHECK(p.M >= 1 && p.K >= kGroup && p.K % kGroup == 0 && p.R >= 1, TRX_E_INVALID,
            "prefill GEMM: M=%d K=%d R=%d", p.M, p.K, p.R);
  TRX_CHECK(p.epi != GM_SWIGLU || p.M % 2 == 0, TRX_E_INVALID, "prefill GEMM: SwiGLU needs an even M");
  TRX_CHECK((size_t)p.R * p.K * 2 < (1ull << 32) && (size_t)p.M * p.row_bytes < (1ull << 32) &&
            (size_t)p.M * p.row_bytes + 16 <= p.w_bytes, TRX_E_INVALID, "prefill GEMM: operands too large");
  int cus = 0, dev = 0;
  TRX_HIP(hipGetDevice(&dev));
  TRX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  // The tile with the least estimated time: rounds of blocks over the CUs times a round's length, in
  // us per 128 columns as measured at one to twelve rounds: 2.55 for the 128 x 256 tiles, 0.65, 0.43 and
  // 0.34 for the K-split tiles of 32 x 128, 64 and 32 (of 8, 4, 2 and 1 times the smallest's products per
  // wave's step: small tiles fill the chip on short prompts and narrow matrices only. 512 positions
  // of a 2048 x 2048 matrix: 61 us in 32 large tiles, 23, 27 and 33 in 256, 512 and 1024 split ones;
  // 2048 of a 24576 x 4096: 503 us against 930).
  const int tiles = p.epi == GM_SWIGLU ? 2 * cdiv(p.M / 2, 32) : cdiv(p.M, 32), npt = cdiv(p.R, 32);
  const float len[4] = {2.55f, 0.65f, 0.43f, 0.34f};
  const int per[4] = {8, 4, 2, 1};
  int nb = -1;
  float best = 0.f;
  const bool far = (size_t)min(p.R, 32) * p.K * 4 >= (1ull << 32);   // a whole tile's planes: K-split only
  for (int i = far ? 1 : 0; i < (p.epi == GM_SWIGLU ? 3 : 4); ++i) {
    const long long blocks = (long long)cdiv(tiles, per[i]) * (i == 0 ? cdiv(p.R, 128) : npt);
    const float t = len[i] * (float)((blocks + cus - 1) / cus);
    if (nb < 0 || t < best) {
      best = t;
      nb = i == 0 ? 0 : per[i];
    }
  }
  if (p.kind == TRX_KIND_TERNARY5) gemm_ternary_epi<TRX_KIND_TERNARY5>(p, nb, s);
  else gemm_ternary_epi<TRX_KIND_TERNARY>(p, nb, s);
  TRX_LAUNCHED();
  return TRX_OK;
}

}  // namespace trx
