// Exact engine matvec of one to eight int8 activation vectors (model/bitexact.py:101-125 matvec_ternary
// and matvec_ternary_rows, the engine's op 0 and its multi-row mode) on the matrix cores: one pass
// over a tensor's row packets. Every output is, bit for bit, per-group exact sums, the fp16 scale
// split, the shift by e16 + B, the int48 accumulator and >> R.
//
// A block takes 32 weight rows at a time and its waves split K. Per 128-column group and 32 rows a wave decodes the codes to int8 (a table read per code byte, a byte permute per four weights),
// multiplies them by the x vectors with four v_mfma_i32_32x32x32_i8, multiplies the sums by the
// scales' mantissas and adds them, shifted, to int64 accumulators; the waves' accumulators are added
// through LDS (exact in any order). The x vectors take the first eight of the instruction's 32 rows
// (vector r its row (r / 2) + 4 (r % 2), so that a lane holds every second vector's sum); the idle
// rows cost nothing that bounds it, which is the weights' decode and, for small matrices, latency.
// Measured against one v_dot4 pass per vector (up to four) or a v_dot4 pass over LDS-staged vectors:
// eight vectors of a 6144 x 2048 trit5 matrix 18.3 -> 5.2 us, two of it 14.1 -> 5.3, one 7.3 -> 5.1.

#include "trx_internal.h"
#include "trx_rows_dev.h"

namespace trx {

int gemv_check(int kind, int M, int K);

typedef int i32x16_t __attribute__((ext_vector_type(16)));

constexpr int kRowsWaves = 8;
constexpr int kRowsMax = 8;
constexpr int kRowsStaged = 114688;    // n * K of a multi-row call

struct RowsParams {
  const uint8_t* W;
  uint32_t w_bytes;
  const int8_t* x8;     // n rows of K int8
  int32_t* y;           // n rows of M int32
  int32_t* status;
  int n, M, K, G, row_bytes, code_off, B, R;
};

// Eight codes (nibbles) as int8 weights: the even ones, the odd ones.
__device__ __forceinline__ void weights8(uint32_t d, int& even, int& odd) {
  constexpr uint32_t kW = 0x020100FFu;                // codes 0 .. 3: -1, 0, 1, 2
  even = (int)__builtin_amdgcn_perm(kW, kW, d & 0x0F0F0F0Fu);
  odd = (int)__builtin_amdgcn_perm(kW, kW, (d >> 4) & 0x0F0F0F0Fu);
}

// E: sums per lane, half the vectors (rounded up). Few registers on purpose (up to eight waves a SIMD):
// loads four groups ahead, tiles in turn over resident blocks, two tiles a wave and sixteen waves a
// block all measured slower.
template <int KIND, int E>
__global__ __launch_bounds__(64 * kRowsWaves) void gemv_rows_kernel(RowsParams p) {
  constexpr int W = kRowsWaves, kRed = W * 64 * E * 2;                // dwords of the waves' accumulators
  __shared__ __align__(16) uint32_t sm[kRed > kLut ? kRed : kLut];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, j = lane & 31;
  const int g0 = p.G * w / W, g1 = p.G * (w + 1) / W;
  RowReader<KIND> row;
  row.init(p, min(32 * (int)blockIdx.x + j, p.M), h);
  // The vector of the instruction's row j; rows past the last vector repeat it (unread sums).
  const int v = j < 8 ? 2 * (j & 3) + (j >> 2) : 0;
  const int8_t* xr = p.x8 + (size_t)min(v, p.n - 1) * p.K + 64 * h;
  Codes codes;
  i32x4_t x[4];
  auto load = [&](int g) {
    row.load(codes, g);
    // Any alignment: a single vector may start anywhere.
#pragma unroll
    for (int i = 0; i < 4; ++i) __builtin_memcpy(&x[i], xr + (size_t)kGroup * g + 16 * i, 16);
  };
  load(min(g0, p.G - 1));
  fill_lut<KIND, false, 64 * W>(sm);
  __syncthreads();
  long long acc[E] = {};
  for (int g = g0; g < g1; ++g) {
    // x in the order of the decoded weights: from 65 on in half 1 of a trit5 group (64 last), the even
    // columns of each eight, then the odd ones.
    uint32_t d[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t lo = (uint32_t)x[i >> 2][i & 3], hi = (uint32_t)x[((i + 1) & 15) >> 2][(i + 1) & 3];
      d[i] = KIND == TRX_KIND_TERNARY5 ? __builtin_amdgcn_alignbyte(hi, lo, (uint32_t)h) : lo;
    }
    i32x4_t a[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a[i >> 1][2 * (i & 1)] = (int)__builtin_amdgcn_perm(d[2 * i + 1], d[2 * i], 0x06040200u);
      a[i >> 1][2 * (i & 1) + 1] = (int)__builtin_amdgcn_perm(d[2 * i + 1], d[2 * i], 0x07050301u);
    }
    const Codes now = codes;
    load(min(g + 1, g1 - 1));
    uint32_t D[8];
    row.decode(now, g, sm, D);
    i32x16_t t = {};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      int e0, o0, e1, o1;
      weights8(D[2 * s], e0, o0);
      weights8(D[2 * s + 1], e1, o1);
      t = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[s], i32x4_t{e0, o0, e1, o1}, t, 0, 0, 0);
    }
    int m11, e16;
    fp16_split((uint16_t)now.sc, m11, e16);
    const int sh = e16 + p.B, left = max(sh, 0), right = min(max(-sh, 0), 63);
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] += ((long long)__mul24(t[e], m11) << left) >> right;
  }
  long long* red = (long long*)sm;                    // [wave][e][lane]
  __syncthreads();                                    // the table's reads are done
#pragma unroll
  for (int e = 0; e < E; ++e) red[(w * E + e) * 64 + lane] = acc[e];
  __syncthreads();
  if (w >= E) return;
  const int r = 2 * w + h, m = 32 * (int)blockIdx.x + j;
  if (r >= p.n || m >= p.M) return;
  long long s = 0;
#pragma unroll
  for (int k = 0; k < W; ++k) s += red[(k * E + w) * 64 + lane];
  const long long res = s >> p.R;
  const int bad = (((s >= (1LL << 47)) || (s <= -(1LL << 47))) ? 1 : 0) |
                  ((res >= (1LL << 31) || res <= -(1LL << 31)) ? 2 : 0);
  p.y[(size_t)r * p.M + m] = (int32_t)res;
  if (bad) atomicOr(p.status, bad);
}

template <int KIND, int E>
static int launch_rows(const RowsParams& p, hipStream_t s) {
  hipLaunchKernelGGL((gemv_rows_kernel<KIND, E>), dim3(cdiv(p.M, 32)), dim3(64 * kRowsWaves), 0, s, p);
  TRX_LAUNCHED();
  return TRX_OK;
}

template <int KIND>
static int dispatch_rows(const RowsParams& p, hipStream_t s) {
  switch ((p.n + 1) / 2) {
    case 1: return launch_rows<KIND, 1>(p, s);
    case 2: return launch_rows<KIND, 2>(p, s);
    case 3: return launch_rows<KIND, 3>(p, s);
    default: return launch_rows<KIND, 4>(p, s);
  }
}

// n vectors (arguments checked by the callers).
int gemv_exact_any(const uint8_t* rows, int kind, int M, int K, const int8_t* x8, int n, int B, int R, int32_t* y,
                   int32_t* status, hipStream_t s) {
  TRX_CHECK(B >= -48 && B <= 48 && R >= 0 && R < 63, TRX_E_INVALID, "gemv_exact: B=%d R=%d out of range", B, R);
  const RowGeom rg = row_geom(kind, K);
  RowsParams p = {};
  p.W = rows;
  // A row's last read ends with its padding at the latest (26 bytes a group, padded to 32).
  p.w_bytes = (uint32_t)((unsigned long long)M * rg.row_bytes + 32);
  p.x8 = x8;
  p.y = y;
  p.status = status;
  p.n = n;
  p.M = M;
  p.K = K;
  p.G = rg.G;
  p.row_bytes = rg.row_bytes;
  p.code_off = rg.code_off;
  p.B = B;
  p.R = R;
  return kind == TRX_KIND_TERNARY5 ? dispatch_rows<TRX_KIND_TERNARY5>(p, s) : dispatch_rows<TRX_KIND_TERNARY>(p, s);
}

int gemv_exact(const uint8_t* rows, int kind, int M, int K, const int8_t* x8, int B, int R,
               int32_t* y, int32_t* status, hipStream_t s);

int gemv_exact_rows(const uint8_t* rows, int kind, int M, int K, const int8_t* x8, int n, int B,
                    int R, int32_t* y, int32_t* status, hipStream_t s) {
  TRX_CHECK(rows && x8 && y && status, TRX_E_INVALID, "gemv_exact_rows: null argument");
  int rc = gemv_check(kind, M, K);
  if (rc) return rc;
  TRX_CHECK(n >= 1 && n <= kRowsMax, TRX_E_INVALID, "gemv_exact_rows: %d x rows (1..%d)", n, kRowsMax);
  TRX_CHECK((long long)n * K <= kRowsStaged, TRX_E_INVALID,
            "gemv_exact_rows: %d x rows of K=%d exceed %d staged bytes", n, K, kRowsStaged);
  TRX_CHECK(((uintptr_t)x8 & 15) == 0, TRX_E_INVALID, "gemv_exact_rows: x8 must be 16-byte aligned");
  // One vector of a large matrix: the single-vector kernel's resident blocks, where their rounds of 4096 rows are
  // nearly full. Weights from memory, trit5 and 2-bit, us there against here: 151936 x 4096 49.8 and 49.9 against
  // 82 and 75, 34816 x 5120 25.6 and 21.4 against 26.9 and 26.6, 4096 x 12288 13.0 and 10.8 against 14.7 and
  // 13.0; with a round of 1024 rows, 5120 x 17408 28.6 and 22.3 against 20.1 and 18.2.
  const int rounds = cdiv(M, 4096);
  if (n == 1 && (long long)M * K >= (1ll << 25) && M >= rounds * 3584)
    return gemv_exact(rows, kind, M, K, x8, B, R, y, status, s);
  return gemv_exact_any(rows, kind, M, K, x8, n, B, R, y, status, s);
}

}  // namespace trx

extern "C" __attribute__((visibility("default"))) int trx_gemv_ternary_exact_rows(
    const uint8_t* rows, int kind, int M, int K, const int8_t* x8_rows, int n_rows, int B, int R,
    int32_t* y, int32_t* status, trx_stream_t s) {
  return trx::gemv_exact_rows(rows, kind, M, K, x8_rows, n_rows, B, R, y, status, (hipStream_t)s);
}
