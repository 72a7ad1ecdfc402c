// fp32 Dense on the f16 matrix cores: each fp32 operand is written as two f16 terms of a power-of-two
// multiple of it, x 2^e = hi + lo + r (|r| <= 2^-23 |x 2^e|: 11 + 11 significant bits and lo's sign), and
//   x . w = 2^-(ex + ew) (hi_x . hi_w + hi_x . lo_w + lo_x . hi_w) + (lo_x . lo_w and r terms)
// runs as three v_mfma_f32_32x32x16_f16 products: hi . hi into one fp32 accumulator, the two cross products into another
// (256x256 tiles, whose registers do not hold both, add all three into one). The dropped terms are at most 2^-22 of a
// product, random in sign; the f16 products themselves are exact in fp32. The large sums then round K / 16 times (3 K / 16
// on 256x256 tiles) against K / 2 for v_mfma_f32_32x32x2_f32, so the result is nearer to float64 than the fp32 MFMA's:
// normal operands, K = 1024 / 4096: 2e-7 / 4e-7 of the result's norm (3.6e-7 / 7.1e-7 with one accumulator; less where K
// is split) against 5.7e-7 / 1.1e-6, at 3/16 of its matrix time (MI355X: 2.5 PFLOP/s f16 against 157 TFLOP/s fp32).
//
// Split rows: a row of K values (K a multiple of 32) is K / 32 groups of [32 hi | 32 lo] f16, 128 bytes a
// group: the same bytes as the fp32 row, and one group is one k-step's LDS row of the bf16 GEMM's layout. The
// exponent is per row, so that the row's largest value lands in [2^14, 2^15): values down to 2^-17 of it keep
// 22 bits, smaller ones an absolute error of 2^-39 of it. Rows that this does not suit go by fp32 (row_is_wide,
// group_max).
#include <math.h>

#include <algorithm>

#include "qvl_split.h"

namespace qvl {

// The sum, or the maximum of the bits, over the threads of a row (T = 64: a wave; 256: the workgroup, through
// 4 floats of LDS).
template <int T>
__device__ __forceinline__ float row_sum(float v, float* tmp) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  if constexpr (T > 64) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
    __syncthreads();
    v = (tmp[0] + tmp[1]) + (tmp[2] + tmp[3]);
  }
  return v;
}

__device__ __forceinline__ uint32_t wave_max_bits(uint32_t m) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
  return m;
}

__device__ __forceinline__ uint32_t block_max_bits(uint32_t m, float* tmp) {
  m = wave_max_bits(m);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = __uint_as_float(m);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) m = max(m, __float_as_uint(tmp[i]));
  return m;
}

// Which rows the split does not serve as well as fp32 does. An entry below 2^-17 of its row's largest has fewer than 22
// bits left (an absolute error of 2^-39 of the largest): nothing beside the others' rounding where such entries are few,
// but all there is where most of the row is that small and what multiplies its few large entries is zero. So a row
// is wide, and its outputs are computed from the fp32 operands, where more than a quarter of its entries (zeros, which
// have no error, aside) are below that line, or where it holds an infinity or a NaN. Normal values: an entry in 40000
// is below it; under one entry 2^16 above the rest of them a row is wide.
__device__ __forceinline__ uint32_t count_small(const f32x4& v, float s) {
  uint32_t n = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) n += (__float_as_uint(v[e] * s) & 0x7fffffffu) - 1u < 0x3e7fffffu;   // 0 < |v s| < 0.25
  return n;
}

template <int T>
__device__ __forceinline__ uint32_t row_count(uint32_t n, float* tmp) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) n += (uint32_t)__shfl_xor((int)n, o);
  if constexpr (T > 64) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = __uint_as_float(n);
    __syncthreads();
    n = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) n += __float_as_uint(tmp[i]);
  }
  return n;
}

// mb: the bits of the row's maximum; small: this thread's count; v[CH]: this thread's entries, zeros past the row.
template <int T, int CH>
__device__ __forceinline__ bool row_is_wide(uint32_t mb, uint32_t small, const f32x4 (&v)[CH], float* tmp) {
  if (T == 64 && !__builtin_amdgcn_ballot_w64(small != 0)) return mb >= 0x7f800000u;
  small = row_count<T>(small, tmp);
  if (small == 0 || mb >= 0x7f800000u) return mb >= 0x7f800000u;
  uint32_t some = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) some += v[i][e] != 0.f;
  return 4 * small > row_count<T>(some, tmp);
}

// store_split4 of columns c..c+3 by lane t, c = 4 t + a multiple of 8: a pair of lanes trades halves, so that each stores 16
// bytes and 8 lanes a whole 128-byte group.
__device__ __forceinline__ void store_split_pair(f16* row, int c, const f16x4& hi, const f16x4& lo, int t) {
  const u32x2 h = __builtin_bit_cast(u32x2, hi), l = __builtin_bit_cast(u32x2, lo);
  const bool odd = t & 1;
  const uint32_t g0 = __builtin_amdgcn_mov_dpp(odd ? h.x : l.x, 0xB1, 0xF, 0xF, true);    // quad_perm 1 0 3 2
  const uint32_t g1 = __builtin_amdgcn_mov_dpp(odd ? h.y : l.y, 0xB1, 0xF, 0xF, true);
  f16* at = row + (c >> 5) * 64 + (odd ? 28 : 0) + (c & 31);
  *reinterpret_cast<u32x4*>(at) = odd ? u32x4{g0, g1, l.x, l.y} : u32x4{h.x, h.y, g0, g1};
}

// ---------------------------------------------------------------------------------------------
// fp32 rows -> split rows: a row's maximum, then its values scaled and split. Memory bound (each row read
// and written once): T = 64 or 256 threads hold a row in registers, CH chunks of 4 values each, so that
// every load is in flight at once and long rows have as many waves as short ones. Rows of x (the first) and
// of w share one launch.
// ---------------------------------------------------------------------------------------------
struct SplitRowsParams {
  const float* src[2];
  int64_t ld[2];
  f16* dst[2];
  float* inv[2];      // 2^-e of each row; NaN for a row that goes by fp32 (row_is_wide)
  int rows[2];
  int K;
};

template <int T, int CH>
__global__ __launch_bounds__(256) void split_rows_kernel(SplitRowsParams p) {
  constexpr int RPB = 256 / T;
  __shared__ float tmp[4];
  const int first = (p.rows[0] + RPB - 1) / RPB, which = (int)blockIdx.x >= first;
  const int t = threadIdx.x % T;
  const int row = ((int)blockIdx.x - (which ? first : 0)) * RPB + threadIdx.x / T;
  if (row >= p.rows[which]) return;                 // (a whole wave, or with T = 256 never)
  const float* src = p.src[which] + (int64_t)row * p.ld[which];
  f32x4 v[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + i * T) * 4;
    v[i] = c < p.K ? *reinterpret_cast<const f32x4*>(src + c) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // (the bits of |x| order as the values do, infinities and NaN above every finite one)
  uint32_t mb = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) mb = max(mb, __float_as_uint(v[i][e]) & 0x7fffffffu);
  if constexpr (T == 256) mb = block_max_bits(mb, tmp);
  else mb = wave_max_bits(mb);
  const float s = split_scale(__uint_as_float(mb));
  f16* dst = p.dst[which] + (int64_t)row * 2 * p.K;
  uint32_t small = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + i * T) * 4;
    if (c >= p.K) break;
    f16x4 hi, lo;
    split4(v[i], s, hi, lo);
    store_split_pair(dst, c, hi, lo, t);
    small += count_small(v[i], s);
  }
  const bool wide = row_is_wide<T>(mb, small, v, tmp);
  if (t == 0) p.inv[which][row] = wide ? __uint_as_float(0x7fc00000u) : 1.0f / s;
}

static int split_rows(const SplitRowsParams& p, hipStream_t stream) {
  const int waves = (p.rows[0] + 3) / 4 + (p.rows[1] + 3) / 4, blocks = p.rows[0] + p.rows[1];
  if (p.K <= 1024) hipLaunchKernelGGL((split_rows_kernel<64, 4>), dim3(waves), dim3(256), 0, stream, p);
  else if (p.K <= 2048) hipLaunchKernelGGL((split_rows_kernel<64, 8>), dim3(waves), dim3(256), 0, stream, p);
  else if (p.K <= 4096) hipLaunchKernelGGL((split_rows_kernel<256, 4>), dim3(blocks), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((split_rows_kernel<256, 8>), dim3(blocks), dim3(256), 0, stream, p);
  return check_launch("split_rows");
}

// ---------------------------------------------------------------------------------------------
// Packed fp32 weights [n][k] -> split rows, with a bound on |LN(x) . w + b|, the Dense's output for any x: the
// normalised row has a norm of at most sqrt(k), so |.| <= sqrt(k) |gamma w| + |beta . w| + |b| (one per row, to
// row_bound). It lets the outputs be split by one exponent that is known before they are. Non-finite weights make
// it non-finite, and their row's factor NaN.
// A tower splits each layer's weights on the stream right before they are used, so that a forward (or a graph's
// replay) reads the weights as they are then; all Dense weights of a layer share one launch, a wave or a workgroup
// holds a row.
// Memory bound: a 1024-wide block's 48 MB are read and written in 21 us, a copy's 4.7 TB/s (28 us with a wave on every
// row: 16 chunks of a 4096-wide row are too many registers for the waves that keep the loads in flight). A 784-patch
// forward of 24 blocks takes 4.76 ms with it, 4.12 with weights split beforehand, and 8.8 on the fp32 MFMA kernels.
template <int CH>
__global__ __launch_bounds__(256) void split_weights_kernel(SplitWeights p) {
  __shared__ float tmp[4];
  int which = 0;
  while (which + 1 < p.count && (int)blockIdx.x >= p.e[which + 1].first) ++which;
  const SplitWeight& e = p.e[which];
  const int k = e.k, T = k <= 256 * CH ? 64 : 256;                 // (uniform over the workgroup)
  const int t = threadIdx.x & (T - 1), row = ((int)blockIdx.x - e.first) * (256 / T) + threadIdx.x / T;
  if (row >= e.n) return;                                          // (a whole wave, or with T = 256 never)
  const float* src = e.w + (int64_t)row * k;
  f32x4 v[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + i * T) * 4;
    v[i] = c < k ? *reinterpret_cast<const f32x4*>(src + c) : f32x4{};
  }
  const auto max_bits = [&](uint32_t m) { return T == 64 ? wave_max_bits(m) : block_max_bits(m, tmp); };
  const auto sum = [&](float x) { return T == 64 ? row_sum<64>(x, tmp) : row_sum<256>(x, tmp); };
  uint32_t mb = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) mb = max(mb, __float_as_uint(v[i][j]) & 0x7fffffffu);
  mb = max_bits(mb);
  if (e.out) {
    const float s = split_scale(__uint_as_float(mb));
    f16* dst = e.out + (int64_t)row * 2 * k;
    uint32_t small = 0;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = (t + i * T) * 4;
      if (c >= k) break;
      f16x4 hi, lo;
      split4(v[i], s, hi, lo);
      store_split_pair(dst, c, hi, lo, t);
      small += count_small(v[i], s);
    }
    const bool wide = T == 64 ? row_is_wide<64>(mb, small, v, tmp) : row_is_wide<256>(mb, small, v, tmp);
    if (t == 0) e.inv[row] = wide && (p.mark_wide || mb >= 0x7f800000u) ? __uint_as_float(0x7fc00000u) : 1.0f / s;
  }
  if (!e.row_bound) return;
  uint32_t gb = 0;                                                 // the bits of max |gamma w|
  float norm = 0.f, dot = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + i * T) * 4;
    if (c >= k) break;
    int lc = c;
    while (e.gamma && lc >= e.ln_cols) lc -= e.ln_cols;
    const f32x4 g = e.gamma ? *reinterpret_cast<const f32x4*>(e.gamma + lc) : f32x4{1.f, 1.f, 1.f, 1.f};
    const f32x4 b = e.beta ? *reinterpret_cast<const f32x4*>(e.beta + lc) : f32x4{};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      dot = fmaf(b[j], v[i][j], dot);
      v[i][j] *= g[j];
      gb = max(gb, __float_as_uint(v[i][j]) & 0x7fffffffu);
    }
  }
  // (the squares are taken of multiples of up to 2^15: neither weights of 1e-25 nor of 1e25 leave the range)
  const float gs = split_scale(__uint_as_float(max_bits(gb)));
#pragma unroll
  for (int i = 0; i < CH; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) norm = fmaf(v[i][j] * gs, v[i][j] * gs, norm);
  norm = sum(norm);
  dot = sum(dot);
  if (t == 0) e.row_bound[row] = 1.001f * sqrtf(norm * (float)k) / gs + fabsf(dot) + fabsf(e.bias[row]);
}

// One exponent for all outputs of a Dense suits them while their bounds are alike: an output's absolute error is 2^-39 of
// the largest bound, and the outputs themselves are some 2^-5 of theirs, so bounds down to 2^-9 of the largest keep fp32's
// 24 bits. kGroupAlike: NaN where more than a quarter of them (zeros aside) are lower, or one is not finite: the Dense
// then writes fp32 rows in place of split rows, and its reader takes them as such. (An atomic maximum per row on one
// address took the launch above from 10 to 45 us.)
__device__ __forceinline__ void group_max(const float* __restrict__ v, int n, int kind, float* __restrict__ out, float* tmp) {
  uint32_t mb = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += 256) mb = max(mb, __float_as_uint(v[i]) & 0x7fffffffu);
  mb = block_max_bits(mb, tmp);
  if (kind == kGroupInf) mb = min(mb, 0x7f800000u);
  if (kind == kGroupAlike) {
    const float low = __uint_as_float(mb) * 0x1p-9f;
    uint32_t lower = 0;
#pragma unroll 4
    for (int i = threadIdx.x; i < n; i += 256) lower += v[i] < low;
    lower = row_count<256>(lower, tmp);
    if (mb >= 0x7f800000u) {
      mb = 0x7fc00000u;
    } else if (4 * lower > (uint32_t)n) {               // (zeros count as lower: how many there are is seldom asked)
      uint32_t some = 0;
      for (int i = threadIdx.x; i < n; i += 256) some += v[i] > 0.f;
      some = row_count<256>(some, tmp);
      if (4 * (lower - ((uint32_t)n - some)) > some) mb = 0x7fc00000u;
    }
  }
  if (threadIdx.x == 0) *out = __uint_as_float(mb);
}

__global__ __launch_bounds__(256) void group_max_kernel(GroupMaxes g) {
  __shared__ float tmp[4];
  group_max(g.v[blockIdx.x], g.n[blockIdx.x], g.kind[blockIdx.x], g.out[blockIdx.x], tmp);
}

int split_weights(SplitWeights p, hipStream_t stream) {
  int k = 0, blocks = 0;
  for (int i = 0; i < p.count; ++i) k = std::max(k, p.e[i].k);
  const int ch = k <= 4096 ? 4 : k <= 5120 ? 5 : 8;
  for (int i = 0; i < p.count; ++i) {
    p.e[i].first = blocks;
    blocks += p.e[i].k <= 256 * ch ? (p.e[i].n + 3) / 4 : p.e[i].n;
  }
  if (ch == 4) hipLaunchKernelGGL(split_weights_kernel<4>, dim3(blocks), dim3(256), 0, stream, p);
  else if (ch == 5) hipLaunchKernelGGL(split_weights_kernel<5>, dim3(blocks), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(split_weights_kernel<8>, dim3(blocks), dim3(256), 0, stream, p);
  return check_launch("split_weights");
}

int group_maxes(const GroupMaxes& g, hipStream_t stream) {
  hipLaunchKernelGGL(group_max_kernel, dim3((unsigned)g.count), dim3(256), 0, stream, g);
  return check_launch("group_max");
}

// ---------------------------------------------------------------------------------------------
// LayerNorm fp32 (the arithmetic of layernorm_f32_kernel) written as split rows for the Dense that reads it:
// no fp32 copy of the normalised rows, and no pass to split them. T threads hold a row; MERGE: the 4 waves of a
// workgroup normalise 4 consecutive rows that form one row of the output (the 2x2 merge), with one exponent.
// A row that is wide (row_is_wide) is written as it is, fp32, with a NaN factor.
// Workgroups past the rows take the maxima of `gm` (a layer's output bounds, needed by the launches after this one).
// ---------------------------------------------------------------------------------------------
template <int T, int CH, bool MERGE>
__global__ __launch_bounds__(256) void layernorm_split_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                              const float* __restrict__ beta, f16* __restrict__ y,
                                                              float* __restrict__ inv, int rows, int cols, float eps,
                                                              GroupMaxes gm) {
  static_assert(!MERGE || T == 64, "a wave per merged row");
  __shared__ float tmp[4];
  const int first_max = gridDim.x - gm.count;         // the last workgroups: the layer's output bounds
  if ((int)blockIdx.x >= first_max) {
    const int g = blockIdx.x - first_max;
    return group_max(gm.v[g], gm.n[g], gm.kind[g], gm.out[g], tmp);
  }
  const int t = threadIdx.x % T, row = blockIdx.x * (256 / T) + threadIdx.x / T;
  if (row >= rows) return;                            // (MERGE: rows % 4 == 0, all waves or none)
  const float* xr = x + (int64_t)row * cols;
  f32x4 v[CH];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + T * i) * 4;
    v[i] = c < cols ? *reinterpret_cast<const f32x4*>(xr + c) : f32x4{};
    s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  }
  const float inv_n = 1.0f / (float)cols;
  const float mean = row_sum<T>(s, tmp) * inv_n;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if ((t + T * i) * 4 < cols) {
#pragma unroll
      for (int e = 0; e < 4; ++e) { const float d = v[i][e] - mean; q += d * d; }
    }
  const float rstd = 1.0f / sqrtf(row_sum<T>(q, tmp) * inv_n + eps);
  uint32_t mb = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + T * i) * 4;
    if (c >= cols) break;
    const f32x4 g = *reinterpret_cast<const f32x4*>(gamma + c), b = *reinterpret_cast<const f32x4*>(beta + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[i][e] = (v[i][e] - mean) * rstd * g[e] + b[e];
      mb = max(mb, __float_as_uint(v[i][e]) & 0x7fffffffu);
    }
  }
  if constexpr (T > 64 || MERGE) mb = block_max_bits(mb, tmp);
  else mb = wave_max_bits(mb);
  const float sc = split_scale(__uint_as_float(mb));
  uint32_t small = 0;
#pragma unroll
  for (int i = 0; i < CH; ++i) small += count_small(v[i], sc);
  const bool wide = row_is_wide<MERGE ? 256 : T>(mb, small, v, tmp);
  const int orow = MERGE ? row / 4 : row, ocol = MERGE ? (row & 3) * cols : 0;
  f16* dst = y + (int64_t)orow * 2 * (MERGE ? 4 * cols : cols);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = (t + T * i) * 4;
    if (c >= cols) break;
    if (wide) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(dst) + ocol + c) = v[i];
      continue;
    }
    f16x4 hi, lo;
    split4(v[i], sc, hi, lo);
    store_split_pair(dst, ocol + c, hi, lo, t);
  }
  if (t == 0 && (!MERGE || (row & 3) == 0)) inv[orow] = wide ? __uint_as_float(0x7fc00000u) : 1.0f / sc;
}

// cols a multiple of 64 (32-column groups), at most kSplitMaxK; merge: rows % 4 == 0, cols <= 2048.
int layer_norm_split(const float* x, const float* g, const float* b, void* y, float* inv, int rows, int cols, float eps,
                     bool merge, const GroupMaxes& gm, hipStream_t stream) {
  if (rows == 0) return QVL_OK;
#define QVL_LN_SPLIT(T, CH, MERGE)                                                                                  \
  hipLaunchKernelGGL((layernorm_split_kernel<T, CH, MERGE>), dim3((rows + 256 / T - 1) / (256 / T) + gm.count),     \
                     dim3(256), 0, stream, x, g, b, (f16*)y, inv, rows, cols, eps, gm)
  if (merge) {
    if (cols <= 1024) QVL_LN_SPLIT(64, 4, true);
    else QVL_LN_SPLIT(64, 8, true);
  } else if (cols <= 1024) QVL_LN_SPLIT(64, 4, false);
  else if (cols <= 2048) QVL_LN_SPLIT(64, 8, false);
  else if (cols <= 5120) QVL_LN_SPLIT(256, 5, false);
  else QVL_LN_SPLIT(256, 8, false);
#undef QVL_LN_SPLIT
  return check_launch("layernorm_split");
}

// ---------------------------------------------------------------------------------------------
// GEMM on split rows.
// ---------------------------------------------------------------------------------------------
template <int BM, int BN, int WM, int WN>
struct SplitShape {
  static constexpr int THREADS = 64 * WM * WN;
  static constexpr int TM = BM / WM, TN = BN / WN, MB = TM / 32, NB = TN / 32;
  static constexpr int PASS = THREADS / 8;               // rows one DMA pass covers
  static constexpr int XPT = BM / PASS, WPT = BN / PASS;
  static constexpr int STAGE = (BM + BN) * 64;           // f16 elements of one stage
  static_assert(BM % PASS == 0 && BN % PASS == 0 && TM % 32 == 0 && TN % 32 == 0, "tile shape");
};

// LDS element offset of (row, 16-byte chunk) in 128-byte rows, swizzled as in the bf16 GEMM: the 16 rows
// one clock of a fragment read touches fall on 16 distinct bank groups.
__device__ __forceinline__ int split_lds_off(int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 1) & 7)) << 3); }

// y[m, n..n+3] = epi(v + bias), v already scaled back; OUTS: as split rows, scaled by the exponent of p.ybound.
template <int EPI, bool OUTS>
__device__ __forceinline__ void split_store4(const GemmSplitParams& p, int m, int n, f32x4 v, const f32x4& bias) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] += bias[e];
    if constexpr (EPI == kEpiBiasGelu) v[e] = gelu_tanh(v[e]);
  }
  if constexpr (EPI == kEpiBiasResidual) v += *reinterpret_cast<const f32x4*>(p.res + (int64_t)m * p.ldr + n);
  if constexpr (OUTS) {
    const float bound = *p.ybound;
    if (bound != bound) {                                // (kGroupAlike: fp32 rows)
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.ys) + (int64_t)m * p.N + n) = v;
      return;
    }
    f16x4 hi, lo;
    split4(v, split_scale(bound), hi, lo);
    store_split4(p.ys + (int64_t)m * 2 * p.N, n, hi, lo);
  } else {
    *reinterpret_cast<f32x4*>(p.y + (int64_t)m * p.ldc + n) = v;
  }
}

// The factor of row m of x: its own, or one for every row from a bound on |x|. NaN: the row goes by fp32.
__device__ __forceinline__ float split_row_factor(const GemmSplitParams& p, int m) {
  if (p.sx) return p.sx[m];
  const float b = *p.xbound;
  return b == b ? 1.0f / split_scale(b) : b;
}

// acc 2^-(ex + ew): the smaller factor first, so that neither step leaves the range unless the result does
// (sums below 1 in the scaled domain are rounding noise of products of up to 2^30).
__device__ __forceinline__ f32x4 split_unscale(f32x4 v, float sx, const f32x4& sw) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = v[e] * fminf(sx, sw[e]) * fmaxf(sx, sw[e]);
  return v;
}

__device__ __forceinline__ bool any_nan(const f32x4& v) { return v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3]; }

// Whether outputs (m, n .. n + 3) come from the fp32 operands.
__device__ __forceinline__ bool by_fp32(const GemmSplitParams& p, int m, int n) {
  const float sx = split_row_factor(p, m);
  return sx != sx || any_nan(*reinterpret_cast<const f32x4*>(p.sw + n));
}

// Rows of x and columns of w whose factor is NaN (row_is_wide): their outputs come from the fp32 operands, on
// v_mfma_f32_32x32x2_f32, 32 tokens (from m1) x 32 features (from n1) of one wave at a time over k in [k0, k1). x comes
// from xf, or without it from p.x: a row with a NaN factor lies there as fp32, any other as a split row. Lane l32 holds
// row l32 of both, hh the k's half of 8. Rare: no LDS, one step of 32 k loaded ahead. Every row wide: 784 x 4096 x 1024
// 158 us (fp32 MFMA kernel 88), 4096 x 4096 x 1024 569 (300).
__device__ __forceinline__ f32x16 split_fp32_block(const GemmSplitParams& p, int m1, int n1, int k0, int k1, int l32, int hh) {
  const int m = min(m1 + l32, p.M - 1);
  const float* w = p.wf + (int64_t)min(n1 + l32, p.N - 1) * p.K + 4 * hh;
  const float fx = split_row_factor(p, m);
  const float* xf = p.xf ? p.xf + (int64_t)m * p.ldx + 4 * hh
                         : fx != fx ? reinterpret_cast<const float*>(p.x) + (int64_t)m * p.K + 4 * hh : nullptr;
  const f16* xs = p.x + (int64_t)m * 2 * p.K + 4 * hh;
  struct Step { f32x4 w[4], x[4]; };
  auto load = [&](int k, Step& s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s.w[i] = *reinterpret_cast<const f32x4*>(w + k + 8 * i);
      if (xf) {
        s.x[i] = *reinterpret_cast<const f32x4*>(xf + k + 8 * i);
      } else {
        const f16* g = xs + (k >> 5) * 64 + 8 * i;
        const f16x4 hi = *reinterpret_cast<const f16x4*>(g), lo = *reinterpret_cast<const f16x4*>(g + 32);
#pragma unroll
        for (int e = 0; e < 4; ++e) s.x[i][e] = ((float)hi[e] + (float)lo[e]) * fx;
      }
    }
  };
  f32x16 acc = {};
  Step cur, nxt;
  load(k0, cur);
#pragma unroll 1
  for (int k = k0; k < k1; k += 32) {
    if (k + 32 < k1) load(k + 32, nxt);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(cur.w[i][e], cur.x[i][e], acc, 0, 0, 0);
    cur = nxt;
  }
  return acc;
}

template <int BM, int BN, int WM, int WN, int NS, int EPI, bool OUTS>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_split_kernel(GemmSplitParams p) {
  using S = SplitShape<BM, BN, WM, WN>;
  extern __shared__ __attribute__((aligned(16))) f16 smem_h[];   // [NS][BM + BN][64]
  const int tiles_n = (p.N + BN - 1) / BN, tiles_m = (p.M + BM - 1) / BM;
  const int tiles = tiles_m * tiles_n;
  // split-K: the units of one K part are consecutive, so one XCD's units share operand rows
  const int unit = xcd_remap(blockIdx.x, tiles * p.split);
  const int tile = unit % tiles, part_i = unit / tiles;
  int tm, tn;
  tile_coords(tile, tiles_m, tiles_n, p.group_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int l32 = lane & 31, hh = lane >> 5;

  // Operand DMA, as in the bf16 GEMM: one wave instruction fills 8 LDS rows of 128 bytes; rows past M or N
  // lie past the resource's range and arrive as zeros.
  const int lrow = wave * 8 + (lane >> 3);
  const int lch = (lane & 7) ^ ((lrow >> 1) & 7);
  const uint32_t rowb = (uint32_t)p.K * 4;
  const uint32_t xv = (uint32_t)(m0 + lrow) * rowb + lch * 16, wv = (uint32_t)(n0 + lrow) * rowb + lch * 16;
  const u32x4 rx = rsrc_words(p.x, (uint32_t)p.M * rowb), rw = rsrc_words(p.w, (uint32_t)p.N * rowb);
  const uint32_t lds_base = lds_addr_of(smem_h);
  auto dma_stage = [&](int kt, int stage) {
    const uint32_t xa = lds_base + stage * S::STAGE * 2, wa = xa + BM * 128;
#pragma unroll
    for (int i = 0; i < S::XPT; ++i)
      dma16(rx, xv, (uint32_t)(i * S::PASS) * rowb + kt * 128, xa + (i * S::PASS + wave * 8) * 128);
#pragma unroll
    for (int i = 0; i < S::WPT; ++i)
      dma16(rw, wv, (uint32_t)(i * S::PASS) * rowb + kt * 128, wa + (i * S::PASS + wave * 8) * 128);
  };
  const int KT = p.K / 32;
  const int kt0 = part_i * KT / p.split, kt1 = (part_i + 1) * KT / p.split;
  // Whether a row or column of the wave's sub-tile goes by fp32: loaded here, where the products hide it.
  const int mw = m0 + wm * S::TM, nw = n0 + wn * S::TN;
  float marks = p.sx ? 0.f : *p.xbound;
#pragma unroll
  for (int r = 0; r < S::TM; r += 64)
    if (p.sx && r + lane < S::TM && mw + r + lane < p.M) marks += p.sx[mw + r + lane];
#pragma unroll
  for (int c = 0; c < S::TN; c += 64)
    if (c + lane < S::TN && nw + c + lane < p.N) marks += p.sw[nw + c + lane];
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (kt0 + s < kt1) dma_stage(kt0 + s, s);

  // The hi . hi products and (where the registers hold both) the 2^-11 smaller cross products in accumulators of
  // their own: the large sums then round K / 16 times and not 3 K / 16.
  constexpr bool TWO = S::NB * S::MB <= 4;
  f32x16 acc[S::NB][S::MB], low[TWO ? S::NB : 1][TWO ? S::MB : 1];
#pragma unroll
  for (int a = 0; a < S::NB; ++a)
#pragma unroll
    for (int b = 0; b < S::MB; ++b) {
      acc[a][b] = f32x16{};
      if constexpr (TWO) low[a][b] = f32x16{};
    }

  // Half step h of a k-step (16 of its 32 values): hi fragments in chunks 2h + hh, lo in 4 + 2h + hh.
  constexpr int NFR = S::NB + S::MB;
  f16x8 fh[2][NFR], fl[2][NFR];
  auto read_frags = [&](const f16* xs, int h, int slot) {
    const f16* ws = xs + BM * 64;
    const int ch = 2 * h + hh;
#pragma unroll
    for (int a = 0; a < S::NB; ++a) {
      fh[slot][a] = *reinterpret_cast<const f16x8*>(ws + split_lds_off(wn * S::TN + a * 32 + l32, ch));
      fl[slot][a] = *reinterpret_cast<const f16x8*>(ws + split_lds_off(wn * S::TN + a * 32 + l32, ch + 4));
    }
#pragma unroll
    for (int b = 0; b < S::MB; ++b) {
      fh[slot][S::NB + b] = *reinterpret_cast<const f16x8*>(xs + split_lds_off(wm * S::TM + b * 32 + l32, ch));
      fl[slot][S::NB + b] = *reinterpret_cast<const f16x8*>(xs + split_lds_off(wm * S::TM + b * 32 + l32, ch + 4));
    }
  };
  auto mfmas = [&](int slot) {
    const f16x8 *wh = fh[slot], *wl = fl[slot], *xh = fh[slot] + S::NB, *xl = fl[slot] + S::NB;
    auto products = [&](const f16x8* w, const f16x8* x, auto& sum) {
#pragma unroll
      for (int a = 0; a < S::NB; ++a)
#pragma unroll
        for (int b = 0; b < S::MB; ++b) sum[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[a], x[b], sum[a][b], 0, 0, 0);
    };
    if constexpr (TWO) {
      products(wl, xh, low);
      products(wh, xl, low);
    } else {
      products(wl, xh, acc);
      products(wh, xl, acc);
    }
    products(wh, xh, acc);
  };
  constexpr int NMF = 3 * S::NB * S::MB;
  auto wait_stage = [&](int kt) {   // every stage up to kt has landed (later ones may be in flight)
    if (NS == 3 && kt + 1 < kt1) asm volatile("s_waitcnt vmcnt(%0)" :: "I"(S::XPT + S::WPT) : "memory");
    else wait_dma();
  };

  wait_stage(kt0);
  __syncthreads();
  read_frags(smem_h, 0, 0);
  int cur = 0;
  for (int kt = kt0; kt < kt1; ++kt) {
    const f16* xs = smem_h + cur * S::STAGE;
    const bool more = kt + 1 < kt1;
    const int nxt = cur + 1 == NS ? 0 : cur + 1;
    if (kt + NS - 1 < kt1) dma_stage(kt + NS - 1, NS == 3 ? (cur == 0 ? 2 : cur - 1) : nxt);
    read_frags(xs, 1, 1);
    mfmas(0);
#pragma unroll
    for (int i = 0; i < NMF; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (i < 2 * NFR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    mfmas(1);
    wait_stage(kt + 1);
    __syncthreads();
    if (more) read_frags(smem_h + nxt * S::STAGE, 0, 0);
    cur = nxt;
  }

  if constexpr (TWO) {
#pragma unroll
    for (int a = 0; a < S::NB; ++a)
#pragma unroll
      for (int b = 0; b < S::MB; ++b) acc[a][b] += low[a][b];
  }

  // Epilogue. Accumulator (a, b), register 4 g + e: token 32 b + l32, feature 32 a + 8 g + 4 hh + e of the
  // wave's sub-tile. Each wave turns 32 tokens at a time through its own piece of the free ring (16-byte
  // chunks XOR-swizzled by row), so that stores go out as whole TN-wide row pieces; no barrier is needed
  // within a wave. A K part stores its raw sums.
  constexpr int CH = S::TN / 4, RPI = 64 / CH;            // 16-byte chunks of a row, rows one read covers
  float* stage = reinterpret_cast<float*>(smem_h) + wave * 32 * S::TN;
  static_assert(WM * WN * 32 * S::TN * 4 <= NS * S::STAGE * 2 && 64 % CH == 0, "epilogue staging");
  const int c = lane % CH, n = n0 + wn * S::TN + 4 * c;
  const bool nok = n < p.N;
  f32x4 sw = {}, bias = {};
  if (p.split == 1 && nok) {
    sw = *reinterpret_cast<const f32x4*>(p.sw + n);
    bias = *reinterpret_cast<const f32x4*>(p.bias + n);
  }
  const bool w_nan = any_nan(sw), marked = __builtin_amdgcn_ballot_w64(marks != marks) != 0;
  const int64_t npad = (int64_t)tiles_n * BN;
#pragma unroll
  for (int b = 0; b < S::MB; ++b) {
#pragma unroll
    for (int a = 0; a < S::NB; ++a)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int cc = 8 * a + 2 * g + hh;
        *reinterpret_cast<f32x4*>(stage + l32 * S::TN + ((cc ^ (l32 % CH)) << 2)) =
            f32x4{acc[a][b][4 * g], acc[a][b][4 * g + 1], acc[a][b][4 * g + 2], acc[a][b][4 * g + 3]};
      }
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
      const int r = i * RPI + lane / CH, m = m0 + wm * S::TM + 32 * b + r;
      const f32x4 v = *reinterpret_cast<const f32x4*>(stage + r * S::TN + ((c ^ (r % CH)) << 2));
      if (m >= p.M) continue;
      if (p.split > 1) {
        if (!marked || !nok || !by_fp32(p, m, n))
          *reinterpret_cast<f32x4*>(p.part + ((int64_t)part_i * p.M + m) * npad + n) = v;
      } else if (nok) {
        const float sx = split_row_factor(p, m);
        if (sx == sx && !w_nan) split_store4<EPI, OUTS>(p, m, n, split_unscale(v, sx, sw), bias);
      }
    }
  }
  if (!marked) return;
#pragma unroll 1
  for (int blk = 0; blk < S::NB * S::MB; ++blk) {
    const int m1 = mw + 32 * (blk % S::MB), n1 = nw + 32 * (blk / S::MB);
    const int at = hh ? n1 + l32 : m1 + l32;
    const float mark = hh ? (at < p.N ? p.sw[at] : 0.f) : (at < p.M ? split_row_factor(p, at) : 0.f);
    if (!__builtin_amdgcn_ballot_w64(mark != mark)) continue;
    const f32x16 v = split_fp32_block(p, m1, n1, kt0 * 32, kt1 * 32, l32, hh);
#pragma unroll
    for (int g = 0; g < 4; ++g)                       // (through LDS as above, 8 chunks of 4 features a row)
      *reinterpret_cast<f32x4*>(stage + l32 * 32 + (((2 * g + hh) ^ (l32 & 7)) << 2)) =
          f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + (lane >> 3), m2 = m1 + r, n2 = n1 + 4 * (lane & 7);
      const f32x4 o = *reinterpret_cast<const f32x4*>(stage + r * 32 + (((lane & 7) ^ (r & 7)) << 2));
      if (m2 >= p.M || n2 >= p.N || !by_fp32(p, m2, n2)) continue;
      if (p.split > 1) *reinterpret_cast<f32x4*>(p.part + ((int64_t)part_i * p.M + m2) * npad + n2) = o;
      else split_store4<EPI, OUTS>(p, m2, n2, o, *reinterpret_cast<const f32x4*>(p.bias + n2));
    }
  }
}

// Sums the K parts in order and applies the epilogue, one thread per 4 consecutive outputs.
template <int EPI, bool OUTS>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(GemmSplitParams p, int64_t npad) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x, quads = (int64_t)p.M * (p.N / 4);
  if (q >= quads) return;
  const int m = (int)(q / (p.N / 4)), n = (int)(q % (p.N / 4)) * 4;
  const float* src = p.part + (int64_t)m * npad + n;
  const int64_t stride = (int64_t)p.M * npad;
  f32x4 v = *reinterpret_cast<const f32x4*>(src);
  for (int s = 1; s < p.split; ++s) v += *reinterpret_cast<const f32x4*>(src + s * stride);
  const f32x4 sw = *reinterpret_cast<const f32x4*>(p.sw + n), bias = *reinterpret_cast<const f32x4*>(p.bias + n);
  const float sx = split_row_factor(p, m);
  if (sx == sx && !any_nan(sw)) v = split_unscale(v, sx, sw);   // (else the parts are fp32 sums)
  split_store4<EPI, OUTS>(p, m, n, v, bias);
}

template <int BM, int BN, int WM, int WN, int NS, int EPI, bool OUTS>
static int launch_gemm_split(GemmSplitParams p, int split, hipStream_t stream) {
  using S = SplitShape<BM, BN, WM, WN>;
  constexpr int lds = NS * S::STAGE * 2;
  static_assert(lds <= 163840, "LDS budget");
  static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_split_kernel<BM, BN, WM, WN, NS, EPI, OUTS>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return set_error(QVL_ERR_LAUNCH, "gemm_split: cannot reserve %d bytes of LDS", lds);
  const int tiles_n = (p.N + BN - 1) / BN, tiles = ((p.M + BM - 1) / BM) * tiles_n;
  const int64_t npad = (int64_t)tiles_n * BN;
  p.split = split;
  p.group_n = std::min(4, tiles_n);
  hipLaunchKernelGGL((gemm_split_kernel<BM, BN, WM, WN, NS, EPI, OUTS>), dim3(tiles * p.split), dim3(S::THREADS), lds, stream, p);
  int rc = check_launch("gemm_split");
  if (rc || p.split == 1) return rc;
  const int64_t blocks = ((int64_t)p.M * (p.N / 4) + 255) / 256;
  hipLaunchKernelGGL((gemm_split_reduce_kernel<EPI, OUTS>), dim3((unsigned)blocks), dim3(256), 0, stream, p, npad);
  return check_launch("gemm_split_reduce");
}

// Tile plan of the calling thread (qvl_set_f32_plan): 0 = the rules below, 1..4 = kSplitTiles[tile - 1],
// 5 = the fp32 MFMA kernel, 6 = kSplitTiles[4].
static thread_local int t_f32_plan = 0;

int gemm_f32_set_plan(int tile) {
  if (tile < 0 || tile > 6) return set_error(QVL_ERR_INVALID_ARG, "f32 plan: tile=%d (0..6)", tile);
  t_f32_plan = tile;
  return QVL_OK;
}

// Tile and K split by a cost model of the launch, in microseconds: start + rounds * (K / split * per_k +
// per_tile), rounds = workgroups per CU, where a last partial round costs its share of the CUs but at least
// `part` of a round, and a launch of less than one round at least `one`; split-K adds its partials' traffic at
// part_rate bytes/us. Fitted to 68 shapes from 49 to 8192 rows with 1 to 8 K parts (MI355X, every tile and part count
// that fits): what it picks is 1.2 % slower than the best measured choice on average, 13 % at worst. For instance
// 8192 x 4096 x 1024 runs in 189 us (1.09 PFLOP/s of f16 products; 609 us on v_mfma_f32_32x32x2_f32), 8192 x 1024 x
// 4096 in 181 us (365 us).
// The small tiles are bound by the operands' way into LDS, not by the matrix units (64x128: 24 KB per 0.4 us and CU),
// so 128x128 tiles, 2/3 of that traffic, win where one round of them covers most CUs; and eight waves a workgroup, each
// with half the DMA to issue, beat four on the same tile. With the split pass: 784 x 3072 x 1024 44.8 -> 37.4 us, 784 x
// 4096 x 1024 46.6 -> 38.9, 1024 x 1024 x 4096 51.3 -> 45.5 (128x128 on four waves: 43.6, 44.1, 47.2); 64x128 on eight
// waves against four: 2048 x 1024 x 1024 29.1 against 32.6, 400 x 4096 x 1024 29.5 against 32.5, 4096 x 1024 x 1024
// 39.8 against 42.4.
struct SplitTile { int bm, bn, slots; double start, per_k, per_tile, part, one, part_rate; };   // slots: workgroups a CU holds
constexpr SplitTile kSplitTiles[] = {
    {64, 128, 3, 13.2, 12.7 / 1024, 0.0, 0.57, 1.49, 34.1e6},     // 4 waves, two-stage ring, 48 KB
    {64, 128, 2, 9.7, 11.8 / 1024, 1.6, 0.65, 0.96, 13.3e6},      // 8 waves, three stages, 72 KB
    {128, 256, 1, 4.8, 38.9 / 1024, 11.3, 0.80, 0.06, 21.6e6},    // 8 waves, three stages, 144 KB
    {256, 256, 1, 5.3, 80.1 / 1024, 11.8, 0.78, 0.22, 14.5e6},    // 8 waves, two stages, 128 KB
    {128, 128, 1, 3.2, 19.9 / 1024, 9.5, 0.83, 0.89, 10.5e6},     // 8 waves, three stages, 96 KB
};

static double split_cost(const SplitTile& t, const GemmSplitParams& p, int cus, int split) {
  const int units = ((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn) * split;
  const int tail = units % cus;
  double rounds = units / cus + (tail ? std::max((double)tail / cus, t.part) : 0.0);
  if (units < cus) rounds = std::max(rounds, t.one);
  return t.start + rounds * (p.K / (double)split * t.per_k + t.per_tile) +
         (split > 1 ? 8.0 * split * p.M * p.N / t.part_rate : 0.0);
}

template <int EPI, bool OUTS = false>
static int dispatch_gemm_split(const GemmSplitParams& p, hipStream_t stream) {
  const int cus = gemm_device_cus();
  int pick = 0, split = 1;
  double best = 1e30;
  const int only = t_f32_plan == 6 ? 4 : t_f32_plan >= 1 && t_f32_plan <= 4 ? t_f32_plan - 1 : -1;
  for (int i = 0; i < 5; ++i) {
    if (only >= 0 && i != only) continue;
    // (256x256 tiles add every product to one accumulator, 3 K / 16 roundings: nearer to float64 than the fp32
    // MFMA kernel where that does not split K, which is where its 128x128 tiles outnumber the CUs)
    if (i == 3 && only < 0 && ((p.M + 127) / 128) * ((p.N + 127) / 128) <= cus) continue;
    const SplitTile& t = kSplitTiles[i];
    const int tiles = ((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn);
    const int64_t npad = round_up(p.N, t.bn);
    for (int s = 1; s <= std::min(8, p.K / 32 / 4) || s == 1; ++s) {
      if (s > 1 && (!p.part || (int64_t)s * p.M * npad > p.part_elems || tiles * s > t.slots * cus)) break;
      const double c = split_cost(t, p, cus, s);
      if (c < best) { best = c; pick = i; split = s; }
    }
  }
  switch (pick) {
    case 0: return launch_gemm_split<64, 128, 2, 2, 2, EPI, OUTS>(p, split, stream);
    case 1: return launch_gemm_split<64, 128, 2, 4, 3, EPI, OUTS>(p, split, stream);
    case 2: return launch_gemm_split<128, 256, 2, 4, 3, EPI, OUTS>(p, split, stream);
    case 4: return launch_gemm_split<128, 128, 2, 4, 3, EPI, OUTS>(p, split, stream);
    default: return launch_gemm_split<256, 256, 4, 2, 2, EPI, OUTS>(p, split, stream);
  }
}

int gemm_split(const GemmSplitParams& p, int epi, hipStream_t stream) {
  if (p.ys) {
    if (epi != kEpiBiasGelu || p.N % 32) return set_error(QVL_ERR_INVALID_ARG, "gemm_split: split outputs need GELU, N %% 32 == 0");
    return dispatch_gemm_split<kEpiBiasGelu, true>(p, stream);
  }
  switch (epi) {
    case kEpiBias: return dispatch_gemm_split<kEpiBias>(p, stream);
    case kEpiBiasGelu: return dispatch_gemm_split<kEpiBiasGelu>(p, stream);
    case kEpiBiasResidual: return dispatch_gemm_split<kEpiBiasResidual>(p, stream);
  }
  return set_error(QVL_ERR_INVALID_ARG, "gemm_split: epilogue %d", epi);
}

// Splits x [M, K] and w [N, K] into the front of the workspace (g.part) and runs the Dense on them; what is
// left of the workspace takes split-K partials.
static int64_t split_scales(int64_t M, int64_t N) { return round_up(M, 4) + round_up(N, 4); }

// Whether a Dense whose operands are both fp32 runs on split rows: the workspace holds them, and splitting the
// weights (N K values, read and written for this one call) pays. It does not for a few rows over many short
// ones, where the fp32 MFMA kernel's time is one tile's K loop: 32 rows x 4096 x 1024 20.0 us against 20.8
// (1: 17.9 against 23.1, 49: 21.7 against 22.2, 100: 25.8 against 24.0), 32 x 3072 x 1024 19.5 against 20.6;
// but 32 x 1024 x 1024 18.2 against 14.9, 32 x 1024 x 4096 51.2 against 25.8, 32 x 4352 x 1152 30.9 against 21.8.
bool gemm_f32_use_split(const GemmF32Params& g) {
  if (t_f32_plan == 5 || !g.part || g.K > kSplitMaxK ||
      g.part_elems < split_scales(g.M, g.N) + ((int64_t)g.M + g.N) * g.K)
    return false;
  return t_f32_plan != 0 || g.M > 64 || g.K > 1024 || g.N <= 2 * g.K;
}

int gemm_f32_split(const GemmF32Params& g, int epi, hipStream_t stream) {
  const int64_t M = g.M, N = g.N, K = g.K, head = split_scales(M, N), used = head + (M + N) * K;
  SplitRowsParams r{};
  r.src[0] = g.x; r.ld[0] = g.lda; r.dst[0] = (f16*)(g.part + head); r.inv[0] = g.part; r.rows[0] = g.M;
  r.src[1] = g.w; r.ld[1] = g.ldw; r.dst[1] = r.dst[0] + 2 * M * K; r.inv[1] = g.part + round_up(M, 4); r.rows[1] = g.N;
  r.K = g.K;
  QVL_TRY_RC(split_rows(r, stream));
  GemmSplitParams p{};
  p.x = r.dst[0]; p.sx = r.inv[0]; p.w = r.dst[1]; p.sw = r.inv[1];
  p.bias = g.bias; p.res = g.res; p.ldr = g.ldr; p.y = g.y; p.ldc = g.ldc;
  p.M = g.M; p.N = g.N; p.K = g.K;
  p.xf = g.x; p.ldx = g.lda; p.wf = g.w;
  p.part = g.part + used;          // (K is a multiple of 64: `used` is a multiple of 4)
  p.part_elems = g.part_elems - used;
  return gemm_split(p, epi, stream);
}

int split_rows_f32(const float* x, int64_t ldx, void* out, float* inv, int rows, const float* w, void* w_out, float* w_inv,
                   int w_rows, int k, hipStream_t stream) {
  SplitRowsParams r{};
  r.src[0] = x; r.ld[0] = ldx; r.dst[0] = (f16*)out; r.inv[0] = inv; r.rows[0] = rows;
  r.src[1] = w; r.ld[1] = k; r.dst[1] = (f16*)w_out; r.inv[1] = w_inv; r.rows[1] = w_rows;
  r.K = k;
  return rows ? split_rows(r, stream) : QVL_OK;
}

}  // namespace qvl
