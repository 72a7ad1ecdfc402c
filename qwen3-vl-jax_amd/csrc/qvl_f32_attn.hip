// fp32 varlen attention (model.py:569-600 in the fp32 dtype) on the f16 matrix cores, for the fp32 tower with
// split weights: q, k, v and the probabilities are two f16 terms each (hi + lo, 22 bits of a power-of-two
// multiple), every product three v_mfma_f32_32x32x16_f16 into fp32 accumulators, softmax in fp32. The exponents
// of q, k and v are one per layer, from the bounds on the qkv Dense's outputs, so nothing has to be searched
// for a maximum first; values down to 2^-17 of the bound keep 22 bits.
//
// Operand layouts (Np = tokens rounded up to 64; rows [n_tokens, Np) zero):
//   Q, K [H][Np][C] 16-byte chunks: per 16 dims (KS = ceil(hd / 16) groups) [16 hi | 16 lo], dims past hd zero,
//     and one unread chunk: C = 4 KS + 1 is odd, so the 16 rows one clock of an LDS fragment read touches fall
//     on 16 distinct bank groups with no swizzle.
//   V^T [H][hd][Np / 32][32 hi | 32 lo]: 128 bytes per 32 keys, keys at vt_pos within 16 (each lane's 8 PV
//     keys are one 16-byte chunk).
#include <math.h>

#include <type_traits>

#include "qvl_split.h"

namespace qvl {

template <int HD>
struct SplitAttn {
  static constexpr int KS = (HD + 15) / 16, C = 4 * KS + 1;     // 16-dim steps, 16-byte chunks of a Q / K row
  static constexpr int NDB = (HD + 31) / 32;                    // 32-row blocks of O^T
  static constexpr int KINSTR = (32 * C * 16 + 1023) / 1024;    // 1 KB DMA instructions of a 32-key K tile
  static constexpr int VINSTR = HD / 8;                         // ... of the V^T tile (8 rows of 128 bytes each)
  static constexpr int KBYTES = KINSTR * 1024, VBYTES = NDB * 32 * 128, STAGE = KBYTES + VBYTES;
  static_assert(HD % 8 == 0, "head_dim");
};

// ---------------------------------------------------------------------------------------------
// Rotary + relayout: the qkv Dense's fp32 rows -> the operands above. x * cos + rotate_half(x) * sin, each product
// and the sum rounded (model.py:579-582). A workgroup takes 64 tokens of one head: 16-byte reads, q / k written in
// 8-byte pieces of a 32-byte run, V turned through LDS. HBM bound: 8192 tokens x 16 heads 45 us (62 us for
// attn_relayout_f32_kernel), 4.6 TB/s.
// ---------------------------------------------------------------------------------------------
template <int HD>
__global__ __launch_bounds__(256) void attn_relayout_split_kernel(const float* __restrict__ qkv, int64_t ld, int D,
                                                                  const f32x2* __restrict__ cs,
                                                                  const float* __restrict__ bound, int N, int Np,
                                                                  f16* __restrict__ Qo, f16* __restrict__ Ko,
                                                                  f16* __restrict__ Vo) {
#pragma clang fp contract(off)
  using A = SplitAttn<HD>;
  constexpr int G = HD / 8, HALF = HD / 2, PAD = A::KS * 16 - HD;   // 4-dim pair groups, zero dims
  constexpr int VS = 72;                                            // LDS row of a V^T row's 64 keys
  __shared__ __attribute__((aligned(16))) f16 tv[2][HD * VS];
  const int n0 = blockIdx.x * 64, head = blockIdx.y, tid = threadIdx.x;
  const float sq = split_scale(1.4143f * bound[0]), sk = split_scale(1.4143f * bound[1]), sv = split_scale(bound[2]);
  for (int i = tid; i < 64 * G; i += 256) {
    const int t = i / G, d = (i % G) * 4, n = n0 + t;
    f32x4 q1{}, q2{}, k1{}, k2{};
    if (n < N) {
      const float* row = qkv + (int64_t)n * ld + head * HD + d;
      const f32x4 c01 = *reinterpret_cast<const f32x4*>(cs + (int64_t)n * HALF + d);
      const f32x4 c23 = *reinterpret_cast<const f32x4*>(cs + (int64_t)n * HALF + d + 2);
      const f32x4 qa = *reinterpret_cast<const f32x4*>(row), qb = *reinterpret_cast<const f32x4*>(row + HALF);
      const f32x4 ka = *reinterpret_cast<const f32x4*>(row + D), kb = *reinterpret_cast<const f32x4*>(row + D + HALF);
      const float co[4] = {c01[0], c01[2], c23[0], c23[2]}, si[4] = {c01[1], c01[3], c23[1], c23[3]};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        q1[e] = qa[e] * co[e] + (-qb[e]) * si[e];
        q2[e] = qb[e] * co[e] + qa[e] * si[e];
        k1[e] = ka[e] * co[e] + (-kb[e]) * si[e];
        k2[e] = kb[e] * co[e] + ka[e] * si[e];
      }
    }
    const int64_t r = ((int64_t)head * Np + n) * (A::C * 8);
    auto put = [&](f16* out, int dim, const f32x4& v, float s) {
      f16x4 hi, lo;
      split4(v, s, hi, lo);
      f16* g = out + r + (dim >> 4) * 32 + (dim & 15);
      *reinterpret_cast<f16x4*>(g) = hi;
      *reinterpret_cast<f16x4*>(g + 16) = lo;
    };
    put(Qo, d, q1, sq);
    put(Qo, d + HALF, q2, sq);
    put(Ko, d, k1, sk);
    put(Ko, d + HALF, k2, sk);
  }
  if constexpr (PAD > 0) {
    for (int i = tid; i < 64 * (PAD / 4); i += 256) {
      const int t = i / (PAD / 4), d = HD + (i % (PAD / 4)) * 4;
      const int64_t r = ((int64_t)head * Np + n0 + t) * (A::C * 8) + (d >> 4) * 32 + (d & 15);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        *reinterpret_cast<f16x4*>(Qo + r + 16 * p) = f16x4{};
        *reinterpret_cast<f16x4*>(Ko + r + 16 * p) = f16x4{};
      }
    }
  }
  for (int i = tid; i < 64 * (HD / 4); i += 256) {
    const int t = i / (HD / 4), d = (i % (HD / 4)) * 4, n = n0 + t;
    const f32x4 v = n < N ? *reinterpret_cast<const f32x4*>(qkv + (int64_t)n * ld + 2 * D + head * HD + d) : f32x4{};
    f16x4 hi, lo;
    split4(v, sv, hi, lo);
    const int p = vt_pos(t);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      tv[0][(d + e) * VS + p] = hi[e];
      tv[1][(d + e) * VS + p] = lo[e];
    }
  }
  __syncthreads();
  for (int i = tid; i < HD * 16; i += 256) {
    const int d = i >> 4, c = i & 15, tile = c >> 3, plane = (c >> 2) & 1, k8 = (c & 3) * 8;   // 16 chunks: 2 tiles x 128 bytes
    *reinterpret_cast<f16x8*>(Vo + ((int64_t)head * HD + d) * 2 * Np + n0 * 2 + c * 8) =
        *reinterpret_cast<const f16x8*>(&tv[plane][d * VS + tile * 32 + k8]);
  }
}

// ---------------------------------------------------------------------------------------------
// The attention kernel: a workgroup of 4 waves takes one work item (128 queries of one segment and head), each wave
// 32 queries; key tiles of 32 by LDS DMA, two stages. S^T = K Q^T, so a lane holds one query and 16 keys; P feeds
// the PV product from registers as its B operand. Online softmax whose shift moves only when a tile's maximum
// passes it by more than 4 (log2 units): P carries a factor 2^10, so it stays within f16 and its smaller terms keep
// their bits. Items past n_whole are key parts (as in the other attention kernels). Bound by its matrix and VALU
// issue together: 24 MFMAs (768 cycles) and about 150 VALU instructions per tile and wave. MI355X, 16 heads, against
// attn_fwd_f32_kernel: 8 x 1024 tokens x 64 358 -> 116 us, 1404 tokens x 72 128 -> 45 us, 784 x 64 (key parts) 42 ->
// 18 us; error against float64 5.9e-7 -> 3.8e-7 at 1024 keys, 1.5e-6 -> 9.8e-7 at 7056.
// ---------------------------------------------------------------------------------------------
constexpr float kPScale = 1024.0f, kLazy = 4.0f;

template <int HD>
__global__ __launch_bounds__(256, 3) void attn_fwd_split_kernel(const f16* __restrict__ Q, const f16* __restrict__ K,
                                                                const f16* __restrict__ Vt, const int* __restrict__ items,
                                                                const float* __restrict__ bound, int Np, float qscale,
                                                                f16* __restrict__ O, int D, int n_whole,
                                                                float* __restrict__ part) {
  using A = SplitAttn<HD>;
  __shared__ __attribute__((aligned(16))) char smem_a[2 * A::STAGE];
  const int item = blockIdx.x;
  const int seg_s = items[4 * item], seg_e = items[4 * item + 1], q0 = items[4 * item + 2];
  const int hraw = items[4 * item + 3];
  const int head = hraw & kAttnHeadMask;
  const int part_i = (hraw >> kAttnSplitShift) & 0xff, parts = (hraw >> kAttnPartsShift) & 0xff;
  if (seg_e <= seg_s || (parts && (!part || item < n_whole))) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;

  const size_t qk_bytes = (size_t)Np * A::C * 16, v_bytes = (size_t)HD * Np * 4;
  const u32x4 rk = rsrc_words((const char*)K + head * qk_bytes, (uint32_t)qk_bytes);
  const u32x4 rv = rsrc_words((const char*)Vt + head * v_bytes, (uint32_t)v_bytes);
  const uint32_t k_lane = lane * 16;
  const int vr = lane >> 3;      // V^T instruction i fills rows [8 i, 8 i + 8): lane j row 8 i + j / 8, swizzled chunk
  const uint32_t v_lane[2] = {(uint32_t)(vr * Np * 4 + (((lane & 7) ^ ((vr >> 1) & 7)) << 4)),
                              (uint32_t)(vr * Np * 4 + (((lane & 7) ^ (((vr >> 1) + 4) & 7)) << 4))};
  const uint32_t lds0 = lds_addr_of(smem_a);
  auto dma_tile = [&](int kb, int stage) {
    const uint32_t kl = lds0 + stage * A::STAGE, vl = kl + A::KBYTES;
#pragma unroll
    for (int j = 0; j < (A::KINSTR + A::VINSTR + 3) / 4; ++j) {
      const int n = wave + 4 * j;            // wave-uniform
      if (n < A::KINSTR) {
        dma16(rk, k_lane, (uint32_t)(kb * A::C * 16 + n * 1024), kl + n * 1024);
      } else if (n < A::KINSTR + A::VINSTR) {
        const int i = n - A::KINSTR;
        dma16(rv, v_lane[i & 1], (uint32_t)(8 * i * Np * 4 + kb * 4), vl + i * 1024);
      }
    }
  };

  const int qrow = q0 + wave * 32 + l32;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc((const char*)Q + head * qk_bytes, (uint32_t)qk_bytes);
  f16x8 qh[A::KS], ql[A::KS];
#pragma unroll
  for (int ks = 0; ks < A::KS; ++ks) {
    qh[ks] = __builtin_bit_cast(f16x8, buf_load16(rq, (uint32_t)(qrow * A::C + 4 * ks + hh) * 16));
    ql[ks] = __builtin_bit_cast(f16x8, buf_load16(rq, (uint32_t)(qrow * A::C + 4 * ks + 2 + hh) * 16));
  }
  // scores in log2 units = c * (scaled products)
  const float c = qscale / split_scale(1.4143f * bound[0]) / split_scale(1.4143f * bound[1]);
  const float vbound = bound[2];

  f32x16 oacc[A::NDB];
#pragma unroll
  for (int db = 0; db < A::NDB; ++db) oacc[db] = f32x16{};
  float m_run = -INFINITY, l_run = 0.f;    // the shift (log2 units) and this lane's share of the row sum (x 2^10)

  const int n_all = (seg_e - (seg_s & ~31) + 31) / 32;
  const int t0 = parts ? n_all * part_i / parts : 0, t1 = parts ? n_all * (part_i + 1) / parts : n_all;
  const int k_begin = (seg_s & ~31) + t0 * 32, n_kt = t1 - t0;

  auto step = [&](int it, int stage) {
    const int kb = k_begin + it * 32;
    if (it + 1 < n_kt) dma_tile(kb + 32, stage ^ 1);
    const char* sk = smem_a + stage * A::STAGE + l32 * A::C * 16 + hh * 16;
    char* const sv = smem_a + stage * A::STAGE + A::KBYTES;
    // An edge tile (uniform over the workgroup) holds keys of another segment: their v terms become zeros, since
    // their probabilities are but 0 * NaN is not.
    const bool edge = kb < seg_s || kb + 32 > seg_e;
    if (edge) {
      for (int i = tid; i < HD * 32; i += 256) {
        const int d = i >> 5, key = i & 31, p = vt_pos(key);
        if (kb + key >= seg_s && kb + key < seg_e) continue;
        char* at = sv + d * 128 + (p & 7) * 2;
        *reinterpret_cast<f16*>(at + (((p >> 3) ^ ((d >> 1) & 7)) << 4)) = (f16)0.f;
        *reinterpret_cast<f16*>(at + (((4 + (p >> 3)) ^ ((d >> 1) & 7)) << 4)) = (f16)0.f;
      }
      __syncthreads();
    }
    f32x16 s = f32x16{};
    // the cross products first: the small terms meet small sums
#pragma unroll
    for (int ks = 0; ks < A::KS; ++ks) {
      const f16x8 kh = *reinterpret_cast<const f16x8*>(sk + ks * 64), kl = *reinterpret_cast<const f16x8*>(sk + ks * 64 + 32);
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[ks], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[ks], s, 0, 0, 0);
    }
#pragma unroll
    for (int ks = 0; ks < A::KS; ++ks)
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8*>(sk + ks * 64), qh[ks], s, 0, 0, 0);
    if (edge) {
      const int lo = seg_s - (kb + 4 * hh);
      const uint32_t span = (uint32_t)(seg_e - seg_s);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if ((uint32_t)(8 * (r >> 2) + (r & 3) - lo) >= span) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32)) * c;
    if (__builtin_amdgcn_ballot_w64(mx > m_run + kLazy) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_run == m_new ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < A::NDB; ++db) oacc[db] *= alpha;
      m_run = m_new;
    }
    f16x8 ph[2], pl[2];
    float ls = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // (the factor is applied after the exponential: 10 more in its argument would cost it 2 to 4 bits)
      const float p = __builtin_amdgcn_exp2f(fmaf(s[r], c, -m_run)) * kPScale;
      ls += p;
      f16 hi, lo;
      split1(p, hi, lo);
      ph[r >> 3][r & 7] = hi;
      pl[r >> 3][r & 7] = lo;
    }
    l_run += ls;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int db = 0; db < A::NDB; ++db) {
        const int row = db * 32 + l32;
        const f16x8 vh = *reinterpret_cast<const f16x8*>(sv + row * 128 + (((2 * g + hh) ^ ((row >> 1) & 7)) << 4));
        const f16x8 vl = *reinterpret_cast<const f16x8*>(sv + row * 128 + (((4 + 2 * g + hh) ^ ((row >> 1) & 7)) << 4));
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph[g], oacc[db], 0, 0, 0);
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[g], oacc[db], 0, 0, 0);
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[g], oacc[db], 0, 0, 0);
      }
    wait_dma();
    __syncthreads();
  };
  dma_tile(k_begin, 0);
  wait_dma();
  __syncthreads();
  for (int it = 0; it < n_kt; it += 2) {
    step(it, 0);
    if (it + 1 < n_kt) step(it + 1, 1);
  }

  const float l_tot = l_run + __shfl_xor(l_run, 32);
  const float vscale = split_scale(vbound);
  if (qrow >= seg_e) return;
  if (parts) {
    float* pp = part + (int64_t)(item - n_whole) * attn_partial_floats(HD);
    const int qi = wave * 32 + l32;
    const float vinv = 1.0f / vscale;
#pragma unroll
    for (int db = 0; db < A::NDB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = db * 32 + 8 * g + 4 * hh;
        if (d < HD)
          *reinterpret_cast<f32x4*>(pp + qi * HD + d) = f32x4{oacc[db][4 * g] * vinv, oacc[db][4 * g + 1] * vinv,
                                                              oacc[db][4 * g + 2] * vinv, oacc[db][4 * g + 3] * vinv};
      }
    if (hh == 0) *reinterpret_cast<f32x2*>(pp + kAttnBM * HD + 2 * qi) = f32x2{m_run, l_tot};
    return;
  }
  // the output is a convex combination of v rows: it splits by v's exponent, which oacc already carries
  const float inv = 1.0f / l_tot;
  f16* orow = O + (int64_t)qrow * 2 * D;
#pragma unroll
  for (int db = 0; db < A::NDB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = db * 32 + 8 * g + 4 * hh;
      if (d >= HD) continue;
      f16x4 hi, lo;
      split4(f32x4{oacc[db][4 * g], oacc[db][4 * g + 1], oacc[db][4 * g + 2], oacc[db][4 * g + 3]}, inv, hi, lo);
      store_split4(orow, head * HD + d, hi, lo);
    }
}

int64_t attn_split_row_halfs(int hd) { return (4 * ((hd + 15) / 16) + 1) * 8; }   // a Q / K row in f16 elements

int attention_relayout_split(const float* qkv, int64_t ld, const f32x2* cs, const float* bound, int N, int Np, int H,
                             int hd, void* Qo, void* Ko, void* Vo, hipStream_t stream) {
  const dim3 grid((unsigned)(Np / 64), (unsigned)H);
#define QVL_RELAYOUT(HD)                                                                                          \
  hipLaunchKernelGGL(attn_relayout_split_kernel<HD>, grid, dim3(256), 0, stream, qkv, ld, H * hd, cs, bound, N, Np, \
                     (f16*)Qo, (f16*)Ko, (f16*)Vo)
  if (hd == 64) QVL_RELAYOUT(64);
  else if (hd == 72) QVL_RELAYOUT(72);
  else if (hd == 80) QVL_RELAYOUT(80);
  else return set_error(QVL_ERR_UNSUPPORTED, "attention split: head_dim=%d", hd);
#undef QVL_RELAYOUT
  return check_launch("attn_relayout_split");
}

// out: [N][2 H hd] split rows with the exponent of bound[2].
int attention_split(const void* Q, const void* K, const void* Vt, const int* items, int64_t n_items, int64_t n_whole,
                    const float* bound, int Np, int H, int hd, float qscale, void* out, float* part,
                    hipStream_t stream) {
  if (n_items == 0) return QVL_OK;
#define QVL_ATTN(HD)                                                                                                  \
  hipLaunchKernelGGL(attn_fwd_split_kernel<HD>, dim3((unsigned)n_items), dim3(256), 0, stream, (const f16*)Q,        \
                     (const f16*)K, (const f16*)Vt, items, bound, Np, qscale, (f16*)out, H * hd, (int)n_whole, part)
  if (hd == 64) QVL_ATTN(64);
  else if (hd == 72) QVL_ATTN(72);
  else QVL_ATTN(80);
#undef QVL_ATTN
  const int rc = check_launch("attn_fwd_split");
  if (rc || n_whole >= n_items || !part) return rc;
  return attention_combine_split(items, n_items, n_whole, part, bound + 2, out, H * hd, hd, stream);
}

}  // namespace qvl
