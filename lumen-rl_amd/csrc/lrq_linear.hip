// The FP8 rollout linear (lumenrl/quantization/fp8_rollout.py:53-78) in one
// launch: y = x_dq @ w_dq^T + b with x_dq = (x / s) * s per 1x128 activation
// block and w_dq = code * scale per 1x128 weight block, float32 sums, y in x's
// 16-bit type.
//
// What makes one launch possible, without dropping a bit of any operand:
//   * An e4m3 code is exact in bf16 and in fp16, and so is 16-bit x: the matrix
//     cores multiply them exactly and add in float32.  The weight's block scale
//     leaves the block's sum as a float32 factor, sum_k x_k (c_k s) =
//     s sum_k x_k c_k, so w_dq (12 significant bits) is never rounded either.
//   * x_dq is x: the emulation divides by s and multiplies by it again without
//     rounding to e4m3 in between, which moves x by at most 2^-23 |x|
//     (1.3e-8 rms, against 6e-7 to 1.9e-6 for a float32 product's own sums over
//     K = 4096 to 12288), whatever s is, power of two or not.  x itself is the
//     exact value of x / s * s.
//   * Only a block with an inf or NaN is not its own image: s is inf or NaN and
//     the whole block becomes NaN.  Such an x makes every output of its row inf
//     or NaN here, so an output that is inf looks its operands over again
//     (`linear_out`).
//   * The block sums leave out the weight's scale, so they could overflow where
//     y does not.  bf16 x is therefore multiplied with code * 2^-17 (exact in
//     bf16), which bounds a block's sum by 2^127 for every finite x, and the
//     result with 2^17; fp16 x cannot overflow a float32 sum.
#include "lrq.h"
#include "lrq_device.hpp"
#include "lrq_internal.hpp"

namespace lrq {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16 bytes of a 2-byte-aligned row, cached (x is read by many work-groups).
__device__ __forceinline__ v4u load_x16(const void* p) { return *(const LRQ_GLOBAL v4u_in*)p; }

template <int DT>
__device__ __forceinline__ float x16_to_f32(uint16_t b) {
  if constexpr (DT == kBF16) return u2f((uint32_t)b << 16);
  else return f16_to_f32(b);
}

// 8 codes (two words) as the matrix cores' second operand, in x's type: the
// code itself (fp16) or 2^-17 times it (bf16), both exact.
template <int DT>
constexpr float kCodeUnit = DT == kBF16 ? 0x1p-17f : 1.0f;
template <int DT, bool HI>
__device__ __forceinline__ uint32_t codes2_to_x16(uint32_t w) {
  if constexpr (DT == kBF16)
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, kCodeUnit<DT>, HI));
  else
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, kCodeUnit<DT>, HI));
}
template <int DT>
__device__ __forceinline__ v4u codes_to_x16(uint32_t lo, uint32_t hi) {
  return v4u{codes2_to_x16<DT, false>(lo), codes2_to_x16<DT, true>(lo), codes2_to_x16<DT, false>(hi),
             codes2_to_x16<DT, true>(hi)};
}

// D[m][n] += sum over 32 k of A[m][k] B[k][n].  Lane l holds k = 8 (l / 16) ..
// + 7 of row m = l % 16 of A and of column n = l % 16 of B (any order of k that
// A and B share gives the same sums), and rows 4 (l / 16) .. + 3 of column
// l % 16 of D.
template <int DT>
__device__ __forceinline__ f32x4 mfma16(v4u a, v4u b, f32x4 c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Orders a wave's LDS accesses for the compiler; the hardware keeps one wave's
// in order by itself.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// True if a row of x (k elements) or a weight row's scales hold an inf or NaN.
template <int DT>
__device__ __forceinline__ bool linear_nonfinite(const uint16_t* x, const uint16_t* s, int k) {
  constexpr uint32_t kInf = DT == kBF16 ? 0x7F80u : 0x7C00u;
  bool bad = false;
  for (int i = 0; i < k && !bad; i += 8) {
    const v4u v = load_x16(x + i);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) bad |= (w[j] & 0x7FFFu) >= kInf || ((w[j] >> 16) & 0x7FFFu) >= kInf;
  }
  for (int b = 0; b < k / kLinBlock && !bad; ++b) bad = (gld<uint16_t>(s + b) & 0x7FFFu) >= 0x7F80u;
  return bad;
}

__device__ __forceinline__ float linear_bias(const LinearArgs& a, int n) {
  if (a.bias_dtype == kF32) return gld<float>(static_cast<const float*>(a.bias) + n);
  const uint16_t b = gld<uint16_t>(static_cast<const uint16_t*>(a.bias) + n);
  return a.bias_dtype == kBF16 ? x16_to_f32<kBF16>(b) : x16_to_f32<kF16>(b);
}

// float32 -> x's 16-bit type, round to nearest even, NaN to the quiet NaN.
template <int DT>
__device__ __forceinline__ uint16_t linear_bits(float v) {
  if constexpr (DT == kBF16) return (f2u(v) & 0x7FFFFFFFu) > 0x7F800000u ? (uint16_t)0x7FC0u : (uint16_t)bf16_bits(v);
  else return (uint16_t)f16_bits(v);
}

// y[m][n] from its sum (in units of kCodeUnit).  An inf is the sum's own
// overflow, as in the reference, unless x's row or the scales are not finite:
// the reference's ops give NaN there (x / inf * inf; a block scale of inf only
// goes with NaN codes).
template <int DT>
__device__ __forceinline__ bool linear_is_nan(const LinearArgs& a, int m, int n) {
  return linear_nonfinite<DT>(static_cast<const uint16_t*>(a.x) + m * a.ldx, a.scales + n * (a.k / kLinBlock), (int)a.k);
}
template <int DT>
__device__ __forceinline__ uint16_t linear_out(const LinearArgs& a, float sum, int m, int n) {
  sum *= 1.0f / kCodeUnit<DT>;
  if ((f2u(sum) & 0x7FFFFFFFu) == 0x7F800000u && linear_is_nan<DT>(a, m, n)) sum = u2f(0x7FC00000u);
  if (a.bias != nullptr) sum += linear_bias(a, n);
  return linear_bits<DT>(sum);
}

// ---------------------------------------------------------------------------
// Few tokens (decoding): bound by the bytes of the weight
// ---------------------------------------------------------------------------
// The weight's e4m3 bytes are all that has to move; dequantizing it to float32
// for a library product wrote and read 8 times as many.  On an MI355X, one token
// through a 4096 x 4096 weight takes 6.6 us (48 us a call before) and 48 tokens
// through 12288 x 4096 17.9 us (105 us), where the weight's bytes alone take
// 2.5 and 7.6 us: at few work-groups per CU the rest is latency, and from about
// 32 tokens on x's passage through each CU's cache and LDS.
//
// A work-group of KW waves makes a (16 MT) x (16 NT) tile of y over the whole
// of K: wave w takes the 128-element K blocks w, w + KW, ... of all its rows,
// and the waves' sums meet in LDS at the end.  A matrix-core operand wants 16
// different rows in 16 neighbouring lanes, and loads in that order fetch one
// cache line per lane; so each wave loads whole 128-byte runs of codes (8 lanes
// a row) and whole 256-byte runs of x (16 lanes a row) into registers, DEPTH
// blocks ahead, and turns them round through its own few KiB of LDS.  A row's
// 16-byte pieces are stored at (piece ^ row)-like places, which makes both the
// writes and the reads free of bank conflicts, and no other wave touches them,
// so no barrier is needed until the end.
template <int NT, int MT>
struct LinStage {
  v4u w[NT][2];  // codes: rows 8 i + lane / 8, 16-byte piece lane % 8
  uint32_t s[NT];
  v4u x[MT][4];  // x: rows 4 i + lane / 16, 16-byte piece lane % 16
};

template <int DT, int MT, int NT, int KW, int DEPTH>
__global__ __launch_bounds__(64 * KW) void k_linear_rows(LinearArgs a) {
  constexpr int COLS = 16 * NT, CELLS = 16 * MT * COLS;
  constexpr int kStageBytes = NT * 2048 + MT * 4096;
  constexpr int kLds = KW * kStageBytes > KW * CELLS * 4 ? KW * kStageBytes : KW * CELLS * 4;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * COLS, m0 = blockIdx.y * (16 * MT);
  const int n_last = (int)a.n - 1 - n0, m_last = (int)a.m - 1 - m0;  // within this tile
  const int kb_n = (int)(a.k / kLinBlock);
  uint8_t* const lw = lds + wave * kStageBytes;
  uint8_t* const lx = lw + NT * 2048;
  // Tile bases in scalar registers and 32-bit offsets per lane.  Rows past the
  // end read the last one again; their sums are not stored.
  const uint8_t* const w0 = a.codes + (int64_t)n0 * a.k;
  const uint16_t* const s0 = a.scales + (int64_t)n0 * kb_n;
  const uint8_t* const x0 = static_cast<const uint8_t*>(a.x) + 2 * (m0 * a.ldx);
  uint32_t wo[NT][2], so[NT], xo[MT][4];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = 16 * j + 8 * h + (lane >> 3);
      wo[j][h] = (uint32_t)(r < n_last ? r : n_last) * (uint32_t)a.k + 16 * (lane & 7);
    }
    const int r = 16 * j + c;
    so[j] = (uint32_t)(r < n_last ? r : n_last) * (uint32_t)kb_n;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = 16 * i + 4 * q + g;
      xo[i][q] = (uint32_t)(r < m_last ? r : m_last) * (uint32_t)(2 * a.ldx) + 16 * c;
    }
  // Every wave runs the same number of steps, so that no load hangs on a branch
  // and the waits between loads and uses stay counted: a step past K reads the
  // last block again and scales its sums with 0.
  const int steps = ((kb_n + KW - 1) / KW + DEPTH - 1) / DEPTH * DEPTH;
  auto load = [&](LinStage<NT, MT>& st, int t) {
    const int kt = wave + t * KW, kb = kt < kb_n ? kt : kb_n - 1;
    const uint32_t keep = kt < kb_n ? 0xFFFFu : 0u;
    const uint8_t* const wb = w0 + kb * kLinBlock;
    const uint8_t* const xb = x0 + 2 * (kb * kLinBlock);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      st.w[j][0] = load_nt(wb + wo[j][0]);
      st.w[j][1] = load_nt(wb + wo[j][1]);
      st.s[j] = gld<uint16_t>(s0 + kb + so[j]) & keep;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) st.x[i][q] = load_x16(xb + xo[i][q]);
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto stash = [&](const LinStage<NT, MT>& st) {
    wave_lds_fence();  // the last step's reads are before these writes
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = 8 * h + (lane >> 3);
        *reinterpret_cast<v4u*>(lw + 2048 * j + 128 * r + 16 * ((lane & 7) ^ (r >> 1))) = st.w[j][h];
      }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<v4u*>(lx + 4096 * i + 256 * (4 * q + g) + 16 * (c ^ (4 * q + g))) = st.x[i][q];
    wave_lds_fence();
  };
  auto multiply = [&](const float (&sc)[NT]) {
    // MFMA (h, q) takes k = 16 (g + 4 h) + 8 q .. + 7 of the block from lane (c, g)
    v4u x[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int hq = 0; hq < 4; ++hq)
        x[i][hq] = *reinterpret_cast<const v4u*>(lx + 4096 * i + 256 * c + 16 * ((2 * (g + 4 * (hq >> 1)) + (hq & 1)) ^ c));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      v4u b[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v4u w = *reinterpret_cast<const v4u*>(lw + 2048 * j + 128 * c + 16 * ((g + 4 * h) ^ (c >> 1)));
        b[2 * h] = codes_to_x16<DT>(w.x, w.y);
        b[2 * h + 1] = codes_to_x16<DT>(w.z, w.w);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        f32x4 p = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < 4; ++q) p = mfma16<DT>(x[i][q], b[q], p);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(p[r], sc[j], acc[i][j][r]);
      }
    }
  };
  LinStage<NT, MT> st[DEPTH];
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(st[d], d);
  auto step = [&](int d, int next) {
    float sc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = u2f(st[d].s[j] << 16);
    stash(st[d]);
    if (next > 0) load(st[d], next);
    multiply(sc);
  };
  for (int t = DEPTH; t < steps; t += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) step(d, t + d);
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) step(d, 0);
  __syncthreads();  // the waves' own LDS becomes the shared sums
  float* const red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave * CELLS + (16 * i + 4 * g + r) * COLS + 16 * j + c] = acc[i][j][r];
  __syncthreads();
  for (int e = threadIdx.x; e < CELLS; e += 64 * KW) {
    const int r = e / COLS, q = e % COLS;
    if (r > m_last || q > n_last) continue;
    float sum = red[e];
#pragma unroll
    for (int w = 1; w < KW; ++w) sum += red[w * CELLS + e];
    gst<uint16_t>(static_cast<uint16_t*>(a.y) + (int64_t)(m0 + r) * a.n + n0 + q, linear_out<DT>(a, sum, m0 + r, n0 + q));
  }
}

// Tile of y per work-group, in units of 16 tokens and 16 weight rows.  Its
// cost is the bytes that its CU moves through the vector cache and LDS, 2 mt +
// nt (x has two bytes an element), times the rounds of work-groups that the 256
// CUs take; the shape with the least cost is within 5 % of the fastest that a
// sweep over all of them found at 1 to 64 tokens and weights of [1024 to 12288,
// 4096 to 12288].
struct RowsShape {
  int mt, nt;
};
static RowsShape rows_shape(int64_t m, int64_t n) {
  RowsShape best{1, 1};
  int64_t least = INT64_MAX;
  for (int mt = 1; mt <= 4 && 16 * (mt - 1) < m; ++mt)
    for (int nt = 1; nt <= 4; ++nt) {
      const int64_t wgs = ((n + 16 * nt - 1) / (16 * nt)) * ((m + 16 * mt - 1) / (16 * mt));
      const int64_t cost = ((wgs + 255) / 256) * (2 * mt + nt);
      if (cost < least) least = cost, best = {mt, nt};
    }
  return best;
}

template <int DT, int MT, int NT>
static void launch_rows(const LinearArgs& a, hipStream_t stream) {
  // 8 waves where their LDS (2 KiB per 16 weight rows and 4 per 16 tokens each) fits the CU's 160 KiB
  constexpr int KW = 8 * (2 * NT + 4 * MT) <= 144 ? 8 : 4;
  const dim3 grid((unsigned)((a.n + 16 * NT - 1) / (16 * NT)), (unsigned)((a.m + 16 * MT - 1) / (16 * MT)));
  hipLaunchKernelGGL((k_linear_rows<DT, MT, NT, KW, 1>), grid, dim3(64 * KW), 0, stream, a);
}
template <int DT, int MT>
static void launch_rows_nt(const LinearArgs& a, int nt, hipStream_t stream) {
  switch (nt) {
    case 1: launch_rows<DT, MT, 1>(a, stream); break;
    case 2: launch_rows<DT, MT, 2>(a, stream); break;
    case 3: launch_rows<DT, MT, 3>(a, stream); break;
    default: launch_rows<DT, MT, 4>(a, stream); break;
  }
}
template <int DT>
static void launch_rows_shape(const LinearArgs& a, hipStream_t stream) {
  const RowsShape s = rows_shape(a.m, a.n);
  switch (s.mt) {
    case 1: launch_rows_nt<DT, 1>(a, s.nt, stream); break;
    case 2: launch_rows_nt<DT, 2>(a, s.nt, stream); break;
    case 3: launch_rows_nt<DT, 3>(a, s.nt, stream); break;
    default: launch_rows_nt<DT, 4>(a, s.nt, stream); break;
  }
}

hipError_t launch_linear(const LinearArgs& a, int dtype, hipStream_t stream) {
  if (dtype == kBF16) launch_rows_shape<kBF16>(a, stream);
  else launch_rows_shape<kF16>(a, stream);
  return hipGetLastError();
}

}  // namespace lrq
