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
//   * x and code together are multiples of 2^-142, so the float32 block sums lose
//     nothing to underflow: the matrix cores keep subnormals.
//   * The block sums leave out the weight's scale, so with bf16 x beyond 2^112 they
//     can overflow where y does not (fp16 x cannot).  A work-group that finds an inf
//     or NaN among its results multiplies once more, with code * 2^-17 (exact in
//     bf16, and every block's sum of finite x below 2^127), and takes those results,
//     times 2^17, from there.  The others stay as they are: in units of 2^-17 all
//     sums would come 17 binades nearer to underflow (with results of 2^-124, a
//     relative error of 5.2e-3 instead of the rounding's 1.7e-3).  Such work-groups
//     take twice as long: 8192 tokens x [12288, 4096] 1.18 ms with one inf and 1.55
//     with NaN in every token (0.80 without), 48 tokens 34 us (18).
#include "lrq.h"
#include "lrq_device.hpp"
#include "lrq_internal.hpp"

namespace lrq {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16 bytes at a 32-bit offset from a wave-uniform base, from any 2-byte-aligned
// address; cached, or past the caches for what one work-group reads once.
typedef const LRQ_GLOBAL uint8_t* GlobalBytes;
__device__ __forceinline__ v4u load_x16(GlobalBytes p, uint32_t off) { return *(const LRQ_GLOBAL v4u_in*)(p + off); }
__device__ __forceinline__ v4u load_x16_nt(GlobalBytes p, uint32_t off) {
  return __builtin_nontemporal_load((const LRQ_GLOBAL v4u_in*)(p + off));
}
__device__ __forceinline__ uint32_t load_scale16(GlobalBytes p, uint32_t off) { return *(const LRQ_GLOBAL uint16_t*)(p + off); }

template <int DT>
__device__ __forceinline__ float x16_to_f32(uint16_t b) {
  if constexpr (DT == kBF16) return u2f((uint32_t)b << 16);
  else return f16_to_f32(b);
}

// 8 codes (two words) as the matrix cores' second operand, in x's type: the
// code itself or, in the second pass that only bf16 has, 2^-17 times it.
template <int DT>
constexpr bool kTwoPasses = DT == kBF16;
constexpr float kSecondUnit = 0x1p-17f, kSecondResult = 0x1p17f;
template <int DT, bool SECOND, bool HI>
__device__ __forceinline__ uint32_t codes2_to_x16(uint32_t w) {
  if constexpr (DT == kBF16)
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, SECOND ? kSecondUnit : 1.0f, HI));
  else
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, HI));
}
template <int DT, bool SECOND>
__device__ __forceinline__ v4u codes_to_x16(uint32_t lo, uint32_t hi) {
  return v4u{codes2_to_x16<DT, SECOND, false>(lo), codes2_to_x16<DT, SECOND, true>(lo),
             codes2_to_x16<DT, SECOND, false>(hi), codes2_to_x16<DT, SECOND, true>(hi)};
}
// The thread's index, which the second pass takes anew: offsets that it shared
// with the first would be kept for it, in registers that the first has no more of.
template <bool SECOND>
__device__ __forceinline__ int linear_tid() {
  int tid = threadIdx.x;
  if constexpr (SECOND) asm volatile("" : "+v"(tid));
  return tid;
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

// Barrier of the work-group for its LDS accesses only: loads from memory stay
// in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// True in every thread if any of the work-group's has `bad`; `flags`: a word of
// LDS for each of its waves, free since the last barrier and until this returns.
template <int WAVES>
__device__ __forceinline__ bool linear_any(uint32_t* flags, bool bad) {
  const uint32_t mine = __any(bad) ? 1u : 0u;
  if ((threadIdx.x & 63) == 0) flags[threadIdx.x >> 6] = mine;
  lds_barrier();
  if (!__any((int)flags[threadIdx.x % WAVES])) return false;
  lds_barrier();
  return true;
}

// True if a row of x (k elements) or a weight row's scales hold an inf or NaN.
template <int DT>
__device__ __forceinline__ bool linear_nonfinite(const uint16_t* x, const uint16_t* s, int k) {
  constexpr uint32_t kInf = DT == kBF16 ? 0x7F80u : 0x7C00u;
  bool bad = false;
  for (int i = 0; i < k && !bad; i += 8) {
    const v4u v = load_x16((GlobalBytes)(x + i), 0);
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

__device__ __forceinline__ bool linear_finite(float v) { return (f2u(v) & 0x7FFFFFFFu) < 0x7F800000u; }
template <int DT>
__device__ __forceinline__ bool linear_bits_finite(uint16_t v) {
  constexpr uint16_t kInf = DT == kBF16 ? 0x7F80u : 0x7C00u;
  return (v & kInf) != kInf;
}

// y[m][n] from its sum; REDO: what is not finite is looked at in the second pass.
// An inf is the sum's own overflow, as in the reference, unless x's row or the
// scales are not finite: the reference's ops give NaN there (x / inf * inf; a
// block scale of inf only goes with NaN codes).
template <int DT>
__device__ __forceinline__ bool linear_is_nan(const LinearArgs& a, int m, int n) {
  return linear_nonfinite<DT>(static_cast<const uint16_t*>(a.x) + m * a.ldx, a.scales + n * (a.k / kLinBlock), (int)a.k);
}
template <int DT, bool REDO>
__device__ __forceinline__ uint16_t linear_out(const LinearArgs& a, float sum, int m, int n) {
  if (!REDO && (f2u(sum) & 0x7FFFFFFFu) == 0x7F800000u && linear_is_nan<DT>(a, m, n)) sum = u2f(0x7FC00000u);
  if (a.bias != nullptr) sum += linear_bias(a, n);
  return linear_bits<DT>(sum);
}

// ---------------------------------------------------------------------------
// Few tokens (decoding): bound by the bytes of the weight
// ---------------------------------------------------------------------------
// The weight's e4m3 bytes are all that has to move; dequantizing it to float32
// for a library product wrote and read 8 times as many.  On an MI355X, one token
// through a 4096 x 4096 weight takes 6.3 us (48 us a call before) and 48 tokens
// through 12288 x 4096 18.8 us (105 us), medians of rocprofv3 traces, where the
// weight's bytes alone take 2.5 and 7.6 us: at few work-groups per CU the rest is latency, and from about
// 32 tokens on x's passage through each CU's cache and LDS.
//
// A work-group of KW waves makes a (16 MT) x (16 NT) tile of y over the whole
// of K: each wave takes a run of 128-element K blocks of all its rows, and the
// waves' sums meet in LDS at the end.  A matrix-core operand wants 16
// different rows in 16 neighbouring lanes, and loads in that order fetch one
// cache line per lane; so each wave loads whole 128-byte runs of codes (8 lanes
// a row) and whole 256-byte runs of x (16 lanes a row) into registers, a block
// ahead, and turns them round through its own few KiB of LDS.  A row's
// 16-byte pieces are stored at (piece ^ row)-like places, which makes both the
// writes and the reads free of bank conflicts, and no other wave touches them,
// so no barrier is needed until the end.  Measured and left: runs of blocks
// taken in turns by the waves (up to 10 % slower at one token), loads two or
// four blocks ahead (the same, or spilled registers), K split over work-groups
// with a second launch for the sums (slower but for K = 12288 at 32 tokens).
//
// ONCE: one work-group reads each weight row, past the caches (5 % faster); with
// more token groups than one the others find the row in L2 (up to 25 % faster).
template <int NT, int MT>
struct LinStage {
  v4u w[NT][2];  // codes: rows 8 i + lane / 8, 16-byte piece lane % 8
  uint32_t s[NT];
  v4u x[MT][4];  // x: rows 4 i + lane / 16, 16-byte piece lane % 16
};

template <int DT, int MT, int NT, int KW, bool ONCE, bool SECOND>
__device__ __forceinline__ bool linear_rows_pass(const LinearArgs& a, uint8_t* lds) {
  constexpr int COLS = 16 * NT, CELLS = 16 * MT * COLS;
  constexpr int kStageBytes = NT * 2048 + MT * 4096;
  const int tid = linear_tid<SECOND>();
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * COLS, m0 = blockIdx.y * (16 * MT);
  const int n_last = (int)a.n - 1 - n0, m_last = (int)a.m - 1 - m0;  // within this tile
  const int kb_n = (int)(a.k / kLinBlock);
  uint8_t* const lw = lds + wave * kStageBytes;
  uint8_t* const lx = lw + NT * 2048;
  // Tile bases in scalar registers and 32-bit offsets per lane.  Rows past the
  // end read the last one again; their sums are not stored.
  const GlobalBytes w0 = (GlobalBytes)a.codes + (int64_t)n0 * a.k;
  const GlobalBytes s0 = (GlobalBytes)a.scales + 2 * ((int64_t)n0 * kb_n);
  const GlobalBytes x0 = (GlobalBytes)a.x + 2 * (m0 * a.ldx);
  uint32_t wo[NT][2], so[NT], xo[MT][4];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = 16 * j + 8 * h + (lane >> 3);
      wo[j][h] = (uint32_t)(r < n_last ? r : n_last) * (uint32_t)a.k + 16 * (lane & 7);
    }
    const int r = 16 * j + c;
    so[j] = (uint32_t)(r < n_last ? r : n_last) * (uint32_t)(2 * kb_n);
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
  const int steps = (kb_n + KW - 1) / KW;
  auto load = [&](LinStage<NT, MT>& st, int t) {
    const int kt = wave * steps + t, kb = kt < kb_n ? kt : kb_n - 1;
    const uint32_t keep = kt < kb_n ? 0xFFFFu : 0u;
    const GlobalBytes wb = w0 + kb * kLinBlock, xb = x0 + 2 * (kb * kLinBlock), sb = s0 + 2 * kb;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      st.w[j][0] = ONCE ? load_x16_nt(wb, wo[j][0]) : load_x16(wb, wo[j][0]);
      st.w[j][1] = ONCE ? load_x16_nt(wb, wo[j][1]) : load_x16(wb, wo[j][1]);
      st.s[j] = load_scale16(sb, so[j]) & keep;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) st.x[i][q] = load_x16(xb, xo[i][q]);
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
        b[2 * h] = codes_to_x16<DT, SECOND>(w.x, w.y);
        b[2 * h + 1] = codes_to_x16<DT, SECOND>(w.z, w.w);
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
  LinStage<NT, MT> st;
  float sc[NT];
  auto turn = [&] {
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = u2f(st.s[j] << 16);
    stash(st);
  };
  load(st, 0);
  for (int t = 1; t < steps; ++t) {
    turn();
    load(st, t);
    multiply(sc);
  }
  turn();
  multiply(sc);
  __syncthreads();  // the waves' own LDS becomes the shared sums
  float* const red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave * CELLS + (16 * i + 4 * g + r) * COLS + 16 * j + c] = acc[i][j][r];
  __syncthreads();
  bool bad = false;  // a result that the second pass replaces
  for (int e = tid; e < CELLS; e += 64 * KW) {
    const int r = e / COLS, q = e % COLS;
    if (r > m_last || q > n_last) continue;
    float sum = red[e];
#pragma unroll
    for (int w = 1; w < KW; ++w) sum += red[w * CELLS + e];
    uint16_t* const y = static_cast<uint16_t*>(a.y) + (int64_t)(m0 + r) * a.n + n0 + q;
    if constexpr (SECOND) {
      if (linear_bits_finite<DT>(gld<uint16_t>(y))) continue;  // what this thread stored in the first pass
      sum *= kSecondResult;
    } else if constexpr (kTwoPasses<DT>) {
      bad |= !linear_finite(sum);
    }
    gst<uint16_t>(y, linear_out<DT, !SECOND && kTwoPasses<DT>>(a, sum, m0 + r, n0 + q));
  }
  return bad;
}

template <int DT, int MT, int NT, int KW, bool ONCE>
__global__ __launch_bounds__(64 * KW) void k_linear_rows(LinearArgs a) {
  constexpr int kStages = KW * (NT * 2048 + MT * 4096), kSums = KW * (16 * MT) * (16 * NT) * 4;
  static_assert(kSums + 4 * KW <= kStages, "the waves' sums and flags fit where their stages were");
  __shared__ __attribute__((aligned(16))) uint8_t lds[kStages];
  const bool bad = linear_rows_pass<DT, MT, NT, KW, ONCE, false>(a, lds);
  if constexpr (kTwoPasses<DT>)
    if (linear_any<KW>(reinterpret_cast<uint32_t*>(lds + kSums), bad)) linear_rows_pass<DT, MT, NT, KW, ONCE, true>(a, lds);
}

// ---------------------------------------------------------------------------
// Many tokens (prefill): bound by the matrix cores
// ---------------------------------------------------------------------------
// A work-group of WM x WN waves makes a tile of y of 16 FM WM tokens and 16 FN
// WN weight rows; each wave its (16 FM) x (16 FN) of it.  Blocks of 128 k go
// through two LDS buffers: x as it is and the weight as e4m3 bytes, which each
// wave converts for itself (half the LDS traffic of 16-bit weights).  A wave
// keeps the block of its own x rows in registers and takes the weight 16 rows
// at a time: 4 FM matrix instructions, whose float32 sums the block's scale
// then multiplies into the accumulators.  That multiplication runs one step
// behind, between the next step's matrix instructions, and so do the
// conversions, the moves of the next block into LDS and the loads of the one
// after: 3 vector instructions fit beside each matrix instruction.
//
// 4 x 4 x (2 x 4): 128 x 256 tiles, one work-group of 8 waves on a CU, two to a
// SIMD, so that one's vector instructions and waits fall beside the other's
// matrix instructions (4 waves of 128 x 64 each: 0.90 ms instead of 0.80).
// 8192 tokens x [12288, 4096] take 0.80 ms (1032 TFLOP/s), 5.6 ms before by way of
// float32 operands and a float32 library product (147 TFLOP/s).  That is 1.67 million
// cycles, at 2.1 GHz: matrix cores busy 47 % of them, other vector instructions 35 %,
// LDS 33 % (rocprofv3 counters; a profiled pass runs at a lower clock, 0.82 to 1.03 ms).
// The smaller tiles are for grids that would leave CUs idle with the large one:
// each CU does less work per byte that passes its LDS, 28 us for 512 tokens x
// [4096, 4096] in 64 x 128 tiles (59 in 128 x 256), 115 us for 1024 x [12288,
// 4096] in 128 x 192 (140).  32 x 32 matrix instructions need 16 more registers
// than there are (1.07 ms with spills; 4 waves 0.96 ms).
//
// The compiler keeps the matrix instructions' results in vector registers
// (-amdgpu-mfma-vgpr-form): in accumulation registers, its own choice here,
// every result needed a move before the scale could multiply it (15 % slower).
// The tile of work-group `wg`.  Work-groups go to the 8 XCDs in turn; each XCD
// takes one run of the tiles, walked 8 tile rows at a time, so that the rows of
// x and of the weight that its work-groups read together stay in its L2.
__device__ __forceinline__ void linear_tile(int wg, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int tiles = tiles_m * tiles_n, per = tiles >> 3;
  const int t = wg < 8 * per ? (wg & 7) * per + (wg >> 3) : wg;
  const int group = 8 * tiles_n, first = t / group * 8;
  const int rows = tiles_m - first < 8 ? tiles_m - first : 8;
  tm = first + (t % group) % rows;
  tn = (t % group) / rows;
}

template <int FM, int FN, int WM, int WN>
constexpr int kTileBuffer = 16 * FM * WM * 256 + 16 * FN * WN * (128 + 4);  // x, codes and scales of a K block
template <int FM, int FN, int WM, int WN>
constexpr int kTileResult = WM * WN * (16 * FM) * (2 * (16 * FN) + 16);  // y, by waves, in rows of a pitch
template <int DT, int FM, int FN, int WM, int WN, bool SECOND>
__device__ __forceinline__ bool linear_tiles_pass(const LinearArgs& a, int tm, int tn, uint8_t* lds) {
  constexpr int T = 64 * WM * WN, BM = 16 * FM * WM, BN = 16 * FN * WN;
  constexpr int PA = BM * 16 / T, PB = BN * 8 / T;   // 16-byte pieces a thread moves per K block
  constexpr int kA = BM * 256, kB = BN * 128, kBuf = kTileBuffer<FM, FN, WM, WN>;
  static_assert(BN <= T && PA * T == BM * 16 && PB * T == BN * 8, "");
  const int tid = linear_tid<SECOND>(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int m0 = tm * BM, n0 = tn * BN;
  const int n_last = (int)a.n - 1 - n0, m_last = (int)a.m - 1 - m0;
  const int kb_n = (int)(a.k / kLinBlock);
  const GlobalBytes w0 = (GlobalBytes)a.codes + (int64_t)n0 * a.k;
  const GlobalBytes s0 = (GlobalBytes)a.scales + 2 * ((int64_t)n0 * kb_n);
  const GlobalBytes x0 = (GlobalBytes)a.x + 2 * (m0 * a.ldx);
  uint32_t xo[PA], wo[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int r = (T / 16) * p + (tid >> 4);
    xo[p] = (uint32_t)(r < m_last ? r : m_last) * (uint32_t)(2 * a.ldx) + 16 * (tid & 15);
  }
#pragma unroll
  for (int p = 0; p < PB; ++p) {
    const int r = (T / 8) * p + (tid >> 3);
    wo[p] = (uint32_t)(r < n_last ? r : n_last) * (uint32_t)a.k + 16 * (tid & 7);
  }
  const int sr = tid < BN ? tid : BN - 1;  // the scale this thread moves
  const uint32_t so = (uint32_t)(sr < n_last ? sr : n_last) * (uint32_t)(2 * kb_n);
  v4u gx[PA], gw[PB];
  uint32_t gs;
  // The moves of a block are spread over the tiles j = 0 .. FN - 2 of the block
  // before: stores into LDS in the first half, loads in the second.
  constexpr int HP = (FN - 1) / 2, HF = FN - 1 - HP;
  // Keeps the widening of a loop-invariant offset at its load: hoisted out of the
  // loop, as the compiler would, it costs two registers and a 64-bit addition at
  // each load.  64 x 128 tiles come to 125 registers, so that two fit a CU (1075
  // instead of 1190 us for 8192 tokens x [12288, 4096]); the largest tile, one on
  // a CU either way, is 2 % faster without.
  auto here = [](uint32_t off) {
    if constexpr (FM * FN < 16) asm volatile("" : "+v"(off));
    return off;
  };
  auto fetch = [&](int kb, int j) {
    kb = kb < kb_n ? kb : kb_n - 1;
    const GlobalBytes wb = w0 + kb * kLinBlock, xb = x0 + 2 * (kb * kLinBlock), sb = s0 + 2 * kb;
#pragma unroll
    for (int p = 0; p < PA; ++p)
      if (j == HP + p * HF / PA) gx[p] = load_x16(xb, here(xo[p]));
#pragma unroll
    for (int p = 0; p < PB; ++p)
      if (j == HP + p * HF / PB) gw[p] = load_x16(wb, here(wo[p]));
    if (j == HP) gs = load_scale16(sb, here(so));
  };
  auto put = [&](uint8_t* buf, int j) {
#pragma unroll
    for (int p = 0; p < PA; ++p) {
      const int r = (T / 16) * p + (tid >> 4);
      if (j == p * HP / PA) *reinterpret_cast<v4u*>(buf + 256 * r + 16 * ((tid & 15) ^ (r & 15))) = gx[p];
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
      const int r = (T / 8) * p + (tid >> 3);
      if (j == p * HP / PB) *reinterpret_cast<v4u*>(buf + kA + 128 * r + 16 * ((tid & 7) ^ ((r >> 1) & 7))) = gw[p];
    }
    if (j == 0 && (BN == T || tid < BN)) *reinterpret_cast<uint32_t*>(buf + kA + kB + 4 * tid) = gs << 16;
  };
  const int wm = (wave / WN) * 16 * FM, wn = (wave % WN) * 16 * FN;
  v4u xa[FM][4], wr[2];
  auto read_x = [&](const uint8_t* buf, int q) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
        xa[i][q] = *reinterpret_cast<const v4u*>(buf + 256 * (wm + 16 * i + c) + 16 * ((2 * (g + 4 * (q >> 1)) + (q & 1)) ^ c));
  };
  auto read_w = [&](const uint8_t* buf, int j) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      wr[h] = *reinterpret_cast<const v4u*>(buf + kA + 128 * (wn + 16 * j + c) + 16 * ((g + 4 * h) ^ (c >> 1)));
  };
  f32x4 acc[FM][FN], p[FM], pp[FM];
  float sp = 0.0f;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    pp[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int j = 0; j + 1 < FN; ++j) fetch(0, j);
#pragma unroll
  for (int j = 0; j + 1 < FN; ++j) put(lds, j);
#pragma unroll
  for (int j = 0; j + 1 < FN; ++j) fetch(1, j);
  lds_barrier();
#pragma unroll
  for (int q = 0; q < 4; ++q) read_x(lds, q);
  read_w(lds, 0);
  for (int kb = 0; kb < kb_n; ++kb) {
    const uint8_t* const cur = lds + (kb & 1) * kBuf;
    uint8_t* const nxt = lds + ((kb + 1) & 1) * kBuf;
    float sc[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) sc[j] = *reinterpret_cast<const float*>(cur + kA + kB + 4 * (wn + 16 * j + c));
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const v4u w[2] = {wr[0], wr[1]};
      if (j + 1 < FN) {
        read_w(cur, j + 1);
        // the next block goes into LDS during the first tiles, the one after it
        // is fetched during the next
        put(nxt, j);
        fetch(kb + 2, j);
      } else {
        lds_barrier();  // every read of `cur` is done and `nxt` is whole
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v4u b = (q & 1) ? codes_to_x16<DT, SECOND>(w[q >> 1].z, w[q >> 1].w) : codes_to_x16<DT, SECOND>(w[q >> 1].x, w[q >> 1].y);
#pragma unroll
        for (int i = 0; i < FM; ++i) p[i] = mfma16<DT>(xa[i][q], b, q ? p[i] : f32x4{0.0f, 0.0f, 0.0f, 0.0f});
        if (j + 1 == FN) {
          if (q == 0) read_w(nxt, 0);
          read_x(nxt, q);
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
          acc[i][(j + FN - 1) % FN][q] = __builtin_fmaf(pp[i][q], sp, acc[i][(j + FN - 1) % FN][q]);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i) pp[i] = p[i];
      sp = sc[j];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[i][FN - 1][r] = __builtin_fmaf(pp[i][r], sp, acc[i][FN - 1][r]);
  // The wave's part of y goes through its own piece of LDS (no block is read
  // any more), so that rows leave in 16-byte stores.
  constexpr int ROWS = 16 * FM, COLS = 16 * FN, PITCH = 2 * COLS + 16, PIECES = COLS / 8;
  static_assert(WM * WN * ROWS * PITCH == kTileResult<FM, FN, WM, WN>, "");
  uint8_t* const out = lds + wave * (ROWS * PITCH);
  constexpr bool kFirst = kTwoPasses<DT> && !SECOND;
  lds_barrier();
  bool inf = false, bad = false;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = wn + 16 * j + c;
    const float bias = a.bias != nullptr && n <= n_last ? linear_bias(a, n0 + n) : 0.0f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float sum = SECOND ? acc[i][j][r] * kSecondResult : acc[i][j][r];
        if constexpr (kFirst) bad |= !linear_finite(sum);
        else inf |= (f2u(sum) & 0x7FFFFFFFu) == 0x7F800000u;
        *reinterpret_cast<uint16_t*>(out + (16 * i + 4 * g + r) * PITCH + 2 * (16 * j + c)) = linear_bits<DT>(sum + bias);
      }
  }
  wave_lds_fence();
  if (__any(inf)) {  // rare: see linear_out
    for (int e = lane; e < ROWS * COLS; e += 64) {
      const int m = e / COLS, n = e % COLS;
      uint16_t* const v = reinterpret_cast<uint16_t*>(out + m * PITCH + 2 * n);
      if (wm + m <= m_last && wn + n <= n_last && (*v & 0x7FFFu) == (DT == kBF16 ? 0x7F80u : 0x7C00u) &&
          linear_is_nan<DT>(a, m0 + wm + m, n0 + wn + n))
        *v = DT == kBF16 ? 0x7FC0u : 0x7E00u;
    }
    wave_lds_fence();
  }
  const bool whole = a.n % 8 == 0;  // pieces of 8 columns are all in or all out, and 16-byte aligned
#pragma unroll 4
  for (int e = lane; e < ROWS * PIECES; e += 64) {
    const int m = e / PIECES, q = e % PIECES, n = wn + 8 * q;
    if (wm + m > m_last || n > n_last) continue;
    uint16_t* const dst = static_cast<uint16_t*>(a.y) + (int64_t)(m0 + wm + m) * a.n + n0 + n;
    const uint8_t* const src = out + m * PITCH + 16 * q;
    if (whole && !SECOND) {
      gst<v4u>(dst, *reinterpret_cast<const v4u*>(src));
    } else {
      for (int k = 0; k < 8 && n + k <= n_last; ++k) {
        // the second pass replaces what this lane stored in the first where that is not finite
        if (SECOND && linear_bits_finite<DT>(gld<uint16_t>(dst + k))) continue;
        gst<uint16_t>(dst + k, reinterpret_cast<const uint16_t*>(src)[k]);
      }
    }
  }
  return bad;
}

template <int DT, int FM, int FN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 1) void k_linear_tiles(LinearArgs a, int tiles_m, int tiles_n) {
  constexpr int kLds = 2 * kTileBuffer<FM, FN, WM, WN>, kResult = kTileResult<FM, FN, WM, WN>;
  static_assert(kResult + 4 * WM * WN <= kLds, "the tile of y and the waves' flags fit where the blocks were");
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  int tm, tn;
  linear_tile(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const bool bad = linear_tiles_pass<DT, FM, FN, WM, WN, false>(a, tm, tn, lds);
  if constexpr (kTwoPasses<DT>)
    if (linear_any<WM * WN>(reinterpret_cast<uint32_t*>(lds + kResult), bad))
      linear_tiles_pass<DT, FM, FN, WM, WN, true>(a, tm, tn, lds);
}

// ---------------------------------------------------------------------------
// Which kernel
// ---------------------------------------------------------------------------
// The shape with the least modelled time per 128-element K block, in ns:
//   * k_linear_rows: kLinearRows ns a round of 256 work-groups.  It grows with the
//     bytes that a CU moves through its vector cache and LDS, 2 mt + nt units (x
//     has two bytes an element); shapes past 8 waves' LDS do not pay any more;
//   * k_linear_tiles: `each` ns for each 256 tiles, and `once` more; of 64 x 64
//     tiles, three fit a CU, 280 ns and 457 once where they do.
// A sweep of every shape over 1 to 8192 tokens and weights of [512 to 12288, 1024 to
// 12288], 197 sizes: the shape this takes is 1.1 % from the fastest in the mean, over
// 5 % in 16 of them, and 31 % at worst (32 tokens x [2560, 2560] in 32 x 16: 6.7 us,
// 5.1 in 16 x 32; one round of work-groups is charged the same however full it is).
// 16 tokens x 64 weight rows are left out (two rounds of 16 x 32 cost no more), and
// 48 x 64 (more registers than there are).
constexpr int kLinearRows[3][4] = {{136, 190, 315, 0}, {165, 280, 400, 465}, {290, 380, 485, 0}};
constexpr int64_t kCus = 256;
struct LinearTile {
  int m, n, each, once;
};
constexpr LinearTile kLinearTiles[] = {
    {128, 256, 2060, -190}, {128, 192, 1680, -80}, {128, 128, 1290, -60}, {64, 128, 670, 205}, {64, 64, 398, 0}};
constexpr int kLinearTileKinds = sizeof(kLinearTiles) / sizeof(kLinearTiles[0]);
struct LinearShape {
  int tile;    // index into kLinearTiles, or -1: k_linear_rows
  int mt, nt;  // k_linear_rows: tokens and weight rows per work-group, in 16s
};
static int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
static LinearShape linear_shape(int64_t m, int64_t n) {
  LinearShape best{0, 0, 0};
  int64_t least = INT64_MAX;
  for (int i = 0; i < kLinearTileKinds; ++i) {
    const LinearTile& t = kLinearTiles[i];
    const int64_t rounds = ceil_div(ceil_div(m, t.m) * ceil_div(n, t.n), kCus);
    int64_t cost = t.each * rounds + t.once;
    if (t.m == 64 && t.n == 64 && 280 * rounds + 457 > cost) cost = 280 * rounds + 457;
    if (cost < least) least = cost, best = {i, 0, 0};
  }
  for (int mt = 1; mt <= 3 && 16 * (mt - 1) < m; ++mt) {
    if (ceil_div(m, 16 * mt) > 65535) continue;  // the grid's second dimension
    for (int nt = 1; nt <= 4 && kLinearRows[mt - 1][nt - 1] > 0; ++nt) {
      const int64_t cost = kLinearRows[mt - 1][nt - 1] * ceil_div(ceil_div(n, 16 * nt) * ceil_div(m, 16 * mt), kCus);
      if (cost < least) least = cost, best = {-1, mt, nt};
    }
  }
  return best;
}

template <int DT, int MT, int NT>
static void launch_rows(const LinearArgs& a, hipStream_t stream) {
  constexpr int KW = 8;  // their LDS, 2 KiB per 16 weight rows and 4 per 16 tokens each, fits the CU's 160 KiB
  const dim3 grid((unsigned)ceil_div(a.n, 16 * NT), (unsigned)ceil_div(a.m, 16 * MT)), block(64 * KW);
  // One token group never takes 48 x 16 (32 x 32 costs less for the same rounds), and
  // several never 16 x 48: ONCE is a hint for the caches, so neither needs the other kernel.
  constexpr bool kOne = !(MT == 3 && NT == 1), kMany = !(MT == 1 && NT == 3);
  if (kOne && (grid.y == 1 || !kMany)) hipLaunchKernelGGL((k_linear_rows<DT, MT, NT, KW, kOne>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((k_linear_rows<DT, MT, NT, KW, !kMany>), grid, block, 0, stream, a);
}
template <int DT, int MT>
static void launch_rows_nt(const LinearArgs& a, int nt, hipStream_t stream) {
  switch (nt) {
    case 1: return launch_rows<DT, MT, 1>(a, stream);
    case 2: return launch_rows<DT, MT, 2>(a, stream);
    case 3: return launch_rows<DT, MT, 3>(a, stream);
    default:
      if constexpr (MT == 2) launch_rows<DT, MT, 4>(a, stream);
  }
}
template <int DT, int FM, int FN, int WM, int WN>
static void launch_tiles(const LinearArgs& a, hipStream_t stream) {
  const int tiles_m = (int)ceil_div(a.m, 16 * FM * WM), tiles_n = (int)ceil_div(a.n, 16 * FN * WN);
  hipLaunchKernelGGL((k_linear_tiles<DT, FM, FN, WM, WN>), dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * WM * WN), 0,
                     stream, a, tiles_m, tiles_n);
}
template <int DT>
static void launch_linear_dt(const LinearArgs& a, const LinearShape& s, hipStream_t stream) {
  switch (s.tile) {
    case 0: return launch_tiles<DT, 4, 4, 2, 4>(a, stream);
    case 1: return launch_tiles<DT, 4, 3, 2, 4>(a, stream);
    case 2: return launch_tiles<DT, 2, 2, 4, 4>(a, stream);
    case 3: return launch_tiles<DT, 2, 2, 2, 4>(a, stream);
    case 4: return launch_tiles<DT, 2, 2, 2, 2>(a, stream);
  }
  switch (s.mt) {
    case 1: return launch_rows_nt<DT, 1>(a, s.nt, stream);
    case 2: return launch_rows_nt<DT, 2>(a, s.nt, stream);
    default: return launch_rows_nt<DT, 3>(a, s.nt, stream);
  }
}

hipError_t launch_linear(const LinearArgs& a, int dtype, hipStream_t stream) {
  const LinearShape s = linear_shape(a.m, a.n);
  if (dtype == kBF16) launch_linear_dt<kBF16>(a, s, stream);
  else launch_linear_dt<kF16>(a, s, stream);
  return hipGetLastError();
}

}  // namespace lrq
