// Pieces shared by the MFMA GEMM kernels: scheme traits, kernel parameters, the segment walk of
// the grouped (MoE) form and the in-register dequantisation of one group.
#pragma once

#include "gq_common.hpp"
#include "gq_internal.hpp"

namespace gq {

template <int BITS>
struct GemmTraits;
template <>
struct GemmTraits<4> {
  static constexpr int G = 32;
};
template <>
struct GemmTraits<3> {
  static constexpr int G = 40;
};

struct GemmParams {
  const uint16_t* x;
  const uint32_t* qw;
  const uint16_t* qs;
  const uint16_t* bias;
  const uint16_t* residual;  // [rows, N] or null
  void* y;
  const void* indptr;
  int64_t expert_w_stride, expert_s_stride;
  int rows, N, K, ng, nw;
  int num_experts;
  int out_f32, indptr_i64;
  // split-K: workgroup z multiplies K tiles [z * kt_per_split, (z + 1) * kt_per_split) and, when
  // `partial` is set, leaves its fp32 tile in partial[z][rows][part_cols] for the reduction kernel
  float* partial;
  int kt_per_split;
  int bm_hint;  // rows, columns per tile chosen by plan_split_k (0: regular tiles)
  int bn_hint = 0;
  // Fused gate/up form: y[rows, N / 2] = silu(x . W[j]) * (x . W[N / 2 + j]).  A tile's columns walk
  // the stored rows in blocks of 32 gate rows then the matching 32 up rows, so both halves of an
  // output element sit in the same lane and register of neighbouring 32 x 32 accumulators (blocks of
  // 16 + 16 in the one tile whose waves own a single accumulator).
  int paired;
  const int32_t* x_rows;  // null, or the row of x each activation row reads (int32 [rows])
  int x_src_rows;         // rows of x when x_rows is set
  int bf16;               // x, q_scale, bias and a 16-bit y are bfloat16 (q4bf16_* models), not float16
  // columns (in tile order) this launch covers: [n_begin, n_end), n_end = 0 for all; a launch can leave the columns
  // of its last, partly filled round of workgroups to a second launch with another tile
  int n_begin = 0;
  // (set by the launcher, which knows the tile) the column tile from which on a launch of both halves of the N, below, is in the
  // second one, and how far that one lies ahead; a launch of adjoining columns counts as all in the second
  int hop_tile = 0, hop = 0;
  int part_cols = 0;  // columns of this launch (the partial sums' row length)
  // every byte offset into x, one expert's q_weight and q_scale fits 32 bits, and K is whole K tiles of two groups
  // (set by the launcher; lets interior workgroups address with a uniform base plus a 32-bit lane offset)
  int fast_ok = 0;
  uint32_t x_bytes = 0;  // size of x (the form without zero-selects, whose offsets fit 32 bits)
  int n_end = 0;
  // columns [half_lo, half_hi) of both halves of the N of a plain matmul, half_hi = 0 for all.  Of a gate_up projection these are the
  // columns [2 half_lo, 2 half_hi) in tile order, so that the fused form, whose launches are cut there, adds up every element in the
  // order in which the plain matmul does.
  int half_lo = 0, half_hi = 0;
};

// column c of the block-interleaved order above -> stored weight row (clamped into its half).
// PB: gate rows per block; 32 where a wave owns pairs of 32-column accumulators, 16 where it owns a
// single one (then lanes l and l ^ 16 hold the two halves of an output element).
template <int PB>
__device__ __forceinline__ int gate_up_row_blk(int c, int N) {
  const int half = N >> 1;
  const int o = min((c / (2 * PB)) * PB + (c % PB), half - 1);
  return (c & PB) ? half + o : o;
}

// partial[split][count / cols][cols] -> y [rows, N]: all columns, or (HALVES, cols < N) the last cols / 2 of either half
template <bool HALVES>
__global__ void splitk_reduce_kernel(const float* partial, int split, int64_t count, int cols, int N,
                                     const uint16_t* bias, const uint16_t* residual, void* y, int out_f32, int bf16);
// fused gate/up form: partial[split][rows][cols] in the block-interleaved column order (its last block filled up) -> the columns of
// y [rows, N / 2] from n_begin / 2 on
__global__ void splitk_reduce_silu_kernel(const float* partial, int split, int64_t rows, int cols, int N, int n_begin, int pb,
                                          uint16_t* y, int bf16);
// gate rows per column block of the tile planned for a matmul: 16 in the one of 32 rows, whose waves own a single accumulator, else 32
constexpr int pair_block(int bm) { return bm == 32 ? 16 : 32; }

// How a plain GEMM is cut: its tile and K splits.
struct SplitPlan {
  int bm, bn;        // 0: no plan, use the regular tiles
  int split;         // workgroups along K (1: no reduction pass)
  int kt_per_split;  // K tiles (2 groups each) per workgroup
  // the first n_head columns, or the first n_head / 2 of either half, run first, unsplit, as whole rounds of workgroups on a tile of
  // their own; bm, bn and split are for the rest
  int64_t n_head = 0;
  bool halves = false;
  int head_bm = 0, head_bn = 0;
};
// scratch_bytes: what the partial sums of a split may take
SplitPlan plan_split_k(int64_t rows, int64_t N, int64_t K, int bits, int group_size, bool grouped, int bf16, int64_t scratch_bytes);
constexpr int64_t kMaxSplitBytes = int64_t(32) << 20;  // no plan of the q4 cost model asks for more

// ---- float32 models: weights as bfloat16 integers

typedef float fp8_f2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t hi_pair(float a, float b) {  // upper halves of two float32: (a, b) as bfloat16, truncated
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}

// one storage word -> 8 bfloat16 numbers (q - 7) 2^-9 in the order (0, 2) (4, 6) (1, 3) (5, 7).  A byte 0 .. 15 read as an fp8
// (e4m3) number is that many 2^-9: the subnormals, then the first binade, whose steps are the same.  The 2^-9 stays on until
// the result is stored: a group's sum is then at most half the largest |x| in it and cannot overflow before its scale is applied.
__device__ __forceinline__ uint4 word_minus7(uint32_t w) {
  constexpr float k7 = 7.0f / 512.0f;
  const uint32_t t0 = w & 0x0f0f0f0fu, t1 = (w >> 4) & 0x0f0f0f0fu;
  const fp8_f2 a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(t0, 1.0f, false), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(t0, 1.0f, true);
  const fp8_f2 c = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(t1, 1.0f, false), d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(t1, 1.0f, true);
  return make_uint4(hi_pair(a.x - k7, a.y - k7), hi_pair(b.x - k7, b.y - k7), hi_pair(c.x - k7, c.y - k7),
                    hi_pair(d.x - k7, d.y - k7));
}

// One group (4 storage words) -> G halves in natural k order, (q - m) * s with fp16 rounding.
template <int BITS>
__device__ __forceinline__ void dequant_group(const uint4 w4, const uint16_t scale_bits,
                                              uint32_t* __restrict__ out /* G/2 half pairs */) {
  constexpr uint32_t kMagic = 0x64006400u;  // 1024.0 in both halves
  const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
  const _Float16 s = __builtin_bit_cast(_Float16, scale_bits);
  const half2_t s2 = {s, s};
  if (BITS == 4) {
    const half2_t off = {static_cast<_Float16>(-1031.0f), static_cast<_Float16>(-1031.0f)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t t1 = w[i] >> 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // byte j of w -> low half (field 2j in its low nibble), byte j of w>>4 -> high half
        const uint32_t sel = 0x0c000c00u | ((4u + j) << 16) | static_cast<uint32_t>(j);
        const uint32_t r = and_or(__builtin_amdgcn_perm(t1, w[i], sel), 0x000f000fu, kMagic);
        out[4 * i + j] = as_u32((as_half2(r) + off) * s2);
      }
    }
  } else {
    const half2_t off = {static_cast<_Float16>(-1027.0f), static_cast<_Float16>(-1027.0f)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 5; ++j) {
        const uint32_t t = w[i] >> (6 * j);
        const uint32_t r = and_or(t << 13, 0x00070000u, and_or(t, 0x00000007u, kMagic));
        out[5 * i + j] = as_u32((as_half2(r) + off) * s2);
      }
    }
  }
}


// 16-byte chunk c (0..4) of a q3 group: halves 8c .. 8c+7 = pairs 4c .. 4c+3 of the group, pair p being
// fields (2j, 2j+1) of word p / 5 with j = p % 5 (a pair never straddles two words).
__device__ __forceinline__ void dequant_chunk3(const uint4 w4, const uint16_t scale_bits, const int c,
                                               uint32_t* __restrict__ out) {
  constexpr uint32_t kMagic = 0x64006400u;
  const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
  const _Float16 s = __builtin_bit_cast(_Float16, scale_bits);
  const half2_t s2 = {s, s};
  const half2_t off = {static_cast<_Float16>(-1027.0f), static_cast<_Float16>(-1027.0f)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int pr = 4 * c + i;
    const uint32_t t = w[pr / 5] >> (6 * (pr % 5));
    const uint32_t r = and_or(t << 13, 0x00070000u, and_or(t, 0x00000007u, kMagic));
    out[i] = as_u32((as_half2(r) + off) * s2);
  }
}

// One q4 storage word -> 8 halves in natural k order (4 half pairs), (q - 7) * s.
__device__ __forceinline__ void dequant_word4(const uint32_t w, const uint16_t scale_bits,
                                              uint32_t* __restrict__ out) {
  constexpr uint32_t kMagic = 0x64006400u;
  const _Float16 s = __builtin_bit_cast(_Float16, scale_bits);
  const half2_t s2 = {s, s};
  const half2_t off = {static_cast<_Float16>(-1031.0f), static_cast<_Float16>(-1031.0f)};
  const uint32_t t1 = w >> 4;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t sel = 0x0c000c00u | ((4u + j) << 16) | static_cast<uint32_t>(j);
    const uint32_t r = and_or(__builtin_amdgcn_perm(t1, w, sel), 0x000f000fu, kMagic);
    out[j] = as_u32((as_half2(r) + off) * s2);
  }
}

// bfloat16 models (q4bf16_*): the same, with the product (q - m) * s formed exactly in float32
// (a 4-bit by an 8-bit significand) and rounded to a bf16 pair by v_cvt_pk_bf16_f32, which is the
// rounding GroupQuantize._dequantize applies in that dtype.  scale_bits are bfloat16 bits.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  const float2_t f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}
__device__ __forceinline__ uint16_t bf16_bits_of(float v) {
  return static_cast<uint16_t>(bf16_pair(v, 0.0f) & 0xffffu);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
  return __builtin_bit_cast(float, static_cast<uint32_t>(b) << 16);
}
__device__ __forceinline__ void dequant_word4_bf16(const uint32_t w, const uint16_t scale_bits,
                                                   uint32_t* __restrict__ out) {
  const float s = bf16_to_f32(scale_bits), ms = -7.0f * s;
  const uint32_t t0 = w & 0x0f0f0f0fu, t1 = (w >> 4) & 0x0f0f0f0fu;  // even / odd fields, one per byte
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float lo = static_cast<float>((t0 >> (8 * j)) & 0xffu), hi = static_cast<float>((t1 >> (8 * j)) & 0xffu);
    out[j] = bf16_pair(fmaf(lo, s, ms), fmaf(hi, s, ms));
  }
}
template <int BITS>
__device__ __forceinline__ void dequant_group_bf16(const uint4 w4, const uint16_t scale_bits,
                                                   uint32_t* __restrict__ out /* G/2 bf16 pairs */) {
  using S = Scheme<BITS>;
  constexpr int E = S::kElem;
  const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
  const float s = bf16_to_f32(scale_bits), ms = -static_cast<float>(S::kMaxInt) * s;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < E / 2; ++j) {
      const float lo = static_cast<float>((w[i] >> (2 * j * BITS)) & S::kMask);
      const float hi = static_cast<float>((w[i] >> ((2 * j + 1) * BITS)) & S::kMask);
      out[(E / 2) * i + j] = bf16_pair(fmaf(lo, s, ms), fmaf(hi, s, ms));
    }
}

// The t-th row tile of BM rows among the experts' segments, taken one after another (python/mlc_llm/op/moe_matmul.py:653-679 of
// the reference does the same walk per tile): its segment [seg_lo, seg_hi), its number mt within the segment, its expert.  False
// when there are fewer tiles; the launch has one row of workgroups per tile that there could be, and most of the surplus ends
// here.  Every wave looks at 64 experts at a time, a lane each: walked expert by expert, each step waits for its own two loads,
// and that walk was longer than the multiplication for many small experts (128 experts of 2048 x 768, 24 rows each: 147 us on
// 32-row tiles for 113 MB of weights, so 44).
template <int BM>
__device__ __forceinline__ bool locate_segment(const void* indptr, int indptr_i64, int num_experts, int rows, int t, int& seg_lo,
                                               int& seg_hi, int& mt, int& expert) {
  const int lane = threadIdx.x & 63;
  for (int e0 = 0; e0 < num_experts; e0 += 64) {
    int lo = 0, hi = 0;
    if (e0 + lane < num_experts) {
      int64_t l, h;
      if (indptr_i64) {
        l = static_cast<const int64_t*>(indptr)[e0 + lane];
        h = static_cast<const int64_t*>(indptr)[e0 + lane + 1];
      } else {
        l = static_cast<const int32_t*>(indptr)[e0 + lane];
        h = static_cast<const int32_t*>(indptr)[e0 + lane + 1];
      }
      l = l < 0 ? 0 : (l > rows ? rows : l);  // a corrupt indptr must not leave the tensors
      h = h < l ? l : (h > rows ? rows : h);
      lo = static_cast<int>(l);
      hi = static_cast<int>(h);
    }
    const int tiles = (hi - lo + BM - 1) / BM;
    int upto = tiles;  // tiles of this block's experts up to and including this lane's
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(upto, off);
      if (lane >= off) upto += o;
    }
    const unsigned long long past = __ballot(upto > t);
    if (past != 0) {
      const int l = __builtin_ctzll(past);
      seg_lo = __builtin_amdgcn_readlane(lo, l);
      seg_hi = __builtin_amdgcn_readlane(hi, l);
      mt = t - (__builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(tiles, l));
      expert = e0 + l;
      return true;
    }
    t -= __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// the same for a launch's parameters; plain linear: one segment
template <int BM>
__device__ __forceinline__ bool locate_tile(const GemmParams& p, int t, int& seg_lo, int& seg_hi,
                                            int& mt, int& expert) {
  seg_lo = 0; seg_hi = p.rows; mt = t; expert = 0;
  if (p.indptr == nullptr) return t * BM < p.rows;
  return locate_segment<BM>(p.indptr, p.indptr_i64, p.num_experts, p.rows, t, seg_lo, seg_hi, mt, expert);
}

// software-pipelined kernel family (needs K % 8 == 0); hipErrorNotSupported otherwise
hipError_t launch_gemm_pipe(const GemmParams& p, int bits, hipStream_t s);

}  // namespace gq
