// GEMM / grouped GEMM of the float32 models (q4f32_1) on the bfloat16 matrix cores, with float32 activations entering
// exactly.
//
// Callers: GroupQuantizeLinear.forward (python/mlc_llm/quantization/group_quantization.py:390-437) and
// moe_matmul.dequantize_group_gemm (python/mlc_llm/op/moe_matmul.py:562-768) of a float32 model.
//
// The float32 matrix instruction runs at a sixteenth of the bfloat16 one's rate and was what bounded these models.  Here x is cut
// into three bfloat16 planes, x = h + m + l: the leading 8 bits of the significand, the next 8 and the last 8, which is all
// 24 of them (the differences are exact), and the weights enter as the integers q - 7 (times 2^-9), which a bfloat16 holds exactly.  The
// three products of a group of 32 weights then carry no rounding but that of the float32 accumulator, smallest plane first,
// and the group's float32 scale multiplies the group's sum: one rounding per group where the kernel this replaced rounded
// every weight.  Three bfloat16 instructions per product instead of one float32 instruction: up to 16 / 3 = 5.3 times the rate.
//
// Workgroup tile BM x BN, K tile = one group.  Activations go global -> registers (two K tiles ahead) -> three planes -> LDS,
// weights global -> registers -> bfloat16 -> LDS, both in the field order in which v_cvt_scalef32_pk_f32_fp8 delivers a
// storage word ((0, 2) (4, 6) (1, 3) (5, 7)): an order of k is free as long as both operands have it.  LDS rows are 80 bytes
// apart: eight consecutive rows of a fragment read start 20 banks apart and meet all banks once.  The split of x is done by
// every workgroup for itself (7.5 vector instructions per element and column tile, two of them for infinities), which is why
// the tile is wide: at 128 x 256 a wave's K tile is 24 matrix instructions (768 cycles) next to 184 to 195 vector instructions (740 to
// 780 cycles), 64 of them the scaling of the results; over whole launches the matrix pipe is busy for 50 to 54 % of the cycles
// and the vector pipe for 51 to 52 %, so that the two together, not memory, bound it.  Interleaving the two by sched_group_barrier (one matrix instruction, 4 / 6 / 8 vector
// instructions) was 4 to 10 % slower than the compiler's own order.
//
// Measured against the float32 matrix instruction's kernel it replaced (us; rows, then N x K): 16 x 4096 x 4096 317 -> 18,
// 64 x 28672 x 4096 352 -> 97, 300 x 4096 x 14336 1197 -> 167, 300 x 28672 x 4096 1189 -> 272 (259 TFLOP/s), 1024 x 28672 x 4096
// 867 (277 TFLOP/s; the float32 matrix instruction's peak is 157).  Relative error against float64 products 1.0e-7 .. 2.1e-7,
// before 8e-7 .. 1.9e-6.
#include "gq_gemm_common.hpp"

namespace gq {

namespace {

typedef __bf16 f3_bf8 __attribute__((ext_vector_type(8)));

struct F32Params {
  const float* x;
  const uint32_t* qw;
  const float* qs;
  const float* bias;      // [N] or null (plain linear only)
  const float* residual;  // [rows, N] or null, may be y (plain linear only)
  float* y;
  float* partial;         // split K: [split][rows][N - n_begin] sums, else null
  const void* indptr;     // [num_experts + 1] or null
  int rows, N, K, ng, nw;
  int num_experts, indptr_i64;
  int kt_per_split;
  int n_begin, n_end;     // columns of this launch
};

constexpr int kRow = 40;  // halves per LDS row: 32 + 8 of padding

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN)) void gemm_f32_kernel(const F32Params p) {
  constexpr int WAVES_N = BN / WN, NT = 64 * (BM / WM) * WAVES_N;
  constexpr int TM = WM / 32, TN = WN / 32;
  static_assert(BN * 2 == NT, "two threads per weight row");
  constexpr int A_CH = (BM * 4 + NT - 1) / NT;  // chunks of 8 activations per thread and K tile
  constexpr bool A_ALL = BM * 4 % NT == 0;      // (else the upper waves have none)
  static_assert(A_ALL || A_CH == 1, "partial rounds only in the single-round tile");
  extern __shared__ uint4 f3_smem[];
  uint16_t* const lds = reinterpret_cast<uint16_t*>(f3_smem);
  // [stage][plane][BM] rows, [stage][BN] rows, [stage][BN] scales
  auto a_rows = [&](int s) { return lds + s * 3 * BM * kRow; };
  auto w_rows = [&](int s) { return lds + 6 * BM * kRow + s * BN * kRow; };
  float* const sc_lds = reinterpret_cast<float*>(lds + (6 * BM + 2 * BN) * kRow);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;

  // ---- segment and row tile (grouped: the tiles of the experts' segments one after another)
  int seg_lo = 0, seg_hi = p.rows, mt = blockIdx.y, expert = 0;
  if (p.indptr != nullptr) {
    const bool found = locate_segment<BM>(p.indptr, p.indptr_i64, p.num_experts, p.rows, mt, seg_lo, seg_hi, mt, expert);
    if (!found) return;  // (uniform: before any barrier)
  }
  const int m0 = seg_lo + mt * BM, n0 = p.n_begin + blockIdx.x * BN;
  const uint32_t* const qw = p.qw + static_cast<int64_t>(expert) * p.N * p.nw;
  const float* const qs = p.qs + static_cast<int64_t>(expert) * p.N * p.ng;

  // ---- this thread's share of a K tile (rows past the segment and columns past N read valid rows: they reach no live
  //      result and the epilogue drops theirs)
  const float* a_src[A_CH];  // the start of the chunk's row
  int a_k[A_CH], a_dst[A_CH];
  const bool a_active = A_ALL || tid < BM * 4;  // (wave-uniform)
#pragma unroll
  for (int i = 0; i < A_CH; ++i) {
    const int idx = a_active ? tid + NT * i : 0;
    const int r = idx >> 2, ch = idx & 3;
    a_src[i] = p.x + static_cast<int64_t>(min(m0 + r, seg_hi - 1)) * p.K;
    a_k[i] = 8 * ch;
    a_dst[i] = r * kRow + 8 * ch;
  }
  const int wrow = tid >> 1, whalf = tid & 1;
  const int64_t wr = min(n0 + wrow, p.N - 1);
  const uint32_t* const w_src = qw + wr * p.nw + 2 * whalf;
  const float* const s_src = qs + wr * p.ng;

  const int kt0 = blockIdx.z * p.kt_per_split, kt1 = min(p.ng, kt0 + p.kt_per_split);

  struct Stage {
    float4 a[A_CH][2];
    uint2 w;
    float s;
  };
  Stage st[2];
  auto load = [&](int kt_raw, Stage& r) {
    const int kt = min(kt_raw, kt1 - 1);  // (tiles past the end re-read the last one: never multiplied)
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const float* const src = a_src[i] + x_chunk(kt * 32 + a_k[i], p.K);
      r.a[i][0] = *reinterpret_cast<const float4*>(src);
      r.a[i][1] = *reinterpret_cast<const float4*>(src + 4);
    }
    r.w = *reinterpret_cast<const uint2*>(w_src + 4 * kt);
    r.s = s_src[kt];
  };
  auto store = [&](int kt, const Stage& r, int s) {
    if (a_active) {
#pragma unroll
      for (int i = 0; i < A_CH; ++i) {
        const uint32_t keep = kt * 32 + a_k[i] < p.K ? 0xffffffffu : 0u;  // x past K counts as zero
        const float raw[8] = {r.a[i][0].x, r.a[i][0].y, r.a[i][0].z, r.a[i][0].w, r.a[i][1].x, r.a[i][1].y, r.a[i][1].z, r.a[i][1].w};
        float h[8], m[8], l[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t xb = __builtin_bit_cast(uint32_t, raw[e]) & keep;
          const float x = __builtin_bit_cast(float, xb);
          h[e] = __builtin_bit_cast(float, xb & 0xffff0000u);
          const float r1 = __builtin_isinf(x) ? 0.0f : x - h[e];  // (inf - inf: an infinity is all in the first plane)
          m[e] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r1) & 0xffff0000u);
          l[e] = r1 - m[e];
        }
        uint16_t* const at = a_rows(s) + a_dst[i];
        *reinterpret_cast<uint4*>(at) = make_uint4(hi_pair(h[0], h[2]), hi_pair(h[4], h[6]), hi_pair(h[1], h[3]), hi_pair(h[5], h[7]));
        *reinterpret_cast<uint4*>(at + BM * kRow) =
            make_uint4(hi_pair(m[0], m[2]), hi_pair(m[4], m[6]), hi_pair(m[1], m[3]), hi_pair(m[5], m[7]));
        *reinterpret_cast<uint4*>(at + 2 * BM * kRow) =
            make_uint4(hi_pair(l[0], l[2]), hi_pair(l[4], l[6]), hi_pair(l[1], l[3]), hi_pair(l[5], l[7]));
      }
    }
    uint16_t* const wt = w_rows(s) + wrow * kRow + 16 * whalf;
    *reinterpret_cast<uint4*>(wt) = word_minus7(r.w.x);
    *reinterpret_cast<uint4*>(wt + 8) = word_minus7(r.w.y);
    if (whalf == 0) sc_lds[s * BN + wrow] = r.s;
  };

  float16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int frow = lane & 31, fk = 8 * (lane >> 5);
  auto multiply = [&](int s) {
    const uint16_t* const at = a_rows(s) + (wm0 + frow) * kRow + fk;
    const uint16_t* const wt = w_rows(s) + (wn0 + frow) * kRow + fk;
    f3_bf8 bf[TN][2];
    float sc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) bf[j][ks] = *reinterpret_cast<const f3_bf8*>(wt + j * 32 * kRow + 16 * ks);
      sc[j] = sc_lds[s * BN + wn0 + 32 * j + frow];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float16_t d[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) d[j][r] = 0.0f;
#pragma unroll
      for (int pl = 2; pl >= 0; --pl) {  // the smallest plane first
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const f3_bf8 af = *reinterpret_cast<const f3_bf8*>(at + (pl * BM + i * 32) * kRow + 16 * ks);
#pragma unroll
          for (int j = 0; j < TN; ++j) d[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf[j][ks], d[j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(sc[j], d[j][r], acc[i][j][r]);
    }
  };

  load(kt0, st[0]);
  load(kt0 + 1, st[1]);
  store(kt0, st[0], 0);
  load(kt0 + 2, st[0]);
  __syncthreads();
  // K tile kt in LDS stage (kt - kt0) & 1, the next two in registers.  Two tiles per round, so that stages are constants; an
  // odd last tile follows the loop.
  int kt = kt0;
  for (; kt + 2 <= kt1; kt += 2) {
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      store(min(kt + d + 1, kt1 - 1), st[(d + 1) & 1], d ^ 1);
      load(kt + d + 3, st[(d + 1) & 1]);
      multiply(d);
      __syncthreads();
    }
  }
  if (kt < kt1) multiply(0);

  // D[r][c] of a 32 x 32 accumulator: lane c + 32 * ((r / 4) % 2), register 4 * (r / 8) + r % 4
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn0 + j * 32 + (lane & 31);
      const float bias = (p.bias != nullptr && p.partial == nullptr && col < p.N) ? p.bias[col] : 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row < seg_hi && col < p.n_end) {
          const int64_t oi = static_cast<int64_t>(row) * p.N + col;
          const float sum = 512.0f * acc[i][j][r];
          if (p.partial != nullptr) {
            p.partial[(static_cast<int64_t>(blockIdx.z) * p.rows + row) * (p.N - p.n_begin) + (col - p.n_begin)] = sum;
          } else {
            float v = sum + bias;
            if (p.residual != nullptr) v += p.residual[oi];
            p.y[oi] = v;
          }
        }
      }
    }
}

template <int BM, int BN, int WM, int WN>
hipError_t launch_tile(const F32Params& p, int split, hipStream_t s) {
  constexpr size_t lds = size_t(2) * (3 * BM + BN) * kRow * 2 + size_t(2) * BN * 4;
  auto kern = gemm_f32_kernel<BM, BN, WM, WN>;
  if (lds > 65536) {
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kern));
    if (e != hipSuccess) return e;
  }
  const int m_tiles = (p.rows + BM - 1) / BM + (p.indptr != nullptr ? p.num_experts : 0);
  if (m_tiles > 65535) return hipErrorNotSupported;
  note_kernel("gq::gemm_f32_kernel<%d,%d,%d,%d> split=%d", BM, BN, WM, WN, split);
  hipLaunchKernelGGL(kern, dim3((p.n_end - p.n_begin + BN - 1) / BN, m_tiles, split), dim3(64 * (BM / WM) * (BN / WN)), lds, s, p);
  return hipGetLastError();
}

// rows of the tile a problem runs on, and how its K is cut so that most CUs have a workgroup
struct F32Plan {
  int bm, split, kt_per_split;
  int64_t n_head = 0;  // columns that run first, unsplit, as whole rounds of workgroups
};
F32Plan plan_f32(int64_t rows, int64_t N, int64_t K, int64_t num_experts, bool grouped) {
  const int64_t per = grouped ? (rows + num_experts - 1) / num_experts : rows;
  F32Plan plan{per <= 32 ? 32 : (per <= 64 ? 64 : 128), 1, 1 << 28};
  const int ng = static_cast<int>((K + 31) / 32);
  plan.kt_per_split = ng;
  if (grouped) return plan;
  const int bn = plan.bm == 128 ? 256 : 128;
  const int64_t tiles = ((rows + plan.bm - 1) / plan.bm) * ((N + bn - 1) / bn);
  const int64_t want = plan.bm == 32 ? 512 : 256;
  int64_t split = want / tiles;
  if (split > ng / 8) split = ng / 8;  // at least eight K tiles per workgroup
  if (plan.bm == 128 && tiles > 256) {
    // A last round of workgroups costs a whole round however few they are (28672 x 4096: 224 tiles 178 us, 336 tiles 334).  The
    // columns of the whole rounds then run on their own, and the K of the rest is cut so that it fills the chip once: worth it
    // while that shorter round, the sums it writes and reads back and the two more launches stay below 0.85 of a round
    // (a round: 1.3 us per K tile; 28672 x 4096 at 300 / 640 / 777 rows: one launch 334 / 535 / 708 us, so 272 / 453 / 625).
    const int64_t mt = (rows + 127) / 128, nt = (N + 255) / 256, head = tiles / 256 * 256 / mt, rest = mt * (nt - head);
    const int64_t cut = rest > 0 ? (256 / rest < ng / 8 ? 256 / rest : ng / 8) : 0;
    if (head > 0 && cut > 1) {
      const double round_us = 1.3 * ng, sums_us = 10.0 + 2e-6 * static_cast<double>(cut * rows * (N - head * 256));
      if (round_us / static_cast<double>(cut) + sums_us < 0.85 * round_us) {
        plan.n_head = head * 256;
        split = cut;
      }
    }
  }
  if (split <= 1) return plan;
  plan.kt_per_split = (ng + static_cast<int>(split) - 1) / static_cast<int>(split);
  plan.split = (ng + plan.kt_per_split - 1) / plan.kt_per_split;
  return plan;
}

}  // namespace

// columns [N - cols, N) of y [rows, N] = sum over slices of part[slice][rows][cols] + bias + residual, all float32 (y may be the
// residual)
__global__ __launch_bounds__(256) void splitk_reduce_f32_kernel(const float* __restrict__ part, int slices, int64_t count, int cols, int N,
                                                                const float* __restrict__ bias, const float* residual, float* y) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < count; i += stride) {
    float v = part[i];
    for (int sl = 1; sl < slices; ++sl) v += part[sl * count + i];
    const int64_t o = cols == N ? i : (i / cols) * N + (N - cols) + i % cols;
    if (bias != nullptr) v += bias[o % N];
    if (residual != nullptr) v += residual[o];
    y[o] = v;
  }
}

hipError_t launch_splitk_reduce_f32(const float* part, int slices, int64_t rows, int64_t cols, int64_t N, const float* bias,
                                    const float* residual, float* y, hipStream_t s) {
  const int64_t count = rows * cols, blocks = (count + 255) / 256;
  hipLaunchKernelGGL(splitk_reduce_f32_kernel, dim3(static_cast<unsigned>(blocks > 8192 ? 8192 : blocks)), dim3(256), 0, s, part,
                     slices, count, static_cast<int>(cols), static_cast<int>(N), bias, residual, y);
  return hipGetLastError();
}

int64_t gemm_f32_workspace_bytes(int64_t rows, int64_t N, int64_t K) {
  if (rows < 1 || N < 1 || K < 1 || (K & 7) != 0) return 0;
  const F32Plan plan = plan_f32(rows, N, K, 1, false);
  return plan.split > 1 ? static_cast<int64_t>(plan.split) * rows * (N - plan.n_head) * 4 : 0;
}

hipError_t launch_gemm_f32(const GemmArgs& a, hipStream_t s) {
  if (a.bits != 4 || a.group_size != 32 || (a.K & 7) != 0 || a.K == 0 || a.rows < 1) return hipErrorNotSupported;
  if ((reinterpret_cast<uintptr_t>(a.x) & 15) != 0 || (reinterpret_cast<uintptr_t>(a.q_weight) & 7) != 0) return hipErrorNotSupported;
  F32Params p{};
  p.x = reinterpret_cast<const float*>(a.x);
  p.qw = a.q_weight;
  p.qs = reinterpret_cast<const float*>(a.q_scale);
  p.bias = reinterpret_cast<const float*>(a.bias);
  p.residual = reinterpret_cast<const float*>(a.residual);
  p.y = static_cast<float*>(a.y);
  p.indptr = a.indptr; p.indptr_i64 = a.indptr_i64; p.num_experts = static_cast<int>(a.num_experts);
  p.rows = static_cast<int>(a.rows); p.N = static_cast<int>(a.N); p.K = static_cast<int>(a.K);
  p.ng = (p.K + 31) / 32;
  p.nw = 4 * p.ng;
  F32Plan plan = plan_f32(a.rows, a.N, a.K, a.num_experts, a.indptr != nullptr);
  if (plan.split > 1) {
    if (a.workspace != nullptr && (reinterpret_cast<uintptr_t>(a.workspace) & 3) == 0 &&
        a.workspace_bytes >= static_cast<int64_t>(plan.split) * a.rows * (a.N - plan.n_head) * 4) {
      p.partial = static_cast<float*>(a.workspace);
    } else {
      plan.split = 1;
      plan.kt_per_split = p.ng;
      plan.n_head = 0;
    }
  }
  p.n_end = p.N;
  if (plan.n_head > 0) {
    F32Params head = p;
    head.partial = nullptr;
    head.kt_per_split = p.ng;
    head.n_end = static_cast<int>(plan.n_head);
    const hipError_t e = launch_tile<128, 256, 64, 64>(head, 1, s);
    if (e != hipSuccess) return e;
    p.n_begin = head.n_end;
  }
  p.kt_per_split = plan.kt_per_split;
  const hipError_t e = plan.bm == 32   ? launch_tile<32, 128, 32, 32>(p, plan.split, s)
                       : plan.bm == 64 ? launch_tile<64, 128, 32, 64>(p, plan.split, s)
                                       : launch_tile<128, 256, 64, 64>(p, plan.split, s);
  if (e != hipSuccess || p.partial == nullptr) return e;
  return launch_splitk_reduce_f32(p.partial, plan.split, a.rows, a.N - plan.n_head, a.N, p.bias, p.residual, p.y, s);
}

}  // namespace gq
