// Matmul for 5..64 activation rows against streamed q4f16_1 (q4bf16_1) weights (batched decode, short prefill chunks):
// v_mfma_f32_16x16x32_f16 on UNSCALED weight operands, the group's scale applied to the matrix instruction's result,
// the activations resident in registers.
//
// Same callers as the few-row tiles of gq_gemm_pipe.hip and as gq_skinny.hip (GroupQuantizeLinear.forward,
// python/mlc_llm/quantization/group_quantization.py:390-437, for the batch buckets above the low-batch GEMV of
// python/mlc_llm/compiler_pass/low_batch_specialization.py:22-57).
//
// Those kernels materialise fp16 weights (q - 7) * s for the matrix core: unpack, subtract, multiply, and for the
// tiles that go through LDS a byte permute into natural k order, 3.4 to 5 vector instructions per weight and lane,
// which is what bounds them in this regime (the weight stream itself would take half their time).  Here the matrix
// instruction multiplies x by the integers 1024 + q (q4 fields OR-ed into the mantissa of 1024.0: one v_and_or per
// field pair, odd fields come out times 16 and meet activations divided by 16), one instruction per quantisation
// group, so that the group's scale multiplies four accumulator values per lane afterwards and the offset
// -(1024 + 7) * sum(x) of the group enters as the instruction's C operand: the arithmetic of the 4x4x4 kernels
// (gq_quadrow.hip), about ten vector instructions per group of 512 weights and wave at 16 rows.
//
// B operand of instruction g = group g of 16 weight rows (a "tile"): lane (c = lane % 16, j = lane / 16) supplies the
// 8 k of storage word j of row c.  A lane LOADS a whole group (128 bits: lane (c, j) group 4 * step + j of row c, so a
// wave instruction covers 16 rows x 64 contiguous bytes); a 4 x 4 transpose across the four 16-lane rows
// (v_permlane32_swap, v_permlane16_swap: four instructions) then leaves register m of lane (c, j) with word j of group
// 4 * step + m.  A operand = 16 activation rows x the same 32 k: lane (i, j) holds x[i][32 g + 8 j ..] in the pair
// order of the unpack masks, the odd fields' activations divided by 16; x is read once, in whole cache lines, and comes into
// that order through a wave's own 2 KiB of LDS (against 16-byte reads of sixteen rows at a time: 28672 x 4096 at 16 / 32 rows
// 22.6 / 30.1 -> 20.5 / 28.2 us, 6144 x 4096 10.6 / 14.8 -> 8.6 / 10.4, 4096 x 4096 9.6 / 13.9 -> 7.5 / 9.9).  The offset
// term needs no cross-lane sum either: the same matrix instruction on a constant B operand (-1031 for the even fields,
// -16 * 71 for the odd ones) leaves -(offset) of rows 4 j .. 4 j + 3 in
// lane (c, j), which is where the C operand wants it.  D: lane (c, j) receives rows 4 j .. 4 j + 3 of column c, four
// values of the lane's own weight row: its scale of the group multiplies them into the fp32 accumulators.
//
// That is the form of one batch tile with the offsets kept (float16).  The float16 forms without them (two batch tiles, and two rounds
// at most: midonce_kernel) take the offset and the factor 16 off the weight operand, four packed instructions per group, and x as it is.
//
// A wave owns U consecutive groups of K (its x: 4 registers per group and batch tile, the offsets as many where they are
// kept) and walks tiles with RT tiles of loads in flight.  The 16 waves of a workgroup (8 of twice the K where the walk
// is long) are KW neighbouring K shares x 16 / KW tiles side by side; results wait in LDS until the walk is over (a store inside the walk would turn every wait
// for a load into a wait for all of them), then the K shares are added and leave.  K beyond a workgroup's KW * U groups
// is walked in phases: each phase loads its share of x and visits every tile again (its own K range of it: the weights
// are still read once), adding to the sums in LDS.  Expert segments (moe_matmul.dequantize_group_gemm,
// python/mlc_llm/op/moe_matmul.py:562-768): grid row = expert, rows from indptr, more rows than the batch tiles hold in
// passes.  Float32 models (q4f32_1): x = h + m + l, three bfloat16 planes that together are x exactly, so five activation
// rows make fifteen rows of the bfloat16 operand; the weights are the integers q, times 2^-9 (v_cvt_scalef32_pk_bf16_fp8, two
// fields per instruction), the offset -7 * sum(x), and the planes of a row meet where the K shares do: products and scales as exact as
// float32 dot products make them (relative error 8e-8 against float64 at K = 4096), at the price of the weight stream
// (4 rows: 28672 x 4096 76.7 us on the dot-product kernel's passes -> 23, 128256 x 4096 237 -> 77, 4096 x 14336 1168 -> 18.4).
// The fused gate/up form walks a gate tile and its up tile in consecutive rounds and folds silu(gate) * up into
// the step that adds the K shares.
#include "gq_gemm_common.hpp"
#include "gq_gemv_common.hpp"

namespace gq {

namespace {

struct MidParams {
  const uint16_t* x;
  const uint32_t* qw;
  const uint16_t* qs;
  const uint16_t* bias;
  const uint16_t* residual;
  void* y;
  const void* indptr;      // null: one segment [0, rows)
  const int32_t* x_rows;   // null, or the row of x each activation row reads
  const int32_t* ids;      // (float32) null, or one expert per row: grid row = activation row, its expert ids[row]
  int64_t expert_w_stride, expert_s_stride;
  int rows, N, K, ng, nw;
  int ntiles;              // tiles of 16 weight rows a walk visits: ceil(N / 16); the fused gate/up form: N / 32 pairs
  int rounds;              // tiles a wave walks per chunk (a multiple of the tiles in flight; the fused form: even)
  int chunks;              // chunks of rounds (1 when K takes phases)
  int total_rounds;        // rounds in all chunks: the last one may be shorter (a multiple of the tiles in flight too)
  int phases;              // passes over K (a workgroup covers KW * U groups per phase)
  int slices;              // workgroups along K (plain linears with a workspace: grid z; each covers slice_shares shares of
                           // K, one phase's worth at most, and leaves fp32 partial sums [slice][rows][N] in y for the reduction kernel)
  int slice_shares;        // shares of U groups of K in a slice (without slices: kw, the shares of a phase)
  int kw_log2;             // log2 of the waves that share a tile's K
  int out_f32, paired, indptr_i64, x_src_rows;
  int num_experts, x_one_row;  // with ids: experts in the stack; every row reads row 0 of x
};

// T[j][m] (register m of the lanes 16 j .. 16 j + 15) -> T[m][j]
__device__ __forceinline__ void mid_transpose(uint32_t& r0, uint32_t& r1, uint32_t& r2, uint32_t& r3) {
  auto a = __builtin_amdgcn_permlane32_swap(r0, r2, false, false);  // upper half of r0 <-> lower half of r2
  auto b = __builtin_amdgcn_permlane32_swap(r1, r3, false, false);
  auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);  // odd rows of the first <-> even rows of the second
  auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  r0 = c[0]; r1 = c[1]; r2 = d[0]; r3 = d[1];
}

typedef uint32_t mid_u4 __attribute__((ext_vector_type(4)));

template <bool BF>
__device__ __forceinline__ float4_t mid_mfma(const mid_u4 a, const mid_u4 b, const float4_t c) {
  if constexpr (BF) {
    typedef __bf16 mid_bf8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mid_bf8, a), __builtin_bit_cast(mid_bf8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
  }
}

// the eight fields of a storage word as bfloat16 numbers q 2^-9, fields (0, 2) (4, 6) (1, 3) (5, 7): a byte 0 .. 15 read as an
// fp8 (e4m3) number is that many 2^-9 (subnormals, then the first binade, whose steps are the same), so the scaled
// conversion delivers two fields per instruction.  The 2^-9 stays on until the K shares meet: a group's sum, offset
// included, then stays below the largest |x| in it and cannot overflow before its scale is applied.
__device__ __forceinline__ mid_u4 mid_word_bf16(uint32_t w) {
  const uint32_t t0 = w & 0x0f0f0f0fu, t1 = (w >> 4) & 0x0f0f0f0fu;
  return mid_u4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(t0, 1.0f, false)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(t0, 1.0f, true)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(t1, 1.0f, false)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(t1, 1.0f, true))};
}

// NBT: batch tiles of 16 rows (float32: of five); U: groups of K a wave owns (8 or, with eight waves, 16); RT: tiles of loads in flight per wave;
// DT: the model's type (x, scales, bias, residual and the result).  bfloat16: 0x4300 | q is the bfloat16 128 + q, so
// every field is shifted down to bit 0 of its half (no x16 trick, x is not rescaled) and all carry the offset 128 + 7;
// KEEP_C: the offset terms stay in registers (else, in bfloat16 and float32 the constant-operand instruction runs again in front of each group, in float16
// the weight operand is rid of the offset);
// PHASED: K takes more than one phase (the sums of all of a wave's rounds stay in LDS between phases: one chunk of rounds);
// else a wave's rounds come in chunks of p.rounds, each followed by the step that adds the K shares and stores, with x
// and the ring of loads carried across
// WV: waves of a workgroup (16 or 8)
// ONCE: every tile of a wave is in its first ring of loads (p.rounds == RT): nothing is loaded behind it (a round without a tile is
// walked over zeros all the same)
// OWN_X (float32; the phases always): a lane loads its own x instead of taking it from LDS
template <int NBT, int U, int RT, bool KEEP_C, bool PHASED, int DT, int WV, bool ONCE, bool OWN_X>
__device__ __forceinline__ void midrow_body(const MidParams& p) {
  static_assert(!ONCE || (!PHASED && DT != MODEL_F32), "one chunk, and no look at the last round's sums");
  constexpr bool BF = DT == MODEL_BF16, F32 = DT == MODEL_F32;
  static_assert(U % 8 == 0 && RT % 2 == 0 && (U == 8 || !F32), "scales in whole 16-byte loads; float32 loads them for pairs of tiles");
  constexpr int STEPS = U / 4;
  constexpr int EL = F32 ? 4 : 2;     // bytes of an activation, a scale
  constexpr bool PAIR = F32;        // scales come for pairs of tiles (see issue_scales)
  constexpr int BR = F32 ? 5 : 16;    // activation rows a batch tile holds
  constexpr int SW = F32 ? U : U / 2; // registers of a row's U scales
  // the weight operands carry no offset (else it is the C operand's, kept or made anew ahead of each group)
  constexpr bool SUB = !KEEP_C && DT == MODEL_F16;
  constexpr uint32_t kMagic = BF ? 0x43004300u : 0x64006400u;
  // element i of a tensor in the model dtype
  auto elem = [](const uint16_t* t, int64_t i) -> float {
    if constexpr (F32) return reinterpret_cast<const float*>(t)[i];
    else return BF ? bf2f(t[i]) : h2f(t[i]);
  };
  extern __shared__ float4 res_lds[];  // [round][wave][NBT][64 lanes]

  // (the wave index in a scalar register: everything derived from it - K share, tiles, the loads' scalar offsets - is
  //  then uniform for the compiler as well, which would otherwise wrap every buffer load in a loop over lanes)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, j = lane >> 4;
  const int kw = 1 << p.kw_log2, tw = WV >> p.kw_log2;
  const int ks = wave & (kw - 1), ti = wave >> p.kw_log2;
  const int tstride = gridDim.x * tw;
  const int base = blockIdx.x * tw + ti;  // this wave's first tile (the fused form: its first gate / up pair)
  const int half_tiles = p.N >> 5;        // (the fused form: tiles of gate rows)

  // ---- this workgroup's expert and rows
  int expert = blockIdx.y;
  int seg_lo = 0, seg_hi = p.rows;
  if (F32 && p.ids != nullptr) {
    seg_lo = expert;
    seg_hi = seg_lo + 1;
    expert = min(max(p.ids[seg_lo], 0), p.num_experts - 1);
  } else if (p.indptr != nullptr) {
    if (p.indptr_i64) {
      seg_lo = static_cast<int>(static_cast<const int64_t*>(p.indptr)[expert]);
      seg_hi = static_cast<int>(static_cast<const int64_t*>(p.indptr)[expert + 1]);
    } else {
      seg_lo = static_cast<const int32_t*>(p.indptr)[expert];
      seg_hi = static_cast<const int32_t*>(p.indptr)[expert + 1];
    }
    seg_lo = max(seg_lo, 0);
    seg_hi = min(seg_hi, p.rows);
  }
  if (seg_hi <= seg_lo) return;  // (uniform: before any barrier)

  // ---- weight / scale loads of one tile, through buffer descriptors: the tensor in scalar registers, the tile as the
  //      scalar offset, one 32-bit lane offset for all tiles.  The descriptors carry the tensors' sizes: rows past N read
  //      zeros, and a tile past the end (a wave's last rounds issue for tiles that do not exist) gets the tensor's size
  //      as its offset, which puts every lane out of range: zeros, and no memory traffic.  Nothing of either is kept.
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const uint32_t w_bytes = static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.nw) * 4u;
  const uint32_t s_bytes = static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.ng) * EL;
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(p.qw + expert * p.expert_w_stride), short(0), static_cast<int>(w_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.qs + expert * p.expert_s_stride * (EL / 2)), short(0), static_cast<int>(s_bytes), 0x00020000);
  const uint32_t w_tile = 16u * static_cast<uint32_t>(p.nw) * 4u, s_tile = 16u * static_cast<uint32_t>(p.ng) * EL;
  // round r of this wave -> tile (the fused form: rounds 2 i, 2 i + 1 = gate tile, up tile of pair i); -1 past the end.
  // Straight-line scalar arithmetic: a branch here would sit inside the walk, where every join makes the wait for one
  // tile's loads a wait for all of them.
  const int pair_shift = p.paired ? 1 : 0;
  const int up_tiles = p.paired ? half_tiles : 0;
  auto tile_from = [&](int first, int r) -> int {
    const int item = first + (r >> pair_shift) * tstride;
    const int t = item + (r & pair_shift) * up_tiles;
    return item < p.ntiles ? t : -1;
  };
  auto tile_of = [&](int r) -> int { return tile_from(base, r); };

  constexpr uint32_t kLoLo = 0x05040100u, kHiHi = 0x07060302u;
  const half2_t r16 = {static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
  const mid_u4 neg_off = F32  ? mid_u4{0xbc60bc60u /* -7 2^-9 */, 0xbc60bc60u, 0xbc60bc60u, 0xbc60bc60u}
                         : BF ? mid_u4{0xc307c307u /* -135 */, 0xc307c307u, 0xc307c307u, 0xc307c307u}
                              : mid_u4{0xe407e407u /* -1031 */, 0xe407e407u, 0xe470e470u /* -16 * 71 */, 0xe470e470u};

  for (int pass_lo = seg_lo; pass_lo < seg_hi; pass_lo += BR * NBT) {
    for (int ph = 0; ph < (PHASED ? p.phases : 1); ++ph) {
      // (slices > 1: each p.slice_shares of K's shares; the phases: kw each.  Uniform; ng % U == 0: a share is whole or empty)
      const int ga_raw = (static_cast<int>(blockIdx.z) * p.slice_shares + ph * kw + ks) * U;
      const bool k_live = ga_raw < p.ng && (PHASED || ks < p.slice_shares);
      const int ga = k_live ? ga_raw : p.ng - U;
      // (a wave without a share of K walks tiles past the end, see above: it loads zeros, and no traffic)
      const int walk_base = k_live ? base : p.ntiles;
      const int w_lane = (c * p.nw + 4 * (ga + j)) * 4;
      u32x4 w[RT][STEPS];  // (kept as whole register tuples until the point of use, see walk_tile)
      auto issue = [&](int r, u32x4 (&wv)[STEPS]) {
        const int tile = tile_from(walk_base, r);
        const int w_off = static_cast<int>(tile >= 0 ? static_cast<uint32_t>(tile) * w_tile : w_bytes);
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
          wv[st] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_lane + 64 * st, w_off, 0);
        }
      };
      // scales: the U of this lane's row c.  float32 (PAIR): of the tiles of rounds r and r + 1 in one load, lane (c, j) taking
      // half j % 2 of row c of tile j / 2, handed round when a tile's turn comes.  A lane's own 32 bytes would be two loads per
      // tile, which all four lanes of a row make to the same addresses; the exchange halves those requests (with it the
      // texture unit is busy for 48 to 53 % of the cycles, the vector pipe for 44 to 49 %; four rows: 128256 x 4096 88 -> 77 us, 28672 x 4096 28 -> 23, 4096 x 14336 20.1 -> 18.4; the
      // 16-bit scales are one load per tile, and the exchange's registers spill there)
      const int s_lane = (c * p.ng + ga) * EL + (PAIR ? (j & 1) * (U / 2 * EL) : 0);
      constexpr int NS = PAIR ? RT / 2 : RT;
      constexpr int SR = PAIR ? SW / 2 : SW;
      uint32_t sraw[NS][SR];
      auto issue_scales = [&](int r, uint32_t (&sv)[SR]) {
        const int t0 = tile_from(walk_base, r);
        const uint32_t o0 = t0 >= 0 ? static_cast<uint32_t>(t0) * s_tile : s_bytes;
        if constexpr (PAIR) {
          const int t1 = tile_from(walk_base, r + 1);
          const uint32_t o1 = t1 >= 0 ? static_cast<uint32_t>(t1) * s_tile : s_bytes;
          const u32x4 v =
              __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, s_lane + static_cast<int>(j < 2 ? o0 : o1), 0, 0);
          sv[0] = v.x; sv[1] = v.y; sv[2] = v.z; sv[3] = v.w;
        } else {
#pragma unroll
          for (int q = 0; q < SR; q += 4) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, s_lane + 4 * q, static_cast<int>(o0), 0);
            sv[q] = v.x; sv[q + 1] = v.y; sv[q + 2] = v.z; sv[q + 3] = v.w;
          }
        }
      };
      auto issue_all = [&]() {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          issue(r, w[r]);
          if (!PAIR || r % 2 == 0) issue_scales(r, sraw[PAIR ? r / 2 : r]);
        }
      };
      mid_u4 xa[NBT][U];
      float4_t cc[KEEP_C ? NBT : 1][KEEP_C ? U : 1];
      if constexpr (F32) {
        // ---- x as three bfloat16 planes, x = h + m + l: the leading 8 bits of the significand, the next 8, the last 8
        //      (differences of float32 values that share their exponent range are exact, so the planes lose nothing).  A
        //      batch tile's matrix rows are (activation row, plane): row i of the operand is plane i % 3 of row i / 3.
        //      The products of an infinity and their offset are inf - inf: such rows are made anew in redo_odd_rows below.
        const int pl = c % 3;
        static_assert(!F32 || (NBT == 1 && !KEEP_C), "one batch tile, offsets from the operand");
        const int b = pass_lo + c / 3;
        const bool ok = k_live && c < 3 * BR && b < seg_hi;
        uint4 lo[U], hi[U];
        if constexpr (PHASED || OWN_X) {
          const int64_t xr = p.x_one_row ? 0 : x_row(p.x_rows, p.x_src_rows, ok ? b : seg_lo);
          const float* const xrow = reinterpret_cast<const float*>(p.x) + xr * p.K + ga * 32 + 8 * j;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            lo[u] = *reinterpret_cast<const uint4*>(xrow + u * 32);
            hi[u] = *reinterpret_cast<const uint4*>(xrow + u * 32 + 4);
          }
          issue_all();  // (behind the loads of x: those are needed first, and loads retire in issue order)
        } else {
          // Each row's 1 KiB is one load (a lane's own two 16 bytes per group would be sixteen of them, three lanes asking for
          // the same), and the lanes take theirs from LDS: the wave's own slots for the sums of rounds 0 .. 4, a KiB each,
          // are free until its walk begins.  Chunk k of row i sits at chunk k + 3 i: five rows at one k meet no bank twice.
          // (5 rows: 4096 x 4096 11.0 -> 10.3 us, 6144 x 4096 11.4 -> 10.3, 28672 x 4096 23.8 -> 23.2, 128256 x 4096 80.5 -> 78.0, 4096 x 14336
          // 19.4 -> 18.6.  The phases keep sums in these slots, and a lane's own loads.)
          int xl = threadIdx.x & 63;
          asm volatile("" : "+v"(xl));  // (what follows from it is made here, not kept in registers through the walk)
          const int bl = pass_lo + (xl < BR ? xl : 0);
          const int row_of_lane = p.x_one_row ? 0 : static_cast<int>(x_row(p.x_rows, p.x_src_rows, bl < seg_hi ? bl : seg_lo));
          uint4 xw[BR];
#pragma unroll
          for (int i = 0; i < BR; ++i) {
            const int64_t xr = __builtin_amdgcn_readlane(row_of_lane, i);
            xw[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const float*>(p.x) + xr * p.K + ga * 32 + 4 * xl);
          }
          issue_all();
          char* const x_lds = reinterpret_cast<char*>(res_lds) + wave * 1024;
#pragma unroll
          for (int i = 0; i < BR; ++i) *reinterpret_cast<uint4*>(x_lds + i * 16384 + (((xl + 3 * i) & 63) << 4)) = xw[i];
          __builtin_amdgcn_wave_barrier();
          const int xi = min((xl & 15) / 3, BR - 1);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int at = 8 * u + 2 * (xl >> 4) + 3 * xi;
            lo[u] = *reinterpret_cast<const uint4*>(x_lds + xi * 16384 + ((at & 63) << 4));
            hi[u] = *reinterpret_cast<const uint4*>(x_lds + xi * 16384 + (((at + 1) & 63) << 4));
          }
          __builtin_amdgcn_wave_barrier();
        }
        // (masks: selects become branches behind the loads, which wait for all of them, the ring's included)
        uint32_t live_x = ok ? 0xffffffffu : 0u, minus_h = pl > 0 ? 0xffff0000u : 0u, minus_m = pl > 1 ? 0xffff0000u : 0u;
        asm volatile("" : "+v"(live_x), "+v"(minus_h), "+v"(minus_m));
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t raw[8] = {lo[u].x, lo[u].y, lo[u].z, lo[u].w, hi[u].x, hi[u].y, hi[u].z, hi[u].w};
          uint32_t v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t xb = raw[e] & live_x;
            const float r = __builtin_bit_cast(float, xb) - __builtin_bit_cast(float, xb & minus_h);
            const float l = r - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & minus_m);
            v[e] = __builtin_bit_cast(uint32_t, l);
          }
          // fields (0, 2) (4, 6) (1, 3) (5, 7): the order in which the conversion delivers a word
          xa[0][u][0] = __builtin_amdgcn_perm(v[2], v[0], kHiHi);
          xa[0][u][1] = __builtin_amdgcn_perm(v[6], v[4], kHiHi);
          xa[0][u][2] = __builtin_amdgcn_perm(v[3], v[1], kHiHi);
          xa[0][u][3] = __builtin_amdgcn_perm(v[7], v[5], kHiHi);
        }
      } else {
        // ---- this wave's share of x goes out first (it is needed first, and loads retire in issue order).  Lane (i = c, j) of
        //      batch tile bt wants x[row 16 bt + i][32 g + 8 j .. + 7], but loads that way would touch sixteen cache lines
        //      per quarter of a wave: all of x (32 rows of K = 4096) arrives in 5.9 us that way and in 1.7 with eight lanes
        //      side by side on the 128 bytes of a row (a kernel of these loads alone, less its launch).  So load i of a lane is 16 bytes of row 8 (i % 2) +
        //      lane / 8, groups 2 (i / 2) and the next, and a tile of LDS of the wave's own (16 rows x 128 bytes, no barrier:
        //      a wave's LDS instructions execute in order) turns two loads into the operands of two groups.
        uint4 xraw[NBT][U];
        bool x_ok[NBT];
        int xl = threadIdx.x & 63;
        asm volatile("" : "+v"(xl));  // (what follows from it is made here, not kept in registers through the walk)
#pragma unroll
        for (int bt = 0; bt < NBT; ++bt) {
          x_ok[bt] = k_live && pass_lo + 16 * bt + (xl & 15) < seg_hi;
          const uint16_t* xrow[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int b = pass_lo + 16 * bt + 8 * h + (xl >> 3);
            xrow[h] = p.x + x_row(p.x_rows, p.x_src_rows, b < seg_hi ? b : seg_lo) * p.K + ga * 32 + 8 * (xl & 7);
          }
#pragma unroll
          for (int u = 0; u < U; ++u) xraw[bt][u] = *reinterpret_cast<const uint4*>(xrow[u & 1] + (u >> 1) * 64);
        }
        issue_all();

        // ---- x in operand order, (x0, x4) (x2, x6) (x1, x5) / 16 (x3, x7) / 16, and the offset terms
        // (16-byte chunk k of row r sits at chunk k ^ (r / 2 % 8): the reads of sixteen rows at one k then meet no bank twice)
        char* const x_lds = reinterpret_cast<char*>(res_lds) + (p.rounds * NBT * WV + 2 * wave) * 1024;
        const int x_put = (xl >> 3) * 128, x_get = (xl & 15) * 128;
#pragma unroll
        for (int bt = 0; bt < NBT; ++bt) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if (u % 2 == 0) {
              __builtin_amdgcn_wave_barrier();
#pragma unroll
              for (int h = 0; h < 2; ++h)
                *reinterpret_cast<uint4*>(x_lds + x_put + 1024 * h + (((xl & 7) ^ ((4 * h + (xl >> 4)) & 7)) << 4)) = xraw[bt][u + h];
              __builtin_amdgcn_wave_barrier();
#pragma unroll
              for (int h = 0; h < 2; ++h)
                xraw[bt][u + h] = *reinterpret_cast<const uint4*>(x_lds + x_get + (((4 * h + (xl >> 4)) ^ ((xl >> 1) & 7)) << 4));
            }
            uint4 v = xraw[bt][u];
            if (!x_ok[bt]) v = make_uint4(0, 0, 0, 0);
            xa[bt][u][0] = __builtin_amdgcn_perm(v.z, v.x, kLoLo);
            xa[bt][u][1] = __builtin_amdgcn_perm(v.w, v.y, kLoLo);
            xa[bt][u][2] = __builtin_amdgcn_perm(v.z, v.x, kHiHi);
            xa[bt][u][3] = __builtin_amdgcn_perm(v.w, v.y, kHiHi);
            if constexpr (!BF && !SUB) {
              xa[bt][u][2] = as_u32(as_half2(xa[bt][u][2]) * r16);
              xa[bt][u][3] = as_u32(as_half2(xa[bt][u][3]) * r16);
            }
            if constexpr (KEEP_C) cc[bt][u] = mid_mfma<BF>(xa[bt][u], neg_off, float4_t{0.f, 0.f, 0.f, 0.f});
          }
        }
      }

      // one tile from a ring slot; round `next` goes into the registers it leaves
      // (PAIR: first: the first of a pair of tiles; `odd`: the pair's scales after the exchange that splits them by tile, kept for
      //  the second)
      uint32_t odd[SR];
      auto walk_tile = [&](bool first, int next, u32x4 (&wv)[STEPS], uint32_t (&sp)[SR], float4_t (&acc)[NBT]) __attribute__((always_inline)) {
        uint32_t sv[SW];
        if constexpr (PAIR) {
          // to every lane: rows of 16 lanes hold (tile 0 half 0, tile 0 half 1, tile 1 half 0, tile 1 half 1)
#pragma unroll
          for (int q = 0; q < SW / 2; ++q) {
            uint32_t mine = first ? sp[q] : odd[q];
            if (first) {
              auto e = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);  // (0 0, 0 1, 0 0, 0 1) (1 0, 1 1, 1 0, 1 1)
              mine = e[0];
              odd[q] = e[1];
            }
            auto e = __builtin_amdgcn_permlane16_swap(mine, mine, false, false);  // half 0 everywhere, half 1 everywhere
            sv[q] = e[0];
            sv[SW / 2 + q] = e[1];
          }
        } else {
#pragma unroll
          for (int q = 0; q < SW; ++q) sv[q] = sp[q];
        }
#pragma unroll
        for (int bt = 0; bt < NBT; ++bt) acc[bt] = float4_t{0.f, 0.f, 0.f, 0.f};
        // (a zero the compiler cannot see through: the offset instruction would otherwise be hoisted out of the walk,
        //  into the registers this form is there to save)
        float zero = 0.f;
        asm volatile("" : "+v"(zero));
        const float4_t zero4 = {zero, zero, zero, zero};
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
          // (the loaded tuple becomes a new value HERE and is taken apart after that: the in-place lane swaps below
          //  otherwise make the compiler copy parts of a load into other registers right behind the load itself, and
          //  that copy waits for the load)
          u32x4 t = wv[st];
          asm volatile("" : "+v"(t));
          uint32_t r[4] = {t.x, t.y, t.z, t.w};
          mid_transpose(r[0], r[1], r[2], r[3]);
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const int u = 4 * st + m;
            const uint32_t w8 = r[m] >> 8;
            const mid_u4 bw = F32  ? mid_word_bf16(r[m])
                              : BF ? mid_u4{and_or_c(r[m], 0x000f000fu, kMagic), and_or_c(w8, 0x000f000fu, kMagic),
                                            and_or_c(r[m] >> 4, 0x000f000fu, kMagic), and_or_c(r[m] >> 12, 0x000f000fu, kMagic)}
                                   : mid_u4{and_or_c(r[m], 0x000f000fu, kMagic), and_or_c(w8, 0x000f000fu, kMagic),
                                            and_or_c(r[m], 0x00f000f0u, kMagic), and_or_c(w8, 0x00f000f0u, kMagic)};
            float s;
            if constexpr (F32) {
              s = __builtin_bit_cast(float, sv[u]);
            } else {
              const uint16_t sb = static_cast<uint16_t>((u & 1) ? sv[u >> 1] >> 16 : sv[u >> 1] & 0xffffu);
              s = BF ? bf2f(sb) : h2f(sb);
            }
            // (float16 without the kept offsets: they come off the weight operand instead, exactly, four packed instructions per group
            //  whatever the batch tiles, in place of one more matrix instruction per group and batch tile: 1024 + q - 1031 and
            //  (1024 + 16 q) / 16 - 71 are small integers, and x is taken as it is, infinities and the smallest values included)
            mid_u4 bo = bw;
            if constexpr (SUB) {
              const half2_t o_lo = {static_cast<_Float16>(-1031.f), static_cast<_Float16>(-1031.f)};
              const half2_t o_hi = {static_cast<_Float16>(-71.f), static_cast<_Float16>(-71.f)};
              bo[0] = as_u32(as_half2(bw[0]) + o_lo); bo[1] = as_u32(as_half2(bw[1]) + o_lo);
              bo[2] = as_u32(__builtin_elementwise_fma(as_half2(bw[2]), r16, o_hi));
              bo[3] = as_u32(__builtin_elementwise_fma(as_half2(bw[3]), r16, o_hi));
            }
#pragma unroll
            for (int bt = 0; bt < NBT; ++bt) {
              float4_t c0;
              if constexpr (KEEP_C) c0 = cc[bt][u];
              else if constexpr (SUB) c0 = float4_t{0.f, 0.f, 0.f, 0.f};
              else c0 = mid_mfma<BF || F32>(xa[bt][u], neg_off, zero4);
              const float4_t d = mid_mfma<BF || F32>(xa[bt][u], SUB ? bo : bw, c0);
#pragma unroll
              for (int q = 0; q < 4; ++q) acc[bt][q] = fmaf(s, d[q], acc[bt][q]);
            }
          }
        }
        // (after the arithmetic: the loads then land in the very registers the tile has left, with no copies whose
        //  wait would drain the queue)
        if constexpr (!ONCE) {
          issue(next, wv);
          if (!PAIR || first) issue_scales(next, sp);
        }
      };

      // (float32) the sums of a chunk of rounds in the rows whose shares of x hold infinities or NaNs, which are then all that
      // counts: from the weights with their offset taken off, an infinity's products are infinities and, with a weight of zero, NaN.
      // Rare, so the tiles are read a second time and x with them.  What calls for it is a NaN in the sums of the walk's last round, a
      // tile past the end included: whatever the tile, the offset alone makes one.  (Tests of x ahead of the walk cost the
      // phases 4 to 9 % of their time.)
      auto redo_odd_rows = [&](int r0) {
        int lane_here = threadIdx.x & 63;
        asm volatile("" : "+v"(lane_here));  // (what follows from it is made here, not kept in registers through the walk)
        const int c = lane_here & 15, j = lane_here >> 4;
        const int b = pass_lo + c / 3;
        const bool ok = c < 3 * BR && b < seg_hi;
        const int64_t xr = p.x_one_row ? 0 : x_row(p.x_rows, p.x_src_rows, ok ? b : seg_lo);
        const uint32_t keep = ok ? 0x7fffffffu : 0u;
#pragma unroll 1
        for (int round = 0; round < p.rounds; ++round) {
          const int tile = tile_of(r0 + round);
          if (tile < 0) break;
          float4_t acc = {0.f, 0.f, 0.f, 0.f}, odd_x = {0.f, 0.f, 0.f, 0.f};  // odd_x: NaN in the rows in question
#pragma unroll 1
          for (int g = ga_raw - ph * kw * U, ph2 = 0; (PHASED || k_live) && ph2 <= ph && g < p.ng; ++ph2, g += kw * U) {
            const uint32_t* const xrow = reinterpret_cast<const uint32_t*>(p.x) + xr * p.K + g * 32 + 8 * j;
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
              const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (c * p.nw + 4 * (g + j)) * 4 + 64 * st,
                                                                    static_cast<int>(static_cast<uint32_t>(tile) * w_tile), 0);
              const u32x4 sv = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, (c * p.ng + g + 4 * st) * 4,
                                                                     static_cast<int>(static_cast<uint32_t>(tile) * s_tile), 0);
              uint32_t r[4] = {t.x, t.y, t.z, t.w};
              mid_transpose(r[0], r[1], r[2], r[3]);
#pragma unroll
              for (int m = 0; m < 4; ++m) {
                uint32_t v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                  const uint32_t raw = xrow[(4 * st + m) * 32 + e];
                  const uint32_t quiet = (raw & 0x7fffffu) != 0 ? raw | 0x400000u : raw;  // (a NaN's upper half is to stay a NaN)
                  v[e] = (raw & keep) >= 0x7f800000u ? quiet : 0u;
                }
                const mid_u4 xi = {__builtin_amdgcn_perm(v[2], v[0], kHiHi), __builtin_amdgcn_perm(v[6], v[4], kHiHi),
                                   __builtin_amdgcn_perm(v[3], v[1], kHiHi), __builtin_amdgcn_perm(v[7], v[5], kHiHi)};
                odd_x = mid_mfma<true>(xi, mid_u4{0u, 0u, 0u, 0u}, odd_x);
                const uint4 w7 = word_minus7(r[m]);
                const float4_t d = mid_mfma<true>(xi, mid_u4{w7.x, w7.y, w7.z, w7.w}, float4_t{0.f, 0.f, 0.f, 0.f});
                const float s = __builtin_bit_cast(float, m == 0 ? sv.x : (m == 1 ? sv.y : (m == 2 ? sv.z : sv.w)));
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[q] = d[q] != 0.f ? fmaf(s, d[q], acc[q]) : acc[q];
              }
            }
          }
          float* const at = reinterpret_cast<float*>(res_lds + (round * WV + wave) * 64 + lane_here);
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (odd_x[q] != odd_x[q]) at[q] = acc[q];
        }
      };

      // ---- the K shares of a tile meet: 256 values per (round, tile lane, batch tile); thread (jq, cq) takes row
      //      16 bt + jq of column cq, so that 16 neighbouring threads store 16 neighbouring columns
      auto finish = [&](int r0, int rounds) __attribute__((always_inline)) {
        const float* const res = reinterpret_cast<const float*>(res_lds);
        const int sub = threadIdx.x & 255, cq = sub & 15, jq = sub >> 4;
        auto at_row = [&](int r) { return (((r >> 2) * 16 + cq) << 2) + (r & 3); };  // lane (cq, r / 4), value r % 4
        const int at = at_row(F32 ? 0 : jq);
        if (jq >= BR) return;
        auto share_sum = [&](int round, int tl, int bt) {
          float v = 0.f;
          if constexpr (F32) {  // the row's three planes, the smallest first
#pragma unroll
            for (int pl = 2; pl >= 0; --pl) {
              const int ap = at_row(3 * jq + pl);
              for (int k = 0; k < kw; ++k) v += res[(((round * WV + (tl << p.kw_log2) + k) * NBT + bt) << 8) + ap];
            }
          } else {
            for (int k = 0; k < kw; ++k) v += res[(((round * WV + (tl << p.kw_log2) + k) * NBT + bt) << 8) + at];
          }
          return F32 ? 512.0f * v : v;
        };
        if (p.paired) {
          const int items = (rounds >> 1) * tw * NBT;
          const int half = p.N >> 1;
          for (int it = threadIdx.x >> 8; it < items; it += WV / 4) {
            const int bt = it % NBT, rest = it / NBT, tl = rest % tw, pr = rest / tw;
            const int pair = blockIdx.x * tw + tl + ((r0 >> 1) + pr) * tstride;
            const int col = pair * 16 + cq, b = pass_lo + BR * bt + jq;
            if (pair >= p.ntiles || b >= seg_hi) continue;
            const float gate = share_sum(2 * pr, tl, bt), up = share_sum(2 * pr + 1, tl, bt);
            if constexpr (!F32) static_cast<uint16_t*>(p.y)[static_cast<int64_t>(b) * half + col] = silu_mul_t<BF>(gate, up);
          }
        } else {
          const int items = rounds * tw * NBT;
          for (int it = threadIdx.x >> 8; it < items; it += WV / 4) {
            const int bt = it % NBT, rest = it / NBT, tl = rest % tw, round = rest / tw;
            const int t = blockIdx.x * tw + tl + (r0 + round) * tstride;
            const int col = t * 16 + cq, b = pass_lo + BR * bt + jq;
            if (t >= p.ntiles || col >= p.N || b >= seg_hi) continue;
            float v = share_sum(round, tl, bt);
            const int64_t oi = static_cast<int64_t>(b) * p.N + col;
            if (p.slices > 1) {  // (bias, residual and the cast belong to the reduction)
              static_cast<float*>(p.y)[static_cast<int64_t>(blockIdx.z) * p.rows * p.N + oi] = v;
              continue;
            }
            if (p.bias != nullptr) v += elem(p.bias, col);
            if (p.residual != nullptr) v += elem(p.residual, oi);
            if (F32 || p.out_f32) static_cast<float*>(p.y)[oi] = v;
            else static_cast<uint16_t*>(p.y)[oi] = BF ? f2bf(v) : f2h(v);
          }
        }
      };

      // ---- the walk: p.rounds is a multiple of RT (rounds past the last tile read nothing and leave zeros in LDS slots
      //      that nobody reads).  Later phases add to what the earlier ones left (the read is unconditional and the
      //      first phase drops it: no branch inside the walk).
      const int chunks = ONCE ? 1 : p.chunks;
      for (int chunk = 0; chunk < chunks; ++chunk) {
        const int r0 = chunk * p.rounds;
        const int rounds = ONCE ? RT : min(p.rounds, p.total_rounds - r0);
        for (int round = 0; round < rounds; round += RT) {
#pragma unroll
          for (int slot = 0; slot < RT; ++slot) {
            float4_t acc[NBT];
            walk_tile((slot & 1) == 0, r0 + round + slot + RT, w[slot], sraw[PAIR ? slot / 2 : slot], acc);
#pragma unroll
            for (int bt = 0; bt < NBT; ++bt) {
              float4* const at = res_lds + (((round + slot) * WV + wave) * NBT + bt) * 64 + lane;
              if constexpr (PHASED) {
                const float4 old = *at;
                const bool add = ph > 0;
                *at = make_float4(acc[bt][0] + (add ? old.x : 0.f), acc[bt][1] + (add ? old.y : 0.f),
                                  acc[bt][2] + (add ? old.z : 0.f), acc[bt][3] + (add ? old.w : 0.f));
              } else {
                *at = make_float4(acc[bt][0], acc[bt][1], acc[bt][2], acc[bt][3]);
              }
            }
            __builtin_amdgcn_sched_barrier(0);  // (each refill stays ahead of the next tile's arithmetic)
          }
        }
        if (!PHASED || ph + 1 == p.phases) {  // (uniform)
          if constexpr (F32) {
            const float4 last = res_lds[((rounds - 1) * WV + wave) * 64 + lane];
            const float sum = (last.x + last.y) + (last.z + last.w);
            if (__ballot(sum != sum) != 0) redo_odd_rows(r0);  // (uniform; the sums are this wave's own until the barrier)
          }
          __syncthreads();
          finish(r0, rounds);
          __syncthreads();  // (the next chunk, or the next pass, writes the same LDS slots)
        }
      }
    }
  }
}

template <int NBT, int U, int RT, bool KEEP_C, bool PHASED, int DT, int WV, bool OWN_X>
__global__ __launch_bounds__(64 * WV) void midrow_kernel(const MidParams p) {
  midrow_body<NBT, U, RT, KEEP_C, PHASED, DT, WV, false, OWN_X>(p);
}

template <int NBT, int U, int RT, bool KEEP_C, int DT>
__global__ __launch_bounds__(1024) void midonce_kernel(const MidParams p) {
  midrow_body<NBT, U, RT, KEEP_C, false, DT, 16, true, false>(p);
}

// y[b][j] = silu(sum over slices of part[s][b][j]) * (sum over slices of part[s][b][N / 2 + j]), in the model dtype
__global__ __launch_bounds__(256) void mid_reduce_silu_kernel(const float* __restrict__ part, int slices, int64_t rows, int N,
                                                              uint16_t* __restrict__ y, int bf16) {
  const int half = N >> 1;
  const int64_t count = rows * N, outs = rows * half;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < outs; i += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t b = i / half;
    const int64_t at = b * N + (i - b * half);
    float g = 0.f, u = 0.f;
    for (int sl = 0; sl < slices; ++sl) {
      g += part[sl * count + at];
      u += part[sl * count + at + half];
    }
    y[i] = bf16 ? silu_mul_bf(g, u) : silu_mul_h(g, u);
  }
}

template <int NBT, int U, int RT, bool KEEP_C, bool PHASED, int DT = MODEL_F16, int WV = 16, bool OWN_X = false>
hipError_t launch_mid(const MidParams& p, int wgx, int experts, hipStream_t s) {
  // the sums, and 2 KiB of x per wave (float32: x in the slots of five rounds' sums)
  const int slots = DT == MODEL_F32 ? (PHASED || OWN_X || p.rounds > 5 ? p.rounds : 5) : p.rounds * NBT + 2;
  const size_t lds = static_cast<size_t>(slots) * WV * 1024;
  if (lds > 160 * 1024) return hipErrorNotSupported;
  if (lds > 64 * 1024) {
    static bool raised = false;  // (idempotent; a race sets the same attribute twice)
    if (!raised) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&midrow_kernel<NBT, U, RT, KEEP_C, PHASED, DT, WV, OWN_X>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      if (e != hipSuccess) return e;
      raised = true;
    }
  }
  note_kernel("gq::midrow_kernel<%d,%d,%d,%d,%d%s> rounds=%d chunks=%d phases=%d slices=%d kw=%d%s", NBT, U, RT, int(KEEP_C),
              int(PHASED), DT == MODEL_BF16 ? ",true" : (DT == MODEL_F32 ? ",f32" : ""), p.rounds, p.chunks, p.phases, p.slices, 1 << p.kw_log2, OWN_X ? " own x" : "");
  hipLaunchKernelGGL((midrow_kernel<NBT, U, RT, KEEP_C, PHASED, DT, WV, OWN_X>), dim3(wgx, experts, p.slices), dim3(64 * WV), lds, s, p);
  return hipGetLastError();
}

template <int NBT>
hipError_t launch_mid_once(const MidParams& p, int wgx, hipStream_t s) {
  constexpr int RT = 2;
  constexpr size_t lds = (RT * NBT + 2) * 16 * 1024;  // (64 or 96 KiB)
  if (lds > 64 * 1024) {
    static bool raised = false;  // (idempotent; a race sets the same attribute twice)
    if (!raised) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&midonce_kernel<NBT, 8, RT, false, MODEL_F16>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      if (e != hipSuccess) return e;
      raised = true;
    }
  }
  note_kernel("gq::midonce_kernel<%d,8,%d,0> slices=%d kw=%d", NBT, RT, p.slices, 1 << p.kw_log2);
  hipLaunchKernelGGL((midonce_kernel<NBT, 8, RT, false, MODEL_F16>), dim3(wgx, 1, p.slices), dim3(1024), lds, s, p);
  return hipGetLastError();
}

}  // namespace

// q4f16_1 / q4bf16_1 / q4f32_1 (activations, scales and results of one type), K % 256 == 0 (a wave's eight groups: 16-byte runs of scales), N % 16 == 0 for expert
// segments and N % 32 == 0 for the fused gate/up form; any number of rows (more than the batch tiles hold: passes that read
// the weights again, so callers keep it to few rows per segment).  hipErrorNotSupported otherwise.  Tuning overrides:
// quad_ksplit (log2 of the waves that share a tile's K, minus one), gemv_waves (workgroups per expert x 16),
// gemv_rows_per_wave (2: the float16 instance of one batch tile with a ring of four tiles).
hipError_t launch_midrow(const GemmArgs& a, int rows_max, hipStream_t s) {
  if (a.bits != 4 || a.group_size != 32) return hipErrorNotSupported;
  if (a.rows < 1 || a.N < 16 || (a.K & 255) != 0 || a.K == 0) return hipErrorNotSupported;
  const bool grouped = a.indptr != nullptr;
  if (grouped && (a.N & 15) != 0) return hipErrorNotSupported;  // (an expert's tensor ends where the next begins)
  if (a.paired && ((a.N & 31) != 0 || a.bias != nullptr || a.residual != nullptr || a.out_f32)) return hipErrorNotSupported;
  if ((reinterpret_cast<uintptr_t>(a.x) & 15) != 0 || (reinterpret_cast<uintptr_t>(a.q_weight) & 15) != 0 ||
      (reinterpret_cast<uintptr_t>(a.q_scale) & 15) != 0)
    return hipErrorNotSupported;
  if (a.N * (a.K / 8) >= (int64_t(1) << 29)) return hipErrorNotSupported;  // (32-bit byte offsets with room to add)
  // (workgroup rows: one per expert, or per activation row where each names its expert)
  const int experts = grouped ? static_cast<int>(a.num_experts) : (a.expert_ids != nullptr ? static_cast<int>(a.rows) : 1);
  if (experts < 1 || experts > 65535) return hipErrorNotSupported;
  if (a.f32 && (a.paired || a.bf16)) return hipErrorNotSupported;
  if (a.expert_ids != nullptr && (!a.f32 || grouped || (a.N & 15) != 0)) return hipErrorNotSupported;
  MidParams p{};
  p.x = a.x; p.qw = a.q_weight; p.qs = a.q_scale; p.bias = a.bias; p.residual = a.residual; p.y = a.y;
  p.indptr = a.indptr; p.indptr_i64 = a.indptr_i64; p.x_rows = a.x_rows; p.x_src_rows = static_cast<int>(a.x_src_rows);
  p.ids = a.expert_ids; p.x_one_row = a.x_one_row; p.num_experts = static_cast<int>(a.num_experts);
  p.rows = static_cast<int>(a.rows); p.N = static_cast<int>(a.N); p.K = static_cast<int>(a.K);
  p.ng = p.K / 32; p.nw = 4 * p.ng;
  p.expert_w_stride = static_cast<int64_t>(p.N) * p.nw;
  p.expert_s_stride = static_cast<int64_t>(p.N) * p.ng;
  p.paired = a.paired;
  p.ntiles = a.paired ? p.N / 32 : (p.N + 15) / 16;
  p.out_f32 = a.out_f32;
  // batch tiles per pass: one for up to 16 rows per segment, else two (more rows: passes)
  const int nbt = rows_max <= 16 || a.f32 ? 1 : 2;  // (float32: one, of five rows)
  constexpr int U = 8;
  // waves that share a tile's K: the power of two that covers K's shares of U groups, at most 16 (a wave whose share lies
  // past K idles: one phase with 14 of 16 waves at work is ahead of two phases of 8)
  int kwl = 0;
  while (kwl < 4 && (1 << kwl) < p.ng / U) ++kwl;
  if (options().quad_ksplit >= 0) kwl = options().quad_ksplit + 1;  // (tuning override: 2, 4, 8 or 16 waves)
  p.kw_log2 = kwl;
  const int phase_groups = (1 << kwl) * U;
  p.phases = (p.ng + phase_groups - 1) / phase_groups;
  // A plain linear whose K takes several phases and whose caller brings the scratch: as many workgroup rows as
  // phases, each with an equal share of K, instead (x stays in registers for all of a workgroup's tiles, the walk comes in chunks), fp32 partial sums in the
  // workspace and a second, small launch that adds them; the fused gate/up form then runs as a plain one and the reduction
  // folds the activation in.  The slices are as long as one another (K = 14336: four of 14 shares, not three of 16 and one
  // of 8, whose workgroups would be done first and leave their CUs idle: 15360 x 5120 at 7 / 16 / 32 rows 20.7 / 21.9 / 29.4 -> 18.8 /
  // 20.1 / 27.5 us, 27648 x 5120 31.9 / 33.4 / 44.4 -> 29.4 / 31.2 / 42.5, 4096 x 14336 16.0 / 16.3 / 20.9 -> 15.5 / 15.6 / 20.2, a K of
  // whole phases as before).  Tuning override: gemv_ksplit 0 keeps the phases.
  p.slices = 1;
  p.slice_shares = 1 << kwl;
  bool fold_silu = false;
  if (p.phases > 1 && experts == 1 && !grouped && p.phases <= 64 && options().gemv_ksplit != 0 && a.workspace != nullptr &&
      a.workspace_bytes >= static_cast<int64_t>(p.phases) * p.rows * p.N * 4 &&
      (reinterpret_cast<uintptr_t>(a.workspace) & 15) == 0) {
    p.slices = p.phases;
    p.slice_shares = (p.ng / U + p.slices - 1) / p.slices;
    p.phases = 1;
    p.y = a.workspace;
    p.bias = nullptr; p.residual = nullptr; p.out_f32 = 1;
    if (p.paired) {
      fold_silu = true;
      p.paired = 0;
      p.ntiles = (p.N + 15) / 16;
    }
  }
  const bool paired_walk = p.paired != 0;
  const int tw = 16 >> kwl;
  const int form = options().gemv_rows_per_wave;  // (tuning override: which one-batch-tile instance)
  const int rt = form == 2 ? 4 : 2;
  // workgroups in all: one per CU (sixteen waves of up to 128 registers fill it), each with at most 128 KiB of sums in LDS
  const int want_wg = options().gemv_waves > 0 ? options().gemv_waves / 16 : 256;
  int wgx = want_wg / (experts * p.slices);
  if (wgx < 1) wgx = 1;
  const int per_round = paired_walk ? 2 : 1;           // rounds per walked item
  const int sets = (p.ntiles + tw - 1) / tw;        // items per tile lane
  if (wgx > sets) wgx = sets;
  const int unit = paired_walk ? (rt % 2 == 0 ? rt : 2 * rt) : rt;  // rounds come in whole rings (and whole pairs)
  const int max_rounds = (128 / (16 * nbt)) / unit * unit;
  if (max_rounds < unit) return hipErrorNotSupported;
  int items = (sets + wgx - 1) / wgx;               // items per wave
  if (p.phases > 1 && items * per_round > max_rounds) {  // (one chunk: more workgroups instead)
    items = max_rounds / per_round;
    wgx = (sets + items - 1) / items;
  }
  wgx = (sets + items - 1) / items;
  // (chunks of one length, the last one shorter by what is over: walked to its full length as well, 18 rounds of eight waves were 20, and
  //  66560 x 4096 took 38.1 / 38.7 us at 5 / 8 rows, where the quad-row kernel takes 36.4 / 37.3; now 35.3 / 36.4)
  int rounds = (items * per_round + unit - 1) / unit * unit;
  p.chunks = (rounds + max_rounds - 1) / max_rounds;
  // One batch tile and more than one chunk of rounds: eight waves of sixteen groups each instead, whose sums take half the LDS
  // (twice the rounds per chunk, half as many stops where the shares meet; the sums of half as many shares): 128256 x 4096 at 7 /
  // 16 rows 63.8 / 67.1 -> 61.1 / 66.5 us, 27648 x 5120 29.4 / 31.2 -> 25.9 / 27.0, 57344 x 8192 61.3 / 65.9 -> 56.7 / 60.9; where one chunk
  // does, sixteen waves hide more (4096 x 4096 7.4 against 8.1, 28672 x 4096 at 16 rows 19.4 against 19.7).  Two batch tiles lose
  // with eight waves (128256 x 4096 at 32 rows 81.5 against 86.6).  A K of one or two such shares leaves little between the stops
  // either way, and sixteen waves stay ahead (180224 x 1024 at 7 / 16 rows 25.1 / 26.1 against 26.5 / 28.2).  Expert segments alike (rows per
  // expert): 8 of 28672 x 4096 at 4..8 106-108 -> 104-107, 64 of 5120 x 3584 at 4.5 147 -> 139, 64 of 5120 x 1536 at 4.5 66.9 -> 65.9, but 64 of
  // 9952 x 1024 at 4.5 84.4 against 88.0, 64 of 9952 x 512 49.1 against 54.3.
  // (The fused gate/up form walks half as many items of two rounds each, so it takes more than one chunk exactly where the plain
  // form does, and the two add in the same order.)
  const bool wide = nbt == 1 && !a.f32 && p.phases == 1 && p.chunks > 1 && a.K >= 1536 && (a.K & 511) == 0 && options().quad_ksplit < 0 && form < 0;
  if (wide) {
    --p.kw_log2;
    p.slice_shares = p.slices > 1 ? (p.ng / 16 + p.slices - 1) / p.slices : 1 << p.kw_log2;
    p.chunks = (rounds + 2 * max_rounds - 1) / (2 * max_rounds);
  }
  p.rounds = ((rounds + p.chunks - 1) / p.chunks + unit - 1) / unit * unit;
  p.total_rounds = rounds;
  auto run = [&]() -> hipError_t {
    // Two rounds of a plain float16 linear.  One batch tile only of 9 rows on below 24 M weights: with 24 M and more, rows with an
    // infinity have always been NaN there (the kept offsets' inf - inf), below they went to a kernel that gave infinities, which this form
    // gives too (and the dispatch sends no other shapes of those sizes: midrow_two_rounds).
    const bool once = !a.f32 && !a.bf16 && experts == 1 && !grouped && p.phases == 1 && p.chunks == 1 && p.rounds == 2 &&
                      options().gemv_variant < 0;
    if (once && nbt == 2) return launch_mid_once<2>(p, wgx, s);
    if (once && a.rows > 8 && a.N * a.K < (24ll << 20)) return launch_mid_once<1>(p, wgx, s);
    if (a.f32) {
      if (p.phases > 1)
        return launch_mid<1, 8, 2, false, true, MODEL_F32>(p, wgx, experts, s);
      // One or two rows of up to 12 M weights: a lane's own loads of x.  The way through LDS is ahead once more rows or more workgroups want
      // it (in us, own loads against LDS, 2 rows: 4096 x 768 8.5 / 8.8, 4096 x 2304 10.0 / 10.1, 1 row 1024 x 9216 11.4 / 11.9; 2 rows 4096 x 4096
      // 10.8 / 10.4, 28672 x 768 10.5 / 10.1, 3 rows 4096 x 1024 9.2 / 8.9).  Three and four rows too where a wave has one tile and a quarter
      // of the waves or more no share of a K below 3072, so that fewer of them load (3 rows 1216 x 1280 8.30 / 8.65, 672 x 2304 9.11 / 9.42,
      // 4 rows 7360 x 1280 9.01 / 9.22, 192 x 2560 9.07 / 9.24; but two tiles, 3 rows 9408 x 1280 9.29 / 9.14, no such waves, 3 rows 1968 x 2048
      // 9.28 / 8.98, and 4 rows 160 x 3072 9.31 / 9.22, 5 rows 336 x 2560 level).
      // Expert segments of about one row on average (two with such waves), one tile per wave: own loads as well, ahead while the longest segment
      // has one or two rows (4 experts at 3 rows: 1056 x 768 8.16 / 8.52, 656 x 1280 8.22 / 8.70, 192 x 2304 8.87 / 9.45, 592 x 3584 9.61 / 10.06; 8 at 5
      // rows of 176 x 4096 9.21 / 9.63, at 14 of 736 x 1280 9.24 / 9.47; but 8 at 14 of 176 x 4096 10.44 / 9.95, 16 at 24 of 192 x 3072 10.42 / 10.21).
      const bool one_tile = p.slices == 1 && items == 1;
      const bool idle_waves = a.K < 3072 && 4 * (p.ng / U) <= 3 << kwl;
      const bool own_x = grouped ? one_tile && a.rows <= (idle_waves ? 2 * a.num_experts : a.num_experts + 1)
                                 : (a.expert_ids != nullptr || a.rows <= (one_tile && idle_waves ? 4 : 2)) && a.N * a.K * experts < (12ll << 20);
      if (own_x)
        return launch_mid<1, 8, 2, false, false, MODEL_F32, 16, true>(p, wgx, experts, s);
      return launch_mid<1, 8, 2, false, false, MODEL_F32>(p, wgx, experts, s);
    }
    if (wide)
      return a.bf16 ? launch_mid<1, 16, 2, true, false, MODEL_BF16, 8>(p, wgx, experts, s)
                    : launch_mid<1, 16, 2, true, false, MODEL_F16, 8>(p, wgx, experts, s);
    if (a.bf16) {  // (the bfloat16 instances: q4bf16_*)
      if (p.phases > 1)
        return nbt == 2 ? launch_mid<2, 8, 2, false, true, MODEL_BF16>(p, wgx, experts, s)
                        : launch_mid<1, 8, 2, true, true, MODEL_BF16>(p, wgx, experts, s);
      return nbt == 2 ? launch_mid<2, 8, 2, false, false, MODEL_BF16>(p, wgx, experts, s)
                      : launch_mid<1, 8, 2, true, false, MODEL_BF16>(p, wgx, experts, s);
    }
    if (p.phases > 1) {
      if (form == 2) return hipErrorNotSupported;
      if (nbt == 2) return launch_mid<2, 8, 2, false, true>(p, wgx, experts, s);
      return launch_mid<1, 8, 2, true, true>(p, wgx, experts, s);
    }
    if (nbt == 2) return launch_mid<2, 8, 2, false, false>(p, wgx, experts, s);
    if (form == 2) return launch_mid<1, 8, 4, false, false>(p, wgx, experts, s);
    return launch_mid<1, 8, 2, true, false>(p, wgx, experts, s);
  };
  const hipError_t e = run();
  if (e != hipSuccess || p.slices == 1) return e;
  const int64_t count = static_cast<int64_t>(p.rows) * p.N;
  if (a.f32)
    return launch_splitk_reduce_f32(static_cast<const float*>(a.workspace), p.slices, p.rows, p.N, p.N, reinterpret_cast<const float*>(a.bias),
                                    reinterpret_cast<const float*>(a.residual), static_cast<float*>(a.y), s);
  if (fold_silu) {
    const int64_t outs = count / 2;
    hipLaunchKernelGGL(mid_reduce_silu_kernel, dim3(static_cast<unsigned>((outs + 255) / 256 > 4096 ? 4096 : (outs + 255) / 256)),
                       dim3(256), 0, s, static_cast<const float*>(a.workspace), p.slices, static_cast<int64_t>(p.rows), p.N,
                       static_cast<uint16_t*>(a.y), a.bf16);
  } else {
    const int64_t blocks = ((p.N & 3) == 0 ? (count / 4 + 255) / 256 : (count + 255) / 256);
    hipLaunchKernelGGL(splitk_reduce_kernel<false>, dim3(static_cast<unsigned>(blocks > 4096 ? 4096 : blocks)), dim3(256), 0, s,
                       static_cast<const float*>(a.workspace), p.slices, count, p.N, p.N, a.bias, a.residual, a.y, a.out_f32, a.bf16);
  }
  return hipGetLastError();
}

// whether a dense float16 linear (K a positive multiple of 256, beyond 4096 as K slices) is two rounds per wave at most
bool midrow_two_rounds(int64_t N, int64_t K) {
  const int64_t shares = K / 256, slices = (shares + 15) / 16;
  int64_t tw = 16;  // tiles side by side in a workgroup
  while (tw > 1 && 16 / tw < shares) tw /= 2;
  return slices <= 256 && (N + 15) / 16 <= 2 * tw * (256 / slices);
}

// scratch for the K slices of a plain linear (0: K is one phase)
int64_t midrow_workspace_bytes(int64_t rows, int64_t N, int64_t K) {
  if (rows < 1 || N < 16 || K <= 0 || (K & 255) != 0) return 0;
  const int64_t phases = (K / 32 + 127) / 128;
  return phases > 1 ? phases * rows * N * 4 : 0;
}

}  // namespace gq
