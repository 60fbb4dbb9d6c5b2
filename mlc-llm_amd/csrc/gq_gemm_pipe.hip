// Prefill GEMM / MoE grouped GEMM, software-pipelined form (the one that normally runs).
//
// Same tiling and LDS layout as gq_gemm.hip; what differs is how latency is hidden:
//  * global loads run TWO K tiles ahead of the MFMAs (register ping-pong), because one tile of
//    MFMA work (~0.4 us) is shorter than a trip to L2 / HBM;
//  * every load is branch-free (addresses are clamped, out-of-range data is zeroed when it is
//    written to LDS) so that the compiler's wait-count insertion can leave the newest loads in
//    flight instead of draining the queue at every join;
//  * the MFMA fragments of k-step s+1 are read from LDS before the MFMAs of step s are issued.
// Requires K % 8 == 0 (16-byte aligned activation rows); other K take the kernel in gq_gemm.hip.
#include <type_traits>

#include "gq_gemm_common.hpp"

namespace gq {

// DEPTH: K tiles of global loads in flight (register stages); even, 2 for the large tiles, more
// for few-row tiles whose MFMA work per tile is far shorter than a trip to memory
// BF: bfloat16 model (operands and 16-bit outputs are bf16; see dequant_word4_bf16)
// SKIP: waves leave out the 32-row blocks of their sub-tile that lie past the segment's last row
// WX: extra register stages for the weights alone.  Loads return in issue order, so each iteration issues its
// activation loads first and the weight loads (WX tiles further ahead) after them: waiting for the activations of
// the next tile then leaves the newer weight loads in flight.  For matmuls whose weights are read once and come
// straight from HBM (grouped, one row tile per expert) while the activations come from L2.
// FAST: K is whole K tiles and whole rounds of the register rings, and every byte offset is below 4 GiB (checked by the
// launcher).  The K loop then has no zero-selects and no clamps, and loads through buffer descriptors (tensor in scalar
// registers, K tile as the scalar offset, one 32-bit lane offset): 122 -> 62 VALU instructions per wave and K tile.  Rows
// past the segment and columns past N need no zeros: their loads are clamped to valid rows when the offsets are set up, a
// row of x or of W only ever reaches its own row or column of the result, and the epilogue drops those; only k past K
// would reach live results: q4 runs this form only when there is none; q3f16_1, whose 80-wide K tiles divide no power of two
// (K = 4096 is 51.2 tiles), masks the activation chunks at k >= K and gives a group past the last one scale 0 (one AND per
// chunk word, one select per group), and its descriptors carry the tensors' sizes, so that the last row's overrun reads
// zeros instead of the bytes behind the tensor.  A separate instantiation rather than a branch: the general
// form's addresses and flags would otherwise stay in registers next to this one's, and the large tile has none to spare
// (a spill reload inside the loop waits for every global load in flight).
// q4 in that form also reads its scales in bulk: the two lanes of a weight row load the row's 16 bytes of scales for FOUR
// K tiles at once (one request: both lanes name the same address) instead of 2 bytes per lane and K tile.  A 2-byte load
// costs the memory pipeline what a 16-byte one does (a wave's instruction touches 32 rows = 32 cache lines either way),
// and those loads alone were 9 % of the plain 256 x 256 GEMM, 18 % of down_proj's and a third of a grouped GEMM with few
// rows per expert (timing-only builds without them).  Needs K in whole blocks of four K tiles and 16-byte aligned scale
// rows (checked by the launcher).
template <int BITS, int BM, int BN, int WM, int WN, int DEPTH = 2, bool BF = false, bool SKIP = false, int WX = 0,
          bool FAST = false>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN)) void gemm_pipe_kernel(const GemmParams p) {
  using T = GemmTraits<BITS>;
  constexpr int G = T::G;
  constexpr int BK = 2 * G;        // 64 | 80
  constexpr int KSTEPS = BK / 16;  // MFMA k = 16
  constexpr int CPR = BK / 8;      // 16-byte chunks per tile row
  constexpr int LDA = BK + 8;      // padded row, in halves
  constexpr int WAVES_N = BN / WN;
  constexpr int NT = 64 * (BM / WM) * (BN / WN);
  static_assert(NT == 256 || NT == 512, "4 or 8 waves per workgroup");
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int A_CHUNKS = (BM * CPR + NT - 1) / NT;  // the last round may cover part of the threads only
  constexpr bool A_EXACT = BM * CPR % NT == 0;
  // groups of W per thread and K tile; a tile with fewer groups than threads (256 x 128) leaves the upper waves
  // without any (W_ALL false: a wave-uniform test, every SIMD still hosts one wave that dequantises)
  constexpr int W_GROUPS = BN * 2 >= NT ? BN * 2 / NT : 1;
  constexpr bool W_ALL = BN * 2 >= NT;
  static_assert(BN * 2 % NT == 0 || BN * 2 * 2 == NT, "tile / thread mismatch");
  constexpr bool SCV = FAST && BITS == 4;  // scales of four K tiles per load

  extern __shared__ uint4 smem[];
  uint16_t* lds = reinterpret_cast<uint16_t*>(smem);
  // [A stage 0][A stage 1][W stage 0][W stage 1]: the two stages of an operand lie less than 64 KiB apart, so a
  // stage is an immediate offset of the LDS instruction and both share one address register
  auto a_tile = [&](int s) { return lds + s * BM * LDA; };
  auto w_tile = [&](int s) { return lds + 2 * BM * LDA + s * BN * LDA; };

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;
  const bool w_active = W_ALL || tid < BN * 2;  // (wave-uniform)

  int seg_lo, seg_hi, mt, expert;
  if (!locate_tile<BM>(p, blockIdx.y, seg_lo, seg_hi, mt, expert)) return;  // uniform
  const int m0 = seg_lo + mt * BM;
  // 32-row blocks of this wave that hold rows of the segment: the others are skipped by the matrix core
  // (SKIP; a ragged expert segment or a last row tile leaves most of a tall tile empty)
  const int live = SKIP ? min(TM, max(0, (seg_hi - (m0 + wm0) + 31) / 32)) : TM;
  const bool second = static_cast<int>(blockIdx.x) >= p.hop_tile;
  const int n0 = p.n_begin + blockIdx.x * BN + (second ? p.hop : 0);
  const uint32_t* qw = p.qw + expert * p.expert_w_stride;
  const uint16_t* qs = p.qs + expert * p.expert_s_stride;

  // ---- per-thread load slots: where each 16-byte chunk of x / each group of W comes from
  const uint16_t* a_src[A_CHUNKS];  // chunk address at K tile 0 (row clamped into the segment)
  bool a_row_ok[A_CHUNKS];
  bool a_in_tile[A_CHUNKS];         // false: this thread has no chunk in round i (loads a valid address, stores nothing)
  int a_k[A_CHUNKS];                // k offset of the chunk inside a tile
  int a_dst[A_CHUNKS];              // offset (halves) inside the LDS tile
#pragma unroll
  for (int i = 0; i < A_CHUNKS; ++i) {
    const int idx_raw = tid + NT * i;
    a_in_tile[i] = A_EXACT || idx_raw < BM * CPR;
    const int idx = a_in_tile[i] ? idx_raw : 0;
    // (q4: a thread's chunks sit NT / CPR rows apart in the same column, written out so that their LDS addresses
    //  become one register plus constants instead of a register each)
    constexpr bool AFFINE = A_EXACT && NT % CPR == 0;
    const int r = AFFINE ? tid / CPR + i * (NT / CPR) : idx / CPR;
    const int c = AFFINE ? tid % CPR : idx - r * CPR;
    a_row_ok[i] = m0 + r < seg_hi;
    a_k[i] = 8 * c;
    a_src[i] = p.x + x_row(p.x_rows, p.x_src_rows, a_row_ok[i] ? m0 + r : m0) * p.K + 8 * c;
    a_dst[i] = r * LDA + 8 * c;
  }
  const uint32_t* w_src[W_GROUPS];
  const uint16_t* s_src[W_GROUPS];
  int w_g[W_GROUPS];  // group index at K tile 0
  int w_dst[W_GROUPS];
#pragma unroll
  for (int i = 0; i < W_GROUPS; ++i) {
    const int idx = w_active ? tid + NT * i : 0;
    const int r = idx >> 1, gsel = idx & 1;
    int row = min(n0 + r, p.N - 1);  // rows past N are computed and dropped
    if (p.paired) row = gate_up_row_blk<(TN % 2 == 0) ? 32 : 16>(n0 + r, p.N);
    w_src[i] = qw + static_cast<int64_t>(row) * p.nw;
    s_src[i] = qs + static_cast<int64_t>(row) * p.ng;
    w_g[i] = gsel;
    // (offset from the start of LDS, made opaque: left to itself the compiler folds the W region's 72 KiB into the
    //  constants, finds them past the 64 KiB an LDS instruction's immediate holds, and keeps a register per store)
    w_dst[i] = 2 * BM * LDA + r * LDA + gsel * G;
    asm volatile("" : "+v"(w_dst[i]));
  }

  uint32_t a_off[A_CHUNKS], w_off[W_GROUPS], s_off[W_GROUPS];
  uint32_t sc_shift[W_GROUPS];  // (SCV) bit position of this lane's group inside a K tile's word of two scales
#pragma unroll
  for (int i = 0; i < A_CHUNKS; ++i)
    a_off[i] = static_cast<uint32_t>(reinterpret_cast<const char*>(a_src[i]) - reinterpret_cast<const char*>(p.x));
#pragma unroll
  for (int i = 0; i < W_GROUPS; ++i) {
    w_off[i] = static_cast<uint32_t>(reinterpret_cast<const char*>(w_src[i] + 4 * w_g[i]) - reinterpret_cast<const char*>(qw));
    s_off[i] = static_cast<uint32_t>(reinterpret_cast<const char*>(s_src[i] + (SCV ? 0 : w_g[i])) - reinterpret_cast<const char*>(qs));
    sc_shift[i] = 16u * static_cast<uint32_t>(w_g[i]);
  }

  // this workgroup's share of K (all of it unless the launch splits K)
  const int nk = (p.ng + 1) / 2;
  const int kt0 = blockIdx.z * p.kt_per_split;
  const int kt1 = min(nk, kt0 + p.kt_per_split);
  const int k_lim = min(p.K, kt1 * BK);  // k and groups from here on contribute nothing
  const int g_lim = min(p.ng, 2 * kt1);

  struct StageA {
    uint4 a[A_CHUNKS];
  };
  struct StageW {
    uint4 w[W_GROUPS];
    uint32_t s[W_GROUPS];  // fp16 scale bits (32 bits wide on purpose: in flight, never re-packed)
  };
  static_assert(DEPTH >= 2 && DEPTH % 2 == 0, "register stages pair up with the two LDS stages");
  constexpr int WD = DEPTH + WX;
  static_assert(WD % DEPTH == 0, "the unrolled loop walks whole rounds of both register rings");
  StageA ra[DEPTH];
  StageW rw[WD];

  // K tile kt into registers.  Always valid addresses; validity is re-derived at store time.
  // (buffer loads: the descriptor of each tensor sits in scalar registers, the K tile is the scalar offset and the lane
  //  offset one 32-bit register, so no 64-bit address is formed or kept per load)
  constexpr bool KTAIL = FAST && BITS == 3;  // the last K tile may reach past K
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.x), short(0), KTAIL ? static_cast<int>(p.x_bytes) : -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(qw), short(0), KTAIL ? static_cast<int>(static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.nw) * 4u) : -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(qs), short(0), KTAIL ? static_cast<int>(static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.ng) * 2u) : -1, 0x00020000);
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  auto load_a_fast = [&](int kt, StageA& st) {  // (tiles past the end re-read the last one: never multiplied)
    const int soff = min(kt, kt1 - 1) * (BK * 2);
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, static_cast<int>(a_off[i]), soff, 0);
      st.a[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
  };
  auto load_w_fast = [&](int kt, StageW& st) {
    if (w_active) {
      const int ktc = min(kt, kt1 - 1);
#pragma unroll
      for (int i = 0; i < W_GROUPS; ++i) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, static_cast<int>(w_off[i]), ktc * 32, 0);
        st.w[i] = make_uint4(v.x, v.y, v.z, v.w);
        if constexpr (!SCV) st.s[i] = __builtin_amdgcn_raw_buffer_load_b16(s_rsrc, static_cast<int>(s_off[i]), ktc * 4, 0);
      }
    }
  };
  // (SCV) the scales of K tiles kt0 + 4 blk .. + 3 of this lane's weight row: word c = the two groups of tile c
  struct ScaleBlock {
    uint4 v[W_GROUPS];
  };
  auto load_scales = [&](int blk, ScaleBlock& sb) {
    if (w_active) {
      const int t = min(kt0 + 4 * blk, kt1 - 4);
#pragma unroll
      for (int i = 0; i < W_GROUPS; ++i) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(s_rsrc, static_cast<int>(s_off[i]), t * 4, 0);
        sb.v[i] = make_uint4(v.x, v.y, v.z, v.w);
      }
    }
  };
  auto scale_of = [&](const ScaleBlock& sb, int i, int c) -> uint32_t {  // c: K tile inside the block (compile-time)
    const uint32_t word = c == 0 ? sb.v[i].x : (c == 1 ? sb.v[i].y : (c == 2 ? sb.v[i].z : sb.v[i].w));
    return (word >> sc_shift[i]) & 0xffffu;
  };
  auto load_a = [&](int kt, StageA& st) {
    if constexpr (FAST) {
      load_a_fast(kt, st);
      return;
    }
    const int k_base = kt * BK;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      st.a[i] = *reinterpret_cast<const uint4*>(a_src[i] + (x_chunk(k_base + a_k[i], k_lim) - a_k[i]));
    }
  };
  auto load_w = [&](int kt, StageW& st) {
    if constexpr (FAST) {
      load_w_fast(kt, st);
      return;
    }
    if (w_active) {
#pragma unroll
      for (int i = 0; i < W_GROUPS; ++i) {
        const int g = 2 * kt + w_g[i];
        const int gc = g < p.ng ? g : 0;
        st.w[i] = *reinterpret_cast<const uint4*>(w_src[i] + 4 * gc);
        st.s[i] = s_src[i][gc];
      }
    }
  };
  // One of KSTEPS slices of "tile kt: registers -> LDS stage s".  The slices are issued between the
  // MFMA k-steps of the tile being multiplied, so that dequantisation (VALU) and the LDS stores
  // run in the shadow of the matrix pipe instead of after it.
  auto store_part = [&](int kt, const StageA& sa, const StageW& st, int s, int part, const ScaleBlock& scb, int sc_c) {
    uint16_t* at = a_tile(s);
    uint16_t* wt = lds + s * BN * LDA;  // (w_dst holds the offset of the W region)
    const int k_base = kt * BK;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
      if (i % KSTEPS != part) continue;
      // (the zero for rows past the segment and k past K as an AND with a lane mask: written as a select of the four
      //  words it becomes a branch around four moves, and control flow inside the loop makes the wait-count insertion
      //  drain every load in flight at the loop header)
      const bool kept = KTAIL ? k_base + a_k[i] < p.K : (FAST || (a_row_ok[i] && (k_base + a_k[i] < k_lim)));
      const uint32_t keep = kept ? 0xffffffffu : 0u;
      if (A_EXACT || a_in_tile[i])
        *reinterpret_cast<uint4*>(at + a_dst[i]) =
            (FAST && !KTAIL) ? sa.a[i] : make_uint4(sa.a[i].x & keep, sa.a[i].y & keep, sa.a[i].z & keep, sa.a[i].w & keep);
    }
    if (!w_active) return;
#pragma unroll
    for (int i = 0; i < W_GROUPS; ++i) {
      const bool ok = KTAIL ? 2 * kt + w_g[i] < p.ng : (FAST || 2 * kt + w_g[i] < g_lim);
      // a group past the end gets scale +0.0: every value becomes (q - m) * 0 = +-0
      const uint16_t sb = SCV ? static_cast<uint16_t>(scale_of(scb, i, sc_c)) : (ok ? static_cast<uint16_t>(st.s[i]) : uint16_t(0));
      uint4* dst = reinterpret_cast<uint4*>(wt + w_dst[i]);
      if (BITS == 4) {
        // word `part` of the group -> 8 halves = one 16-byte chunk
        const uint32_t w4[4] = {st.w[i].x, st.w[i].y, st.w[i].z, st.w[i].w};
        uint32_t d[4];
        if constexpr (BF) dequant_word4_bf16(w4[part], sb, d);
        else dequant_word4(w4[part], sb, d);
        dst[part] = make_uint4(d[0], d[1], d[2], d[3]);
      } else if constexpr (!BF) {
        // q3: 16-byte chunk `part` of the group (5 chunks, 5 k-steps)
        uint32_t d[4];
        dequant_chunk3(st.w[i], sb, part, d);
        dst[part] = make_uint4(d[0], d[1], d[2], d[3]);
      } else if (part == 0) {
        uint32_t d[G / 2];
        dequant_group_bf16<BITS>(st.w[i], sb, d);
#pragma unroll
        for (int c = 0; c < G / 8; ++c) dst[c] = make_uint4(d[4 * c], d[4 * c + 1], d[4 * c + 2], d[4 * c + 3]);
      }
    }
  };
  auto store_tile = [&](int kt, const StageA& sa, const StageW& st, int s, const ScaleBlock& scb, int sc_c) {
#pragma unroll
    for (int part = 0; part < KSTEPS; ++part) store_part(kt, sa, st, s, part, scb, sc_c);
  };

  float16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int frag_row = lane & 31, frag_k = 8 * (lane >> 5);
  // MFMAs of the tile in stage s; slice ks of the next tile's store is issued after k-step ks
  // full: every 32-row block of the wave is live (the straight-line form); otherwise blocks >= live are skipped by
  // wave-uniform branches, fragments and all
  auto mfma_tile = [&](auto full, int s, int kt_store, const StageA& sa_store, const StageW& st_store,
                       const ScaleBlock& scb, int sc_c) {
    constexpr bool FULL = decltype(full)::value;
    const uint16_t* at = a_tile(s) + (wm0 + frag_row) * LDA + frag_k;
    const uint16_t* wt = w_tile(s) + (wn0 + frag_row) * LDA + frag_k;
    auto mma = [&](const half8_t& av, const half8_t& bv, float16_t& c) {
      if constexpr (BF)
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, av), __builtin_bit_cast(bf16x8_t, bv), c,
                                                    0, 0, 0);
      else
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, c, 0, 0, 0);
    };
    if constexpr (TM == 4) {
      // Four row blocks per wave: the kernel runs close to the 256-register limit, and a spill reload inside this loop
      // would wait for every global load in flight.  The activation fragments therefore live in ONE set of registers:
      // block i of the next k-step is read right after the MFMAs that used block i of this one (six MFMAs ahead of its
      // own use); only the weight fragments are double-buffered (same speed as two sets, 16 registers fewer).
      half8_t af[TM], bf[2][TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        if (FULL || i < live) af[i] = *reinterpret_cast<const half8_t*>(at + i * 32 * LDA);
      if (FULL || live > 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[0][j] = *reinterpret_cast<const half8_t*>(wt + j * 32 * LDA);
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int cur = ks & 1, nxt = cur ^ 1;
        if (ks + 1 < KSTEPS && (FULL || live > 0)) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            bf[nxt][j] = *reinterpret_cast<const half8_t*>(wt + j * 32 * LDA + (ks + 1) * 16);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if (FULL || i < live) {
#pragma unroll
            for (int j = 0; j < TN; ++j) mma(af[i], bf[cur][j], acc[i][j]);
            if (ks + 1 < KSTEPS) af[i] = *reinterpret_cast<const half8_t*>(at + i * 32 * LDA + (ks + 1) * 16);
          }
        }
        store_part(kt_store, sa_store, st_store, s ^ 1, ks, scb, sc_c);
        __builtin_amdgcn_sched_barrier(0);  // keep the slices where they were written
      }
    } else {  // fragments of k-step s+1 are read while the MFMAs of step s run
      half8_t af[2][TM], bf[2][TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        if (FULL || i < live) af[0][i] = *reinterpret_cast<const half8_t*>(at + i * 32 * LDA);
      if (FULL || live > 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[0][j] = *reinterpret_cast<const half8_t*>(wt + j * 32 * LDA);
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int cur = ks & 1, nxt = cur ^ 1;
        if (ks + 1 < KSTEPS) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
            if (FULL || i < live) af[nxt][i] = *reinterpret_cast<const half8_t*>(at + i * 32 * LDA + (ks + 1) * 16);
          if (FULL || live > 0) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
              bf[nxt][j] = *reinterpret_cast<const half8_t*>(wt + j * 32 * LDA + (ks + 1) * 16);
          }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if (FULL || i < live) {
#pragma unroll
            for (int j = 0; j < TN; ++j) mma(af[cur][i], bf[cur][j], acc[i][j]);
          }
        }
        store_part(kt_store, sa_store, st_store, s ^ 1, ks, scb, sc_c);
        __builtin_amdgcn_sched_barrier(0);  // keep the slices where they were written
      }
    }
  };

  // ---- pipeline: tile t in LDS stage t&1, tiles t+1 .. t+DEPTH-1 in registers, tile t+DEPTH in flight
  ScaleBlock sc_cur{}, sc_nxt{};  // (SCV) scales of the block of four K tiles being stored, and of the block after it
  if constexpr (SCV) {
    load_scales(0, sc_cur);
    load_scales(1, sc_nxt);
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load_a(kt0 + d, ra[d]);
#pragma unroll
  for (int d = 0; d < WD; ++d) load_w(kt0 + d, rw[d]);
  store_tile(kt0, ra[0], rw[0], 0, sc_cur, 0);
  load_a(kt0 + DEPTH, ra[0]);
  load_w(kt0 + WD, rw[0]);
  __syncthreads();
  // (a register stage is refilled right after the MFMA/store block that drains it; a tile past
  //  the end is stored as zeros and adds nothing)
  constexpr int TRIP = SCV ? 4 : WD;  // K tiles per trip: whole rounds of the register rings, and of a scale block
  static_assert(TRIP % WD == 0, "a trip walks whole rounds of the register rings");
  // one trip; SCV: the four tiles stored are 1..3 of block `cur` and the first of block `nxt`, after which `cur` is free
  // and takes the block after `nxt` (consumed four K tiles from there)
  auto trip = [&](auto full, int kt, ScaleBlock& cur, ScaleBlock& nxt) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < TRIP; ++d) {
      // the tile stored during this step is kt + d + 1
      mfma_tile(full, d & 1, kt + d + 1, ra[(d + 1) % DEPTH], rw[(d + 1) % WD], (SCV && d == 3) ? nxt : cur, (d + 1) & 3);
      load_a(kt + d + 1 + DEPTH, ra[(d + 1) % DEPTH]);
      load_w(kt + d + 1 + WD, rw[(d + 1) % WD]);
      if constexpr (SCV) {
        if (d == 3) load_scales((kt - kt0) / 4 + 2, cur);
      }
      __syncthreads();
    }
  };
  auto k_loop = [&](auto full) {
    if constexpr (SCV) {
      // the two scale blocks swap roles from trip to trip: written out as two trips per round (no register copies, which
      // the compiler would place right behind the load they wait for); an odd last trip follows the loop (an exit in
      // the middle of the round would make the loop a join of two paths, where the wait-count insertion drains the queue)
      int kt = kt0;
      for (; kt + 2 * TRIP <= kt1; kt += 2 * TRIP) {
        trip(full, kt, sc_cur, sc_nxt);
        trip(full, kt + TRIP, sc_nxt, sc_cur);
      }
      if (kt < kt1) trip(full, kt, sc_cur, sc_nxt);
    } else {
      for (int kt = kt0; kt < kt1; kt += TRIP) trip(full, kt, sc_cur, sc_nxt);
    }
  };
  if (!SKIP || live == TM) k_loop(std::true_type{});
  else k_loop(std::false_type{});

  // ---- epilogue: D[i][j] of a 32x32 tile sits in lane (j + 32*((i/4)%2)), register 4*(i/8) + i%4
  if (p.paired && p.partial == nullptr) {
    const int half = p.N >> 1;
    if constexpr (TN % 2 == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int jj = 0; jj < TN / 2; ++jj) {
          const int col = ((n0 + wn0) >> 1) + jj * 32 + (lane & 31);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = m0 + wm0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (row < seg_hi && col < half)
              static_cast<uint16_t*>(p.y)[static_cast<int64_t>(row) * half + col] =
                  silu_mul_t<BF>(acc[i][2 * jj][r], acc[i][2 * jj + 1][r]);
          }
        }
      }
    } else {
      static_assert(TN % 2 == 0 || TN == 1, "one accumulator per wave, or pairs of them");
      // columns 0..15 of the accumulator are gate rows, 16..31 the matching up rows
      const int col = ((n0 + wn0) >> 1) + (lane & 15);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float up = __shfl_xor(acc[i][0][r], 16, 64);  // every lane takes part
          const int row = m0 + wm0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          if ((lane & 16) == 0 && row < seg_hi && col < half)
            static_cast<uint16_t*>(p.y)[static_cast<int64_t>(row) * half + col] = silu_mul_t<BF>(acc[i][0][r], up);
        }
      }
    }
    return;
  }
  // (one loop nest per output form keeps each fully unrolled nest small)
  // (a launch of the first columns is whole tiles and stays below any of these; the fused form comes here with partial sums only)
  const int n_lim = p.paired ? p.n_begin + p.part_cols : (second ? p.N : p.N >> 1);
  auto for_each = [&](auto&& body) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = n0 + wn0 + j * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + wm0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          if (row < seg_hi && col < n_lim) body(row, col, acc[i][j][r]);
        }
      }
    }
  };
  if (p.partial != nullptr) {
    const int part_at = second && !p.paired ? p.N - p.part_cols : p.n_begin;  // the column that the sums' first one would be
    float* part = p.partial + static_cast<int64_t>(blockIdx.z) * p.rows * p.part_cols - part_at;
    for_each([&](int row, int col, float v) { part[static_cast<int64_t>(row) * p.part_cols + col] = v; });
  } else if (p.bias == nullptr && p.residual == nullptr) {
    if (p.out_f32)
      for_each([&](int row, int col, float v) { static_cast<float*>(p.y)[static_cast<int64_t>(row) * p.N + col] = v; });
    else
      for_each([&](int row, int col, float v) {
        static_cast<uint16_t*>(p.y)[static_cast<int64_t>(row) * p.N + col] = BF ? bf16_bits_of(v) : f2h(v);
      });
  } else {
    for_each([&](int row, int col, float v) {
      const int64_t o = static_cast<int64_t>(row) * p.N + col;
      const float t = v + (p.bias != nullptr ? (BF ? bf16_to_f32(p.bias[col]) : h2f(p.bias[col])) : 0.f) +
                      (p.residual != nullptr ? (BF ? bf16_to_f32(p.residual[o]) : h2f(p.residual[o])) : 0.f);
      if (p.out_f32) static_cast<float*>(p.y)[o] = t;
      else static_cast<uint16_t*>(p.y)[o] = BF ? bf16_bits_of(t) : f2h(t);
    });
  }
}

template <int BITS, int BM, int BN, int WM, int WN, int DEPTH, bool BF, bool SKIP, int WX, bool FAST>
static hipError_t launch_pipe_form(const GemmParams& p, hipStream_t s) {
  constexpr int BK = 2 * GemmTraits<BITS>::G;
  constexpr int LDA = BK + 8;
  constexpr size_t lds = size_t(2) * (BM + BN) * LDA * 2;
  auto kern = gemm_pipe_kernel<BITS, BM, BN, WM, WN, DEPTH, BF, SKIP, WX, FAST>;
  if (lds > 65536) {
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kern));
    if (e != hipSuccess) return e;
  }
  const int m_tiles = p.indptr ? (p.rows + BM - 1) / BM + p.num_experts : (p.rows + BM - 1) / BM;
  const int nk = (p.ng + 1) / 2;
  const int split = p.partial ? (nk + p.kt_per_split - 1) / p.kt_per_split : 1;
  // the fused gate/up form walks whole 64-column blocks (32 gate + 32 up rows)
  constexpr int PB = ((WN / 32) % 2 == 0) ? 32 : 16;
  const int n_cols = p.paired ? ((p.N / 2 + PB - 1) / PB) * 2 * PB : p.N;
  const int n_last = p.n_end > 0 ? p.n_end : n_cols;
  if (n_last <= p.n_begin) return hipSuccess;
  GemmParams q = p;
  int n_tiles = (n_last - p.n_begin + BN - 1) / BN, first = p.n_begin;  // (first: columns that another launch has done)
  if (p.half_hi > 0) {
    q.hop_tile = (p.half_hi - p.half_lo + BN - 1) / BN;
    q.hop = p.N / 2 - q.hop_tile * BN;
    q.n_begin = p.half_lo;
    n_tiles = 2 * q.hop_tile;
    first = 2 * p.half_lo;
  }
  const dim3 grid(n_tiles, m_tiles, split);
  if (first > 0)
    note_kernel("gq::gemm_pipe_kernel<%d,%d,%d,%d,%d,%d,%s,%s,%d,%s> split=%d after %d columns", BITS, BM, BN, WM, WN, DEPTH,
                BF ? "true" : "false", SKIP ? "true" : "false", WX, FAST ? "true" : "false", split, first);
  else
    note_kernel("gq::gemm_pipe_kernel<%d,%d,%d,%d,%d,%d,%s,%s,%d,%s>", BITS, BM, BN, WM, WN, DEPTH, BF ? "true" : "false",
                SKIP ? "true" : "false", WX, FAST ? "true" : "false");
  hipLaunchKernelGGL(kern, grid, dim3(64 * (BM / WM) * (BN / WN)), lds, s, q);
  return hipGetLastError();
}

template <int BITS, int BM, int BN, int WM, int WN, int DEPTH = 2, bool BF = false, bool SKIP = false, int WX = 0>
static hipError_t launch_pipe_cfg(const GemmParams& p, hipStream_t s) {
  // the form without zero-selects: K in whole K tiles (fast_ok), and every workgroup's share of them in whole rounds of
  // the register rings (all of K, or the split's share; the last split gets what is left)
  constexpr int WD = DEPTH + WX;
  const int nk = (p.ng + 1) / 2;
  const bool whole_rounds = nk % WD == 0 && (p.partial == nullptr || p.kt_per_split % WD == 0);
  // q4 reads its scales 16 bytes (four K tiles) at a time there: whole blocks of four K tiles, 16-byte aligned scale rows
  const bool scale_blocks = BITS != 4 || (nk % 4 == 0 && (p.partial == nullptr || p.kt_per_split % 4 == 0) &&
                                          (reinterpret_cast<uintptr_t>(p.qs) & 15) == 0 && p.ng % 8 == 0);
  if (p.fast_ok && whole_rounds && scale_blocks)
    return launch_pipe_form<BITS, BM, BN, WM, WN, DEPTH, BF, SKIP, WX, true>(p, s);
  return launch_pipe_form<BITS, BM, BN, WM, WN, DEPTH, BF, SKIP, WX, false>(p, s);
}

// y = sum over splits of partial[s] + bias + residual, in the output type (y may be the residual
// buffer itself: every element is read before the same thread writes it)
template <bool HALVES>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int split,
                                                            int64_t count /* rows * cols */, int cols, int N,
                                                            const uint16_t* __restrict__ bias,
                                                            const uint16_t* residual, void* y, int out_f32, int bf16) {
  // bias, residual and a 16-bit y carry the model dtype: float16, or bfloat16 when bf16 is set
  auto in = [bf16](uint16_t bits) { return bf16 ? bf2f(bits) : h2f(bits); };
  auto out = [bf16](float v) { return bf16 ? f2bf(v) : f2h(v); };
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  // element i of the sums -> element of y
  const int w = cols >> 1, half = N >> 1;
  auto at = [&](int64_t i) -> int64_t {
    if (!HALVES) return i;
    const int c = static_cast<int>(i % cols);
    return (i / cols) * N + (c < w ? half - w + c : N - w + (c - w));
  };
  if (((N | (HALVES ? cols : 0)) & (HALVES ? 7 : 3)) == 0) {  // runs of columns are 16-byte aligned: four per thread
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; 4 * i < count; i += stride) {
      float4 a = *reinterpret_cast<const float4*>(partial + 4 * i);
      for (int sidx = 1; sidx < split; ++sidx) {
        const float4 b = *reinterpret_cast<const float4*>(partial + sidx * count + 4 * i);
        a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
      }
      const int64_t o4 = at(4 * i);
      if (bias != nullptr) {
        const int col = static_cast<int>(o4 % N);
        const uint2 bb = *reinterpret_cast<const uint2*>(bias + col);
        a.x += in(static_cast<uint16_t>(bb.x & 0xffffu)); a.y += in(static_cast<uint16_t>(bb.x >> 16));
        a.z += in(static_cast<uint16_t>(bb.y & 0xffffu)); a.w += in(static_cast<uint16_t>(bb.y >> 16));
      }
      if (residual != nullptr) {
        const uint2 rr = *reinterpret_cast<const uint2*>(residual + o4);
        a.x += in(static_cast<uint16_t>(rr.x & 0xffffu)); a.y += in(static_cast<uint16_t>(rr.x >> 16));
        a.z += in(static_cast<uint16_t>(rr.y & 0xffffu)); a.w += in(static_cast<uint16_t>(rr.y >> 16));
      }
      if (out_f32) {
        *reinterpret_cast<float4*>(static_cast<float*>(y) + o4) = a;
      } else {
        uint2 o;
        o.x = static_cast<uint32_t>(out(a.x)) | (static_cast<uint32_t>(out(a.y)) << 16);
        o.y = static_cast<uint32_t>(out(a.z)) | (static_cast<uint32_t>(out(a.w)) << 16);
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(y) + o4) = o;
      }
    }
  } else {
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < count; i += stride) {
      float a = partial[i];
      for (int sidx = 1; sidx < split; ++sidx) a += partial[sidx * count + i];
      const int64_t o = at(i);
      if (bias != nullptr) a += in(bias[o % N]);
      if (residual != nullptr) a += in(residual[o]);
      if (out_f32) static_cast<float*>(y)[o] = a;
      else static_cast<uint16_t*>(y)[o] = out(a);
    }
  }
}

template __global__ void splitk_reduce_kernel<false>(const float* __restrict__, int, int64_t, int, int, const uint16_t* __restrict__, const uint16_t*,
                                                    void*, int, int);
template __global__ void splitk_reduce_kernel<true>(const float* __restrict__, int, int64_t, int, int, const uint16_t* __restrict__, const uint16_t*,
                                                   void*, int, int);

__global__ __launch_bounds__(256) void splitk_reduce_silu_kernel(const float* __restrict__ partial, int split,
                                                                 int64_t rows, int cols, int N, int n_begin, int pb,
                                                                 uint16_t* __restrict__ y, int bf16) {
  const int half = (N - n_begin) >> 1;
  const int64_t count = rows * cols, outs = rows * half;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < outs; i += stride) {
    const int64_t row = i / half;
    const int oc = static_cast<int>(i - row * half);
    const int64_t at = row * cols + (oc / pb) * 2 * pb + oc % pb;  // pb gate columns, then their pb up columns
    float g = partial[at], u = partial[at + pb];
    for (int sidx = 1; sidx < split; ++sidx) {
      g += partial[sidx * count + at];
      u += partial[sidx * count + at + pb];
    }
    y[row * (N >> 1) + (n_begin >> 1) + oc] = bf16 ? silu_mul_bf(g, u) : silu_mul_h(g, u);
  }
}

// The plain q4 GEMM's tiles beyond 64 rows, each with its fitted cost (us): a launch of `tiles x split` workgroups of `kt` K
// tiles takes
//   base + whole * kt * pairs + odd * kt * odd_one + filled * kt * per_cu + live * kt * per_cu * (rows / tile rows) + round * rounds
//        + (split: reduce + 1e-6 * traffic * split * rows * N) + 1e-6 * store * rows * N
// per_cu = workgroups / 256 (fractional), rounds = per_cu rounded up; the tiles of four waves sit two on a CU (pairs = rounds / 2, a
// lone one `odd_one`), the others one (pairs = rounds).  The last, partly filled round is what decides between tiles; the terms in
// the fractional per_cu are the part's power limit (a round on half the CUs runs faster than a full one) and, for the tiles whose waves
// skip row blocks past the last row, the matrix work that is left out.
struct TileCost {
  int bm, bn;
  int skip;  // waves skip the 32-row blocks past the last row (256-row tiles: for a row count that leaves such blocks)
  float base, whole, odd, filled, live, round, reduce, traffic, store;
};
// Least squares (non-negative) over 22 shapes (N 2048..37888, K 2048..28672, the projections of 1.5B to 70B models) x 19 row counts from
// 72 to 4096 x splits of 1 to 16: 7700 timings, 5-6 % rms.  Choosing by it instead of by the rules it replaced (128 x 128 tiles split up to
// 256 workgroups to 1024 rows, three unsplit tiles beyond) makes those launches 7.5 % (bfloat16 11 %) faster on average, where
// the best of all measured choices would make 8.3 % (11.3 %).  For instance (us): 4096 x 14336 at 160 / 300 / 640 / 777 rows 43.6 / 77.8 /
// 113.5 / 129 -> 36.9 / 62 / 89.8 / 117 (bfloat16 46.3 / 85.2 / 122.5 / 143 -> 37.0 / 61.2 / 91.9 / 113), 4096 x 4096 at 300 rows 37.1 -> 27.2, 28672 x
// 4096 at 160 / 300 / 777 rows 66.3 / 112.5 / 219.8 -> 54.3 / 92.7 / 207.4; from 1536 rows on the choice is mostly the old one.
constexpr TileCost kTilesF16[] = {
    {128, 128, 0, 6.83f, 0.593f, 0.37f, 0.219f, 0, 0, 2.51f, 0.858f, 0.33f},
    {128, 256, 0, 5.43f, 0.549f, 0, 0.419f, 0, 2.18f, 2.62f, 0.719f, 0.149f},
    {256, 256, 0, 0, 0.922f, 0, 0.681f, 0, 11.9f, 2.66f, 0.37f, 0.0425f},
    {256, 256, 1, 0.992f, 0.934f, 0, 0, 0.712f, 10.5f, 3.68f, 0.405f, 0},
    {256, 128, 1, 7.7f, 0.57f, 0, 0, 0.437f, 1.24f, 2.91f, 0.569f, 0},
    {64, 128, 0, 5.69f, 0.446f, 0.298f, 0.119f, 0, 0.175f, 2.0f, 1.22f, 0.604f},
};
constexpr TileCost kTilesBf16[] = {  // (more vector instructions per weight: the tiles that dequantise it less often are ahead)
    {128, 128, 0, 8.01f, 0.621f, 0.4f, 0.224f, 0, 0, 2.51f, 0.73f, 0.371f},
    {128, 256, 0, 6.05f, 0.625f, 0, 0.385f, 0, 2.47f, 2.64f, 0.578f, 0.23f},
    {256, 256, 0, 0.544f, 1.01f, 0, 0.574f, 0, 10.2f, 3.75f, 0.395f, 0.152f},
    {256, 256, 1, 6.61f, 0.969f, 0, 0, 0.692f, 4.4f, 4.43f, 0.384f, 0.0978f},
    {256, 128, 1, 7.17f, 0.552f, 0, 0, 0.412f, 2.2f, 2.87f, 0.518f, 0},
    {64, 128, 0, 6.81f, 0.507f, 0.338f, 0.128f, 0, 0.183f, 1.99f, 0.916f, 0.339f},
};

// tiles of `bn` columns that N columns take, in one run of columns or in two of half of them
static int64_t column_tiles(int64_t N, int bn, int runs) { return runs * ((N / runs + bn - 1) / bn); }

static float tile_us(const TileCost& c, int64_t rows, int64_t N, int nk, int kt, int split, int runs) {
  const int64_t mt = (rows + c.bm - 1) / c.bm, wgs = mt * column_tiles(N, c.bn, runs) * split, rounds = (wgs + 255) / 256;
  const float live = static_cast<float>(rows) / static_cast<float>(mt * c.bm), mn = 1e-6f * static_cast<float>(rows) * static_cast<float>(N);
  const bool pairs = c.bm * c.bn <= 128 * 128;  // (four waves: two workgroups on a CU)
  const float ktf = static_cast<float>(split > 1 ? kt : (nk + 3) / 4 * 4), per_cu = static_cast<float>(wgs) / 256.f;
  const float us = c.base + ktf * (c.whole * static_cast<float>(pairs ? rounds / 2 : rounds) + (pairs ? c.odd * static_cast<float>(rounds % 2) : 0.f) +
                                   per_cu * (c.filled + c.live * live)) +
                   c.round * static_cast<float>(rounds) + c.store * mn;
  // (a split has to be 2 % ahead on paper)
  return split > 1 ? (us + c.reduce + c.traffic * static_cast<float>(split) * mn) * 1.02f : us;
}
static bool tile_applies(const TileCost& c, int64_t rows, int nk) {
  // (fitted from K = 2048 on: what a workgroup costs before and behind its K loop is not told apart there, and for a short K this tile,
  //  whose weight loads run four K tiles ahead, looks a quarter of its time: 16272 x 128 at 3596 rows 74 us, 256 x 256 47)
  if (c.bm == 256 && c.bn == 128 && nk < 16) return false;
  return c.bm < 256 || (c.skip != 0) == (c.bn == 128 || rows % 256 != 0);
}

// one launch for all of N columns
static SplitPlan plan_one(const TileCost* costs, int64_t rows, int64_t N, int nk, int64_t scratch_bytes, int runs, float* best_us) {
  SplitPlan best{0, 0, 1, 1 << 28};
  for (int t = 0; t < 6; ++t) {
    const TileCost& c = costs[t];
    if (!tile_applies(c, rows, nk)) continue;
    const int64_t tiles = ((rows + c.bm - 1) / c.bm) * column_tiles(N, c.bn, runs);
    int last = 0;
    for (int want = 1; want <= 16; ++want) {
      const int kt = ((nk + want - 1) / want + 3) / 4 * 4;  // (the K loop advances four tiles at a time)
      const int split = (nk + kt - 1) / kt;
      // at least four K tiles per workgroup, and no more workgroups than two and a half rounds of one per CU
      if (split > 1 && (want > nk / 4 || tiles * split > 640 || split * rows * N * 4 > scratch_bytes)) break;
      if (split == last) continue;
      last = split;
      const float us = tile_us(c, rows, N, nk, kt, split, runs);
      if (best.bm == 0 || us < *best_us) {
        *best_us = us;
        best = SplitPlan{c.bm, c.bn, split, split > 1 ? kt : 1 << 28};
      }
    }
  }
  return best;
}

// ... or two: a last round of workgroups that is far from full costs about what a full one does, so the columns of the whole rounds run
// first on one of the large tiles and the rest on whatever suits it (a smaller tile, K split).  Taken where the model puts it 7 % ahead
// (it is some 5 % too optimistic about two launches).  Measured (us, one launch -> two): 6144 x 4096 at 2700 rows 181 -> 153, 22016 x 4096 at
// 1536 326 -> 275, 10240 x 8192 at 2048 377 -> 327, 15360 x 5120 at 1200 230 -> 205, 37888 x 3584 at 450 164 -> 145; 28672 x 4096 at 2048 (3.5
// rounds) within the noise either way, and left alone by the 7 %.
// A rest that splits K takes the same columns of both halves of the N (runs = 2): of a gate_up projection those are whole pairs, as
// the fused form needs them, and either form then adds up an element in the same order.  Unsplit, the order is the same everywhere and the
// columns adjoin.  (The model puts this 0.1 % behind a rest of adjoining columns that may split: 9 % where none of the split fits two
// halves, 5120 x 13824 at 3107 rows 419 -> 456, and mostly nothing, 22016 x 4096 at 380 rows 89.0 -> 87.6.)
static SplitPlan plan_by_cost(int64_t rows, int64_t N, int nk, int bf16, int64_t scratch_bytes) {
  if (scratch_bytes > kMaxSplitBytes) scratch_bytes = kMaxSplitBytes;
  const TileCost* const costs = bf16 ? kTilesBf16 : kTilesF16;
  float one_us = 0.f;
  SplitPlan best = plan_one(costs, rows, N, nk, scratch_bytes, 1, &one_us);
  float best_us = one_us / 1.07f;
  for (int t = 1; t <= 4; ++t) {  // (the tiles of one workgroup per CU)
    const TileCost& c = costs[t];
    if (!tile_applies(c, rows, nk)) continue;
    const int64_t mt = (rows + c.bm - 1) / c.bm;
    for (int runs = 1; runs <= (N % 2 == 0 ? 2 : 1); ++runs) {
      const int64_t nt = column_tiles(N, c.bn, runs), head = mt * nt / 256 * 256 / mt / runs * runs;  // column tiles of the whole rounds
      if (head < 1 || head >= nt) continue;
      const int64_t n_head = head * c.bn;
      const float head_us = tile_us(c, rows, n_head, nk, 0, 1, runs) - 3.f;  // (its launch overlaps the other's)
      if (head_us >= best_us) continue;
      float rest_us = 0.f;
      SplitPlan rest = plan_one(costs, rows, N - n_head, nk, runs == 2 ? scratch_bytes : 0, runs, &rest_us);
      if (head_us + rest_us < best_us) {
        best_us = head_us + rest_us;
        best = rest;
        best.n_head = n_head;
        best.halves = runs == 2;
        best.head_bm = c.bm;
        best.head_bn = c.bn;
      }
    }
  }
  return best;
}

// K up to 512 and several rounds of workgroups, where the output's stores weigh as much as the K loop: rounds x (time of one tile), rounds =
// ceil(tiles / resident workgroups) (256, 512 for 128 x 128, a lone one of which takes 0.72 of a pair's time), tile times from the rates
// measured with balanced rounds (1035 / 870 / 806 TFLOP/s); the smaller tile has to win by 8 %.  (us, by the cost above / by this: 28800 x 80 at 2734
// rows 92 / 58, 35712 x 360 at 760 60 / 41, 20120 x 272 at 3751 138 / 99, 27376 x 64 at 1732 55 / 35.)
constexpr int kShortTiles = 8;
static SplitPlan plan_by_rounds(int64_t rows, int64_t N) {
  const int64_t mt = (rows + 127) / 128, big = ((rows + 255) / 256) * ((N + 255) / 256), mid = mt * ((N + 255) / 256), small = mt * ((N + 127) / 128);
  const int64_t per_cu = (small + 255) / 256;
  const double t_small = 16384.0 / (806.0 / 512);
  const double c_big = static_cast<double>((big + 255) / 256) * (65536.0 / (1035.0 / 256)), c_mid = static_cast<double>((mid + 255) / 256) * (32768.0 / (870.0 / 256)),
               c_small = static_cast<double>(per_cu / 2) * t_small + static_cast<double>(per_cu % 2) * 0.72 * t_small;
  SplitPlan plan{256, 256, 1, 1 << 28};
  double best = c_big;
  if (c_mid < 0.92 * best) { plan.bm = 128; best = c_mid; }
  if (c_small < 0.92 * best) plan.bm = plan.bn = 128;
  return plan;
}

SplitPlan plan_split_k(int64_t rows, int64_t N, int64_t K, int bits, int group_size, bool grouped, int bf16, int64_t scratch_bytes) {
  SplitPlan plan{0, 0, 1, 1 << 28};
  if (grouped || rows <= 0 || N <= 0 || K <= 0 || (K & 7) != 0) return plan;
  const int ng = static_cast<int>((K + group_size - 1) / group_size);
  const int nk = (ng + 1) / 2;
  if (bits == 4 && rows > 64 && options().gemm_split_k <= 0) {
    if (nk <= kShortTiles && ((rows + 127) / 128) * ((N + 127) / 128) >= 200) return plan_by_rounds(rows, N);
    return plan_by_cost(rows, N, nk, bf16, scratch_bytes);
  }
  // few rows: the GEMM is bound by streaming the weights, and 128-wide column tiles alone leave
  // most CUs idle (o_proj / down have 32 of them).  Match the tile height to the rows and cut K
  // until about one workgroup per CU exists.
  // (up to 1024 rows: down_proj, 32 column tiles and a long K, ran 150 us flat from 257 to 512 rows unsplit)
  if (rows > 1024) return plan;
  const int bm = rows <= 32 ? 32 : (rows <= 64 ? 64 : 128);
  const int64_t tiles = ((rows + bm - 1) / bm) * ((N + 127) / 128);
  if (rows > 128 && tiles >= 200) return plan;  // the regular tiles already fill the chip
  plan.bm = bm;
  plan.bn = 128;
  // Splitting K pays with partial sums (split * rows * N * 8 bytes written and read back): only
  // when the tiles alone leave CUs idle, and never beyond about twice the weight bytes.
  int split = 1;
  if (tiles < 200 || options().gemm_split_k > 0) {
    // one workgroup per CU: measured 8-20 % faster than two (o_proj, qkv, down at 17..128 rows), whose
    // partial sums cost more than the second workgroup hides
    const int64_t want = options().gemm_split_k > 0 ? options().gemm_split_k : 256;  // (tuning override)
    split = static_cast<int>((want + tiles - 1) / tiles);
    const int64_t cap = K / (7 * rows);
    if (options().gemm_split_k <= 0 && split > cap) split = static_cast<int>(cap);
    if (split > nk / 4) split = nk / 4;  // at least four K tiles per workgroup
    if (split < 1) split = 1;
  }
  // the K loop advances four tiles at a time in the few-row kernels: whole rounds per workgroup
  plan.kt_per_split = ((nk + split - 1) / split + 3) / 4 * 4;
  plan.split = (nk + plan.kt_per_split - 1) / plan.kt_per_split;
  return plan;
}

// q3: 128 x 256 tiles rather than 128 x 128 (a K tile is 80 wide and the 256 x 256 tile does not fit LDS)?  A launch costs rounds x
// (time of one tile), rounds = ceil(tiles / resident workgroups) (256, 512 for 128 x 128), tile times from the rates measured with
// balanced rounds, 739 / 566 TFLOP/s.
static bool q3_wide_tile(int64_t rows, int64_t N) {
  const int64_t mid = ((rows + 127) / 128) * ((N + 255) / 256), small = ((rows + 127) / 128) * ((N + 127) / 128);
  const double t_mid = 32768.0 / (739.0 / 256), t_small = 16384.0 / (566.0 / 512);
  // 128 x 128: two workgroups share a CU; one on its own runs faster than its half of a pair (0.72 of the pair's time)
  const int64_t per_cu = (small + 255) / 256;
  const double c_small = static_cast<double>(per_cu / 2) * t_small + static_cast<double>(per_cu % 2) * 0.72 * t_small;
  // a partly filled last round runs faster than a full one (the part is power-limited), which favours the larger
  // tile: the smaller one has to win by 8 % on paper
  return c_small >= 0.92 * static_cast<double>((mid + 255) / 256) * t_mid;
}

// the planned tile of a plain q4 matmul (see plan_split_k)
template <bool BF>
static hipError_t launch_planned_q4(const GemmParams& p, hipStream_t s) {
  if (p.bm_hint == 32) return launch_pipe_cfg<4, 32, 128, 32, 32, 4, BF>(p, s);
  if (p.bm_hint == 64) return launch_pipe_cfg<4, 64, 128, 32, 64, 4, BF>(p, s);
  if (p.bm_hint == 128 && p.bn_hint == 256) return launch_pipe_cfg<4, 128, 256, 64, 64, 2, BF>(p, s);
  if (p.bm_hint == 256 && p.bn_hint == 128) return launch_pipe_cfg<4, 256, 128, 64, 64, 2, BF, true, 2>(p, s);
  if (p.bm_hint == 256)
    return p.rows % 256 != 0 && (p.ng + 1) / 2 > kShortTiles ? launch_pipe_cfg<4, 256, 256, 128, 64, 2, BF, true, 2>(p, s) : launch_pipe_cfg<4, 256, 256, 128, 64, 2, BF>(p, s);
  return launch_pipe_cfg<4, 128, 128, 64, 64, 2, BF>(p, s);
}

// Expert segments of a q4 model: the tile height follows the rows per expert on average, r.  Measured on 8 / 16 / 64 / 128 experts of 768
// x 2048 to 28672 x 4096 (f16, us; tiles of 32 / 64 / 128 / 256 rows): 64 experts of 2816 x 2048 at r = 20 63.7 / 81.0 / 107 / 108, at r =
// 32 93.9 / 84.0 / 111 / 125, at r = 64 145 / 121 / 116 / 125, at r = 96 - / 163 / 120 / 140, at r = 128 - / 194 / 175 / 151; 8 experts of 4096 x
// 14336 at r = 20 89.5 / 103, r = 64 183 / 158 / 142 / 170, r = 96 - / 177 / 150 / 185, r = 128 - / 258 / 232 / 189.  Beyond r = 100 a segment no longer fits
// 128 rows, and 256-row tiles whose waves skip the 32-row blocks past the segment's end are ahead: matrix work is the segment's rows
// rounded up to 32, and the expert's weights are dequantised once.  bfloat16 the same (64 experts of 5120 x 3584 at r = 128 / 192: 468 / 561
// against 560 / 728 for 128 rows).  A short K the same: tiles of 128 / 256 rows at r = 64 / 96 on 64 experts of 2048 x 704 38.6 / 46.7, 42.9 / 51.5,
// on 128 of 1024 x 384 28.9 / 38.1, 34.4 / 41.2, on 32 of 4096 x 640 34.2 / 45.5, 42.4 / 48.9.
template <bool BF>
static hipError_t launch_grouped_q4(const GemmParams& p, hipStream_t s) {
  const int64_t rows = p.rows, experts = p.num_experts;
  if (rows <= 24 * experts) return launch_pipe_cfg<4, 32, 128, 32, 32, 4, BF>(p, s);
  if (rows <= 48 * experts) return launch_pipe_cfg<4, 64, 128, 32, 64, 4, BF>(p, s);
  // (a K of one K tile keeps the 256-row form and its two launches)
  if (rows <= 100 * experts && p.K > 64) return launch_pipe_cfg<4, 128, 128, 64, 64, 2, BF>(p, s);
  // 256 columns per tile while that gives every CU a workgroup, else 128 (e2 of a Mixtral layer, 128 wide tiles: r = 128 189
  // against 270 us; 16 experts of 4096 x 2048, 256 of them: 53 against 63)
  const int64_t tiles_x = (p.N + 255) / 256, live = experts > rows / 256 ? experts : rows / 256;  // row tiles that hold rows
  if (tiles_x * live < 256) {
    // ... and for bfloat16 128 rows where those tiles, one and a half per expert at r = 128, have a CU each or take one round where the tall
    // ones take two (128 rows / 256: 4 experts of 2048 x 2048 at r = 128 and 256 0.85 and 0.81 of the time, 8 of 64..2048 x 4096 0.84..0.87, 17
    // of 2048 x 1024 0.69, 12 of 2048 x 4096 at r = 256 0.72; on the other side 12 of 2048 x 2048 at r = 128 1.26, 8 of 4096 x 4096 1.28;
    // float16 measures alike, 0.78 and 0.69, and keeps the tall tiles it has had there)
    const int64_t n_tiles = (p.N + 127) / 128, wg128 = (rows / 128 + experts / 2) * n_tiles;
    const int64_t tall = rows / 256 + experts / 2, wg256 = (tall > experts ? tall : experts) * n_tiles;
    if (BF && (wg128 <= 256 || (wg256 > 256 && wg128 <= 512))) return launch_pipe_cfg<4, 128, 128, 64, 64, 2, BF>(p, s);
    return launch_pipe_cfg<4, 256, 128, 64, 64, 2, BF, true, 2>(p, s);
  }
  // A last round of workgroups that is at most about half full costs a whole round here (the kernel waits on
  // memory, not on the matrix pipe): its columns go to a second launch on the narrow tile, whose workgroups take
  // half as long.  (Mixtral's e1_e3, 112 column tiles x 8 experts = 3.5 rounds of 256.)
  const int64_t rounds = tiles_x * live / 256, rest = tiles_x * live % 256;
  if (rest > 0 && rest <= 144) {
    GemmParams a = p, b = p;
    a.n_end = static_cast<int>(rounds * 256 / live * 256);
    b.n_begin = a.n_end;
    if (a.n_end > 0 && a.n_end < p.N) {
      const hipError_t e = launch_pipe_cfg<4, 256, 256, 128, 64, 2, BF, true, 2>(a, s);
      if (e != hipSuccess) return e;
      return launch_pipe_cfg<4, 256, 128, 64, 64, 2, BF, true, 2>(b, s);
    }
  }
  // (both tiles' weight loads run two more K tiles ahead than their activation loads: Mixtral's e2 on the narrow tile
  // at 64 / 128 / 256 rows per expert 201 -> 177, 236 -> 213, 320 -> 305 us; e1_e3 on the wide one 1-2 %)
  return launch_pipe_cfg<4, 256, 256, 128, 64, 2, BF, true, 2>(p, s);
}

hipError_t launch_gemm_pipe(const GemmParams& p, int bits, hipStream_t s) {
  if ((p.K & 7) != 0 || p.ng == 0) return hipErrorNotSupported;
  const int variant = options().gemm_variant;
  if (p.paired && (p.N & 1)) return hipErrorNotSupported;
  if (p.bf16) {
    // bfloat16 models: plain and grouped matmul (no folded activation)
    if (p.indptr == nullptr && bits == 4) return launch_planned_q4<true>(p, s);
    if (p.bm_hint > 0 && p.indptr == nullptr) {  // few rows, K possibly split (see plan_split_k)
      if (p.bm_hint == 32) return launch_pipe_cfg<3, 32, 128, 32, 32, 4, true>(p, s);
      if (p.bm_hint == 64) return launch_pipe_cfg<3, 64, 128, 32, 64, 4, true>(p, s);
      return launch_pipe_cfg<3, 128, 128, 64, 64, 2, true>(p, s);
    }
    if (p.partial != nullptr) return hipErrorNotSupported;
    if (p.indptr != nullptr) {
      if (bits == 4) return launch_grouped_q4<true>(p, s);
      const bool wide = p.rows >= 96 * p.num_experts &&
                        (static_cast<int64_t>(p.rows) / 128 + p.num_experts) * ((p.N + 255) / 256) >= 768;
      return wide ? launch_pipe_cfg<3, 128, 256, 64, 64, 2, true>(p, s)
                  : launch_pipe_cfg<3, 128, 128, 64, 64, 2, true>(p, s);
    }
    if (q3_wide_tile(p.rows, p.N)) return launch_pipe_cfg<3, 128, 256, 64, 64, 2, true>(p, s);
    return launch_pipe_cfg<3, 128, 128, 64, 64, 2, true>(p, s);
  }
  if (p.indptr == nullptr && bits == 4 && variant != 6 && variant != 7 && variant != 9) return launch_planned_q4<false>(p, s);
  if (p.bm_hint > 0 && variant < 0) {
    if (p.bm_hint == 32) return launch_pipe_cfg<3, 32, 128, 32, 32, 4>(p, s);
    if (p.bm_hint == 64) return launch_pipe_cfg<3, 64, 128, 32, 64, 4>(p, s);
    return launch_pipe_cfg<3, 128, 128, 64, 64>(p, s);
  }
  if (p.indptr != nullptr && bits == 4) {
    // (tuning override: 6 / 9 / 10 / 11 force 128 x 128, 128 x 256, 256 x 256 and 256 x 128 tiles)
    if (variant == 6) return launch_pipe_cfg<4, 128, 128, 64, 64>(p, s);
    if (variant == 9) return launch_pipe_cfg<4, 128, 256, 64, 64>(p, s);
    if (variant == 10) return launch_pipe_cfg<4, 256, 256, 128, 64, 2, false, true, 2>(p, s);
    if (variant == 11) return launch_pipe_cfg<4, 256, 128, 64, 64, 2, false, true, 2>(p, s);
    if (variant != 7) return launch_grouped_q4<false>(p, s);
  }
  // q3, from about 64 rows per expert on: 256-row tiles whose waves skip the row blocks past the segment's end
  if (p.indptr != nullptr && ((variant < 0 && p.rows > 48 * p.num_experts) || variant == 10 || variant == 11))
    return launch_pipe_cfg<3, 256, 128, 64, 64, 2, false, true>(p, s);
  if (bits == 4) {  // (tuning override: the forced tiles of a plain matmul)
    if (variant == 9) return launch_pipe_cfg<4, 128, 256, 64, 64>(p, s);
    if (variant == 7) return launch_pipe_cfg<4, 256, 256, 128, 64>(p, s);
    return launch_pipe_cfg<4, 128, 128, 64, 64>(p, s);
  }
  if (p.indptr != nullptr && (variant < 0 || variant == 1)) {  // grouped, few rows per expert
    if (p.rows <= 16 * p.num_experts) return launch_pipe_cfg<3, 32, 128, 32, 32, 4>(p, s);
    if (p.rows <= 48 * p.num_experts) return launch_pipe_cfg<3, 64, 128, 32, 64, 4>(p, s);
  }
  // q3: a K tile is 80 wide, so the 256 x 256 tile does not fit LDS; 128 x 256 does
  const bool plain_wide = p.indptr == nullptr && q3_wide_tile(p.rows, p.N);
  const bool grouped_wide = p.indptr != nullptr && p.rows >= 96 * p.num_experts &&
                            (static_cast<int64_t>(p.rows) / 128 + p.num_experts) * ((p.N + 255) / 256) >= 768;
  if (variant == 9 || (variant != 6 && (plain_wide || grouped_wide)))
    return launch_pipe_cfg<3, 128, 256, 64, 64>(p, s);
  return launch_pipe_cfg<3, 128, 128, 64, 64>(p, s);
}

}  // namespace gq
