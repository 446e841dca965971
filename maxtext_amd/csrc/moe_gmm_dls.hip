// Grouped matmul: the persistent kernel on tiles of 256, 192 or 160 rows x 256 channels for operands that need no conversion (int8 x int8, bf16 x bf16 and
// fp8 x fp8 with per-row x per-channel scales, prefill) with the stages of a block's consecutive tiles as ONE request
// stream.
//
// Both operands go global -> LDS without passing through registers (buffer_load ... lds, 1 KB = 8 rows of 128 bytes per
// wave instruction; XOR-swizzled unpadded rows; two buffers of 64 KB, 56 KB for lower tiles).  8 waves as 2 x 4, each 128 (96,
// 80) x 64 of the tile in 16 x 16 MFMAs (16x16x64 i8 / 16x16x32 bf16 / 16x16x128 f8f6f4).
//
// Schedule: the two waves of a SIMD take turns.  A stage (128 bytes of K) is four phases, one 64 x 32 quadrant of the
// wave's tile each (16 MFMAs, 8 of fp8: 256 cycles); a phase is a fetching side (fragment reads, two requests, waits), a
// barrier, a multiplying side and a barrier, and waves 4 .. 7 run one barrier behind waves 0 .. 3, so that while one
// wave of a SIMD multiplies the other fetches.  Everything that can stall a wave in order (a request that finds the
// address unit's queue full, a fragment that is not there yet) then stalls it while the matrix unit works for its
// neighbour.  Before, both waves ran one mixed stream (a request behind every third MFMA, one barrier per stage) and
// stalled together.  Mixtral shape, 16384 routed rows, same box: int8 first projection + SwiGLU 1.63 -> 1.50 ms, second
// 0.88 -> 0.78; bf16 1.52 -> 1.40 and 1.76 -> 1.51; fp8 1.54 -> 1.46 and 0.87 -> 0.76, 6000 rows 0.36 -> 0.30 (bf16
// 1.37 PFLOP/s, int8 2.57, fp8 2.64 with the padding of ragged groups not counted).  What bounds it now is power: wave
// priorities, the place of the waits and the spread of the reads over the phases all measure within 1 %.
//
// Slots and waits.  A stage arrives in four halves of two requests per wave, requested in the order they become free two
// stages earlier: activation rows h = 0 in phase 2 (read in phase 1), weight rows g = 0 in phase 3, g = 1 in phase 4 (read
// in phases 1 and 2), activation rows h = 1 in phase 1 of the next stage (read in phase 3).  A wave ends the reads of a phase
// before its hand-over barrier, so a slot is requested again only behind every wave's reads.  At most five halves may be
// outstanding where the next phase reads new data (vmcnt 10), i.e. a request has at least five phases (2500 cycles).
//
// The requests run ahead ACROSS tile boundaries: a tile's first two stages arrive while the previous tile is still being
// multiplied, and the record of the next tile is read a whole tile ahead.  Addresses go through buffer descriptors that
// end where the tile's rows (the expert's weight matrix) end: rows past the end read as zeros, the lane-dependent part of
// an address is the same for every tile and the tile-dependent part is scalar, so moving the stream on to the next tile
// costs no vector work (with a row index: one index load per request).  What is left between two tiles is the epilogue,
// which both waves of a SIMD run side by side.
//
// fp8: e4m3 weights, e4m3 or e5m2 activations; scales per row / per tensor x per channel / per tensor, applied in the
// epilogue: what gmm() quantises to, kernels/megablox/ops.py:232-267, and the e5m2 gradient times e4m3 weights of its
// backward, ops.py:583-604.

#include "moe_gmm_common.h"

namespace moe {

template <int OP_, bool GLU_, int LF_ = 0, bool KN_ = false, int TM_ = 8>
struct DlsCfg {
  static constexpr int OP = OP_;
  static constexpr bool GLU = GLU_;
  static constexpr int LF = LF_;  // fp8 activations: 0 = e4m3, 1 = e5m2 (format selector of the MFMA's second operand)
  // weights given as [G, K, N] (the contraction index as the row: dlhs of a layer whose weights are [G, N, K], read as they
  // are).  The weight half of a stage then holds 128 (bf16: 64) contraction rows x 256 output channels (four rows of 256 or two
  // of 512 bytes per wave instruction) and the weight fragments come out of it through ds_read_b64_tr_b8 / _b16.
  static constexpr bool KN = KN_;
  // Row tiles of a wave: 8, 6 or 5, i.e. 256, 192 or 160 rows to a tile.  Row tile i of wave row wm holds the tile's rows
  // 32 i + 16 wm .. + 15; the first four are half h = 0 of the activations (128 rows), the others half h = 1.
  static constexpr int TM = TM_, H1 = TM - 4;
  static constexpr int BM = TM * 32, BN = 256, BKB = 128, MI = 16;
  static constexpr int ESZ = OP == OP_BF16 ? 2 : 1, BK = BKB / ESZ;
  static constexpr int WAVES_M = 2, WAVES_N = 4, NWAVES = 8, THREADS = NWAVES * kWave;
  static constexpr int WN = BN / WAVES_N, TN = WN / MI;
  // requests per wave and stage: 2 for the first activation half, NA1 for the second (64 rows' worth at least: rows past the
  // tile's are past its descriptor and fetch nothing), 4 for the weights
  static constexpr int NA1 = H1 > 2 ? 2 : 1, A_IPW = 2 + NA1, B_IPW = BN / 8 / NWAVES;
  static constexpr int A_ROWS = 128 + NA1 * 64, A_STAGE = A_ROWS * BKB, STAGE = A_STAGE + BN * BKB, LDS_BYTES = 2 * STAGE;
  static_assert(TM == 8 || TM == 6 || TM == 5, "row tiles");
  static constexpr int OUT_BN = GLU ? BN / 2 : BN;
  static_assert(OP == OP_I8 || OP == OP_BF16 || OP == OP_F8, "operands");
  static_assert(LF == 0 || OP == OP_F8, "only fp8 activations come in two formats");
  static_assert(!KN || (OP != OP_I8 && !GLU), "[G, K, N] weights: fp8 or bf16 without rhs_up");
  // slot of the 16-byte chunk c of contraction row r in a [G, K, N] weight stage: c ^ kn_swz(r); the 8 rows of a transposing
  // 1-byte read and those of the next lane group (16 rows further) then fall into 16 different 16-byte bank groups (bf16: see
  // tr_swz)
  __device__ static __forceinline__ int kn_swz(int row) { return OP == OP_BF16 ? tr_swz(row) : (row & 7) ^ (((row >> 4) & 1) << 3); }
  static constexpr int KN_ROW = BN * ESZ, KN_RPR = 1024 / KN_ROW;  // bytes of a contraction row, rows per request
  __device__ static __forceinline__ int swz(int row) { return (row >> 1) & 7; }
};

template <typename C>
__global__ __launch_bounds__(C::THREADS, 2) void gmm_dls_kernel(const TiledParams p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  constexpr int OP = C::OP;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave % C::WAVES_M, wn = wave / C::WAVES_M;
  const bool late = wave >= C::NWAVES / 2;  // the second wave of its SIMD
  const int N = p.N, K = p.K;
  const uint32_t row_bytes = (uint32_t)K * C::ESZ;
  const int num_tiles = p.header[0];
  const int nk = K / C::BK;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;

  using Tile = StreamTile;
  using Peek = TilePeek;
  auto peek_from = [&](int id0) { return peek_tile<C::OUT_BN>(p, num_tiles, id0, nk); };
  auto resolve = [&](Peek pk, Tile& t) { return resolve_tile<C::OUT_BN, C::THREADS>(p, num_tiles, pk, t, tid, nk); };

  // ---- the loading side of the stream ---------------------------------------------------------------------------
  // A stage arrives in four halves of two requests per wave (1 KB = 8 rows x 128 bytes each; the second half of a lower tile:
  // one request): activation rows 0 .. 127 and 128 .. of the tile, and the weight rows of channel tiles 0, 1 (g = 0) and 2, 3
  // (g = 1) of the four wave columns (with GLU: the first and the second projection).  The lane's 16 bytes: global chunk =
  // LDS slot ^ swizzle of the row.
  // (w: the wave as a scalar for LDS addresses, wave_v for lane offsets: a value the compiler shares between the two ends up in
  // a vector register, which the copy's scalar operand then cannot take)
  int wave_v = wave;
  asm volatile("" : "+v"(wave_v));
  auto a_req_row = [&](int i, int w) { return i < 2 ? w * 16 + i * 8 : 128 + w * 8 * C::NA1 + (i - 2) * 8; };
  auto b_req_row = [&](int i, int w) {
    return C::GLU ? (i / 2) * 128 + w * 16 + (i % 2) * 8 : (w / 2) * 64 + (i / 2) * 32 + (w % 2) * 16 + (i % 2) * 8;
  };
  auto lane_off = [&](int req_row, uint32_t row) {
    return row * row_bytes + (uint32_t)(((lane % 8) ^ C::swz(req_row + lane / 8)) << 4);
  };
  v4i a_desc, b_desc[C::GLU ? 2 : 1];
  uint32_t a_voff[C::A_IPW], b_voff[C::B_IPW], b_soff = 0;
  auto set_a_sources = [&](const Tile& t) {
    if (p.ro.row_idx) {
      a_desc = buffer_desc(p.lhs, clamp_u32((size_t)p.ro.lhs_rows * row_bytes));
      // (opaque: rows and chunks of the requests are made again for each tile; kept, they do not fit the registers of the
      // 256-row instances and come back from scratch memory, each behind the requests in flight)
      int lane_s = lane, wave_s = wave_v;
      asm volatile("" : "+v"(lane_s), "+v"(wave_s));
      int rows[C::A_IPW];
#pragma unroll
      for (int i = 0; i < C::A_IPW; i++) rows[i] = min(t.info.row0 + a_req_row(i, wave_s) + lane_s / 8, p.M - 1);
      lhs_rows_of<C::A_IPW>(p.ro, rows);
      // (rows past the tile's end: one row past the descriptor's, i.e. zeros without a request to memory)
#pragma unroll
      for (int i = 0; i < C::A_IPW; i++) {
        const int r = a_req_row(i, wave_s) + lane_s / 8;
        a_voff[i] = (uint32_t)(r < t.info.nrows ? rows[i] : p.ro.lhs_rows) * row_bytes + (uint32_t)(((lane_s % 8) ^ C::swz(r)) << 4);
      }
    } else {
      a_desc = buffer_desc(p.lhs + (size_t)t.info.row0 * row_bytes, clamp_u32((size_t)t.info.nrows * row_bytes));
    }
  };
  if (!p.ro.row_idx) {
#pragma unroll
    for (int i = 0; i < C::A_IPW; i++) a_voff[i] = lane_off(a_req_row(i, wave_v), (uint32_t)(a_req_row(i, wave_v) + lane / 8));
  }
#pragma unroll
  for (int i = 0; i < C::B_IPW; i++) {
    if constexpr (C::KN) {
      // request i covers KN_RPR contraction rows of the stage, the lane one 16-byte LDS slot of its row
      constexpr int LPR = kWave / C::KN_RPR;
      const int r = (wave_v * C::B_IPW + i) * C::KN_RPR + lane / LPR;
      b_voff[i] = (uint32_t)r * (uint32_t)(N * C::ESZ) + (uint32_t)(((lane % LPR) ^ C::kn_swz(r)) << 4);
    } else {
      b_voff[i] = lane_off(b_req_row(i, wave_v), (uint32_t)((C::GLU ? b_req_row(i, wave_v) % 128 : b_req_row(i, wave_v)) + lane / 8));
    }
  }
  auto set_b_sources = [&](const Tile& t) {
    b_desc[0] = buffer_desc(p.rhs + (size_t)t.info.group * N * row_bytes, clamp_u32((size_t)N * row_bytes));
    if constexpr (C::GLU) b_desc[1] = buffer_desc(p.rhs_up + (size_t)t.info.group * N * row_bytes, clamp_u32((size_t)N * row_bytes));
    b_soff = C::KN ? (uint32_t)t.n0 * C::ESZ : (uint32_t)t.n0 * row_bytes;  // (KN: a byte offset inside every contraction row)
  };
  auto issue_a = [&](int kt, int buf, int h) {
#pragma unroll
    for (int i = 2 * h; i < (h ? C::A_IPW : 2); i++)
      dma16_buffer(a_desc, a_voff[i], (uint32_t)kt * C::BKB, lds_base + buf * C::STAGE + a_req_row(i, wave) * C::BKB);
  };
  auto issue_b = [&](int kt, int buf, int g) {
#pragma unroll
    for (int i = 2 * g; i < 2 * g + 2; i++) {
      const uint32_t dst = lds_base + buf * C::STAGE + C::A_STAGE + (C::KN ? (wave * C::B_IPW + i) * 1024 : b_req_row(i, wave) * C::BKB);
      dma16_buffer(b_desc[C::GLU ? g : 0], b_voff[i], b_soff + (uint32_t)kt * C::BKB * (C::KN ? (uint32_t)N : 1u), dst);
    }
  };

  // ---- the multiplying side --------------------------------------------------------------------------------------
  using T_ = std::true_type;
  using F_ = std::false_type;
  constexpr int NT_OUT = C::GLU ? C::TN / 2 : C::TN;
  constexpr int HN = C::TN / 2;  // channel tiles of a quadrant
  auto row_tiles = [](int h) { return h ? C::H1 : 4; };
  // first LDS row of channel tile j
  const int b_base = C::A_STAGE + (C::GLU ? wn * (C::WN / 2) : wn * C::WN) * C::BKB;
  auto b_tile = [&](int j) { return (C::GLU ? (j / HN) * (C::BN / 2) + (j % HN) * C::MI : j * C::MI) * C::BKB; };
  // fragment of a 64-byte k-step ks: row (lane % 16), chunk q = 4 * ks + lane / 16, stored at slot q ^ swz(row)
  const int frag_lane = (lane % 16) * C::BKB + (((lane / 16) ^ C::swz(lane % 16)) << 4);
  // [G, K, N] weights.  fp8: lane (s, q) addresses row 16 q + s / 2 (+ 8, 64, 72) of the stage's 128 contraction rows, i.e. the
  // K bytes 16 q .. and 64 + 16 q .. its activation fragment holds, and the 8 bytes s % 2 of the fragment's 16-byte channel
  // block.  bf16: row 8 q + s / 4 (+ 4) of the k-step's 32 rows and the 8 bytes s % 4 of the fragment's 32-byte slice.  Channel
  // tile j is 16 * ESZ * j bytes further along the row before the swizzle: an XOR.
  const int kn_s = lane % 16, kn_q = lane / 16;
  const int kn_base = C::A_STAGE + (OP == OP_BF16
      ? (8 * kn_q + kn_s / 4) * C::KN_ROW + ((((8 * wn + (kn_s % 4) / 2) ^ C::kn_swz(8 * kn_q + kn_s / 4)) << 4) | ((kn_s & 1) << 3))
      : (16 * kn_q + kn_s / 2) * C::KN_ROW + (((wn * C::TN) ^ C::kn_swz(16 * kn_q + kn_s / 2)) << 4) + (kn_s % 2) * 8);

  typedef typename std::conditional<OP == OP_I8, v4i, v4f>::type acc_t;
  acc_t acc[C::TN][C::TM];
  // fragments: 8 registers per tile and stage, the two 64-byte k-steps of int8 / bf16 or the one 128-byte operand of fp8
  // (K bytes 16 q .. and 64 + 16 q ..: both operands alike, so the order of K inside the instruction does not matter)
  v8i fa[4], fb[2][HN];
  auto read_frag = [&](v8i& f, const uint8_t* src) {
    const v4i lo = *(const v4i*)(src + frag_lane), hi = *(const v4i*)(src + (frag_lane ^ 64));
    f[0] = lo[0]; f[1] = lo[1]; f[2] = lo[2]; f[3] = lo[3];
    f[4] = hi[0]; f[5] = hi[1]; f[6] = hi[2]; f[7] = hi[3];
  };
  auto read_a = [&](int buf, int h) {
#pragma unroll
    for (int i = 0; i < row_tiles(h); i++) read_frag(fa[i], smem + buf * C::STAGE + ((h * 4 + i) * 32 + wm * 16) * C::BKB);
  };
  auto read_b = [&](int buf, int g) {
#pragma unroll
    for (int jj = 0; jj < HN; jj++) {
      const int j = g * HN + jj;
      if constexpr (C::KN && OP == OP_BF16) {
        const uint8_t* src = smem + buf * C::STAGE + (kn_base ^ (j << 5));
        const v4i lo = __builtin_bit_cast(v4i, tr_read_frag(src, C::KN_ROW)), hi = __builtin_bit_cast(v4i, tr_read_frag(src + 32 * C::KN_ROW, C::KN_ROW));
        fb[g][jj] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      } else if constexpr (C::KN) {
        typedef int v2i_kn __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) v2i_kn* lds_v2i_kn;
        const uint8_t* src = smem + buf * C::STAGE + (kn_base ^ (j << 4));
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const v2i_kn x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_kn)(src + ((t & 1) * 8 + (t >> 1) * 64) * C::KN_ROW));
          fb[g][jj][2 * t] = x[0];
          fb[g][jj][2 * t + 1] = x[1];
        }
      } else {
        read_frag(fb[g][jj], smem + buf * C::STAGE + b_base + b_tile(j));
      }
    }
  };
  auto lo4 = [](const v8i& v) { return __builtin_shufflevector(v, v, 0, 1, 2, 3); };
  auto hi4 = [](const v8i& v) { return __builtin_shufflevector(v, v, 4, 5, 6, 7); };
  // One quadrant: row tiles 4h .. x channel tiles 2g, 2g + 1.  ZC: a tile's first stage starts from zero.
  auto quadrant = [&](auto zc_c, int h, int g) __attribute__((always_inline)) {
    constexpr bool ZC = decltype(zc_c)::value;
    if constexpr (OP == OP_F8) {
#pragma unroll
      for (int i = 0; i < row_tiles(h); i++)
#pragma unroll
        for (int jj = 0; jj < HN; jj++) {
          acc_t& c = acc[g * HN + jj][h * 4 + i];
          c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[g][jj], fa[i], ZC ? acc_t{} : c, 0, C::LF, 0, 127, 0, 127);
        }
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
#pragma unroll
        for (int i = 0; i < row_tiles(h); i++)
#pragma unroll
          for (int jj = 0; jj < HN; jj++) {
            acc_t& c = acc[g * HN + jj][h * 4 + i];
            const v4i b = ks ? hi4(fb[g][jj]) : lo4(fb[g][jj]), a = ks ? hi4(fa[i]) : lo4(fa[i]);
            if constexpr (OP == OP_I8) c = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, ZC && ks == 0 ? acc_t{} : c, 0, 0, 0);
            else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, b), __builtin_bit_cast(v8bf, a), ZC && ks == 0 ? acc_t{} : c, 0, 0, 0);
          }
    }
  };
  // The two sides of a phase.  fetch_end: this wave's fragment reads have landed and so have its requests up to the ones
  // that may still be outstanding (WAIT), then the hand-over barrier; after it the wave multiplies while the other wave of
  // its SIMD fetches.
  auto fetch_end = [&](auto wait_c) {
    constexpr int WAIT = decltype(wait_c)::value;
    if constexpr (WAIT >= 0) wait_vmcnt<WAIT>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
  };
  auto multiply_end = [&](int h, int g) {
    // (the sums are pinned here: at a tile's end their only readers sit behind branches, and the compiler otherwise moves
    // the products down there)
#pragma unroll
    for (int jj = 0; jj < HN; jj++)
#pragma unroll
      for (int i = 0; i < row_tiles(h); i++) asm volatile("" : "+v"(acc[g * HN + jj][h * 4 + i]));
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
  };
  using NOWAIT = std::integral_constant<int, -1>;
  // requests that may be outstanding where a phase ends ahead of new data: those behind the last half that the next phase reads
  using W1 = std::integral_constant<int, 6 + 2 * C::NA1>;                // ahead of phase 2 (weights, g = 1)
  using W2 = std::integral_constant<int, 8 + C::NA1>;                    // ahead of phase 3 (activations, h = 1)
  using W4 = std::integral_constant<int, (C::KN ? 6 : 8) + C::NA1>;      // ahead of phase 1 ([G, K, N]: both weight halves)

  Tile cur, nxt;
  if (!resolve(peek_from(blockIdx.x), cur)) return;
  // ---- head of the stream: the first tile's stage 0, and stage 1 up to the half that its first phase requests ----
  set_a_sources(cur);
  set_b_sources(cur);
  issue_a(cur.k0, 0, 0); issue_b(cur.k0, 0, 0); issue_b(cur.k0, 0, 1); issue_a(cur.k0, 0, 1);
  issue_a(cur.k0 + 1, 1, 0); issue_b(cur.k0 + 1, 1, 0); issue_b(cur.k0 + 1, 1, 1);
  wait_vmcnt<0>();
  asm volatile("s_barrier" ::: "memory");

  auto epilogue = [&]() __attribute__((always_inline)) {
    const int n_out0 = cur.n0 + (C::GLU ? wn * (C::WN / 2) : wn * C::WN);
    EpilogueScales<C::TM, NT_OUT, C::GLU> esc;
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    load_epilogue_scales<C::TM, NT_OUT, C::GLU, true, C::MI, 32>(esc, p, cur.info, wm * C::MI, n_out0, lane_e);
    // the next tile's stage 0 lands ahead of the stores, so that its phases need not count them (stage 1's three halves are
    // waited for in that stage's last phase, the stores with them)
    wait_vmcnt<6>();
    store_epilogue<C::TM, C::TN, NT_OUT, C::GLU, C::TM, 32>(acc, esc, p, cur.info, wm * C::MI, n_out0, lane_e);
  };
  int cb = 0;  // buffer of the current stage
  while (true) {
    // the record of the block's next tile is requested now and looked at two stages before this tile ends
    Peek pk = peek_from(cur.id + gridDim.x);
    bool have_n = false;
    auto stream_kt = [&](int s) { return s < cur.k1 ? s : have_n ? nxt.k0 + s - cur.k1 : cur.k1 - 1; };
    // Stage `it`, in four phases.  first: the stage's data landed before the tile began.  cross: the stream moves on to the next tile after the first phase.
    auto stage_head = [&](int it, auto first_c) __attribute__((always_inline)) {
      using WA = typename std::conditional<decltype(first_c)::value, NOWAIT, W1>::type;
      // 1: both first halves; requests the last half of the next stage (its slot was read two phases ago)
      read_b(cb, 0);
      read_a(cb, 0);
      issue_a(stream_kt(it + 1), cb ^ 1, 1);
      fetch_end(WA{});
      quadrant(first_c, 0, 0);
      multiply_end(0, 0);
    };
    auto stage_rest = [&](int it, auto first_c) __attribute__((always_inline)) {
      constexpr bool FIRST = decltype(first_c)::value;
      using WA = typename std::conditional<FIRST, NOWAIT, W2>::type;
      // 2
      const int kt2 = stream_kt(it + 2);
      read_b(cb, 1);
      issue_a(kt2, cb, 0);
      fetch_end(WA{});
      quadrant(first_c, 0, 1);
      multiply_end(0, 1);
      // 3
      read_a(cb, 1);
      issue_b(kt2, cb, 0);
      fetch_end(NOWAIT{});
      quadrant(first_c, 1, 1);
      multiply_end(1, 1);
      // 4
      issue_b(kt2, cb, 1);
      fetch_end(W4{});
      quadrant(first_c, 1, 0);
      multiply_end(1, 0);
      cb ^= 1;
    };
    if (late) asm volatile("s_barrier" ::: "memory");
    stage_head(cur.k0, T_{});
    stage_rest(cur.k0, T_{});
    for (int it = cur.k0 + 1; it < cur.k1 - 2; it++) {
      stage_head(it, F_{});
      stage_rest(it, F_{});
    }
    stage_head(cur.k1 - 2, F_{});
    have_n = resolve(pk, nxt);
    if (have_n) {
      set_a_sources(nxt);
      set_b_sources(nxt);
    }
    stage_rest(cur.k1 - 2, F_{});
    stage_head(cur.k1 - 1, F_{});
    stage_rest(cur.k1 - 1, F_{});
    if (!late) asm volatile("s_barrier" ::: "memory");
    if (cur.k1 - cur.k0 != nk) break;  // (a part of a tile is the last that a block has)
    epilogue();
    if (!have_n) break;
    cur = nxt;
  }
  if (cur.k1 - cur.k0 != nk && join_parts(acc, p, num_tiles, cur, nk, wave, tid)) epilogue();
  // nothing may still be writing LDS when the block ends
  __builtin_amdgcn_s_waitcnt(0xC07F);
  wait_vmcnt<0>();
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------

template <typename C>
static int prepare_dls_cfg() {
  return reserve_lds(gmm_dls_kernel<C>, C::LDS_BYTES, lds_flags<C>());
}

// Calls f with the configuration of a call: operand, GLU, e5m2 activations, [G, K, N] weights, row tiles.
template <typename F>
static int with_dls_cfg(int op, bool glu, int lhs_e5m2, int rhs_kn, int tm, F&& f) {
  auto rows = [&](auto tm_c) {
    constexpr int TM = decltype(tm_c)::value;
    if (op == OP_F8) {
      if (rhs_kn) return lhs_e5m2 ? f(DlsCfg<OP_F8, false, 1, true, TM>{}) : f(DlsCfg<OP_F8, false, 0, true, TM>{});
      if (lhs_e5m2) return f(DlsCfg<OP_F8, false, 1, false, TM>{});
      return glu ? f(DlsCfg<OP_F8, true, 0, false, TM>{}) : f(DlsCfg<OP_F8, false, 0, false, TM>{});
    }
    if (op == OP_I8) return glu ? f(DlsCfg<OP_I8, true, 0, false, TM>{}) : f(DlsCfg<OP_I8, false, 0, false, TM>{});
    if (rhs_kn) return f(DlsCfg<OP_BF16, false, 0, true, TM>{});
    return glu ? f(DlsCfg<OP_BF16, true, 0, false, TM>{}) : f(DlsCfg<OP_BF16, false, 0, false, TM>{});
  };
  return tm == 5 ? rows(std::integral_constant<int, 5>{}) : tm == 6 ? rows(std::integral_constant<int, 6>{}) : rows(std::integral_constant<int, 8>{});
}

int prepare_dls() {
  auto prep = [](auto cfg) { return prepare_dls_cfg<decltype(cfg)>(); };
  for (int tm : {5, 6, 8})
    for (int op : {OP_I8, OP_BF16, OP_F8})
      for (int v = 0; v < 5; v++) {  // plain, GLU, e5m2, [G, K, N], both
        const bool glu = v == 1, e5m2 = v == 2 || v == 4, kn = v >= 3;
        if ((e5m2 && op != OP_F8) || (kn && op == OP_I8)) continue;
        if (int st = with_dls_cfg(op, glu, e5m2, kn, tm, prep)) return st;
      }
  return MOE_OK;
}

template <typename C>
static int launch_dls_cfg(const TiledParams& p0, int M, int G_total, hipStream_t s) {
  if (int st = prepare_dls_cfg<C>()) return st;
  TiledParams p = p0;
  p.max_m_tiles = max_tiles_for(M, G_total, C::BM);
  p.tiles_n = cdiv(p.N, C::OUT_BN);
  const long long tiles = (long long)p.max_m_tiles * p.tiles_n;
  if (tiles > 0x7fffffffLL) return fail(MOE_ERR_UNSUPPORTED, "gmm: grid too large");
  if (p.tune <= 0) p.tune = default_super_row(M, G_total, C::BM);
  int blocks = 0;
  if (int st = stream_blocks(tiles, p, &blocks)) return st;
  gmm_dls_kernel<C><<<(unsigned)blocks, C::THREADS, C::LDS_BYTES, s>>>(p);
  return check_launch("gmm_dls_kernel");
}

bool dls_takes(int op, int K, int N, long long indexed_lhs_rows) {
  // whole 128-byte stages, at least three of them (the stream looks two stages ahead, into the next tile at most).  Byte
  // offsets are 32-bit: a weight request adds the lane's row (up to 255 rows past the last n-tile's first row, i.e. up to
  // N + 255 in all) times the row pitch to the descriptor's base, an activation request the lane's row of the 256-row
  // tile (or, with a row index, any of the indexed rows); each sum must stay below 2^32 so that a row past the end lands
  // beyond the descriptor's range and reads as zeros instead of wrapping around into it
  const long long esz = op == OP_BF16 ? 2 : 1, pitch = K * esz;
  return (op == OP_I8 || op == OP_BF16 || op == OP_F8) && pitch % 128 == 0 && pitch >= 384 && ((long long)N + 256) * pitch < (1LL << 32) &&
         (indexed_lhs_rows + 256) * pitch < (1LL << 32);
}

bool dls_kn_takes(int op, int K, int N, long long indexed_lhs_rows) {
  // [G, K, N] weights: whole 256-channel tiles, a contraction row's offset inside the expert's matrix in 32 bits
  return op != OP_I8 && dls_takes(op, K, N, indexed_lhs_rows) && N % 256 == 0 && ((long long)K + 128) * N * (op == OP_BF16 ? 2 : 1) < (1LL << 32);
}

int launch_dls(int op, bool glu, int bm, const TiledParams& p, int M, int G_total, hipStream_t s, int lhs_e5m2, int rhs_kn) {
  if (!dls_takes(op, p.K, p.N, p.ro.row_idx ? p.ro.lhs_rows : 0))
    return fail(MOE_ERR_UNSUPPORTED, "gmm: the stream kernel needs int8, bf16 or fp8 operands, whole 128-byte stages (three or more) and 32-bit byte offsets");
  if (lhs_e5m2 && (op != OP_F8 || glu)) return fail(MOE_ERR_UNSUPPORTED, "gmm: e5m2 activations run against e4m3 weights without rhs_up");
  if (rhs_kn && (glu || !dls_kn_takes(op, p.K, p.N, p.ro.row_idx ? p.ro.lhs_rows : 0)))
    return fail(MOE_ERR_UNSUPPORTED, "gmm: [G, K, N] weights on the stream kernel need bf16 or fp8 operands, no rhs_up, N %% 256 == 0 and 32-bit byte offsets");
  if (bm != 256 && bm != 192 && bm != 160) return fail(MOE_ERR_INVALID_ARG, "gmm: the stream kernel has no tiles of %d rows", bm);
  return with_dls_cfg(op, glu, lhs_e5m2, rhs_kn, bm / 32, [&](auto cfg) { return launch_dls_cfg<decltype(cfg)>(p, M, G_total, s); });
}

}  // namespace moe
