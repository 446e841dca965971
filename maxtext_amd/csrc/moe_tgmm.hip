// Transposed grouped matmul (weight gradient): out[g][n][k] = sum over the rows m of group g of
// dout[m][n] * lhs[m][k].  Both operands are row-major with the contraction index m as the ROW index, the
// opposite of what an MFMA fragment wants (8 consecutive contraction values per lane).  The tiles are staged
// in LDS as they are and read back with ds_read_b64_tr_b16, gfx950's transposing LDS load: within 16 lanes,
// lane L receives the L-th 16-bit column of a 4 x 16 block whose rows are addressed by lanes 0-3, 4-7, ...
// Two such reads give a lane its 8 contraction values.  lhs is the MFMA "A" operand (32 k channels), dout
// the "B" operand (32 n channels), so a lane ends up with 4 consecutive k of one n: contiguous stores into
// the [G, N, K] weight layout.

#include "moe_gmm_common.h"

namespace moe {

constexpr int kTgBN = 128, kTgBK = 128, kTgBM = 32;  // output tile [BN x BK], contraction chunk BM rows
constexpr int kTgThreads = 256;
constexpr int kTgLdr = kTgBN * 2 + 32;  // LDS row stride in bytes (the pad spreads the 4 rows of a transposing read over the banks)

struct TgmmParams {
  const uint16_t* lhs;   // [M, K] bf16
  const uint16_t* dout;  // [M, N] bf16
  const int32_t* group_sizes;
  void* out;  // [G_local, N, K] bf16 or f32
  const void* existing;  // NULL, or [G_local, N, K] values added to the products before the store (may be `out` itself)
  const float* n_scale;  // NULL, or [N]: the products of output row n are multiplied by n_scale[n] first
  int M, K, N;
  int G_total, G_local, group_offset;
  int out_f32, existing_f32;
};

// out[off .. off+3] = v * n_scale[n] + existing[off .. off+3]: four values along K of output row n.  A lane reads the
// four values it is about to overwrite, so `existing` may be the output buffer.
__device__ __forceinline__ void tgmm_store4(const TgmmParams& p, size_t off, int n, float v0, float v1, float v2, float v3) {
  if (p.n_scale) {
    const float sc = p.n_scale[n];
    v0 *= sc; v1 *= sc; v2 *= sc; v3 *= sc;
  }
  if (p.existing) {
    if (p.existing_f32) {
      const float4 e = *(const float4*)((const float*)p.existing + off);
      v0 += e.x; v1 += e.y; v2 += e.z; v3 += e.w;
    } else {
      const uint2 e = *(const uint2*)((const uint16_t*)p.existing + off);
      v0 += bf16_bits_to_f32(e.x & 0xffffu); v1 += bf16_bits_to_f32(e.x >> 16);
      v2 += bf16_bits_to_f32(e.y & 0xffffu); v3 += bf16_bits_to_f32(e.y >> 16);
    }
  }
  if (p.out_f32) *(float4*)((float*)p.out + off) = make_float4(v0, v1, v2, v3);
  else *(uint2*)((uint16_t*)p.out + off) = make_uint2(pack_bf16x2(v0, v1), pack_bf16x2(v2, v3));
}

__device__ __forceinline__ v8bf read_tr_frag(const uint8_t* tile, int row0, int col0, int lane) {
  // 8 contraction values (rows row0 + 8*(lane/32) .. +7) of column col0 + lane%32
  const int s = lane % 16, cg = (lane / 16) % 2, half = lane / 32;
  const uint8_t* p = tile + (row0 + half * 8 + s / 4) * kTgLdr + (col0 + cg * 16 + 4 * (s % 4)) * 2;
  const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)p);
  const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)(p + 4 * kTgLdr));
  typedef short v8s __attribute__((ext_vector_type(8)));
  const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(v8bf, v);
}

__global__ __launch_bounds__(kTgThreads) void tgmm_kernel(const TgmmParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[2][2][kTgBM * kTgLdr];  // [buffer][lhs|dout]
  __shared__ int s_red[kTgThreads / kWave];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int wk = wave % 2, wn = wave / 2;  // wave tile: 64 k x 64 n
  const int g_local = blockIdx.z, g = g_local + p.group_offset;
  const int n0 = blockIdx.y * kTgBN, k0 = blockIdx.x * kTgBK;
  const int N = p.N, K = p.K;

  // rows of group g: [start, start + size), clipped to M (sum of the sizes of the groups before it)
  long long part = 0;
  for (int i = tid; i < min(g, p.G_total); i += kTgThreads) part += max(p.group_sizes[i], 0);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
  if (lane == 0) s_red[wave] = (int)min(part, (long long)p.M);
  __syncthreads();
  long long start_ll = 0;
  for (int w = 0; w < kTgThreads / kWave; w++) start_ll += s_red[w];
  const int start = (int)min(start_ll, (long long)p.M);
  const int size = g < p.G_total ? min(max(p.group_sizes[g], 0), p.M - start) : 0;

  // staging: each tile is 32 rows x 256 bytes = 512 16-byte chunks, 2 per thread and operand
  int st_row[2], st_col[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int c = tid + i * kTgThreads;
    st_row[i] = c / 16;
    st_col[i] = (c % 16) * 8;  // element column within the tile
  }
  uint4 ra[2], rb[2];
  auto load_chunk = [&](int m0) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int r = m0 + st_row[i];
      const bool ok = r < size;
      const size_t row = (size_t)(start + (ok ? r : 0));
      const int kc = k0 + st_col[i], nc = n0 + st_col[i];
      uint4 a = make_uint4(0, 0, 0, 0), b = make_uint4(0, 0, 0, 0);
      if (ok && kc < K) a = *(const uint4*)(p.lhs + row * K + kc);
      if (ok && nc < N) b = *(const uint4*)(p.dout + row * N + nc);
      ra[i] = a;
      rb[i] = b;
    }
  };
  auto store_chunk = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      *(uint4*)(&smem[buf][0][st_row[i] * kTgLdr + st_col[i] * 2]) = ra[i];
      *(uint4*)(&smem[buf][1][st_row[i] * kTgLdr + st_col[i] * 2]) = rb[i];
    }
  };

  v16f acc[2][2];  // [n tile][k tile]
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[j][i][r] = 0.f;

  const int nchunks = (size + kTgBM - 1) / kTgBM;
  if (nchunks > 0) {
    load_chunk(0);
    store_chunk(0);
  }
  __syncthreads();
  for (int c = 0; c < nchunks; c++) {
    const int cur = c & 1;
    if (c + 1 < nchunks) load_chunk((c + 1) * kTgBM);
#pragma unroll
    for (int ks = 0; ks < kTgBM / 16; ks++) {
      v8bf fk[2], fn[2];
#pragma unroll
      for (int i = 0; i < 2; i++) fk[i] = read_tr_frag(smem[cur][0], ks * 16, wk * 64 + i * 32, lane);
#pragma unroll
      for (int j = 0; j < 2; j++) fn[j] = read_tr_frag(smem[cur][1], ks * 16, wn * 64 + j * 32, lane);
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fk[i], fn[j], acc[j][i], 0, 0, 0);
    }
    if (c + 1 < nchunks) store_chunk(cur ^ 1);
    __syncthreads();
  }

  // D[i = k][j = n]: lane holds n = lane % 32 and k = 8*q + 4*(lane/32) + r
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int n = n0 + wn * 64 + j * 32 + (lane % 32);
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int k = k0 + wk * 64 + i * 32 + 8 * q + 4 * (lane / 32);
        if (k >= K) continue;
        const size_t off = ((size_t)g_local * N + n) * K + k;
        tgmm_store4(p, off, n, acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
      }
  }
}


// ---------------------------------------------------------------------------------------
// 256 (n) x 256 (k) output tiles for groups of many rows, bf16 (v_mfma_f32_16x16x32_bf16) or 1-byte operands as stored (the
// drhs product of the fp8_full backward, kernels/megablox/ops.py:590-604: float8_e4m3fn activations x float8_e5m2 gradient,
// v_mfma_scale_f32_16x16x128_f8f6f4).  A stage is 64 (1-byte: 128) contraction rows of both operands as they lie in memory,
// 32 KB each, copied by buffer_load ... lds (a wave instruction moves 2 rows of 512 or 4 of 256 bytes: whole 128-byte
// lines) into two buffers of 64 KB.  The descriptor of a stage ends at the group's last row: rows past it arrive as zeros.
// 8 waves of 64 (k) x 128 (n).  Fragments come out of the row-major stage through ds_read_b64_tr_b16 / _b8.
//
// Schedule: the two waves of a SIMD take turns, as in the grouped matmul of prefill.  A stage is four phases of 256
// matrix cycles; a phase is a fetching side (fragment reads, two requests, waits), a barrier, a multiplying side and a
// barrier, and waves 4 .. 7 run one barrier behind waves 0 .. 3.  Phases of bf16: the two k-steps of 32 rows x the two halves
// of the dout fragments, so a stage frees its slots by halves of 32 rows; of the 1-byte operands (one instruction spans
// the stage): pairs of dout fragments, the pair of the third phase read a phase early so that the dout slots are free for
// the whole fourth.  A request has five (1-byte: three) phases to land.
// Persistent blocks, one request stream across tiles: a tile's first two stages arrive behind the previous tile's products,
// and its stores drain behind the next tile's.  Mixtral shape, same box: 16384 rows, bf16 1.68 -> 1.55 / 1.71 -> 1.61 ms (one
// mixed stream per wave, one barrier per stage and a block per tile before; the schedule alone 1 %, the stream across tiles
// 6 %); 1-byte at 6000 rows 0.51 -> 0.47 / 0.53 -> 0.50 ms (six stages a tile: there the descriptors as running scalars gave
// most).  Reading the fragments between the products instead of ahead of them is slower (1.52 -> 1.60).  What bounds bf16 now:
// with the same stage over and over (no misses in L2) 1.40 ms, i.e. 10 % is the latency of the real stream (440 cycles at
// 67 lines in flight per CU, against 330 for the products of the forward pass), the rest the matrix units under the power
// limit and twice as many fragment reads as a row-major operand takes.
//
// bf16 swizzle: the 16-byte chunk q of row r is stored at slot q ^ f(r), f(r) = 4 * (r % 4) ^ 2 * ((r / 8) % 2): the 4 rows x
// 32 bytes that 16 lanes of a transposing read address, and those of the next 16 lanes (8 rows further), then fall into 8
// different 32-byte bank groups.  1-byte: 16 lanes address an 8-row x 16-byte block (lane l: row l / 2, half l % 2) and lane l
// receives column l of the 8 rows; four such reads give the 32 contraction values of a 16 x 16 x 128 fragment.  Lane group q
// takes stage rows 32 q .. 32 q + 31 for BOTH operands (any order of the contraction index does, as long as the fragments
// agree); chunk c of row r sits at slot c ^ (r % 8) ^ 8 * ((r / 32) % 2): the 8 rows of a read and those of the next lane
// group fall into 16 different 16-byte bank groups.
// ---------------------------------------------------------------------------------------

constexpr int kTdTile = 256;                   // output tile edge
constexpr int kTdThreads = 512, kTdWaves = 8;

template <bool F8_, int DF_ = 0>
struct TgCfg {
  static constexpr bool F8 = F8_;
  static constexpr int DF = DF_;               // element format of a 1-byte dout: 0 = e4m3, 1 = e5m2 (lhs is e4m3)
  static constexpr int ESZ = F8 ? 1 : 2;
  static constexpr int BM = F8 ? 128 : 64;     // contraction rows per stage
  static constexpr int ROW = kTdTile * ESZ;    // bytes of one operand row in a stage
  static constexpr int OPERAND = BM * ROW;     // 32 KB
  static constexpr int STAGE = 2 * OPERAND;    // lhs rows | dout rows
  static constexpr int LDS = 2 * STAGE;
  static constexpr int RPR = 1024 / ROW;       // rows per request
  static constexpr int IPW = OPERAND / 1024 / kTdWaves;  // requests per wave, operand and stage
  static_assert(OPERAND == 32768 && IPW == 4, "stage shape");
  __device__ static __forceinline__ int swz(int row) { return F8 ? (row & 7) ^ (((row >> 5) & 1) << 3) : tr_swz(row); }
};

typedef int v2i_t8 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i_t8* lds_v2i_t8;
__device__ __forceinline__ void tr8_read_frag(v8i& f, const uint8_t* p, int row_bytes) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const v2i_t8 x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t8)(p + t * 8 * row_bytes));
    f[2 * t] = x[0];
    f[2 * t + 1] = x[1];
  }
}

template <typename C>
__global__ __launch_bounds__(kTdThreads, 2) void tgmm_dl_kernel(const TgmmParams p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t td_smem[];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wk = wave % 4, wn = wave / 4;  // wave tile: 64 k x 128 n
  const bool late = wave >= kTdWaves / 2;  // the second wave of its SIMD
  const int N = p.N, K = p.K;

  // Persistent blocks: block b works on tile ids b, b + gridDim.x, ..  Ids congruent mod 8 run on one XCD: each XCD owns a
  // contiguous range of tiles, walked in patches of 8 n-tiles x 4 k-tiles of one group, so that the 32 blocks of an XCD
  // share 8 dout and 4 lhs panels in its L2.
  const int tiles_k = K / kTdTile, tiles_n = N / kTdTile, per_group = tiles_k * tiles_n;
  const int total = per_group * p.G_local;
  struct Tile {
    int g_local, n0, k0, start, size, nk;
  };
  // rows of group g: [start, start + size), clipped to M.  A block's tiles come in the order of their groups, so a new start is
  // the old one plus the sizes of the groups in between.
  typedef const __attribute__((address_space(4))) int32_t* const_i32_t;
  const const_i32_t sizes = (const_i32_t)(uintptr_t)p.group_sizes;
  int g_at = 0;          // group that `row_at` is the first row of (clipped to M)
  long long row_at = 0;
  auto locate = [&](int id, Tile& t) __attribute__((always_inline)) {
    const int q8 = total / 8, rem = total % 8, xcd = id % 8, loc = id / 8;
    const int logical = xcd < rem ? xcd * (q8 + 1) + loc : rem * (q8 + 1) + (xcd - rem) * q8 + loc;
    const int r = logical % per_group;
    constexpr int GSM = 8;
    const int width = GSM * tiles_k, first_n = (r / width) * GSM, gsz = min(tiles_n - first_n, GSM);
    t.g_local = logical / per_group;
    t.n0 = (first_n + (r % width) % gsz) * kTdTile;
    t.k0 = ((r % width) / gsz) * kTdTile;
    const int g = t.g_local + p.group_offset;
    for (; g_at < min(g, p.G_total); g_at++) row_at += max(sizes[g_at], 0);
    t.start = (int)min(row_at, (long long)p.M);
    t.size = g < p.G_total ? min(max(sizes[g], 0), p.M - t.start) : 0;
    // (three stages at least: the stream looks two stages ahead, into the next tile at most; a stage past the rows is zeros)
    t.nk = max((t.size + C::BM - 1) / C::BM, 3);
  };
  if (p.group_offset > 0) {  // the groups before the local ones, summed once by every wave
    long long part = 0;
    const int gl = min(p.group_offset, p.G_total);
    for (int i = lane; i < gl; i += kWave) part += max(p.group_sizes[i], 0);
    int lim = (int)min(part, (long long)p.M);  // (a sum past M is as good as M)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lim = min((int)min((long long)lim + __shfl_xor(lim, o), (long long)p.M), p.M);
    row_at = __builtin_amdgcn_readfirstlane(lim);
    g_at = gl;
  }
  const int s16 = lane % 16, gq = lane / 16;
  // the block's first tile from `id` on whose group has rows; the gradients of empty groups are zeros, written on the way
  auto next_tile = [&](int& id, Tile& t) __attribute__((always_inline)) -> bool {
    for (; id < total; id += gridDim.x) {
      locate(id, t);
      if (t.size > 0) return true;
      for (int i = tid; i < kTdTile * (kTdTile / 4); i += kTdThreads) {
        const int n = t.n0 + i / (kTdTile / 4);
        tgmm_store4(p, ((size_t)t.g_local * N + n) * K + t.k0 + (i % (kTdTile / 4)) * 4, n, 0.f, 0.f, 0.f, 0.f);
      }
    }
    return false;
  };

  // ---- requests.  Request i of an operand and wave: half i / 2 of the stage (bf16: 32 rows each), RPR rows of it.
  auto req_row = [&](int i) { return (i / 2) * (C::BM / 2) + (wave * 2 + i % 2) * C::RPR; };
  uint32_t a_off[C::IPW], b_off[C::IPW];
  const uint32_t a_pitch = (uint32_t)K * C::ESZ, b_pitch = (uint32_t)N * C::ESZ;
#pragma unroll
  for (int i = 0; i < C::IPW; i++) {
    constexpr int LPR = kWave / C::RPR;  // lanes per row
    const int r = req_row(i) + lane / LPR;
    const uint32_t chunk = (uint32_t)((lane % LPR) ^ C::swz(r)) * 16;
    a_off[i] = (uint32_t)r * a_pitch + chunk;
    b_off[i] = (uint32_t)r * b_pitch + chunk;
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)td_smem;
  // The loading side: the next stage's first byte of the two panels, and the descriptors of the stage being requested.  A
  // descriptor starts at the stage's first row and ends with the group's last one, so rows past it arrive as zeros; a stage
  // past the end has no bytes at all and fetches nothing.  (Kept as running scalars: formed from the stage number for every
  // request they were 18 scalar instructions in the fetching side, as long as its fragment reads.)
  uint64_t a_next = 0, b_next = 0;
  int a_kt = 0, b_kt = 0, src_full = 0;   // stage numbers; full stages
  uint32_t a_part = 0, b_part = 0;        // bytes of the stage behind them
  v4i a_desc, b_desc;
  auto set_sources = [&](const Tile& t) __attribute__((always_inline)) {
    a_next = (uint64_t)p.lhs + (uint64_t)t.start * a_pitch + (uint64_t)t.k0 * C::ESZ;
    b_next = (uint64_t)p.dout + (uint64_t)t.start * b_pitch + (uint64_t)t.n0 * C::ESZ;
    a_kt = b_kt = 0;
    src_full = t.size / C::BM;
    const int part = t.size % C::BM;
    a_part = part > 0 ? (uint32_t)(part - 1) * a_pitch + C::ROW : 0u;
    b_part = part > 0 ? (uint32_t)(part - 1) * b_pitch + C::ROW : 0u;
  };
  const uint32_t a_full = (uint32_t)(C::BM - 1) * a_pitch + C::ROW, b_full = (uint32_t)(C::BM - 1) * b_pitch + C::ROW;
  auto advance = [&](bool is_a) __attribute__((always_inline)) {
    if (is_a) {
      a_desc = buffer_desc((const void*)a_next, a_kt < src_full ? a_full : a_kt == src_full ? a_part : 0u);
      a_next += (uint64_t)C::BM * a_pitch;
      a_kt++;
    } else {
      b_desc = buffer_desc((const void*)b_next, b_kt < src_full ? b_full : b_kt == src_full ? b_part : 0u);
      b_next += (uint64_t)C::BM * b_pitch;
      b_kt++;
    }
  };
  // half h of an operand of the stage its descriptor stands at
  auto issue = [&](bool is_a, int buf, int h) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 2 * h; i < 2 * h + 2; i++)
      dma16_buffer(is_a ? a_desc : b_desc, is_a ? a_off[i] : b_off[i], lds_base + buf * C::STAGE + (is_a ? 0 : C::OPERAND) + req_row(i) * C::ROW);
  };

  // ---- fragments.  bf16: lane (group gq, s16) addresses row 8 * gq + s16 / 4 (+ 4) of the k-step's 32 rows and the 8 bytes
  // 8 * (s16 % 4) of the fragment's 32-byte row slice; fragment f of an operand is 32 * f bytes further along the row before
  // the swizzle, which turns the step into an XOR of address bits 5 .. 7.  1-byte: row 32 * gq + s16 / 2 (+ 8, 16, 24) and the
  // 8 bytes s16 % 2 of the fragment's 16-byte column block; the step is an XOR of address bits 4 .. 6.
  int k_base, n_base;
  if constexpr (C::F8) {
    const int xmask = (s16 / 2) ^ ((gq & 1) << 3), row_part = (32 * gq + s16 / 2) * C::ROW + (s16 % 2) * 8;
    k_base = row_part + (((4 * wk) ^ xmask) << 4);
    n_base = row_part + (((8 * wn) ^ xmask) << 4);
  } else {
    const int xmask = ((s16 / 4) << 2) ^ ((gq & 1) << 1), piece = s16 % 4, row_part = (gq * 8 + s16 / 4) * C::ROW;
    k_base = row_part + ((((8 * wk + piece / 2) ^ xmask) << 4) | ((piece & 1) << 3));
    n_base = row_part + ((((16 * wn + piece / 2) ^ xmask) << 4) | ((piece & 1) << 3));
  }
  typedef typename std::conditional<C::F8, v8i, v8bf>::type frag_t;
  constexpr int NSLOTS = C::F8 ? 6 : 4;
  frag_t fk[4], fn[NSLOTS];
  auto read_k = [&](int buf, int ks, int f) {
    const uint8_t* src = td_smem + buf * C::STAGE + (k_base ^ ((C::F8 ? 16 : 32) * f));
    if constexpr (C::F8) tr8_read_frag(fk[f], src, C::ROW);
    else fk[f] = tr_read_frag(src + ks * 32 * C::ROW, C::ROW);
  };
  auto read_n = [&](int buf, int ks, int f, int slot) {
    const uint8_t* src = td_smem + buf * C::STAGE + C::OPERAND + (n_base ^ ((C::F8 ? 16 : 32) * f));
    if constexpr (C::F8) tr8_read_frag(fn[slot], src, C::ROW);
    else fn[slot] = tr_read_frag(src + ks * 32 * C::ROW, C::ROW);
  };
  v4f acc[4][8];  // [k fragment][n fragment]
  // n fragments f0 .. of one phase (4 of bf16, 2 of the 1-byte operands) from the slots slot0 ..
  auto multiply = [&](auto zc_c, int f0, int slot0) __attribute__((always_inline)) {
    constexpr bool ZC = decltype(zc_c)::value;  // a tile's first products start from zero
#pragma unroll
    for (int i = 0; i < (C::F8 ? 2 : 4); i++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v4f& c = acc[j][f0 + i];
        if constexpr (C::F8) c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fk[j], fn[slot0 + i], ZC ? v4f{} : c, 0, C::DF, 0, 127, 0, 127);
        else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fk[j], fn[slot0 + i], ZC ? v4f{} : c, 0, 0, 0);
      }
    // (pinned to the phase: at the end the sums' only readers sit behind branches)
#pragma unroll
    for (int i = 0; i < (C::F8 ? 2 : 4); i++)
#pragma unroll
      for (int j = 0; j < 4; j++) asm volatile("" : "+v"(acc[j][f0 + i]));
  };
  auto fetch_end = [&](auto wait_c) {
    constexpr int WAIT = decltype(wait_c)::value;
    if constexpr (WAIT >= 0) wait_vmcnt<WAIT>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
  };
  auto multiply_end = [&]() {
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  using NOWAIT = std::integral_constant<int, -1>;
  using WAIT = std::integral_constant<int, C::F8 ? 6 : 10>;

  // D[k][n]: the lane holds n = s16 and k = 4 * gq + r of each 16 x 16 tile
  auto store_tile = [&](const Tile& t) __attribute__((always_inline)) {
    float sc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) sc[i] = p.n_scale ? p.n_scale[t.n0 + wn * 128 + i * 16 + s16] : 1.0f;
    // the next tile's stage 0 lands ahead of the stores, so that its phases need not count them (stage 1's three halves are
    // waited for in that stage's last phase, the stores with them)
    wait_vmcnt<6>();
    if (!p.out_f32 && !p.existing) {
      // plain bf16 results: neighbouring k-tiles trade halves between lanes 16 apart, so that a lane stores 16 bytes and
      // the 64 bytes of a row n leave in one instruction
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int n = t.n0 + wn * 128 + i * 16 + s16;
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(acc[j][i][0] * sc[i], acc[j][i][1] * sc[i]),
                                                           pack_bf16x2(acc[j + 1][i][0] * sc[i], acc[j + 1][i][1] * sc[i]), false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(acc[j][i][2] * sc[i], acc[j][i][3] * sc[i]),
                                                           pack_bf16x2(acc[j + 1][i][2] * sc[i], acc[j + 1][i][3] * sc[i]), false, false);
          const int k = t.k0 + wk * 64 + (j + (gq & 1)) * 16 + 4 * (gq & ~1);
          *(uint4*)((uint16_t*)p.out + ((size_t)t.g_local * N + n) * K + k) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int n = t.n0 + wn * 128 + i * 16 + s16;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const size_t off = ((size_t)t.g_local * N + n) * K + t.k0 + wk * 64 + j * 16 + 4 * gq;
        tgmm_store4(p, off, n, acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]);
      }
    }
  };

  Tile cur, nxt;
  int id = blockIdx.x;
  if (!next_tile(id, cur)) return;
  // ---- head: stage 0, and stage 1 up to the half that the first phase requests ----
  set_sources(cur);
  advance(true); advance(false);
  issue(true, 0, 0); issue(false, 0, 0); issue(true, 0, 1); issue(false, 0, 1);
  advance(true); advance(false);
  issue(true, 1, 0); issue(false, 1, 0);
  issue(true, 1, 1);
  wait_vmcnt<0>();
  asm volatile("s_barrier" ::: "memory");

  int cb = 0;  // buffer of the current stage
  while (true) {
    bool have_n = false;
    const int nk = cur.nk;
    // the first phase of stage kt: it requests the last half of the next stage; the rest requests stage kt + 2.
    // FIRST: what these phases start with landed before the tile began (no waits)
    auto stage_head = [&](auto first_c) __attribute__((always_inline)) {
#pragma unroll
      for (int f = 0; f < 4; f++) read_k(cb, 0, f);
#pragma unroll
      for (int f = 0; f < (C::F8 ? 2 : 4); f++) read_n(cb, 0, f, f);
      issue(false, cb ^ 1, 1);
      fetch_end(NOWAIT{});
      multiply(first_c, 0, 0);
      multiply_end();
    };
    auto stage_rest = [&](auto first_c) __attribute__((always_inline)) {
      using W = typename std::conditional<decltype(first_c)::value, NOWAIT, WAIT>::type;
      if constexpr (C::F8) {
        // lhs slots are free behind phase 1 (requested in 2 and 3), dout slots behind phase 3 (4 and the next stage's 1)
#pragma unroll
        for (int f = 2; f < 6; f++) read_n(cb, 0, f, f);
        advance(true);
        issue(true, cb, 0);
        fetch_end(NOWAIT{});
        multiply(first_c, 2, 2);
        multiply_end();
        read_n(cb, 0, 6, 0);
        read_n(cb, 0, 7, 1);
        issue(true, cb, 1);
        fetch_end(NOWAIT{});
        multiply(first_c, 4, 4);
        multiply_end();
        advance(false);
        issue(false, cb, 0);
        fetch_end(WAIT{});  // (the next stage's last half is this stage's first request: waited for in every stage)
        multiply(first_c, 6, 0);
        multiply_end();
      } else {
#pragma unroll
        for (int f = 0; f < 4; f++) read_n(cb, 0, 4 + f, f);
        advance(true);
        issue(true, cb, 0);
        fetch_end(W{});
        multiply(first_c, 4, 0);
        multiply_end();
#pragma unroll
        for (int f = 0; f < 4; f++) read_k(cb, 1, f);
#pragma unroll
        for (int f = 0; f < 4; f++) read_n(cb, 1, f, f);
        advance(false);
        issue(false, cb, 0);
        fetch_end(NOWAIT{});
        multiply(F_{}, 0, 0);
        multiply_end();
#pragma unroll
        for (int f = 0; f < 4; f++) read_n(cb, 1, 4 + f, f);
        issue(true, cb, 1);
        fetch_end(WAIT{});
        multiply(F_{}, 4, 0);
        multiply_end();
      }
      cb ^= 1;
    };
    if (late) asm volatile("s_barrier" ::: "memory");
    stage_head(T_{});
    stage_rest(T_{});
    for (int kt = 1; kt < nk - 2; kt++) {
      stage_head(F_{});
      stage_rest(F_{});
    }
    stage_head(F_{});
    // the stream crosses into the next tile
    id += gridDim.x;
    have_n = next_tile(id, nxt);
    if (have_n) set_sources(nxt);
    stage_rest(F_{});
    stage_head(F_{});
    stage_rest(F_{});
    if (!late) asm volatile("s_barrier" ::: "memory");
    store_tile(cur);
    if (!have_n) break;
    cur = nxt;
  }
  wait_vmcnt<0>();  // no request may still be writing LDS when the block ends
}

}  // namespace moe

using namespace moe;

namespace moe {
template <typename C>
static int launch_tgmm_dl(const TgmmParams& p, hipStream_t s) {
  if (int st = reserve_lds(tgmm_dl_kernel<C>, C::LDS, lds_flags<C>())) return st;
  // one persistent block per CU (the LDS footprint allows no more); a multiple of 8 keeps "tile id mod 8" equal to the XCD
  // a block runs on
  int blocks = 0;
  if (int st = device_cu_count(&blocks)) return st;
  const long long tiles = (long long)(p.K / kTdTile) * (p.N / kTdTile) * p.G_local;
  if (tiles < blocks) blocks = (int)tiles;
  if (blocks >= 8) blocks -= blocks % 8;
  tgmm_dl_kernel<C><<<(unsigned)blocks, kTdThreads, C::LDS, s>>>(p);
  return check_launch("tgmm_dl_kernel");
}
int prepare_tgmm() {
  int st = reserve_lds(tgmm_dl_kernel<TgCfg<false>>, TgCfg<false>::LDS, lds_flags<TgCfg<false>>());
  if (!st) st = reserve_lds(tgmm_dl_kernel<TgCfg<true, 0>>, TgCfg<true, 0>::LDS, lds_flags<TgCfg<true, 0>>());
  if (!st) st = reserve_lds(tgmm_dl_kernel<TgCfg<true, 1>>, TgCfg<true, 1>::LDS, lds_flags<TgCfg<true, 1>>());
  return st;
}
}  // namespace moe

static bool tgmm_f8_takes(long long M, int K, int N, int G_total, int G_local) {
  const long long tiles = (long long)(K / kTdTile) * (N / kTdTile) * G_local;
  return K % kTdTile == 0 && N % kTdTile == 0 && K < (1 << 24) && N < (1 << 24) && M >= 128LL * G_total && tiles >= 128 && tiles <= 0x7fffffffLL;
}

extern "C" int moe_tgmm_fp8_supported(int M, int K, int N, int num_groups_total, int num_groups_local) {
  return M >= 0 && K > 0 && N > 0 && num_groups_total > 0 && num_groups_local > 0 && tgmm_f8_takes(M, K, N, num_groups_total, num_groups_local);
}

extern "C" int moe_tgmm_fp8(const void* lhs, const void* dout, int dout_dtype, const int32_t* group_sizes, int M, int K, int N,
                            int num_groups_total, int num_groups_local, int group_offset, const float* out_row_scale,
                            const void* existing_out, int existing_dtype, int out_dtype, void* out, void* stream) {
  if (!lhs || !dout || !group_sizes || !out) return fail(MOE_ERR_INVALID_ARG, "tgmm_fp8: NULL pointer");
  if (M < 0 || K <= 0 || N <= 0 || num_groups_total <= 0 || num_groups_local <= 0 || group_offset < 0)
    return fail(MOE_ERR_INVALID_ARG, "tgmm_fp8: bad sizes");
  if (dout_dtype != MOE_FP8_E4M3 && dout_dtype != MOE_FP8_E5M2) return fail(MOE_ERR_UNSUPPORTED, "tgmm_fp8: dout_dtype %d", dout_dtype);
  if (out_dtype != MOE_BF16 && out_dtype != MOE_F32) return fail(MOE_ERR_UNSUPPORTED, "tgmm_fp8: out_dtype %d", out_dtype);
  if (!tgmm_f8_takes(M, K, N, num_groups_total, num_groups_local))
    return fail(MOE_ERR_UNSUPPORTED, "tgmm_fp8: needs K and N multiples of 256, 128 rows per group on average and 128 output tiles "
                "(M=%d K=%d N=%d groups=%d); widen the operands to bf16 for moe_tgmm_scaled otherwise", M, K, N, num_groups_total);
  if (((uintptr_t)lhs | (uintptr_t)dout | (uintptr_t)out | (uintptr_t)existing_out) & 15) return fail(MOE_ERR_UNSUPPORTED, "tgmm_fp8: pointers must be 16-byte aligned");
  if (existing_out && existing_dtype != MOE_BF16 && existing_dtype != MOE_F32) return fail(MOE_ERR_UNSUPPORTED, "tgmm_fp8: existing_dtype %d", existing_dtype);
  if (existing_out == out && existing_dtype != out_dtype) return fail(MOE_ERR_INVALID_ARG, "tgmm_fp8: existing_out aliases out with another element type");
  TgmmParams p;
  p.lhs = (const uint16_t*)lhs; p.dout = (const uint16_t*)dout; p.group_sizes = group_sizes; p.out = out;
  p.M = M; p.K = K; p.N = N; p.G_total = num_groups_total; p.G_local = num_groups_local; p.group_offset = group_offset;
  p.out_f32 = out_dtype == MOE_F32;
  p.existing = existing_out; p.existing_f32 = existing_dtype == MOE_F32;
  p.n_scale = out_row_scale;
  return dout_dtype == MOE_FP8_E5M2 ? launch_tgmm_dl<TgCfg<true, 1>>(p, (hipStream_t)stream) : launch_tgmm_dl<TgCfg<true, 0>>(p, (hipStream_t)stream);
}

extern "C" int moe_tgmm_scaled(const void* lhs, const void* dout, const int32_t* group_sizes, int M, int K, int N,
                               int num_groups_total, int num_groups_local, int group_offset, const float* out_row_scale,
                               const void* existing_out, int existing_dtype, int out_dtype, void* out, void* stream) {
  if (!lhs || !dout || !group_sizes || !out) return fail(MOE_ERR_INVALID_ARG, "tgmm: NULL pointer");
  if (M < 0 || K <= 0 || N <= 0 || num_groups_total <= 0 || num_groups_local <= 0 || group_offset < 0)
    return fail(MOE_ERR_INVALID_ARG, "tgmm: bad sizes");
  if (K % 8 || N % 8) return fail(MOE_ERR_UNSUPPORTED, "tgmm: K and N must be multiples of 8");
  if (out_dtype != MOE_BF16 && out_dtype != MOE_F32) return fail(MOE_ERR_UNSUPPORTED, "tgmm: out_dtype %d", out_dtype);
  if (num_groups_local > 65535 || cdiv(N, kTgBN) > 65535) return fail(MOE_ERR_UNSUPPORTED, "tgmm: grid too large");
  if (((uintptr_t)lhs | (uintptr_t)dout | (uintptr_t)out) & 15) return fail(MOE_ERR_UNSUPPORTED, "tgmm: pointers must be 16-byte aligned");
  TgmmParams p;
  p.lhs = (const uint16_t*)lhs; p.dout = (const uint16_t*)dout; p.group_sizes = group_sizes; p.out = out;
  p.M = M; p.K = K; p.N = N; p.G_total = num_groups_total; p.G_local = num_groups_local; p.group_offset = group_offset;
  p.out_f32 = out_dtype == MOE_F32;
  if (existing_out && existing_dtype != MOE_BF16 && existing_dtype != MOE_F32)
    return fail(MOE_ERR_UNSUPPORTED, "tgmm: existing_dtype %d", existing_dtype);
  if ((uintptr_t)existing_out & 15) return fail(MOE_ERR_UNSUPPORTED, "tgmm: pointers must be 16-byte aligned");
  if (existing_out == out && existing_dtype != out_dtype)
    return fail(MOE_ERR_INVALID_ARG, "tgmm: existing_out aliases out with another element type");
  p.existing = existing_out; p.existing_f32 = existing_dtype == MOE_F32;
  p.n_scale = out_row_scale;
  // groups of 128 rows and more on average take the 256 x 256 tiles when the shape allows it
  const long long tiles = (long long)(K / kTdTile) * (N / kTdTile) * num_groups_local;
  if (K % kTdTile == 0 && N % kTdTile == 0 && K < (1 << 24) && N < (1 << 24) && (long long)M >= 128LL * num_groups_total && tiles >= 128 && tiles <= 0x7fffffffLL)
    return launch_tgmm_dl<TgCfg<false>>(p, (hipStream_t)stream);
  dim3 grid(cdiv(K, kTgBK), cdiv(N, kTgBN), num_groups_local);
  tgmm_kernel<<<grid, kTgThreads, 0, (hipStream_t)stream>>>(p);
  return check_launch("tgmm_kernel");
}

extern "C" int moe_tgmm(const void* lhs, const void* dout, const int32_t* group_sizes, int M, int K, int N,
                        int num_groups_total, int num_groups_local, int group_offset, const void* existing_out,
                        int existing_dtype, int out_dtype, void* out, void* stream) {
  return moe_tgmm_scaled(lhs, dout, group_sizes, M, K, N, num_groups_total, num_groups_local, group_offset, nullptr, existing_out,
                         existing_dtype, out_dtype, out, stream);
}
