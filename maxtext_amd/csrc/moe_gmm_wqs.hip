// Grouped matmul, decode sizes: bf16 activations x group-128 int4 weights with the weights streamed through LDS.

#include "moe_gmm_wqs.h"
#include "moe_gmm_wqs_run.h"

namespace moe {

template <int FMT, int NSEG, bool GLU>
__global__ __launch_bounds__(kWqsThreads) void gmm_wqs_kernel(const WqSkinnyParams p, int num_groups) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  wqs_run<FMT, NSEG, GLU, 16>(p, num_groups, smem);
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------

// group-128 int4 or MXFP4 with K up to 3072, at least four channel groups per tile (a copy issued three positions ahead
// then never looks past the next tile), scale rows that start on 16-byte boundaries and tensors within 32-bit offsets
bool wqs_takes(int fmt, int K, int N, int G_local, bool glu) {
  const int nkb = (K + 127) / 128;
  const int ncg = cdiv(N, glu ? 32 : 64);
  if (fmt != WQ_I4 && fmt != WQ_MX4) return false;
  const long long srow = fmt == WQ_MX4 ? K / 32 : nkb * 2;
  return K % 32 == 0 && nkb <= kWqsMaxKBlocks && N % 8 == 0 && ncg >= 4 && ((long long)N * srow) % 16 == 0 && (32 * srow) % 16 == 0 &&
         (long long)G_local * N * (K / 2) + 65LL * (K / 2) + 1024 < (1LL << 32);  // (an item's last rows may lie up to 63 rows past N)
}

template <int FMT, int NSEG, bool GLU>
static int launch_wqs_one(const WqSkinnyParams& p, int num_groups, int blocks, hipStream_t s) {
  if (int st = reserve_lds(gmm_wqs_kernel<FMT, NSEG, GLU>, kWqsLds, lds_flags<std::integral_constant<int, 7000 + FMT * 100 + NSEG * 2 + (GLU ? 1 : 0)>>()))
    return st;
  gmm_wqs_kernel<FMT, NSEG, GLU><<<blocks, kWqsThreads, kWqsLds, s>>>(p, num_groups);
  return check_launch("gmm_wqs_kernel");
}

template <int FMT>
static int launch_wqs_fmt(const WqSkinnyParams& p, bool glu, int num_groups, int blocks, hipStream_t s) {
  switch (cdiv(cdiv(p.K, 128), 8)) {
    case 1: return glu ? launch_wqs_one<FMT, 1, true>(p, num_groups, blocks, s) : launch_wqs_one<FMT, 1, false>(p, num_groups, blocks, s);
    case 2: return glu ? launch_wqs_one<FMT, 2, true>(p, num_groups, blocks, s) : launch_wqs_one<FMT, 2, false>(p, num_groups, blocks, s);
    case 3: return glu ? launch_wqs_one<FMT, 3, true>(p, num_groups, blocks, s) : launch_wqs_one<FMT, 3, false>(p, num_groups, blocks, s);
  }
  return fail(MOE_ERR_UNSUPPORTED, "gmm: K = %d is past the LDS-streamed decode kernel", p.K);
}

int launch_wqs(int fmt, int rows, const WqSkinnyParams& p, bool glu, int num_groups, hipStream_t s) {
  if (rows == 32) return launch_wqs32(fmt, p, glu, num_groups, s);
  int cus = 0;
  if (int st = device_cu_count(&cus)) return st;
  return fmt == WQ_MX4 ? launch_wqs_fmt<WQ_MX4>(p, glu, num_groups, cus, s) : launch_wqs_fmt<WQ_I4>(p, glu, num_groups, cus, s);
}

template <int FMT, int NSEG>
static int prepare_wqs_pair() {
  if (int st = reserve_lds(gmm_wqs_kernel<FMT, NSEG, true>, kWqsLds, lds_flags<std::integral_constant<int, 7000 + FMT * 100 + NSEG * 2 + 1>>())) return st;
  return reserve_lds(gmm_wqs_kernel<FMT, NSEG, false>, kWqsLds, lds_flags<std::integral_constant<int, 7000 + FMT * 100 + NSEG * 2>>());
}

int prepare_wqs() {
  if (int st = prepare_wqs32()) return st;
  if (int st = prepare_wqs_pair<WQ_I4, 1>()) return st;
  if (int st = prepare_wqs_pair<WQ_I4, 2>()) return st;
  if (int st = prepare_wqs_pair<WQ_I4, 3>()) return st;
  if (int st = prepare_wqs_pair<WQ_MX4, 1>()) return st;
  if (int st = prepare_wqs_pair<WQ_MX4, 2>()) return st;
  return prepare_wqs_pair<WQ_MX4, 3>();
}

}  // namespace moe
