// Grouped matmul, decode sizes with more than a few rows per expert: the LDS-streamed 4-bit kernel on tiles of up to 32 rows.

#include "moe_gmm_wqs.h"
#include "moe_gmm_wqs_run.h"

namespace moe {

// (instances of their own: the second row tile's code in the 16-row kernels costs a launch of one token 0.8-1 us)
template <int FMT, int NSEG, bool GLU, int ROWS>
__global__ __launch_bounds__(kWqsThreads) void gmm_wqs_kernel(const WqSkinnyParams p, int num_groups) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  wqs_run<FMT, NSEG, GLU, ROWS>(p, num_groups, smem);
}

template <int FMT, int NSEG, bool GLU>
static int launch_wqs_one(const WqSkinnyParams& p, int num_groups, int blocks, hipStream_t s) {
  if (int st = reserve_lds(gmm_wqs_kernel<FMT, NSEG, GLU, 32>, kWqsLds, lds_flags<std::integral_constant<int, 7300 + FMT * 100 + NSEG * 2 + (GLU ? 1 : 0)>>()))
    return st;
  gmm_wqs_kernel<FMT, NSEG, GLU, 32><<<blocks, kWqsThreads, kWqsLds, s>>>(p, num_groups);
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

int launch_wqs32(int fmt, const WqSkinnyParams& p, bool glu, int num_groups, hipStream_t s) {
  int cus = 0;
  if (int st = device_cu_count(&cus)) return st;
  return fmt == WQ_MX4 ? launch_wqs_fmt<WQ_MX4>(p, glu, num_groups, cus, s) : launch_wqs_fmt<WQ_I4>(p, glu, num_groups, cus, s);
}

template <int FMT, int NSEG>
static int prepare_wqs_pair() {
  if (int st = reserve_lds(gmm_wqs_kernel<FMT, NSEG, true, 32>, kWqsLds, lds_flags<std::integral_constant<int, 7300 + FMT * 100 + NSEG * 2 + 1>>())) return st;
  return reserve_lds(gmm_wqs_kernel<FMT, NSEG, false, 32>, kWqsLds, lds_flags<std::integral_constant<int, 7300 + FMT * 100 + NSEG * 2>>());
}

int prepare_wqs32() {
  if (int st = prepare_wqs_pair<WQ_I4, 1>()) return st;
  if (int st = prepare_wqs_pair<WQ_I4, 2>()) return st;
  if (int st = prepare_wqs_pair<WQ_I4, 3>()) return st;
  if (int st = prepare_wqs_pair<WQ_MX4, 1>()) return st;
  if (int st = prepare_wqs_pair<WQ_MX4, 2>()) return st;
  return prepare_wqs_pair<WQ_MX4, 3>();
}

}  // namespace moe
