// Launchers of the block kernels (widths up to 128), the scalar kernels (any width), the partial-sum
// reduction and the fill kernel.
#include "ccv1d_block.h"
#include "ccv1d_launch.h"

namespace ccv1d {

static_assert(blk_lds_bytes(kMaxBlockW, 4, true) <= 160 * 1024, "LDS of one gfx950 CU");

// Whether the x ring holds TX itself: 16-bit x, with initial states (if any) of the same type.
template <typename TX, typename Params>
static bool ring_of_tx(const Params& p) {
  const int dt = __is_same(TX, __bf16) ? DT_BF16 : __is_same(TX, _Float16) ? DT_F16 : -1;
  return dt >= 0 && (!p.has_init || p.i_dt == dt);
}

template <typename TX, typename E>
static hipError_t fwd_block(const FwdParams& p, hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed{0};
  const dim3 grid((unsigned)((int64_t)p.B * p.tl.nT), (unsigned)((p.D + 63) / 64));
  const void* k = reinterpret_cast<const void*>(&fwd_block_kernel<TX, E>);
  const size_t shmem = blk_lds_bytes(p.W, sizeof(E), false);
  const hipError_t e =
      allow_lds(k, shmem, blk_lds_bytes(kMaxBlockW, sizeof(E), false), lds_allowed);
  if (e != hipSuccess) return e;
  return launch(k, grid, dim3(kBlkNW * 64), shmem, s, &p);
}

template <typename TX, typename E>
static hipError_t bwd_block(const BwdParams& p, hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed{0};
  const dim3 grid((unsigned)((int64_t)p.B * p.tl.nT), (unsigned)((p.D + 63) / 64));
  const void* k = reinterpret_cast<const void*>(&bwd_block_kernel<TX, E>);
  const size_t shmem = blk_lds_bytes(p.W, sizeof(E), true);
  const hipError_t e = allow_lds(k, shmem, blk_lds_bytes(kMaxBlockW, sizeof(E), true), lds_allowed);
  if (e != hipSuccess) return e;
  return launch(k, grid, dim3(kBlkNW * 64), shmem, s, &p);
}

template <typename TX>
hipError_t launch_fwd_generic_t(const FwdParams& p, hipStream_t s) {
  if (p.W <= kMaxBlockW && p.tl.vec == 0) {  // vec == 1: few rows, the scalar kernel
    if constexpr (sizeof(TX) == 2) {
      if (ring_of_tx<TX>(p)) return fwd_block<TX, TX>(p, s);
    }
    return fwd_block<TX, float>(p, s);
  }
  const dim3 grid((unsigned)((int64_t)p.B * p.tl.nT), (unsigned)((p.D + 63) / 64));
  return launch(reinterpret_cast<const void*>(&fwd_generic_kernel<TX>), grid, dim3(64), 0, s, &p);
}

// Widths up to kMaxBlockW; wider ones take launch_bwd_wide_t.
template <typename TX>
hipError_t launch_bwd_generic_t(const BwdParams& p, hipStream_t s) {
  if constexpr (sizeof(TX) == 2) {
    if (ring_of_tx<TX>(p)) return bwd_block<TX, TX>(p, s);
  }
  return bwd_block<TX, float>(p, s);
}

template <typename TX>
hipError_t launch_bwd_wide_t(const BwdParams& p, float* G, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.B * p.tl.nT), (unsigned)((p.D + 63) / 64));
  BwdParams pc = p;
  void* args[] = {&pc, &G};
  hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(&bwd_g_kernel<TX>), grid, dim3(64),
                                 args, 0, s);
  if (e != hipSuccess) return e;
  return launch_args(reinterpret_cast<const void*>(&bwd_wide_kernel<TX>), grid, dim3(64), 0, s,
                     args);
}

template hipError_t launch_fwd_generic_t<float>(const FwdParams&, hipStream_t);
template hipError_t launch_fwd_generic_t<_Float16>(const FwdParams&, hipStream_t);
template hipError_t launch_fwd_generic_t<__bf16>(const FwdParams&, hipStream_t);
template hipError_t launch_fwd_generic_t<double>(const FwdParams&, hipStream_t);
template hipError_t launch_bwd_generic_t<float>(const BwdParams&, hipStream_t);
template hipError_t launch_bwd_generic_t<_Float16>(const BwdParams&, hipStream_t);
template hipError_t launch_bwd_generic_t<__bf16>(const BwdParams&, hipStream_t);
template hipError_t launch_bwd_generic_t<double>(const BwdParams&, hipStream_t);
template hipError_t launch_bwd_wide_t<float>(const BwdParams&, float*, hipStream_t);
template hipError_t launch_bwd_wide_t<_Float16>(const BwdParams&, float*, hipStream_t);
template hipError_t launch_bwd_wide_t<__bf16>(const BwdParams&, float*, hipStream_t);
template hipError_t launch_bwd_wide_t<double>(const BwdParams&, float*, hipStream_t);

hipError_t launch_reduce(const ReduceParams& p, hipStream_t s) {
  const int64_t n = (int64_t)(p.W + (p.has_bias ? 1 : 0)) * p.D;
  const dim3 grid((unsigned)((n + 63) / 64));
  return launch(reinterpret_cast<const void*>(&reduce_partials_kernel<kReduceNW>), grid,
                dim3(kReduceNW * 64), 0, s, &p);
}

hipError_t launch_fill(void* dst, int dst_dt, const void* src, int src_dt, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  void* args[] = {&dst, &dst_dt, &src, &src_dt, &n};
  return hipLaunchKernel(reinterpret_cast<const void*>(&fill_kernel), dim3((unsigned)blocks), dim3(256),
                         args, 0, s);
}

}  // namespace ccv1d
