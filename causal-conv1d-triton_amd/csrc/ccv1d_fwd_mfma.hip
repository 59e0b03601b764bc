// Launcher of the matrix-core forward (bf16 x, silu, no seq_idx).
#include "ccv1d_launch.h"
#include "ccv1d_mfma_fwd.h"

namespace ccv1d {

template <int NC, int SUB>
static hipError_t mfma_one(const FwdParams& p, hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed{0};
  constexpr size_t shmem = MmFwdShape<NC, SUB>::BYTES;
  static_assert(shmem <= 160 * 1024, "LDS of one gfx950 CU");
  const void* k = reinterpret_cast<const void*>(&fwd_mfma_kernel<NC, SUB>);
  const hipError_t e = allow_lds(k, shmem, shmem, lds_allowed);
  if (e != hipSuccess) return e;
  return launch(k, dim3((unsigned)p.tl.nBlk), dim3(kMmNW * 64), shmem, s, &p);
}

template <int NC>
static hipError_t mfma_nc(const FwdParams& p, hipStream_t s) {
  return p.tl.L > kMmRows ? mfma_one<NC, 2>(p, s) : mfma_one<NC, 1>(p, s);
}

hipError_t launch_fwd_mfma(const FwdParams& p, hipStream_t s) {
  switch ((p.W - 1 + 15) / 16) {
    case 2: return mfma_nc<2>(p, s);
    case 3: return mfma_nc<3>(p, s);
    case 4: return mfma_nc<4>(p, s);
    case 5: return mfma_nc<5>(p, s);
    case 6: return mfma_nc<6>(p, s);
    case 7: return mfma_nc<7>(p, s);
    case 8: return mfma_nc<8>(p, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ccv1d
