// Launches of the streaming matrix-core kernel (va_stream_tile.h) by itself: plans without wide items.
#include <hip/hip_runtime.h>

#include "va_internal.h"
#include "va_launch.h"
#include "va_stream_tile.h"

namespace va {

template <typename E, int kD, bool kGather>
__global__ __launch_bounds__(kStreamThreads, StreamShape<kD>::kMinBlocks) void attn_stream_kernel(AttnArgs a) {
  stream_block<E, kD, kGather>(a, blockIdx.x);
}

template <typename E, int kD, bool kGather>
__global__ __launch_bounds__(kStreamThreads, (StreamShape<kD, true>::kMinBlocks)) void attn_stream_short_kernel(AttnArgs a) {
  stream_block_short<E, kD, kGather>(a, blockIdx.x);
}

template <typename E, int kD, bool kGather>
static int launch_stream_one(const AttnArgs& a, int n_items, bool short_items, hipStream_t stream) {
  const dim3 grid((unsigned)n_items * (unsigned)a.num_kv_heads), block(kStreamThreads);
  constexpr int bytes = StreamShape<kD>::lds_bytes(kGather), short_bytes = StreamShape<kD, true>::lds_bytes(kGather);
  static std::atomic<unsigned long long> devices{0}, short_devices{0};
  const hipError_t allowed =
      short_items ? allow_lds(reinterpret_cast<const void*>(&attn_stream_short_kernel<E, kD, kGather>), short_bytes, short_devices)
                  : allow_lds(reinterpret_cast<const void*>(&attn_stream_kernel<E, kD, kGather>), bytes, devices);
  if (allowed != hipSuccess) return va_fail(VA_ERR_HIP, "raising the LDS limit: %s", hipGetErrorString(allowed));
  if (short_items) {
    hipLaunchKernelGGL((attn_stream_short_kernel<E, kD, kGather>), grid, block, short_bytes, stream, a);
  } else {
    hipLaunchKernelGGL((attn_stream_kernel<E, kD, kGather>), grid, block, bytes, stream, a);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? VA_OK : va_fail(VA_ERR_HIP, "streaming attention launch: %s", hipGetErrorString(e));
}

template <typename E, int kD>
static int launch_stream_dim(const AttnArgs& a, int n_items, bool short_items, hipStream_t stream) {
  // Pages of at least 16 tokens take one scalar lookup per tile, smaller ones an entry per token.  The choice hangs
  // on the page size alone, so that a recorded launch keeps its kernel; in one kernel, the registers of the second
  // kind spilled into the first at head_dim 256.  (Other page sizes and slot lists beside larger
  // pages go through the first kernel's per-lane lookups.)
  if (a.page_size < kStreamTok && (a.page_size & (a.page_size - 1)) == 0)
    return launch_stream_one<E, kD, true>(a, n_items, short_items, stream);
  return launch_stream_one<E, kD, false>(a, n_items, short_items, stream);
}

template <typename E>
static int launch_stream_typed(const AttnArgs& a, int n_items, bool short_items, hipStream_t stream) {
  switch (a.head_dim) {
    case 64:
      return launch_stream_dim<E, 64>(a, n_items, short_items, stream);
    case 128:
      return launch_stream_dim<E, 128>(a, n_items, short_items, stream);
    case 256:
      return launch_stream_dim<E, 256>(a, n_items, short_items, stream);
    default:
      return va_fail(VA_ERR_ARG, "matrix-core path supports head_dim 64, 128, 256");
  }
}

int launch_mfma_stream(const AttnArgs& a, int dtype, int n_items, bool short_items, hipStream_t stream) {
  if (n_items == 0) return VA_OK;
  return dtype == VA_BF16 ? launch_stream_typed<BF16>(a, n_items, short_items, stream)
                          : launch_stream_typed<F16>(a, n_items, short_items, stream);
}

}  // namespace va
