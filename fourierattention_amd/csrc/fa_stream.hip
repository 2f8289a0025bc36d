// One decode step of the cache for one layer in one launch (CACHE:731-748): the oldest window row of K and of V
// leaves the window -- its compressed dims enter the coefficients as a rank-1 update (TRI:853-856 with K = 1,
// K_start = p), its stored dims are appended to the page store -- and the new token takes a free window slot.
// The window buffer keeps one slot more than the window is long, so the slot that is written is never the slot
// that is read in the same step, and the three pieces of work need no order among themselves: the blocks of
// one grid take one of them each.
#include "fa_stream.h"

namespace {

template <typename E>
__global__ __launch_bounds__(256) void stream_update_kernel(const fa_stream::StreamParams p) {
  __shared__ float2 s_cs[64];
  fa_stream::stream_update_body<E>(p, blockIdx.x, blockIdx.y, s_cs);
}

}  // namespace

extern "C" int fa_stream_update(const fa_stream_args* a, fa_stream_t stream) {
  fa_stream::StreamParams p{};
  const int rc = fa_stream::stream_params(a, false, p);
  if (rc != FA_OK) return rc;
  dim3 grid(p.total, a->B);
  hipStream_t st = fa_hip_stream(stream);
  switch (a->dtype) {
    case FA_BF16: stream_update_kernel<bf16_t><<<grid, 256, 0, st>>>(p); break;
    case FA_FP16: stream_update_kernel<f16_t><<<grid, 256, 0, st>>>(p); break;
    default: stream_update_kernel<float><<<grid, 256, 0, st>>>(p); break;
  }
  return fa_check_launch("fa_stream_update");
}

extern "C" size_t fa_stream_args_size(void) { return sizeof(fa_stream_args); }
