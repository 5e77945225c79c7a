// nbg_split_wide.hip -- three-wave launch for few systems (nbg_split.h): one
// workgroup a compute unit, its waves on different SIMDs with all their
// registers, the Jacobian in LDS at every body count.
#include "nbg_split.h"

namespace nbg {

template <int HI, int LIMIT>
__global__ __launch_bounds__(3 * WAVE, 1) void nbg_run_split_wide(GroupList gl, SysBufs B, int64_t chunk, int64_t bound,
                                                                  unsigned long long* __restrict__ units,
                                                                  unsigned long long* __restrict__ err) {
  __shared__ __attribute__((aligned(16))) unsigned char raw[LIMIT];
  __shared__ int share;
  split_body<HI, false, LIMIT, true>(raw, &share, gl, B, chunk, bound, units, err);
}

}  // namespace nbg

extern "C" hipError_t nbg_launch_split_wide(nbg::GroupList gl, nbg::SysBufs bufs, int64_t chunk, int64_t bound, int grid,
                                            unsigned long long* units, unsigned long long* err, hipStream_t stream) {
  hipLaunchKernelGGL((nbg::nbg_run_split_wide<12, 163776>), dim3(grid), dim3(3 * nbg::WAVE), 0, stream, gl, bufs, chunk, bound, units, err);
  return hipGetLastError();
}
