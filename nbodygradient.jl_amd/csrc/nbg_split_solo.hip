// nbg_split_solo.hip -- two-wave launches of one system per workgroup
// (nbg_split.h): four workgroups a compute unit for up to 11 bodies, three for
// 12.  A translation unit of its own, as for the other launches.
#include "nbg_split.h"

namespace nbg {

// Two waves per SIMD: at most 256 registers each.
template <int HI, int LIMIT>
__global__ __launch_bounds__(2 * WAVE, 2) void nbg_run_split(GroupList gl, SysBufs B, int64_t chunk, int64_t bound,
                                                             unsigned long long* __restrict__ units,
                                                             unsigned long long* __restrict__ err) {
  // records of fewer than JGLOBAL_MIN bodies may have no room for J in HBM
  static_assert(!split_global<JGLOBAL_MIN - 1, false, LIMIT>(), "small systems keep J in LDS");
  __shared__ __attribute__((aligned(16))) unsigned char raw[LIMIT];
  __shared__ int share;
  split_body<HI, false, LIMIT>(raw, &share, gl, B, chunk, bound, units, err);
}

}  // namespace nbg

extern "C" hipError_t nbg_launch_split(int cls, nbg::GroupList gl, nbg::SysBufs bufs, int64_t chunk, int64_t bound,
                                       int grid, unsigned long long* units, unsigned long long* err, hipStream_t stream) {
  if (cls <= 11)
    hipLaunchKernelGGL((nbg::nbg_run_split<11, 40896>), dim3(grid), dim3(2 * nbg::WAVE), 0, stream, gl, bufs, chunk, bound, units, err);
  else if (cls == 12)
    hipLaunchKernelGGL((nbg::nbg_run_split<12, 54528>), dim3(grid), dim3(2 * nbg::WAVE), 0, stream, gl, bufs, chunk, bound, units, err);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}
