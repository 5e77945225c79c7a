// nbg_split_duo.hip -- two-wave launch of two systems per workgroup
// (nbg_split.h), up to 9 bodies, four workgroups a compute unit.
#include "nbg_split.h"

namespace nbg {

template <int HI, int LIMIT>
__global__ __launch_bounds__(2 * WAVE, 2) void nbg_run_split_duo(GroupList gl, SysBufs B, int64_t chunk, int64_t bound,
                                                                 unsigned long long* __restrict__ units,
                                                                 unsigned long long* __restrict__ err) {
  static_assert(split_pairs<HI, LIMIT>(), "two records of HI bodies must fit");
  __shared__ __attribute__((aligned(16))) unsigned char raw[LIMIT];
  __shared__ int share;
  split_body<HI, true, LIMIT>(raw, &share, gl, B, chunk, bound, units, err);
}

}  // namespace nbg

extern "C" hipError_t nbg_launch_split_duo(nbg::GroupList gl, nbg::SysBufs bufs, int64_t chunk, int64_t bound, int grid,
                                           unsigned long long* units, unsigned long long* err, hipStream_t stream) {
  hipLaunchKernelGGL((nbg::nbg_run_split_duo<9, 40896>), dim3(grid), dim3(2 * nbg::WAVE), 0, stream, gl, bufs, chunk, bound, units, err);
  return hipGetLastError();
}
