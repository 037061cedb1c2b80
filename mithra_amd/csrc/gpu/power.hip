// Launches of the radiation power sampler (power.h).
#include "common.h"
#include "power.h"

namespace mithra {

namespace {

__global__ __launch_bounds__(kPowerBlock) void k_power(const float* __restrict__ eb, PowerBufs B,
                                                       double* __restrict__ row, int N0, int N1, unsigned slot,
                                                       bool fresh) {
  power_body(eb, B, row, N0, N1, slot, fresh, blockIdx.x, gridDim.x, blockIdx.y);
}

}  // namespace

// Rows of planes outside the domain keep the zero the set-up gave them, as do all rows when no
// plane or no inner node exists.
hipError_t launch_power(Domain* d, unsigned n_time, unsigned row) {
  const mithra_grid& g = d->g;
  if (d->pN * d->pNl == 0) return hipErrorInvalidConfiguration;  // nothing to sample
  if (d->pNz == 0 || g.N0 <= 4 || g.N1 <= 4) return hipSuccess;
  bool fresh;
  const unsigned slot = sampler_slot(d, n_time, &fresh);
  hipLaunchKernelGGL(k_power, dim3(d->pblocks, d->pNz), dim3(kPowerBlock), 0, d->stream, d->eb, power_bufs(*d),
                     d->history + (size_t)row * d->pN * d->pNl, g.N0, g.N1, slot, fresh);
  return hipGetLastError();
}

}  // namespace mithra
