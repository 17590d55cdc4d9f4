// Batches whose portions all run token by token (step_scan.h); the chunk kernels carry their short portions along.
#include "step_scan.h"

namespace mixk {
namespace ss {

template <typename T, int MODE, int R, bool V4>
__global__ void __launch_bounds__(256)
scan_step_kernel(ChunkArgs a, int max_rows, int portion0) {
  __shared__ StepLds<MODE, R> lds;
  scan_step<T, MODE, R, V4>(a, max_rows, blockIdx.x, portion0 + blockIdx.y, lds);
}

template <typename T, int MODE, int R>
int launch(const ChunkArgs& a, int max_rows, hipStream_t st) {
  const bool v4 = scan_step_v4(a);
  scan_grids(a.H * ((a.dv + kCols - 1) / kCols), a.S, [&](dim3 grid, int first) {
    if (v4)
      hipLaunchKernelGGL((scan_step_kernel<T, MODE, R, true>), grid, dim3(256), 0, st, a, max_rows, first);
    else
      hipLaunchKernelGGL((scan_step_kernel<T, MODE, R, false>), grid, dim3(256), 0, st, a, max_rows, first);
  });
  return static_cast<int>(hipGetLastError());
}

template <typename T, int MODE>
int launch_dk(const ChunkArgs& a, int max_rows, hipStream_t st) {
  if (a.dk <= 64) return launch<T, MODE, 4>(a, max_rows, st);
  if (a.dk <= 128) return launch<T, MODE, 8>(a, max_rows, st);
  return launch<T, MODE, 16>(a, max_rows, st);
}

}  // namespace ss

int launch_step_scan(const ChunkArgs& a, int mode, int max_rows, int dtype, hipStream_t st) {
  if (a.dk > 256 || a.dk <= 0) return -1;
  int rc = -1;
#define MIXK_MODE(M) \
  case M: MIXK_DISPATCH(dtype, rc = (ss::launch_dk<T, M>(a, max_rows, st))); break;
  switch (mode) {
    MIXK_MODE(kModeRetention)
    MIXK_MODE(kModeForget)
    MIXK_MODE(kModeStateSpace)
    MIXK_MODE(kModeDelta)
    MIXK_MODE(kModeDeltaChannel)
  }
#undef MIXK_MODE
  return rc;
}

}  // namespace mixk
