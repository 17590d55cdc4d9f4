// Batches whose portions all run token by token (step_scan.h); the chunk kernels carry their short portions along.
#include "step_scan.h"

namespace mixk {
namespace ss {

template <typename T, int MODE, int R, bool V4>
__global__ void __launch_bounds__(256)
scan_step_kernel(ChunkArgs a, int max_rows) {
  __shared__ StepLds<MODE, R> lds;
  const int s = scan_grid_portion();
  if (s < a.S) scan_step<T, MODE, R, V4>(a, max_rows, blockIdx.x, s, lds);
}

template <typename T, int MODE, int R>
int launch(const ChunkArgs& a, int max_rows, hipStream_t st) {
  const dim3 grid = scan_grid(static_cast<int64_t>(a.H) * ((a.dv + kCols - 1) / kCols), a.S);
  if (scan_step_v4(a))
    hipLaunchKernelGGL((scan_step_kernel<T, MODE, R, true>), grid, dim3(256), 0, st, a, max_rows);
  else
    hipLaunchKernelGGL((scan_step_kernel<T, MODE, R, false>), grid, dim3(256), 0, st, a, max_rows);
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
