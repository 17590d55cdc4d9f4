#include "chunk_scan_kernels.h"

template int mixk::cs::launch_mode<mixk::kModeForget>(const mixk::ChunkArgs&, int, hipStream_t);
