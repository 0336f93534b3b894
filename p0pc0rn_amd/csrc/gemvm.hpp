// gemvm.hpp - the standalone GEMV-M launch (gemvm.hip), for its caller in gemv.hip.
#pragma once
#include "gemv_kernels.hpp"

namespace p0 {
void launch_gemvm(const GemvP& p, hipStream_t s);   // p.mrows = 2..16 rows, both encodings
}
