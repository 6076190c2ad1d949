// GEMM of few rows (vh_skinny.hip), as vh_gemm dispatches to it.
#pragma once

#include "../../include/voyager_hip.h"

namespace vh {

// Whether the few-row kernel takes a validated descriptor.
bool skinny_fits(const vh_gemm_desc* d);

// Runs it (skinny_fits holds and M, N > 0).
int skinny_gemm(const vh_gemm_desc* d, vh_stream_t stream);

}  // namespace vh
