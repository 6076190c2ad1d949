// GEMM of few rows (vh_skinny.hip), as vh_gemm dispatches to it.
#pragma once

#include "../../include/voyager_hip.h"

namespace vh {

// Whether the few-row kernel can run a validated descriptor.
bool skinny_fits(const vh_gemm_desc* d);

// Whether it does: tile_hint asks for it, or there is no hint and it is the
// faster one.
bool skinny_taken(const vh_gemm_desc* d);

// Runs it (skinny_fits holds and M, N > 0).
int skinny_gemm(const vh_gemm_desc* d, vh_stream_t stream);

}  // namespace vh
