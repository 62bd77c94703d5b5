// The int8 step over many known tokens, layer by layer (ygg_scan.hip): what ygg_capi.hip calls.
#pragma once
#include <hip/hip_runtime.h>

#include "ygg_layout.h"

namespace ygg {

// Is a call of B streams and T >= 2 tokens faster layer by layer than token by token? From the two forms' costs in
// microseconds, fitted to the six benchmark and trained models (tables and factored) at 1 to 4096 streams of 16 to 1024
// tokens: of those 220 calls the choice cost 0.6% over the faster form in the geometric mean, and at most 3% where this
// form was chosen and the other was the faster.
bool scan_pays(const YggDevModel &m, int64_t B, int64_t T);
// Workspace bytes of a call of B streams and T tokens (score: with the NLL; sort: its rows always sorted by expert), at
// most cap or what 64 rows take.
int64_t scan_scratch_bytes(const YggDevModel &m, int64_t B, int64_t T, bool score, bool sort, int64_t cap);
// The run or score of io (logits, leaves; targets and nll) in `bytes` of workspace at ws; hipErrorInvalidValue where
// that holds no row. Shapes of YGG_SHAPES with at least two layers.
hipError_t launch_scan(const YggDevModel &m, const int32_t *tokens, int B, int T, int8_t *state, const YggIO &io,
                       bool group, bool sort, void *ws, int64_t bytes, hipStream_t st);

}  // namespace ygg
