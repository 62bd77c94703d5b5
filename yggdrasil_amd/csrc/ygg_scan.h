// The int8 step over many known tokens, layer by layer (ygg_scan.hip): what ygg_capi.hip calls.
#pragma once
#include <hip/hip_runtime.h>

#include "ygg_layout.h"

namespace ygg {

// What a call of known tokens is asked for: a run with its logits, a score, or a run without logits.
enum class ScanCall { run, score, state };
// The kernel that takes it token by token: flow_kernel, pipe_kernel or a per-stream one.
enum class TokenKernel { flow, pipe, stream };
// Is a call of B streams and T >= 2 tokens faster layer by layer than token by token? From the two forms' costs in
// microseconds, fitted to 54 models (2 to 5 layers, depths 3 to 14, every shape of YGG_SHAPES, tables and factored) at 1
// to 4096 streams of 2 to 1024 tokens, run with and without logits and scored: 17 094 times of each form. Over them the
// choice costs 0.5% over the faster form in the geometric mean, more than 10% in 2% of the calls and 1.8 times at most.
// (Without each kernel's layers, rounds and fixed cost, fitted to models of 3 to 5 layers from 16 tokens on, it cost 13%,
// and short calls of few layers took up to 8 times as long.)
bool scan_pays(const YggDevModel &m, int64_t B, int64_t T, ScanCall call, TokenKernel token);
// Workspace bytes of a call of B streams and T tokens (score: with the NLL; sort: its rows always sorted by expert), at
// most cap or what 64 rows take.
int64_t scan_scratch_bytes(const YggDevModel &m, int64_t B, int64_t T, bool score, bool sort, int64_t cap);
// The run or score of io (logits, leaves; targets and nll) in `bytes` of workspace at ws; hipErrorInvalidValue where
// that holds no row. Shapes of YGG_SHAPES with at least two layers.
hipError_t launch_scan(const YggDevModel &m, const int32_t *tokens, int B, int T, int8_t *state, const YggIO &io,
                       bool group, bool sort, void *ws, int64_t bytes, hipStream_t st);

}  // namespace ygg
