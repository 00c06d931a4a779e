// rows.h -- the decode-order forward of many rows at once (rows.hip): the
// multi-row counterpart of the token step, with the same bits.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "prefill.h"

struct Yue2Model;
struct Yue2Cache;

namespace y2 {

// C = DOT(W rows, X rows) in the decode order, through FP32 MFMAs.  epi:
// GEPI_ROUND, GEPI_RESID or GEPI_SWIGLU_BF16.  K a multiple of kGemmTK up to
// 16384, ldx and ldw multiples of 8, operands 16-byte aligned.
hipError_t launch_dot_gemm(hipStream_t s, int epi, const GemmArgs& g);

// Causal attention of `rows` query rows at positions p0 + r over the cache
// (whose rows up to p0 + rows - 1 are written), in the decode order; stats:
// rows x heads float2 scratch.  head_dim 64 or 128.
hipError_t launch_rows_attention(hipStream_t s, const FlashArgs& f, float2* stats, int head_dim);

// The self-tests of yue2_hip_selftest_math numbered 21 to 23: n a multiple of
// 64, 256 and 512.
hipError_t launch_rows_selftest(hipStream_t s, int which, const float* in, float* out, size_t n);

// Whether the multi-row path takes n tokens appended to `context` cached
// ones (the shape allows it and it is the faster way).
bool rows_supported(const Yue2Model* m, int context, int n);

// n ids through the layers, appended to cache c (validated by the caller;
// the model's batch-1 workspace allocated), the last row's logits of the
// phase in the workspace.  Enqueued on the model's stream and waited for;
// c->length is the caller's to advance.  1: no memory for the rows' scratch
// (nothing ran).
int run_rows(Yue2Model* m, Yue2Cache* c, const int32_t* ids, int n, int phase, bool head);

}  // namespace y2
