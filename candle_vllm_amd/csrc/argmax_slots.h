// Greedy sampling in two launches: the first leaves a row's largest logit as (ordered value bits << 32 | ~index) in the row's slot; whoever
// takes it, once, clears the slot for the next step.  Both are enqueued in one turn of (MI355_SCR_ARGMAX, stream), scratch.h: the slots are the stream's.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "scratch.h"

// the slots of (device, stream), filled for `batch` rows behind everything on `stream` (elementwise.hip)
int mi355_internal_argmax_slots(unsigned long long** slots, const float* logits, int32_t batch, int32_t vocab, int64_t stream);

__device__ __forceinline__ uint32_t argmax_take(unsigned long long* slot) {
    const unsigned long long k = *slot;
    *slot = 0;
    return (k >> 32) == 0 ? 0u : (0xFFFFFFFFu - (uint32_t)(k & 0xFFFFFFFFu));
}
