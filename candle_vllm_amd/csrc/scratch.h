// Device scratch registry (scratch.cpp): one buffer per (device, stream, key); growing retires instead of freeing.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

enum {
    MI355_SCR_PA_ARRIVE = 1,     // fused attention merge: arrival tickets (zero-initialised, self-cleaning)
    MI355_SCR_ARGMAX = 2,        // arg-max stage-1 slots (zero-initialised, self-cleaning)
    MI355_SCR_QMM_IMG0 = 3,      // wide mat-mul path: activation image, buffer 0 / 1
    MI355_SCR_QMM_IMG1 = 4,
    MI355_SCR_QMM_PART = 5,      // wide mat-mul path: split-K partial sums
    MI355_SCR_QMM_TICKET = 6,    // wide mat-mul path: split-K arrival tickets (zero-initialised, self-cleaning)
    MI355_SCR_QMP_WS = 7,        // prompt-step GEMM: quantised activation image
    MI355_SCR_DENSE_WS = 8,      // 16-bit prompt GEMM: copies of operands that do not start on 16 bytes
    MI355_SCR_COMM = 9,          // one-shot all-reduce staging
    MI355_SCR_GPTQ_WIDE = 10,    // split-K partial sums: 5..48-token launches of tiled 4-bit and of 16-bit weights, prompt launches of 16-bit weights
    MI355_SCR_PF_FP8 = 11,       // prompt attention over an e4m3 cache: the sequences' blocks as bf16 + their block table (prefill_attention.hip)
    MI355_SCR_GPTQ_GEMM = 13,    // 4-bit prompt GEMM: permuted x, its sums, scale panel, split-K partial sums (gptq_gemm.inc)
    MI355_SCR_DELTA = 12,        // delta rule by pieces: the pieces' records (hybrid_delta.hip)
};

// *out = a device buffer of >= bytes owned by (current device, st, key).  zero_on_create: the buffer is cleared (on `st`)
// when it is first created or grown.  Returns hipErrorStreamCaptureUnsupported when growth would be needed mid-capture.
// `most`: what a caller asks for at most; a buffer that grows is doubled, but not beyond this.
int mi355_scratch_get(void** out, int key, size_t bytes, hipStream_t st, bool zero_on_create, size_t most = (size_t)-1);
extern "C" void mi355_scratch_release_all(void);

// Launches that hand a buffer on to each other (a producer and its consumers) are enqueued under one of these, from before mi355_scratch_get until
// the last of them: two host threads on one stream then take turns with it, instead of one's producer running between the other's two.  A thread
// takes turns of one (stream, key) at a time; it may take that one again.
class Mi355ScratchTurn {
public:
    Mi355ScratchTurn(int key, hipStream_t st);
    ~Mi355ScratchTurn();
    Mi355ScratchTurn(const Mi355ScratchTurn&) = delete;
    Mi355ScratchTurn& operator=(const Mi355ScratchTurn&) = delete;
private:
    int slot_;
};

// void FFI entry points record their first failure here (mi355_last_error / mi355_clear_error in the header)
void mi355_note_error(int code);
