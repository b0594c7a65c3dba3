// Device-side restatement of `prepare_decode` for the greedy loop of both host layers (host_model.cpp, dense_model.cpp):
// positions / slots / context lengths of the NEXT step from the block table, so that a captured graph runs step after step
// without host input.   reference: src/openai/pipelines/inputs.rs:389-423 (`prepare_decode`), backend/graph.rs:592-608 (static inputs)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>
#include "argmax_slots.h"

// The sampled tokens come out of the argmax' slots here: a launch of 4 us less per step.
static __global__ void advance_kernel(uint32_t* tokens, unsigned long long* sampled, int64_t* positions, int64_t* slots,
                                      uint32_t* ctx, const uint32_t* bt, int max_blocks, int block_size, int batch) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= batch) return;
    tokens[b] = argmax_take(sampled + b);
    const uint32_t n = ctx[b] + 1;              // sequence length after appending the sampled token
    ctx[b] = n;
    const int64_t pos = (int64_t)n - 1;
    positions[b] = pos;
    // the step after the last reserved block has no slot (-1 = "do not write", as a padded slot): the host refuses to
    // run that step, and this kernel never reads past the block-table row
    if (pos / block_size >= max_blocks) { slots[b] = -1; return; }
    const int64_t blk = bt[(size_t)b * max_blocks + pos / block_size];
    slots[b] = blk * block_size + pos % block_size;
}

// The static inputs of the greedy loop, one block of device memory (positions | slots | tokens | context lengths | block tables) behind one pinned
// image of it: a change of the batch is one copy, and waits for it.  (Begin, step and read of one sequence of a 1B model, eight layers: 346 us with a
// copy per array from pageable memory, 330 with one; 16 of a 4-bit 7B, seven layers, 752 and 723.  Without the wait 324 and 716, but then nothing orders
// a step on another stream behind the copy -- one whose handle is the same (a per-thread stream of another thread, a new stream in a destroyed one's place) or
// a graph of the step that the caller captured and replays where he likes.)
struct StepInputs {
    uint8_t *dev = nullptr, *host = nullptr;
    int32_t batch = 0, blocks = 0;          // room
    size_t bytes() const { return (size_t)batch * (24 + 4 * (size_t)blocks); }
    int64_t* positions(uint8_t* p) const { return reinterpret_cast<int64_t*>(p); }
    int64_t* slots(uint8_t* p) const { return positions(p) + batch; }
    uint32_t* tokens(uint8_t* p) const { return reinterpret_cast<uint32_t*>(slots(p) + batch); }
    uint32_t* ctx(uint8_t* p) const { return tokens(p) + batch; }
    uint32_t* tables(uint8_t* p) const { return ctx(p) + batch; }
    bool create(int max_batch, int max_blocks) {
        batch = max_batch; blocks = max_blocks;
        return hipMalloc((void**)&dev, bytes()) == hipSuccess && hipHostMalloc((void**)&host, bytes() + (size_t)batch * 4, hipHostMallocDefault) == hipSuccess;
    }
    void destroy() {
        if (host) (void)hipHostFree(host);
        if (dev) (void)hipFree(dev);
        dev = host = nullptr;
    }
    // the inputs of a step over n sequences (checked by the caller: every position has a block in its table's row), behind everything on `st`; waits for it
    hipError_t send(const uint32_t* toks, const uint32_t* lens, const uint32_t* bt, int n, int n_blocks, int block_size, hipStream_t st) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;     // the image is written once, a replay would send what it holds by then
        if (st && hipStreamIsCapturing(st, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone) return hipErrorStreamCaptureUnsupported;
        for (int b = 0; b < n; ++b) {
            const int64_t pos = (int64_t)lens[b] - 1;
            positions(host)[b] = pos;
            slots(host)[b] = (int64_t)bt[(size_t)b * n_blocks + pos / block_size] * block_size + pos % block_size;
            tokens(host)[b] = toks[b];
            ctx(host)[b] = lens[b];
        }
        memcpy(tables(host), bt, (size_t)n * n_blocks * 4);
        const hipError_t e = hipMemcpyAsync(dev, host, (size_t)batch * 24 + (size_t)n * n_blocks * 4, hipMemcpyHostToDevice, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    }
    // the tokens of the n sequences, behind everything on `st`; waits for it
    hipError_t read_tokens(uint32_t* out, int n, hipStream_t st) {
        uint32_t* pin = reinterpret_cast<uint32_t*>(host + bytes());
        hipError_t e = hipMemcpyAsync(pin, tokens(dev), (size_t)n * 4, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e == hipSuccess) memcpy(out, pin, (size_t)n * 4);
        return e;
    }
};
