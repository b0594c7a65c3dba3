// The activation image of a prompt step's next quantised product, handed from one product to the next by the model that runs them (no look-up by
// address: the model owns the buffer and passes it to both calls; whether the second call's x is what the image was made of is checked).
#pragma once
#include <cstddef>
#include <cstdint>

struct Mi355PromptImage {
    uint8_t* buf = nullptr;          // device memory of the owner
    size_t bytes = 0;
    bool valid = false;              // an image is there: of x, `live` rows and K columns, normalised with `norm`, in a layout of `rows` rows
    int32_t live = 0, rows = 0, K = 0;
    int32_t half = 0;                // which of two sets of the rows' factors it has: a product reads its own behind its GEMM, where the next image goes over the last
    const float* norm = nullptr;
    const void* x = nullptr;         // where the call that left the image wrote its output; taken by the next call or by none
    float eps = 0.f;                 // of every norm that an image is made with (the owner's; a product's descriptor has only its own)
    bool next = false;               // the call's output is the next call's x: leave its image
    // a grouped product of a mixture's down projection (group_block_table): its sums of `ks` ranges of K instead of outputs, where that is quicker (0: outputs)
    bool want_parts = false;
    // ... whose groups, so many, are whole tiles of 256 rows (mi355_internal_moe_group_tiles); -1: the kernels of such tiles whatever they take.  16 bits in what was
    // padding: the members around it stay where callers have them (below)
    int16_t tiles = 0;
    int32_t ks = 0, ldp = 0;
    const float* parts = nullptr;    // [ks][num_tokens][ldp], in scratch: read by the caller's next launch, in the same turn of (MI355_SCR_QMP_WS, stream)
    const float* scale = nullptr;    // [num_tokens]
    static constexpr int MAX_ROWS = 1024;
    // two sets of two floats a row, the f16 image, its sub-block sums
    static size_t need(size_t rows, size_t k) { return (size_t)MAX_ROWS * 16 + rows * (k * 2 + k / 256 * 32); }
};
// callers outside these sources share this layout (mi355_internal_qmatmul_prompt is exported): a new member goes behind the last or into padding
static_assert(offsetof(Mi355PromptImage, eps) == 56 && offsetof(Mi355PromptImage, want_parts) == 61 && offsetof(Mi355PromptImage, tiles) == 62 &&
              offsetof(Mi355PromptImage, ks) == 64 && offsetof(Mi355PromptImage, parts) == 72 && offsetof(Mi355PromptImage, scale) == 80 &&
              sizeof(Mi355PromptImage) == 88, "the layout that callers have");
