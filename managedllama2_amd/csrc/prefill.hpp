// Prompt tokens in batches: host interface (prefill.hip).
#pragma once

#include <cstddef>
#include <cstdint>

#include "../../include/llama2_hip.h"

namespace l2 {

constexpr int kPrefillMaxRows = 1024; // tokens per batch; longer prompts go through in batches of equal size
// Fewer known tokens take the decode step one by one.  A batch of one token tile costs about as much as three
// steps and the same for 8 rows as for 32.  8 rows and the step after them, against 9 steps: 7B 3.35 ms (9.32),
// behind 600 rows 3.7 (10.3), behind 3500 rows 4.7 (12.9); 13B 5.55 (16.8); a 2-layer model of width 256
// 0.11 (0.42).  Prompts of a few tokens keep the decode step's sums bit for bit.
constexpr int kPrefillMinRows = 8;

struct PrefillWorkspace {
    uint16_t* x = nullptr;    // residual stream, [rows][dim]
    uint16_t* q = nullptr;    // rotated queries, [rows][dim]
    uint16_t* xf = nullptr;   // normalised input / attention output in fragment order
    uint16_t* hf = nullptr;   // SwiGLU output in fragment order
    float* parts = nullptr;   // fp32 sums of the residual products over pieces of K, of attention over pieces of time
    float* rope = nullptr;    // (cos, sin) of 64 angles per row
    void* base = nullptr;     // the one allocation behind all of them
    int rows = 0;             // capacity, a multiple of 32; 0: no workspace, every token is a step
};

// Sizes `ws` for batches of up to min(seq_len, kPrefillMaxRows) tokens and allocates it (7B 78 MiB, 13B 145 MiB for
// 1024 rows); for fewer, or none, where memory is short.
int prefill_create(PrefillWorkspace& ws, const llama2_config& cfg);
void prefill_destroy(PrefillWorkspace& ws);
// The layers of Transformer.Forward for the `count` tokens at positions position .. position + count - 1,
// which are known: fills their rows of the key and value caches (nothing else of the run state).
int prefill_run(const PrefillWorkspace& ws, const llama2_config& cfg, const llama2_layer_weights* layers,
                const llama2_transformer_weights& w, const llama2_run_state& s, int position, int count);

} // namespace l2
