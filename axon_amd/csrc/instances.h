// Which kernel instance a launch chose.
//
// The products and the attention are templates with many instances (tile shapes, waves a block,
// segments, epilogues), one of which a dispatch picks from the sizes of a call.  An instance that
// no test ever launches is unverified arithmetic: so every launch site names its instance here,
// the library knows every instance that was compiled into it (they register themselves when the
// library is loaded) and which of them have been launched since the last reset, and a test
// asserts that the two lists are the same (the reference tests its products at the sizes of its
// models for the same reason: src/cuda/prefill.cu:1100, src/model.rs:6238-6319).
//
//   AXK_INSTANCE(INST_GEMM_TILE, BM, BN, ...);     // at the launch, inside the launching template
//
// Host code only; costs one store a launch.
#pragma once

#include <initializer_list>

enum {
  INST_GEMM_FMA = 0,         // rows of X a block (16, 32, 64: streaming W; 128: tiles through LDS), gated
  INST_GEMM_TILE,            // BM, BN, waves m, waves n, gated, whole steps of 64 k that the stages hold (five of 32: 2)
  INST_GEMM_STREAM,          // row tiles, tiles of X rows, segments, epilogue
  INST_GEMM_NORMED,          // tile pairs a wave, segments, epilogue, rows of X in LDS, float4 a lane
  INST_GEMM_ROWS,            // row tiles of W a wave, tiles of 16 rows of X, waves, epilogue
  INST_GEMM_SPLIT_REDUCE,    // 0 plain, 1 with the norm, 2 with the rotary store (2, 8 beside it: eight tokens a thread), 3 an element a thread
  INST_ATTENTION_ROWS,       // bfloat16 build, waves a (token, head)
  INST_ATTENTION_PREFILL,    // head_dim, query heads a block, pages of 64 positions or more
  INST_ATTENTION_DECODE,     // head_dim, waves a block
  INST_RMSNORM,              // 1: rows read as float4
  INST_GROUPED_GEMM,         // 2, 3: matrix cores through LDS, 256 and 128 rows of W a block, 5: 256 by tiles of 128 rows, 1, 4: from memory, a long and a short K, 0: 32-bit FMA; gated epilogue
  INST_CAUSAL_CONV,          // 1: runs of tokens, 0: a thread a (token, channel)
  INST_LATENT_PROMPT,        // tiles of 16 latent dims, chunks of 32 key dims, bounds known when compiled, sink
  INST_LATENT_TOKENS,        // tiles of 16 latent dims, chunks of 32 key dims, sink
  INST_GEMM_KEPT,            // tiles of 128 x 128 that keep the sums of K's segments; gated
  INST_ATTENTION_F32_PREFILL,    // float32 build, head_dim
  INST_ATTENTION_F32_DECODE,     // float32 build, head_dim, waves a block
  INST_GEMM_FMA_BY_CHAIN,    // beside gemm_fma: rows of X a block, gated, numbers loaded four at a time
  INST_GEMM_FMA_FLOW,        // beside gemm_fma<128>: rows to LDS by direct loads; gated
  INST_HEADS_PREPARE,        // blocks a token: 1: one, 2: of up to eight or sixteen units, 0: of four
  INST_STATE_CONV,           // 1: runs of tokens, 0: a thread a (token, channel)
  INST_EMBED,                // 1: eight numbers a thread, 0: one
  INST_ATTENTION_F32_WAVES,      // beside attention_f32_prefill: head_dim, waves for sixteen tokens
  INST_LATENT_BLOCKS,        // tiles of 16 latent dims, chunks of 32 key dims: blocks of positions side by side
  INST_GEMM_FMA_FLOW_ROWS,   // beside gemm_fma_flow: rows a block; gated
  INST_GATED_SCAN,           // 1: waves that feed the walk, 0: a thread a channel
  INST_MASKED_BLOCKS,        // maps, tiles of 16 value dims, chunks of 32 key dims: blocks of positions side by side
  INST_MASKED_FOLD,          // maps, value dims a lane
  INST_KINDS
};

int axk_register_instance(int kind, std::initializer_list<int> params);
void axk_note_instance(int id);

template <int KIND, int... P>
struct KernelInstance {
  static const int id;
};
template <int KIND, int... P>
const int KernelInstance<KIND, P...>::id = axk_register_instance(KIND, {P...});

#define AXK_INSTANCE(...) axk_note_instance(KernelInstance<__VA_ARGS__>::id)
