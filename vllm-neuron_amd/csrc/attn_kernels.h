// Block-layout paged-KV attention (the NxDI
// context-encoding and token-generation attention reached through
// /root/reference/vllm_neuron/worker/neuronx_distributed_model_loader.py:339-348 with the
// block_table / slot_mapping / *_context_lens contract of
// /root/reference/vllm_neuron/worker/neuronx_distributed_model_runner.py:739-832).
//
// Pool layout (library-owned, one per layer and per K/V):
//     [num_blocks][nkv][block_size][hd] bf16
// i.e. one (block, kv-head) tile is a dense block_size*hd*2-byte range (8 KiB at 32 x 128),
// which a wave streams as 1 KiB coalesced reads.  Block 0 is vLLM's null block
// (reference platform.py:150-159): valid memory, never referenced by a live position.
#pragma once
#include "mi_common.h"

namespace mi {

constexpr int kAttnMaxSplits = 16;

int attn_decode_splits(int B, int nkv);
size_t attn_scratch_bytes(int B, int nh, int hd);

// launch_attn_decode of B rows and launch_attn_prefill of one sequence's T tokens in one launch (their outputs and partials are apart); scratch as launch_attn_decode's with tickets_zeroed
struct AttnMixed { const uint16_t* q; const int32_t* block_table; const int32_t* ctx_lens; int MB, B, max_ctx, num_blocks; uint16_t* out; void* scratch; };
int attn_mixed_lds(int hd, int kh, int splits);   // bytes its launch asks for: kh waves a head of the prompt's, splits of a request's context
int launch_attn_mixed(const AttnMixed& m, int T, int q_pos0, const uint16_t* q, const int32_t* block_table, uint16_t* out, const uint16_t* kpool, const uint16_t* vpool,
                      int block_size, int nh, int nkv, int hd, hipStream_t s, float* ws, size_t ws_bytes);
// whether a grid too short for the chip still takes each (sequence, kv head) in one work-group, without partials: short contexts
bool attn_decode_short(int B, int nkv, int hd, int max_ctx);
// q [B, nh, hd] bf16 -> out [B, nh*hd] bf16.  ctx_lens[b] = number of keys (incl. the new one); max_ctx: the longest, 0 = not known
int launch_attn_decode(const uint16_t* q, const uint16_t* kpool, const uint16_t* vpool, int block_size,
                       const int32_t* block_table, int MB, const int32_t* ctx_lens, int B, int nh,
                       int nkv, int hd, uint16_t* out, void* scratch, hipStream_t s, bool tickets_zeroed = false,
                       int rows_per_seq = 1, int num_blocks = 0, int max_ctx = 0);
// num_blocks > 0 (blocks of the pool): a wave's first K/V request does not wait for the context length (ids clamped into the pool)
// rows_per_seq R > 1: batch rows b R .. b R + R - 1 are one sequence at consecutive positions (block_table row b R
// serves them all); their heads share the MFMA columns and the sequence's K/V is read once
// tickets_zeroed: the first 4 KiB of `scratch` (the merge tickets) were zeroed once by the owner and
// only ever touched by these launches (which leave them at zero): enables the in-launch merge

// One sequence: q [T, nh, hd] at absolute positions q_pos0.., keys 0..q_pos0+T-1 from the pool.
// ws: room for the partial results of slices of the keys (none: one slice).
// The sequence's block table is staged in LDS once: at most kPrefillMaxBlocks blocks (131072 tokens at block_size 32).
constexpr int kPrefillMaxBlocks = 4096;
int launch_attn_prefill(const uint16_t* q, int T, int q_pos0, const uint16_t* kpool,
                        const uint16_t* vpool, int block_size, const int32_t* block_table, int nh,
                        int nkv, int hd, uint16_t* out, hipStream_t s, float* ws = nullptr, size_t ws_bytes = 0);

// k, v [T, nkv, hd] bf16 -> pool at slots [T] (-1 skips)
int launch_kv_write(const uint16_t* k, const uint16_t* v, const int64_t* slots, int T, int nkv, int hd,
                    uint16_t* kpool, uint16_t* vpool, int block_size, hipStream_t s);

}  // namespace mi
