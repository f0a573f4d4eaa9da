// paged_attention.hip — GQA decode attention over the paged KV pool (gfx950).
//
// The decode-step hot kernel of the per-GPU worker engine. Memory-bound: the
// whole point is streaming each sequence's K/V exactly once per step at
// near-HBM rate.
#include "decode_core.h"

namespace {

using decode::D;
using decode::Work;

template <bool SPLIT>
hipError_t attend(const void* q, const void* k_cache, const void* v_cache,
                  const int32_t* block_tables, const int32_t* seq_lens,
                  void* out, float* part_o, float* part_ml, int n_seqs,
                  int n_q_heads, int kvh, int bs, int head_dim, int max_blocks,
                  int n_parts, int part_tokens, int spread, int probe,
                  int kv_fp8, int waves, float scale, hipStream_t stream) {
  if (n_seqs == 0) return hipSuccess;
  const int qpg = n_q_heads / kvh;
  if (head_dim != D || n_parts > 64 || (waves != 4 && waves != 8) ||
      (qpg != 1 && qpg != 2 && qpg != 4 && qpg != 8))
    return hipErrorInvalidValue;
  auto run = [&](auto zero) {
    typedef decltype(zero) CT;
    const int64_t head = (int64_t)bs * D;
    const Work<CT> w{(const short*)q, (int64_t)n_q_heads * D, (const CT*)k_cache,
                     (const CT*)v_cache, kvh * head, head, block_tables, seq_lens,
                     nullptr, 0, max_blocks, bs, (short*)out, part_o, part_ml, kvh,
                     qpg, part_tokens, spread && n_seqs % 2 == 0,
                     probe < max_blocks ? probe : max_blocks - 1, scale, 0.f, 0};
    return decode::attend<SPLIT, D>(w, n_seqs, n_parts, waves, stream);
  };
  return kv_fp8 ? run((unsigned char)0) : run((short)0);
}

}  // namespace

extern "C" {

hipError_t lds_paged_attention(const void* q, const void* k_cache,
                               const void* v_cache, const int32_t* block_tables,
                               const int32_t* seq_lens, void* out, int n_seqs,
                               int n_q_heads, int kvh, int bs, int head_dim,
                               int max_blocks, int probe, int kv_fp8, int waves,
                               float scale, hipStream_t stream) {
  return attend<false>(q, k_cache, v_cache, block_tables, seq_lens, out,
                       nullptr, nullptr, n_seqs, n_q_heads, kvh, bs, head_dim,
                       max_blocks, 1, 0, 0, probe, kv_fp8, waves, scale, stream);
}

hipError_t lds_paged_attention_split(
    const void* q, const void* k_cache, const void* v_cache,
    const int32_t* block_tables, const int32_t* seq_lens, void* out,
    float* part_o, float* part_ml, int n_seqs, int n_q_heads, int kvh, int bs,
    int head_dim, int max_blocks, int n_parts, int part_tokens, int spread,
    int probe, int kv_fp8, int waves, float scale, hipStream_t stream) {
  return attend<true>(q, k_cache, v_cache, block_tables, seq_lens, out, part_o,
                      part_ml, n_seqs, n_q_heads, kvh, bs, head_dim,
                      max_blocks, n_parts, part_tokens, spread, probe, kv_fp8,
                      waves, scale, stream);
}

}  // extern "C"
