// The vector RoPE + K/V write looked at on the host.
#include "rope_vec_items.h"

// out: kernel, non-temporal, workgroups, workgroups a token.
extern "C" void plan_of(uint64_t tokens, uint64_t query_heads, uint64_t kv_heads, uint64_t rot_items,
                        uint64_t tail_chunks, uint64_t value_chunks, uint64_t bytes, uint64_t fp8, uint64_t whole_lines,
                        uint32_t* out) {
  const auto p = loom_hip_rope::write_plan({tokens, query_heads, kv_heads, rot_items, tail_chunks, value_chunks, bytes,
                                            fp8 != 0, whole_lines != 0});
  out[0] = static_cast<uint32_t>(p.kernel);
  out[1] = p.nt;
  out[2] = p.grid;
  out[3] = p.splits;
}

// Walks every lane of a launch and counts how often it reads each item's source:
// counts[token][query rotary | key rotary | key tail | value].

extern "C" int walk_items(uint32_t tokens, uint32_t cache_tokens, const int64_t* slots, uint32_t num_blocks,
                          uint32_t block_size, uint32_t query_heads, uint32_t kv_heads, uint32_t rot_items,
                          uint32_t tail_chunks, uint32_t value_chunks, uint8_t* counts) {
  using namespace loom_hip_rope;
  const VecCounts n{query_heads, kv_heads, rot_items, tail_chunks, value_chunks};
  const VecDivisors div = vec_divisors(query_heads, kv_heads, rot_items, tail_chunks, value_chunks);
  const uint32_t rows[4] = {query_heads, kv_heads, kv_heads, kv_heads};
  const uint32_t per[4] = {rot_items, rot_items, tail_chunks, value_chunks};
  uint32_t first[5] = {0, 0, 0, 0, 0};
  for (int k = 0; k < 4; ++k) first[k + 1] = first[k] + rows[k] * per[k];
  const uint32_t units = (tokens * div.waves_per_token + 3) / 4 * 4;  // whole workgroups of four waves
  for (uint32_t unit = 0; unit < units; ++unit) {
    uint32_t wave = 0;
    const uint32_t token = vec_token(div, unit, &wave);
    if (token >= tokens) continue;
    const int64_t slot = token < cache_tokens ? slots[token] : -1;
    for (uint32_t lane = 0; lane < 64; ++lane) {
      const VecItem it = vec_item(n, div, wave * 64U + lane);
      if (it.kind == kNoItem || !vec_reads(it.kind, vec_writes(slot, num_blocks, block_size))) continue;
      if (it.kind > kValueChunk || it.head >= rows[it.kind] || it.chunk >= per[it.kind]) return 1;
      ++counts[static_cast<uint64_t>(token) * first[4] + first[it.kind] + it.head * per[it.kind] + it.chunk];
    }
  }
  return 0;
}
