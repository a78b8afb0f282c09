// The launch shape of a streaming decode call, looked at on the host.
#include "stream_plan.h"

// out: waves per item, items per workgroup, stages, pairs.
extern "C" void plan_of(uint64_t items, uint32_t steps, uint32_t head_size, uint32_t group, uint32_t kv_heads,
                        uint64_t parts, uint32_t fp8, uint32_t dense, uint32_t index_order, uint32_t* out) {
  const auto p = loom_hip_decode::stream_plan(
      {items, steps, head_size, group, kv_heads, parts, fp8 != 0, dense != 0, index_order != 0});
  out[0] = p.waves;
  out[1] = p.items;
  out[2] = p.stages;
  out[3] = p.pairs;
}
