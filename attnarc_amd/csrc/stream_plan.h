// Launch shape of the streaming decode kernels for groups of up to 16 query heads
// over 16-bit and FP8 caches, as a function of the call alone. Plain C++, so that a
// host program can look at any call.
#pragma once

#include <cstdint>

namespace loom_hip_decode {

struct StreamCall {
  uint64_t items;        // sequences x partitions x KV heads
  uint32_t steps;        // 16-token steps of the longest item
  uint32_t head_size;    // 64, 80, 96, 112, 128 or 256
  uint32_t group;        // query heads per KV head
  uint32_t kv_heads;
  uint64_t parts;        // partitions of the longest sequence
  bool fp8;              // FP8 cache, else 16-bit
  bool dense;            // each KV head's token rows are contiguous (HND)
  bool index_order;      // the library's own split: items in index order
};

struct StreamPlan {
  uint32_t waves;   // per item
  uint32_t items;   // per workgroup (one wave each where more than one)
  uint32_t stages;  // pipeline stages per wave
  bool pairs;       // a workgroup folds two consecutive partitions of two KV heads
};

// What decides is how many items a CU holds at once. A stage takes 8 KiB of LDS at
// head size 128 (16 tokens of a 16-bit cache, 32 of an FP8 one), so a CU holds two
// workgroups of four two-stage waves, and four of one-stage waves; two stages hide
// more of a load's latency. Sequence lengths are on the device: a ragged batch has
// fewer and shorter items than the call says. Figures below are geometric means of
// call times over some 30,000 calls of generic shapes; those of FP8 caches are
// relative to the form with steps of 16 tokens (see Fp8StreamDecoder), whose
// two-stage waves took 12 KiB.

// FP8 workgroups fold pairs of partitions (pair_item, head size 128) where the
// states they save are worth the coarser workgroups: all short partitions, and
// groups of more than four heads, or four in an HND cache, where a partition
// holds eight steps or more. None -> pairs (one stage): four-step partitions, 1 head
// 0.83 -> 0.83, 2 0.85 -> 0.85, 6 0.97 -> 0.86, 8 1.04 -> 0.87; eight steps from 4,096
// items, NHD, 1 / 2 / 4 heads 0.88 / 0.90 / 0.94 -> 0.89 / 0.88 / 0.93, 6 1.01 -> 0.92, 8
// 0.98 -> 0.92; HND, 4 0.94 -> 0.89, 6 0.97 -> 0.90.
inline bool folds_pairs(const StreamCall& c) {
  if (!c.fp8 || c.head_size != 128 || c.parts <= 2 || c.kv_heads % 2 != 0) return false;
  return c.steps < 8 || c.group > 4 || (c.group == 4 && c.dense);
}

// Items of fewer than eight steps on grids that leave CUs idle: four waves share
// the steps although some take one or none, since a wave alone walks them one
// after another. The reduction costs more with more heads, so wide groups need
// more steps. Call us, one wave -> four, 100-token contexts: BF16 head size 128 8
// items 8.0 -> 6.1, 256 9.0 -> 8.0 (512 9.7 -> 9.9); 64 8 items 6.6 -> 4.9, 512 8.2 ->
// 7.5; FP8 128 8 items 7.4 -> 5.6, 256 8.5 -> 7.0. Four waves over one by group and
// steps, up to 256 items: 16-bit 2 heads 0.91 / 0.83 at 4 / 5 steps, 8 heads 1.01 /
// 0.94, 16 heads 1.13 / 1.06 / 1.03 / 0.91 at 4 / 5 / 6 / 7; FP8 8 heads 0.82 at 5, 16
// heads 0.96 / 0.85 at 5 / 6.
inline bool splits_short(const StreamCall& c) {
  if (c.steps >= 8 || c.items > (c.head_size == 64 ? 512U : 256U)) return false;
  if (c.fp8) return c.steps >= (c.group > 8 ? 6U : 5U);
  return c.steps >= (c.group > 8 ? 7U : c.group > 6 ? 5U : 4U);
}

inline StreamPlan stream_plan(const StreamCall& c) {
  // One wave per item, four items (adjacent KV heads) to a workgroup, from 4,096
  // items, and from 1,024 (four per CU) where partitions have at least eight steps
  // (10% faster there than the 4-wave split). Smaller grids split an item over four
  // waves when that leaves each two steps or more, else run one wave per
  // workgroup: there the number of CUs in use matters more than co-locating heads.
  const bool grouped = c.items >= 4096 || (c.items >= 1024 && c.steps >= 8);
  if (c.head_size == 256) {
    // A stage takes 16 KiB: five two-stage waves fit a CU, ten one-stage ones.
    // 1,025-1,280 items, two stages -> one: ragged 16-bit 0.98 -> 1.07, fixed
    // lengths 0.99 -> 0.89; FP8 0.95 -> 0.88. The 4-wave split under 4 items per
    // CU (128 items as single waves 1.6x slower).
    if (c.items >= 4096) return {1, 2, 1, false};
    if (c.items >= 1024) return {1, 1, c.fp8 || c.items > 1280 ? 1U : 2U, false};
    return c.steps < 8 ? StreamPlan{1, 1, 2, false} : StreamPlan{4, 1, 2, false};
  }
  if (grouped && c.fp8) {
    // One stage where items are short or fill the waves. Two stages -> one: four
    // steps at 128 1.06 -> 0.85 (as pairs), 64 1.00 -> 0.90, 112 0.85 -> 0.64; from
    // 4,096 items, 8 / 16 steps, 64 0.98 / 0.94 -> 0.91 / 0.90, 96 0.71 / 0.68 -> 0.65 / 0.63,
    // 128 0.98 / 0.93 -> 0.89 / 0.88; but 32 steps at 80 and 96 0.70 / 0.76 -> 0.71 / 0.77
    // (32 x <= 4,001 tokens of 32/32 heads at 96 100.6 -> 102.9 us); 2,048-4,095 items at
    // 64 0.83 -> 0.86, at 128 0.88 -> 0.82;
    // pairs of 1,024-2,047 items 0.87 -> 0.87, the worst call 1.10 -> 0.93.
    const bool pairs = folds_pairs(c);
    const bool one = pairs || c.steps < 8 ||
                     (c.head_size == 128 ? c.items >= 2048 : c.items >= 4096 && c.steps <= 16);
    return {1, 4, one ? 1U : 2U, pairs};
  }
  if (grouped) {
    // 16-bit one-stage waves, two items to a workgroup, over two-stage ones, four to
    // a workgroup: from 8,192 items (four rounds of the latter) 0.98, at most 1.01,
    // for groups of four heads and more; 1.02 and up to 1.09 for fewer, and between
    // 4,096 and 8,191 0.96-1.05 by how the last round fills, up to 1.11.
    const bool one = c.head_size == 128 && !c.index_order && c.items >= 8192 && c.steps >= 32 && c.group >= 4;
    return one ? StreamPlan{1, 2, 1, false} : StreamPlan{1, 4, 2, false};
  }
  if (c.steps < 8 && !splits_short(c)) {
    // FP8: one 32-token step, or a few, in half the LDS. Two stages -> one at 128:
    // 2,560-4,095 items of 1 / 2 / 4 steps 1.22 / 1.16 / 0.99 -> 0.91 / 0.86 / 0.88,
    // 257-512 items 1.02 / 0.94 / 0.90 -> 0.98 / 0.91 / 0.87.
    return {1, 1, c.fp8 ? 1U : 2U, false};
  }
  if (c.fp8) {
    // Past two 64 KiB workgroups per CU. Two stages -> one at 80-128, 513-767 items
    // of 16 / 32 / 64 steps 1.02 / 0.98 / 0.91 -> 0.90 / 0.89 / 0.88, 768-1,023 1.00 / 0.93 /
    // 0.91 -> 0.81 / 0.82 / 0.85 (as single waves 0.80 / 0.88 / 0.95, ragged batches up to
    // 1.43); at 64 (32 KiB) 0.93 and 0.93.
    return {4, 1, c.head_size > 64 && c.items > 512 ? 1U : 2U, false};
  }
  // 16-bit caches, from three items per CU: more of them at once on one-stage
  // waves. Two stages -> one at 128, 8 / 16 / 32 steps: fixed lengths 0.81 / 0.89 /
  // 0.95, ragged 0.83 / 0.82 / 0.97; at 80 (48 KiB, three per CU) 0.84 / 0.93 / 0.97 and
  // 1.00 / 0.93 / 1.02. (Single waves at 128: fixed 0.75 / 0.85 / 0.93, but ragged
  // batches up to 1.30, at 80 up to 1.43.)
  const bool one = c.items >= 768 && c.steps <= (c.head_size >= 112 ? 32U : 24U) && c.head_size > 64;
  return {4, 1, one ? 1U : 2U, false};
}

}  // namespace loom_hip_decode
