// The RoPE + paged K/V write as a launch: which kernel a call takes, and which
// 16-byte chunks each lane of rope_paged_kv_vec_kernel reads. Plain C++, so that a
// host program can look at any call and go through every lane of a launch.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define LOOM_ROPE_HD __host__ __device__ __forceinline__
#else
#define LOOM_ROPE_HD inline
#endif

namespace loom_hip_rope {

// Divisions of the item decode as multiplications by rounded inverses.
struct VecDivisors {
  uint32_t waves_per_token;
  uint32_t token_inverse;      // floor(2^32 / waves_per_token), saturated
  uint32_t rot, tail, value;   // floor(2^32 / chunks) + 1: exact below 2^16 items a token; 0: divide
};

// Chunks of a head's row and their counts.
struct VecCounts {
  uint32_t query_heads, kv_heads;
  uint32_t rot_items, tail_chunks, value_chunks;  // a head's rotary items, K tail chunks and V chunks
};

inline VecDivisors vec_divisors(uint64_t query_heads, uint64_t kv_heads, uint64_t rot_items, uint64_t tail_chunks,
                                uint64_t value_chunks) {
  const uint64_t items = query_heads * rot_items + kv_heads * (rot_items + tail_chunks + value_chunks);
  const uint64_t waves_per_token = (items + 63) / 64;
  // chunks == 1 would need 2^32 + 1: divided by one instead
  auto inverse = [&](uint64_t chunks) -> uint32_t {
    return chunks > 1 && items < (1ULL << 16) ? static_cast<uint32_t>((1ULL << 32) / chunks + 1U) : 0U;
  };
  const uint64_t token_inverse = (1ULL << 32) / waves_per_token;
  return {static_cast<uint32_t>(waves_per_token),
          static_cast<uint32_t>(token_inverse > 0xffffffffULL ? 0xffffffffULL : token_inverse), inverse(rot_items),
          inverse(tail_chunks), inverse(value_chunks)};
}

LOOM_ROPE_HD uint32_t mul_high(uint32_t a, uint32_t b) {
  return static_cast<uint32_t>((static_cast<uint64_t>(a) * b) >> 32);
}

// The token of wave `unit` of the launch, and the wave's place in it.
LOOM_ROPE_HD uint32_t vec_token(const VecDivisors& div, uint32_t unit, uint32_t* wave) {
  uint32_t token = mul_high(unit, div.token_inverse);  // unit / waves_per_token, or one less
  *wave = unit - token * div.waves_per_token;
  if (*wave >= div.waves_per_token) {
    ++token;
    *wave -= div.waves_per_token;
  }
  return token;
}

enum : uint32_t { kQueryRotary, kKeyRotary, kKeyTail, kValueChunk, kNoItem };

struct VecItem {
  uint32_t kind, head, chunk;
};

// Item `item` of a token: its rotary items of Q, then of K, then K tail and V
// chunks.
LOOM_ROPE_HD VecItem vec_item(const VecCounts& n, const VecDivisors& div, uint32_t item) {
  const uint32_t q_items = n.query_heads * n.rot_items;
  const uint32_t k_items = n.kv_heads * n.rot_items;
  const uint32_t t_items = n.kv_heads * n.tail_chunks;
  uint32_t r = item, kind = kQueryRotary, per = n.rot_items, inverse = div.rot;
  if (r >= q_items) {
    r -= q_items;
    kind = kKeyRotary;
    if (r >= k_items) {
      r -= k_items;
      kind = kKeyTail;
      per = n.tail_chunks;
      inverse = div.tail;
      if (r >= t_items) {
        r -= t_items;
        kind = kValueChunk;
        per = n.value_chunks;
        inverse = div.value;
        if (r >= n.kv_heads * n.value_chunks) return {kNoItem, 0, 0};
      }
    }
  }
  const uint32_t head = inverse != 0 ? mul_high(r, inverse) : r / per;
  return {kind, head, r - head * per};
}

// Whether the token of slot entry `slot` (-1: it has none) goes to the caches.
LOOM_ROPE_HD bool vec_writes(int64_t slot, uint32_t num_blocks, uint32_t block_size) {
  return slot >= 0 && static_cast<uint64_t>(slot) < static_cast<uint64_t>(num_blocks) * block_size;
}

// Whether a lane reads its item's source row. K tail and V serve the caches
// only; V need not hold a row for a token that does not go there.
LOOM_ROPE_HD bool vec_reads(uint32_t kind, bool writes) { return kind <= kKeyRotary || writes; }

enum class WriteKernel : uint32_t {
  kGeneral,  // rope_paged_kv_kernel
  kWaves,    // rope_paged_kv_vec_kernel
  kTokens,   // rope_paged_kv_token_kernel
};

struct WriteShape {
  uint64_t tokens, query_heads, kv_heads;
  uint64_t rot_items, tail_chunks, value_chunks;  // a head's, as in VecCounts
  uint64_t bytes;                                 // that the call touches
  bool fp8;                                       // the caches hold FP8
  bool whole_lines;  // rotated rows and cache rows are whole 128-byte lines
};

struct WritePlan {
  WriteKernel kernel;
  bool nt;        // kWaves: non-temporal hint
  uint32_t grid;  // workgroups
  uint32_t splits;  // kTokens: workgroups a token
};

// Calls of whole 128-byte lines that touch more than this many bytes take the
// non-temporal hint on the rows and the caches: past it the 256 MiB Infinity
// Cache keeps little of them for the next kernel. Us without / with the hint at
// 32/8 heads, head size 128: BF16 cache 134 MB 22.8 / 24.5, 161 MB 27.9 / 28.8, 188
// MB 34.3 / 33.1, 215 MB 41.6 / 37.4, 323 MB 62.7 / 54.7; FP8 124 MB 22.9 / 24.6,
// 199 MB 37.8 / 35.4. Stores of part of a line are not joined under the hint: 32/8
// heads, head size 96, half rotary, 300 MB 100 / 135.
constexpr uint64_t kNtBytes = 192ULL << 20;

// The workgroup-per-token kernel (two items a thread) against waves of 64 chunks:
//   - 480 to 512 chunks a token, or a multiple of 512, leave it no idle thread.
//     From 24 MiB on. Us, waves -> workgroups a token: 16/16 heads, head size 128,
//     30 MB 8.7 -> 8.5 (12 MB 4.4 -> 5.0), 100 MB 22.7 -> 20.6; 32/32 at 128, half
//     rotary, FP8 300 MB 94 -> 74; 32/32 at 64, 300 MB 69 -> 60; but 768 chunks
//     (32/32 at 96, half rotary) waves by 2-9%.
//   - native caches from 256 chunks a token, 44 to 186 MiB, mostly in the Infinity
//     Cache: 20/20 at 80, 100 MB 19.6 -> 18.2, 32/8 at 128, 100 MB 19.0 -> 18.1 (300
//     MB: waves by 4-11%), 32/8 at 80, 30 MB 8.4 against 11.3 (waves), FP8 at 80 25.3
//     against 25.8 (waves).
constexpr uint64_t kFullTokenBytes = 24ULL << 20;
constexpr uint64_t kNativeTokenChunks = 256, kNativeTokenBytes = 44ULL << 20, kNativeTokenMaxBytes = 186ULL << 20;

inline bool prefers_tokens(const WriteShape& s, uint64_t items) {
  if (items % 512 == 0 || (items >= 480 && items < 512)) return s.bytes > kFullTokenBytes;
  return !s.fp8 && items >= kNativeTokenChunks && s.bytes > kNativeTokenBytes && s.bytes <= kNativeTokenMaxBytes;
}

// The kernel of a call whose rows, strides and bases are whole 16-byte chunks.
// Both vector kernels number a token's items in 32 bits, and a launch takes fewer
// than 2^32 threads: past either the call goes to the other one, or to the
// general kernel.
inline WritePlan write_plan(const WriteShape& s) {
  constexpr uint64_t kMaxItems = 1ULL << 31, kThreads = 256, kMaxGroups = 0xffffffffULL / kThreads;
  const uint64_t items = s.query_heads * s.rot_items + s.kv_heads * (s.rot_items + s.tail_chunks + s.value_chunks);
  const WritePlan general{WriteKernel::kGeneral, false, 0, 0};
  if (items > kMaxItems) return general;
  const uint64_t wave_groups = (s.tokens * ((items + 63) / 64) + 3) / 4;
  const uint64_t max_splits = (items + kThreads - 1) / kThreads;
  uint64_t splits = (2048 + s.tokens - 1) / s.tokens;  // cover the chip
  if (splits > max_splits) splits = max_splits;
  const bool waves_fit = wave_groups <= kMaxGroups, tokens_fit = s.tokens * splits <= kMaxGroups;
  if (!waves_fit && !tokens_fit) return general;
  if ((prefers_tokens(s, items) && tokens_fit) || !waves_fit)
    return {WriteKernel::kTokens, false, static_cast<uint32_t>(s.tokens * splits), static_cast<uint32_t>(splits)};
  return {WriteKernel::kWaves, s.whole_lines && s.bytes > kNtBytes, static_cast<uint32_t>(wave_groups), 0};
}

}  // namespace loom_hip_rope
