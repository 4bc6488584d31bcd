// Plan of the long-chunk attention (dkv_attn_prompt.hip), shared by its kernels and by dkv_attend.
#pragma once
#include "dkv_common.h"

namespace dkv {

constexpr int PROMPT_WAVES = 8;                 // per workgroup, each 32 tokens of one Q head
constexpr int PROMPT_ROWS = 32 * PROMPT_WAVES;  // query rows of one KV head per workgroup
// Ranges come to one workgroup per CU, or to two (twice the partials to merge) when there are at least
// this many units of 256 rows x 64 keys per CU. One against two per CU, us per call (15 Q / 5 KV heads,
// bf16): 4 units per CU (1000 tokens past 640) 23.8 / 25.5, 15 (512 past 8128) 36.5 / 39.8, 16 (2048 past
// 1000) 40.2 / 39.4, 32 (1000 past 8128) 58.6 / 57.1, 67 (2048 past 8128) 106.4 / 100.1. At precision 0 two
// workgroups share a CU (48 KB of LDS each) and overlap each other's waits. At precision 1 (96 KB) only one
// fits and the second half runs after the first, which still evens out ranges of unequal length: 2048 past
// 1000 64.8 / 65.1, 900 past 500 (32 / 8 heads) 42.9 / 42.6, 8192 tokens 287 / 287, 2048 past 8128
// 193.8 / 189.5.
constexpr int PROMPT_TWO_FROM = 16;
constexpr int PROMPT_MIN_LEN = 2;  // units per range, at least (512 tokens past 1024: 4 units 20.5 us, 2 units 19.7)

__host__ __device__ inline int64_t prompt_image_bytes(int precision) { return precision ? 32768 : 16384; }

// Wave tasks (32 tokens of one Q head) of a KV head, token blocks first, and groups of PROMPT_WAVES.
__host__ __device__ inline int prompt_tasks(int G, int nq) { return G * ((nq + 31) / 32); }
__host__ __device__ inline int prompt_groups(int G, int nq) {
  return (prompt_tasks(G, nq) + PROMPT_WAVES - 1) / PROMPT_WAVES;
}
// Units of 64 keys (history, then the chunk) that some row of group i sees: up to its last token.
__host__ __device__ inline int prompt_group_units(int i, int G, int nq, int past) {
  const int last = PROMPT_WAVES * (i + 1) - 1, tasks = prompt_tasks(G, nq);
  const int tb = (last < tasks ? last : tasks - 1) / G;
  const int end = 32 * (tb + 1) < nq ? 32 * (tb + 1) : nq;
  return (past + end + DKV_TILE_TOKENS - 1) / DKV_TILE_TOKENS;
}
__host__ __device__ inline int prompt_splits(int units, int unit_len) { return (units + unit_len - 1) / unit_len; }

struct PromptPlan {
  int groups, units, unit_len, max_splits;
  int ranges;  // of one KV head, over all groups
  // Partials of groups with several ranges as fp16 O / sum (half_slot() order) rather than fp32 O: only
  // where the frame-chunk plan of the same call stores fp16 partials too. Longer chunks (about 24600 query
  // rows over all Q heads, 256 CUs) run one split there, whose O stays in fp32, and keep it so here; fp16
  // would take 2048 tokens past 1000 from 45.3 to 43.4 us and 8192 tokens from 186 to 180 (15 Q / 5 KV
  // heads, bf16) at an error against float64 of 2.682e-3 instead of 2.677e-3.
  bool half;
  int64_t image_bytes, part_o_bytes, part_ml_bytes;
  int64_t bytes() const { return image_bytes + part_o_bytes + part_ml_bytes; }
};

PromptPlan prompt_plan(const dkv_attn_args& a, int cus, bool half);
// ws: PromptPlan::bytes() bytes, 16-byte aligned.
int launch_attn_prompt(const dkv_attn_args& a, const PromptPlan& p, void* ws, hipStream_t s);

}  // namespace dkv
