// How a prefill call's work is cut: the kernel family, its workgroups and key
// ranges. Plain host code, so that the rules can be checked without a GPU.
#ifndef PDA_PREFILL_PLAN_H
#define PDA_PREFILL_PLAN_H

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace pda_prefill {

constexpr int kWaves = 4;  // waves per workgroup (D <= 256)
// Waves that split the head dim: at D = 512 the query fragments and output
// accumulators of 32 queries do not fit one wave's registers, so four waves
// share 32 queries, each holding 128 dims of Q and O; a D = 512 workgroup has
// eight waves (two such query blocks). (Split the same way, D = 256 runs two
// waves per SIMD instead of one but was 2-5% slower: the score exchange
// costs more than the second wave hides.)
constexpr int slices_for(int d) { return d > 256 ? 4 : 1; }
constexpr int waves_for(int d) { return d > 256 ? 2 * kWaves : kWaves; }
// Queries per workgroup: 32 per query block.
constexpr int queries_for(int d) { return 32 * waves_for(d) / slices_for(d); }
// Workgroups per CU that the key ranges are planned for. The pipelined
// kernels' launch bounds hold them to it (with one query block a wave).
constexpr int occupancy_for(int d) { return d == 64 ? 3 : d <= 128 ? 2 : 1; }

constexpr int kCus = 256;  // MI355X compute units
constexpr int kMaxSplits = 64;

// The kernel width serving a head dim: the head dim itself when a kernel
// has it, else the next wider one (GEN kernels; odd head dims the odd
// kernels); 0 for head dims the library does not serve (above 512).
inline int prefill_dim(int head_dim) {
  if (head_dim < 1 || head_dim > 512) return 0;
  for (int d : {64, 96, 128, 256, 512})
    if (head_dim <= d) return d;
  return 0;
}

// Key ranges per (query tile, head): 1 when the tiles and heads alone give
// every workgroup slot of the GPU (CUs x the kernel's occupancy) its work,
// else as many as fit the slots in one round: the ranges of a chunk over a
// long prefix are all alike, so a partly filled second round would cost a
// whole range's time. One exception: a causal chunk that fills at most one
// round and whose first query tile sees at most half the keys of its last
// (a prompt from position 0) takes 2 ranges, so that the halves of its
// longest tiles run beside its short ones. Each range holds at least 8 key
// tiles. `request` > 0 forces a count. The same for 16-bit and 8-bit K/V
// (`width`: prefill_dim's).
inline int prefill_splits(int start, int count, int q_heads, int width, int window, int request) {
  if (request > 0) return request < kMaxSplits ? request : kMaxSplits;
  const int queries = queries_for(width);
  const int64_t wgs = ((int64_t)count + queries - 1) / queries * q_heads;
  const int64_t slots = (int64_t)kCus * occupancy_for(width);
  const int keys = 32 * (width <= 128 ? 2 : 1);
  // Keys seen by the chunk's first and last query tiles.
  const int64_t cap = window > 0 ? (int64_t)window + queries : INT64_MAX;
  const int64_t first = std::min<int64_t>((int64_t)start + std::min(count, queries), cap);
  const int64_t span = std::min<int64_t>((int64_t)start + count, cap);
  const int64_t by_keys = (span + keys - 1) / keys / 8;
  if (wgs * 2 > slots) return wgs <= slots && 2 * first <= span && by_keys >= 2 ? 2 : 1;
  int64_t s = slots / wgs;
  if (s > by_keys) s = by_keys;
  if (s > kMaxSplits) s = kMaxSplits;
  return s < 1 ? 1 : (int)s;
}

inline size_t prefill_workspace(int splits, int count, int q_heads, int width) {
  if (splits <= 1) return 0;
  const size_t pairs = (size_t)count * q_heads;
  // Partial outputs, then the (max, sum) pairs, each 256-byte aligned.
  const size_t o_bytes = ((size_t)splits * pairs * width * 4 + 255) & ~(size_t)255;
  return o_bytes + (((size_t)splits * pairs * 8 + 255) & ~(size_t)255);
}

// The pipelined kernels serve 16-bit K/V at head dims 64, 96, 128 and 256.
inline bool pipelined(int head_dim, bool q8) {
  return !q8 && (head_dim == 64 || head_dim == 96 || head_dim == 128 || head_dim == 256);
}

// Query blocks per wave of the pipelined kernels. At D = 128 a wave may hold
// two (a workgroup of 256 queries alone on its CU, half the LDS reads per
// product). Taken where all of these hold (us, one / two blocks; 28/4 heads
// where none are named):
//  * 8192 keys or more, and ranges of 960 or more: fewer do not make up for the
//    longer way in and out (512 tokens at 0: 15 / 25; at 32256: 245 / 228; 8/8
//    heads, 256 at 8192 in ranges of 528: 33 / 42).
//  * No window shorter than the keys, however many those are: of a 256-query
//    workgroup's tiles each wave sees fewer (8192 at 0, window 1024: 146 / 226;
//    1024 at 8192, window 8192: 142 / 172).
//  * No softcap: a wave alone on its SIMD has nothing to run beside it (512 at
//    32256, softcap 50: 342 / 382).
//  * A CU's queries and keys are no more than with one block, counted in whole
//    workgroups: 1152 at 32256 is 280 workgroups of 256 queries in 2 ranges
//    and 504 of 128, 528 / 802; 640 at 32256 252 and 420, 313 / 299; 3000 at
//    32256 336 and 672, 1494 / 1681; 384 at 32256 336 and 504 (in 6 ranges),
//    183 / 233.
inline int query_blocks(int start, int count, int q_heads, int head_dim, int window, float softcap,
                        int splits) {
  if (head_dim != 128 || softcap > 0.0f) return 1;
  const int64_t keys = (int64_t)start + count;
  if (keys < 8192 || keys / splits < 960 || (window > 0 && window < keys)) return 1;
  const int64_t wgs1 = ((int64_t)count + 127) / 128 * q_heads * splits;
  const int64_t wgs2 = ((int64_t)count + 255) / 256 * q_heads * splits;
  return 2 * ((wgs2 + kCus - 1) / kCus) <= (wgs1 + kCus - 1) / kCus ? 2 : 1;
}

}  // namespace pda_prefill

#endif
