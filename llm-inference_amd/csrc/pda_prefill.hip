// Paged prefill attention for MI355X (gfx950), C-ABI in pda.h
// (pda_paged_prefill_attention).
//
// Reference: PrefillBatch.attend (python/instinct/batches.py:84-132): a chunk
// of one sequence's prompt, tokens at positions [start, start + count), whose
// keys and values were written to the paged arena first; query p attends
// keys [first(p), p] (causal, aligned to the newest key; with a window W,
// first(p) = p - W + 1), the score is softcapped when asked
// (portable.py:173-188), and the output is [count, q_heads * head_dim]. The
// CUDA engine's counterpart is its prefill attention kernel
// (cuda/kernels.cu:260-304).
//
// MI355X design (a flash-attention tile loop on the matrix cores):
//  * Workgroup = 4 waves = one query head and 128 queries (32 per wave).
//    Keys are streamed in tiles of 64 (32 at D >= 256) through LDS, K and V
//    rows gathered from the pages of the sequence's table (either arena
//    layout). The LDS holds two tiles: the loads of tile t + 1 are issued
//    into registers before the math of tile t and stored to the other half
//    after it, one barrier per tile.
//  * D = 512: eight waves, two blocks of 32 queries; the four waves of a
//    block split the head dim (128 dims of Q and O each) and sum their
//    partial scores through LDS, so every wave of the block holds the same
//    scores and probabilities (see slices_for).
//  * Each wave computes S^T = K Q^T for its 32 queries with
//    v_mfma_f32_32x32x16_f16 (D / 16 instructions per key tile), Q held in
//    registers. In that product's accumulator a lane holds 16 keys of one
//    query; 8 of them per 16-key step are the B operand of the next product
//    O^T += V^T P^T (D / 32 x 2 instructions per tile), so the probabilities
//    never leave registers. The contraction pairs A and B by k-slot, so the
//    V^T operand takes the keys in the order the accumulator holds them:
//    two ds_read_b64_tr_b16 per operand give a lane four consecutive keys of
//    one dimension each.
//  * Online softmax per query in the log2 domain with a lazy running max
//    (rescale only when a score passes the max by 2^8), fp16 probabilities
//    into the matrix core, fp32 accumulation, normalised fp16 output. Masks
//    (causality, the window, unusable pages) are evaluated only on the tiles
//    that need them; a wave skips the math of tiles none of its queries see.
//  * Work order: the query tiles with the most keys start first, and the G
//    query heads that read one kv head's tile are dispatched back to back to
//    one XCD (workgroups go round robin over the 8 XCDs), so the L2 of that
//    XCD serves the tile to all of them.
//  * 16-bit K/V at D <= 256 runs the pipelined form of this loop
//    (prefill_pipe_body); 8-bit K/V, D = 512 and the generic head dims run
//    the form described so far (prefill_body).
//  * LDS rows are padded so that the 16 lanes of a 16-byte K read, and the
//    four rows of a transposed V read, fall on distinct banks.
//  * Other even head dims up to 512 (GEN) run the kernel of the next of
//    those widths: rows are gathered as element pairs (the row length is a
//    multiple of 4 bytes only), the pairs past the head dim are zero in Q, K
//    and V, and only the real dims are written. Odd head dims (ODD) do the
//    same one element at a time (paged_prefill_odd_kernel).

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "pda.h"
#include "pda_internal.h"
#include "pda_prefill_plan.h"

namespace {

using namespace pda_prefill;

typedef _Float16 f16;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kSlack = 8.0f;
constexpr int kXcds = 8;

struct PrefillParams {
  const f16* q;        // [count, hq, D]
  const void* k;       // arena: fp16, or int8 with per-(row, kv head) fp16 scales
  const void* v;
  const f16* kscale;   // 8-bit only: scale arenas
  const f16* vscale;
  int64_t scale_page;  // scale elements between pages,
  int32_t scale_head;  //   between kv heads of one page,
  int32_t scale_row;   //   between rows of one page and kv head
  const int32_t* table;
  const int32_t* images;  // [num_images, 2] image spans [begin, end) of positions
  int32_t num_images;
  f16* out;            // [count, hq, D]
  float* part_o;       // [splits, count, hq, D] unnormalised partial outputs (splits > 1)
  float2* part_ml;     // [splits, count, hq] (running max, sum) of each partial
  int64_t arena_pages;
  int64_t page_elems;  // elements between pages of the arena
  int32_t head_elems;  // between kv heads of one page
  int32_t row_elems;   // between rows of one page and kv head
  int32_t table_len;
  int32_t start;
  int32_t count;
  int32_t tiles;       // query tiles = ceil(count / queries per workgroup)
  int32_t splits;      // key ranges per (query tile, head)
  int32_t page_step;   // keys per tile / page_size when that divides, else 0
  int32_t hq;
  int32_t hkv;
  int32_t head_dim;    // row length of Q, K, V and the output (GEN: below D)
  int32_t page_size;
  int32_t window;
  float scale_log2;
  float softcap;
  float cap_in;   // 2 log2(e) scale / softcap
  float cap_out;  // softcap log2(e)
};

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ f16x4 read_tr(const f16* p) {
  return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p));
}

// One 32x32x16 matrix-core step on 16-bit operands held as fp16 bit patterns:
// fp16, or bf16 (BF) for bf16 models.
template <bool BF>
__device__ __forceinline__ f32x16 mfma16(const f16x8& a, const f16x8& b, const f32x16& c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// f32 -> the 16-bit element type (to nearest even), as an fp16 bit pattern.
template <bool BF>
__device__ __forceinline__ f16 round16(float x) {
  if constexpr (BF)
    return __builtin_bit_cast(f16, (bf16)x);
  else
    return (f16)x;
}

// Keys per tile: 64 (two 32-key blocks) where the registers allow it.
template <int D>
constexpr int blocks_per_tile() { return D <= 128 ? 2 : 1; }

// LDS byte address of a shared object.
__device__ __forceinline__ uint32_t lds_address(const void* at) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)at;
}

// 16 bytes per lane from global memory straight into LDS: lane i's, from src +
// kOff bytes, to dst + kOff + kPlus + 16 i (dst: wave-uniform; the
// instruction adds its offset to both addresses). The caller waits
// (wait_vmem) before the barrier that publishes them.
template <int kOff, int kPlus>
__device__ __forceinline__ void copy_to_lds(const void* src, uint32_t dst) {
  asm volatile("s_add_u32 m0, %0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:%3" ::"s"(
                   dst),
               "v"(src), "n"(kPlus), "n"(kOff)
               : "memory", "m0", "scc");
}

// The same product added to c; kAcc: c in accumulator registers, which the
// compiler would otherwise copy to vector registers and back. The compiler
// neither knows what such an instruction still has in flight nor that its
// operands need two wait states after a VALU instruction wrote them. So c is
// only read by further products until outputs_done, the weights' sum or
// operands_done comes between their last write and the first product that reads
// them, and the fragments come from LDS.
// (Two wait states in front of every product instead: 565 against 556 us for
// 4096 tokens at 8192, 28/4 heads of 128.) A test reads the distances from the
// built kernels.
template <bool BF, bool kAcc>
__device__ __forceinline__ void mfma_to(const f16x8& a, const f16x8& b, f32x16& c) {
  if constexpr (!kAcc)
    c = mfma16<BF>(a, b, c);
  else if constexpr (BF)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// f(0), f(1), ... with compile-time arguments.
template <class F, int... kI>
__device__ __forceinline__ void each(F& f, std::integer_sequence<int, kI...>) {
  (f(std::integral_constant<int, kI>{}), ...);
}

// Until at most kLeft of the wave's loads and copies are under way.
template <int kLeft>
__device__ __forceinline__ void wait_vmem() {
  static_assert(kLeft < 64, "the count has six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (kLeft & 15) | (kLeft >> 4) << 14);
}

// Output of one query: normalised, or the unnormalised partial of a key range.
template <int D, bool BF, bool GEN, bool ODD>
__device__ __forceinline__ void finish(const PrefillParams& p,
                                       const f32x16 (&o)[D / slices_for(D) / 32], float m, float l,
                                       int qi, int h, int split, int hh, int sl, bool q_live) {
  constexpr int kDW = D / slices_for(D);
  if (!q_live) return;
  l += __shfl_xor(l, 32);
  if (p.splits > 1) {
    // Unnormalised partial and its (max, sum) for the merge; an empty or
    // fully masked range leaves m = -inf, l = 0 and zeros.
    const int64_t at = ((int64_t)split * p.count + qi) * p.hq + h;  // partials are D wide
    float* dst = p.part_o + at * D + sl * kDW;
#pragma unroll
    for (int b = 0; b < kDW / 32; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(dst + 32 * b + 8 * g + 4 * hh) =
            make_float4(o[b][4 * g], o[b][4 * g + 1], o[b][4 * g + 2], o[b][4 * g + 3]);
    if (hh == 0 && sl == 0) p.part_ml[at] = make_float2(m, l);
    return;
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  if constexpr (ODD) {
    // Rows of an odd number of elements: one element per store.
    const int hd = p.head_dim;
    f16* dst = p.out + ((int64_t)qi * p.hq + h) * hd;
#pragma unroll
    for (int b = 0; b < kDW / 32; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int d = sl * kDW + 32 * b + 8 * (v / 4) + 4 * hh + v % 4;
        if (d < hd) dst[d] = round16<BF>(o[b][v] * inv);
      }
    return;
  }
  if constexpr (GEN) {
    // Rows of head_dim elements: element pairs, the real dims only.
    const int hd = p.head_dim;
    f16* dst = p.out + ((int64_t)qi * p.hq + h) * hd;
#pragma unroll
    for (int b = 0; b < kDW / 32; ++b) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = sl * kDW + 32 * b + 8 * g + 4 * hh;
        const f16x2 y0 = {round16<BF>(o[b][4 * g] * inv), round16<BF>(o[b][4 * g + 1] * inv)};
        const f16x2 y1 = {round16<BF>(o[b][4 * g + 2] * inv),
                          round16<BF>(o[b][4 * g + 3] * inv)};
        if (d < hd) *reinterpret_cast<f16x2*>(dst + d) = y0;
        if (d + 2 < hd) *reinterpret_cast<f16x2*>(dst + d + 2) = y1;
      }
    }
    return;
  }
  f16* dst = p.out + ((int64_t)qi * p.hq + h) * D + sl * kDW;
  // O^T rows: element 32 b + 8 (v / 4) + 4 hh + v % 4 of query n (of the slice).
#pragma unroll
  for (int b = 0; b < kDW / 32; ++b) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f16x4 y;
#pragma unroll
      for (int t = 0; t < 4; ++t) y[t] = round16<BF>(o[b][4 * g + t] * inv);
      *reinterpret_cast<f16x4*>(dst + 32 * b + 8 * g + 4 * hh) = y;
    }
  }
}

// Q8: the arena holds int8 rows and fp16 scales; the gather dequantizes each
// row to fp16(int8 x scale) on its way into LDS, the values the reference's
// 8-bit gather hands to attention (paged_kv.py:285-292), and the rest of the
// kernel is the fp16 one.
// BF: queries, K/V and output in bf16 (bf16 models); every 16-bit value is
// moved as raw bits and only the matrix-core steps, the probabilities and the
// output rounding differ.
// GEN: head dim p.head_dim below D; D-wide tiles, zero past it.
// ODD (with GEN): an odd head dim; rows are 2-byte aligned (1-byte at 8
// bits), so the queries, the gather and the output move single elements.
template <int D, bool Q8, bool BF, bool GEN, bool ODD>
__device__ __forceinline__ void prefill_body(const PrefillParams p) {
  static_assert(!ODD || GEN, "odd head dims run the generic kernels");
  static_assert(!(Q8 && BF), "8-bit K/V dequantizes to fp16");
  constexpr int KB = blocks_per_tile<D>();  // 32-key blocks per tile
  constexpr int kKeys = 32 * KB;            // keys per tile
  constexpr int kSlices = slices_for(D);    // waves sharing one query block
  constexpr int kDW = D / kSlices;          // head dims per wave
  constexpr int kQ = queries_for(D);        // queries per workgroup
  constexpr int kW = waves_for(D);          // waves per workgroup
  constexpr int kT = 64 * kW;               // threads per workgroup
  // D = 512: one V tile in LDS (the partials take the second one's room); V
  // of tile t + 1 is stored at the top of iteration t + 1, after every wave
  // is done with V of tile t.
  constexpr bool kOneV = D > 256;
  constexpr int kGroups = 4 * KB;             // float4 groups of a lane's scores
  constexpr int kPer = kGroups / kSlices;     // groups each slice sums
  static_assert(kPer * kSlices == kGroups, "score groups per slice");
  constexpr int kKRow = D + 8;    // K row in LDS (halves): 16-lane 16-byte reads hit distinct banks
  // V row: the 4 rows of a transposed read hit distinct banks (a row is 16
  // banks past the previous one modulo 64).
  constexpr int kVRow = D % 64 == 32 ? D + 64 : D + 32;
  constexpr int kTpk = kT / kKeys;                     // gather threads per key
  constexpr int kPieces = D / 8 / kTpk;                // 16-byte pieces per thread and tile
  constexpr int kKeysPerWave = 64 / kTpk;              // keys one wave gathers
  static_assert(kPieces >= 1 && kPieces * kTpk * 8 == D, "tile shape");
  typedef typename std::conditional<kKeysPerWave == 16, uint16_t, uint8_t>::type okbits;
  typedef typename std::conditional<KB == 2, uint64_t, uint32_t>::type okword;
  static_assert(kKeysPerWave * kW == kKeys, "usable-key bits");
  __shared__ __align__(16) f16 s_k[2][kKeys * kKRow];
  __shared__ __align__(16) f16 s_v[kOneV ? 1 : 2][kKeys * kVRow];
  __shared__ __align__(8) okbits s_ok[2][kW];  // usable-key bits of the tile
  // D = 512: each wave's partial scores (over its dims), and the sums of
  // the query block's partials, kPer groups per wave.
  __shared__ __align__(16) float4 s_x[kSlices > 1 ? kW * kGroups : 1][64];
  __shared__ __align__(16) float4 s_y[kSlices > 1 ? kW * kPer : 1][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int n = lane & 31;   // query column of this lane
  const int hh = lane >> 5;  // which half of the key rows this lane holds
  const int qb = w / kSlices;       // this wave's 32-query block
  const int sl = w - qb * kSlices;  // and its head dims: [sl kDW, (sl + 1) kDW)

  // Work item. Logical order: query tiles from the last (most keys) to the
  // first, then key range, then kv head, then the G query heads of that kv
  // head. Workgroup ids go round robin over the XCDs; whole runs of G (the
  // workgroups reading the same K/V tiles) go to one XCD.
  const int G = p.hq / p.hkv;
  int item = blockIdx.x;
  const int runs = p.tiles * p.splits * p.hkv;
  const int full = runs / kXcds * kXcds;
  if (item < full * G) {
    const int x = item % kXcds, j = item / kXcds;
    item = ((j / G) * kXcds + x) * G + j % G;
  }
  const int run = item / G;
  const int h = (run % p.hkv) * G + (item - run * G);
  const int kvh = run % p.hkv;
  const int split = (run / p.hkv) % p.splits;
  const int tile = p.tiles - 1 - run / p.hkv / p.splits;

  const int q0 = tile * kQ;
  const int q1 = min(q0 + kQ, p.count);
  const int qi = q0 + 32 * qb + n;  // this lane's query (may be past count)
  const bool q_live = qi < p.count;
  const int qpos = p.start + qi;
  const int wq0 = q0 + 32 * qb;
  const bool wave_live = wq0 < p.count;
  const int wfirst = p.start + wq0;
  const int wlast = p.start + min(wq0 + 31, p.count - 1);

  // Query fragments (B operand of S^T = K Q^T): dims 16 c + 8 hh .. + 7 of
  // the wave's slice.
  f16x8 qf[kDW / 16];
  if constexpr (GEN) {
    // Element pairs, clamped into the row; zero past the head dim.
    const int hd = p.head_dim;
    const f16* qp = p.q + ((int64_t)(q_live ? qi : 0) * p.hq + h) * hd;
#pragma unroll
    for (int c = 0; c < kDW / 16; ++c) {
      i32x4 x;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = sl * kDW + 16 * c + 8 * hh + 2 * j;
        if constexpr (ODD) {
          const uint16_t* q16 = reinterpret_cast<const uint16_t*>(qp);
          const uint32_t lo = q16[min(d, hd - 1)], hi = q16[min(d + 1, hd - 1)];
          x[j] = (int)((q_live && d < hd ? lo : 0u) | (q_live && d + 1 < hd ? hi : 0u) << 16);
        } else {
          const int y = *reinterpret_cast<const int*>(qp + min(d, hd - 2));
          x[j] = q_live && d < hd ? y : 0;
        }
      }
      qf[c] = __builtin_bit_cast(f16x8, x);
    }
  } else {
    const f16* qp = p.q + ((int64_t)(q_live ? qi : 0) * p.hq + h) * D + sl * kDW + 8 * hh;
#pragma unroll
    for (int c = 0; c < kDW / 16; ++c) {
      const f16x8 x = *reinterpret_cast<const f16x8*>(qp + 16 * c);
      qf[c] = q_live ? x : f16x8{};
    }
  }

  f32x16 o[kDW / 32];
#pragma unroll
  for (int b = 0; b < kDW / 32; ++b) o[b] = f32x16{};
  float m = -INFINITY, l = 0.0f;

  // Keys this workgroup needs: from the first visible key of its first query
  // (rounded down to a tile) to its last query.
  int last = p.start + q1 - 1;
  int kfirst = p.window > 0 ? max(0, p.start + q0 - p.window + 1) : 0;
  // Image spans (batches.py:107-118): a query inside one also sees the
  // span's later keys, whatever the window. The lane keeps its query's span
  // [img_lo, img_hi); the workgroup and each wave extend their key ranges to
  // the spans their queries touch (keys stop at the chunk's end).
  int img_lo = 0, img_hi = 0, wave_last = wlast;
  bool wave_img = false;
  for (int i = 0; i < p.num_images; ++i) {
    const int a = p.images[2 * i], b = min(p.images[2 * i + 1], p.start + p.count);
    if (a >= b) continue;
    if (qpos >= a && qpos < b) img_lo = a, img_hi = b;
    if (a <= last && b > p.start + q0) {
      last = max(last, b - 1);
      kfirst = min(kfirst, a);
    }
    if (wave_live && a <= wlast && b > wfirst) {
      wave_last = max(wave_last, b - 1);
      wave_img = true;
    }
  }
  const int kbase = kfirst / kKeys * kKeys;
  const int ntile = (last - kbase) / kKeys + 1;
  // This workgroup's key range: tiles [t_begin, t_end) of the ntile.
  const int t_begin = (int)((int64_t)ntile * split / p.splits);
  const int t_end = (int)((int64_t)ntile * (split + 1) / p.splits);

  // Gather: thread tid moves key tid / kTpk of a tile, 16-byte pieces
  // tid % kTpk + kTpk i (consecutive lanes read consecutive pieces of a row).
  // The page of that key is looked up two tiles ahead (lookup), its rows
  // loaded one tile ahead (fetch), so neither load is waited for in the
  // iteration that issues it.
  const int gk = tid / kTpk;
  const int gp = tid % kTpk;
  // Staged rows: 16 bytes (8 fp16) per piece, or 8 bytes (8 int8) and the
  // key's two scales.
  typedef typename std::conditional<Q8, uint2, f16x8>::type piece_t;
  piece_t kr[kPieces], vr[kPieces];
  f16 ksc = (f16)0.0f, vsc = (f16)0.0f;
  bool gok = false;
  // The table read is unconditional (index clamped, table_len >= 1) and its
  // range check a separate flag, so the loaded page id is never merged with
  // another value, which would wait for the load. The cursor (key kp, page
  // index pi, row r in the page) advances one tile per lookup; when the page
  // size divides the tile, r stays fixed and pi steps by a constant.
  int kp = kbase + t_begin * kKeys + gk;
  int pi = kp / p.page_size;
  int r = kp - pi * p.page_size;
  auto lookup = [&](int& page, bool& in, int& row_off, int& scale_off) {
    in = kp <= last && pi < p.table_len;
    page = p.table[min(pi, p.table_len - 1)];
    row_off = r * p.row_elems + kvh * p.head_elems + (GEN ? 0 : gp * 8);
    scale_off = r * p.scale_row + kvh * p.scale_head;
    kp += kKeys;
    if (p.page_step > 0) {
      pi += p.page_step;
    } else {
      pi = kp / p.page_size;
      r = kp - pi * p.page_size;
    }
  };
  // GEN: dim of element pair j of piece i, clamped into the row (pairs past
  // the head dim reload the last pair; trim zeroes them).
  auto pair_dim = [&](int i, int j) { return min(8 * (gp + kTpk * i) + 2 * j, p.head_dim - 2); };
  // ODD: dim of element e of piece i, clamped into the row (elements past
  // the head dim reload the last one; trim zeroes them).
  auto elem_dim = [&](int i, int e) { return min(8 * (gp + kTpk * i) + e, p.head_dim - 1); };
  auto fetch = [&](int page, bool in, int row_off, int scale_off) {
    gok = in && page >= 0 && page < p.arena_pages;
    const uint32_t pg = (uint32_t)(gok ? page : 0);
    const uint64_t at = (uint64_t)pg * (uint64_t)p.page_elems + row_off;
    if constexpr (ODD && Q8) {
      const uint8_t* kb = static_cast<const uint8_t*>(p.k) + at;
      const uint8_t* vb = static_cast<const uint8_t*>(p.v) + at;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        uint32_t kw[2] = {0u, 0u}, vw[2] = {0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          kw[e / 4] |= (uint32_t)kb[elem_dim(i, e)] << (8 * (e % 4));
          vw[e / 4] |= (uint32_t)vb[elem_dim(i, e)] << (8 * (e % 4));
        }
        kr[i] = uint2{kw[0], kw[1]};
        vr[i] = uint2{vw[0], vw[1]};
      }
      const uint64_t sat = (uint64_t)pg * (uint64_t)p.scale_page + scale_off;
      ksc = p.kscale[sat];
      vsc = p.vscale[sat];
    } else if constexpr (ODD) {
      const uint16_t* kb = reinterpret_cast<const uint16_t*>(static_cast<const f16*>(p.k) + at);
      const uint16_t* vb = reinterpret_cast<const uint16_t*>(static_cast<const f16*>(p.v) + at);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        i32x4 kw, vw;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kw[j] = (int)((uint32_t)kb[elem_dim(i, 2 * j)] | (uint32_t)kb[elem_dim(i, 2 * j + 1)] << 16);
          vw[j] = (int)((uint32_t)vb[elem_dim(i, 2 * j)] | (uint32_t)vb[elem_dim(i, 2 * j + 1)] << 16);
        }
        kr[i] = __builtin_bit_cast(f16x8, kw);
        vr[i] = __builtin_bit_cast(f16x8, vw);
      }
    } else if constexpr (GEN && Q8) {
      const uint8_t* kb = static_cast<const uint8_t*>(p.k) + at;
      const uint8_t* vb = static_cast<const uint8_t*>(p.v) + at;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        uint32_t kw[4], vw[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kw[j] = *reinterpret_cast<const uint16_t*>(kb + pair_dim(i, j));
          vw[j] = *reinterpret_cast<const uint16_t*>(vb + pair_dim(i, j));
        }
        kr[i] = uint2{kw[0] | kw[1] << 16, kw[2] | kw[3] << 16};
        vr[i] = uint2{vw[0] | vw[1] << 16, vw[2] | vw[3] << 16};
      }
      const uint64_t sat = (uint64_t)pg * (uint64_t)p.scale_page + scale_off;
      ksc = p.kscale[sat];
      vsc = p.vscale[sat];
    } else if constexpr (GEN) {
      const f16* kb = static_cast<const f16*>(p.k) + at;
      const f16* vb = static_cast<const f16*>(p.v) + at;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        i32x4 kw, vw;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kw[j] = *reinterpret_cast<const int*>(kb + pair_dim(i, j));
          vw[j] = *reinterpret_cast<const int*>(vb + pair_dim(i, j));
        }
        kr[i] = __builtin_bit_cast(f16x8, kw);
        vr[i] = __builtin_bit_cast(f16x8, vw);
      }
    } else if constexpr (Q8) {
      const uint8_t* kb = static_cast<const uint8_t*>(p.k) + at;
      const uint8_t* vb = static_cast<const uint8_t*>(p.v) + at;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        kr[i] = *reinterpret_cast<const uint2*>(kb + 8 * kTpk * i);
        vr[i] = *reinterpret_cast<const uint2*>(vb + 8 * kTpk * i);
      }
      const uint64_t sat = (uint64_t)pg * (uint64_t)p.scale_page + scale_off;
      ksc = p.kscale[sat];
      vsc = p.vscale[sat];
    } else {
      const f16* kb = static_cast<const f16*>(p.k) + at;
      const f16* vb = static_cast<const f16*>(p.v) + at;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        kr[i] = *reinterpret_cast<const f16x8*>(kb + 8 * kTpk * i);
        vr[i] = *reinterpret_cast<const f16x8*>(vb + 8 * kTpk * i);
      }
    }
  };
  // A staged piece as 8 fp16 values (8-bit: fp16(int8 x scale), one
  // rounding of the exact product).
  auto as_f16 = [&](const piece_t& x, f16 scale, int i) -> f16x8 {
    f16x8 y;
    if constexpr (Q8) {
      const f16x2 s2 = {scale, scale};
      const uint32_t lo = x.x ^ 0x80808080u, hi = x.y ^ 0x80808080u;
      const f16x2 e0 = pda_internal::bytes_to_f16x2(lo, 0x04010400u) * s2;
      const f16x2 e1 = pda_internal::bytes_to_f16x2(lo, 0x04030402u) * s2;
      const f16x2 e2 = pda_internal::bytes_to_f16x2(hi, 0x04010400u) * s2;
      const f16x2 e3 = pda_internal::bytes_to_f16x2(hi, 0x04030402u) * s2;
      y = f16x8{e0[0], e0[1], e1[0], e1[1], e2[0], e2[1], e3[0], e3[1]};
    } else {
      (void)scale;
      y = x;
    }
    if constexpr (ODD) {  // zero the elements past the head dim
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = 8 * (gp + kTpk * i) + e < p.head_dim ? y[e] : (f16)0.0f;
    } else if constexpr (GEN) {  // zero the pairs past the head dim
      i32x4 w4 = __builtin_bit_cast(i32x4, y);
#pragma unroll
      for (int j = 0; j < 4; ++j) w4[j] = 8 * (gp + kTpk * i) + 2 * j < p.head_dim ? w4[j] : 0;
      y = __builtin_bit_cast(f16x8, w4);
    }
    return y;
  };
  auto stash_v = [&](int vbuf) {
    f16* vd = s_v[vbuf] + gk * kVRow + gp * 8;
    if (__ballot(gok) == ~0ull) {
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        *reinterpret_cast<f16x8*>(vd + 8 * kTpk * i) = as_f16(vr[i], vsc, i);
    } else {
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        *reinterpret_cast<f16x8*>(vd + 8 * kTpk * i) = gok ? as_f16(vr[i], vsc, i) : f16x8{};
    }
  };
  auto stash = [&](int buf) {
    // Unusable keys are stored as zeros (their weight is 0; zero V keeps
    // 0 * V finite whatever the arena holds there).
    f16* kd = s_k[buf] + gk * kKRow + gp * 8;
    const uint64_t bits = __ballot(gok);
    if constexpr (kOneV) {
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        *reinterpret_cast<f16x8*>(kd + 8 * kTpk * i) = gok ? as_f16(kr[i], ksc, i) : f16x8{};
    } else {
      f16* vd = s_v[buf] + gk * kVRow + gp * 8;
      if (bits == ~0ull) {  // wave-uniform: the usual case stores without selects
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
          *reinterpret_cast<f16x8*>(kd + 8 * kTpk * i) = as_f16(kr[i], ksc, i);
          *reinterpret_cast<f16x8*>(vd + 8 * kTpk * i) = as_f16(vr[i], vsc, i);
        }
      } else {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
          *reinterpret_cast<f16x8*>(kd + 8 * kTpk * i) = gok ? as_f16(kr[i], ksc, i) : f16x8{};
          *reinterpret_cast<f16x8*>(vd + 8 * kTpk * i) = gok ? as_f16(vr[i], vsc, i) : f16x8{};
        }
      }
    }
    if (lane == 0) {
      uint32_t mk = 0;
#pragma unroll
      for (int j = 0; j < kKeysPerWave; ++j) mk |= (uint32_t)((bits >> (kTpk * j)) & 1) << j;
      s_ok[buf][w] = (okbits)mk;
    }
  };

  // Lane part of the transposed V read: group g = lane / 16 reads dims
  // 16 (g % 2) + 4 (s % 4) of key 4 (g / 2) + s / 4, s = lane % 16.
  const int g16 = lane >> 4, s16 = lane & 15;
  const int v_lane =
      (4 * (g16 >> 1) + (s16 >> 2)) * kVRow + 16 * (g16 & 1) + 4 * (s16 & 3) + sl * kDW;
  const int k_lane = n * kKRow + 8 * hh + sl * kDW;
  const int qlo = p.window > 0 ? qpos - p.window : INT32_MIN;  // keys > qlo are in the window
  const float c = p.softcap <= 0.0f && p.scale_log2 > 0.0f ? p.scale_log2 : 1.0f;

  int page0, r0, s0, page1, r1, s1;
  bool in0, in1;
  page0 = page1 = r0 = r1 = s0 = s1 = 0;
  in0 = in1 = false;
  // Only tiles of the range are looked up: the key after them may be 2^31,
  // past what the cursor holds.
  if (t_begin < t_end) lookup(page0, in0, r0, s0);
  if (t_begin + 1 < t_end) lookup(page1, in1, r1, s1);
  fetch(page0, in0, r0, s0);
  stash(0);
  if constexpr (kOneV) stash_v(0);
  __syncthreads();
  for (int t = t_begin; t < t_end; ++t) {
    const int buf = (t - t_begin) & 1;
    const int k0 = kbase + t * kKeys;
    const bool more = t + 1 < t_end;
    // V of this tile, staged in the previous iteration (every wave finished
    // that tile's V at its closing barrier; the score exchange's barrier
    // below publishes these stores before any wave reads them).
    if constexpr (kOneV)
      if (t > t_begin) stash_v(0);
    if (more) fetch(page1, in1, r1, s1);
    if (t + 2 < t_end) lookup(page1, in1, r1, s1);

    const bool work = wave_live && k0 <= wave_last &&
                      (p.window <= 0 || wave_img || k0 + kKeys - 1 > wfirst - p.window);
    const f16* sk = s_k[buf];
    const f16* sv = s_v[kOneV ? 0 : buf];
    // S^T per 32-key block kb: lane holds keys 32 kb + 8 (v / 4) + 4 hh + v % 4.
    f32x16 s[KB];
    if (work) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        f16x8 ka[kDW / 16];
#pragma unroll
        for (int c = 0; c < kDW / 16; ++c)
          ka[c] = *reinterpret_cast<const f16x8*>(sk + k_lane + 32 * kb * kKRow + 16 * c);
        s[kb] = f32x16{};
        // Raised wave priority while this wave issues matrix-core work: the
        // SIMD's other wave, in its softmax, then yields the issue slots and
        // the matrix core is fed while the VALU phase of one wave overlaps
        // the MFMA phase of the other (2-4% on config 2's chunks).
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int c = 0; c < kDW / 16; ++c)
          s[kb] = mfma16<BF>(ka[c], qf[c], s[kb]);
        __builtin_amdgcn_s_setprio(0);
      }
    }
    if constexpr (kSlices > 1) {
      // Sum the slices' partial scores in slice order, so that every wave of
      // the block holds the same scores, maximum, sum and probabilities.
      // `work` is the same for all of them (it depends on the queries only).
      // Reduce-scatter then gather: 12 adds per lane instead of 48. Slice sl
      // sums groups [sl kPer, (sl + 1) kPer) of the block's partials in
      // slice order; then every wave reads all the sums.
      if (work) {
#pragma unroll
        for (int i = 0; i < kGroups; ++i)
          s_x[w * kGroups + i][lane] = make_float4(s[i / 4][4 * (i % 4)], s[i / 4][4 * (i % 4) + 1],
                                                   s[i / 4][4 * (i % 4) + 2],
                                                   s[i / 4][4 * (i % 4) + 3]);
      }
      __syncthreads();
      if (work) {
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
          const int i = sl * kPer + r;
          float4 acc = s_x[qb * kSlices * kGroups + i][lane];
#pragma unroll
          for (int j = 1; j < kSlices; ++j) {
            const float4 y = s_x[(qb * kSlices + j) * kGroups + i][lane];
            acc.x += y.x;
            acc.y += y.y;
            acc.z += y.z;
            acc.w += y.w;
          }
          s_y[w * kPer + r][lane] = acc;
        }
      }
      __syncthreads();
      if (work) {
#pragma unroll
        for (int i = 0; i < kGroups; ++i) {
          const float4 acc = s_y[(qb * kSlices + i / kPer) * kPer + i % kPer][lane];
          s[i / 4][4 * (i % 4)] = acc.x;
          s[i / 4][4 * (i % 4) + 1] = acc.y;
          s[i / 4][4 * (i % 4) + 2] = acc.z;
          s[i / 4][4 * (i % 4) + 3] = acc.w;
        }
      }
    }
    if (work) {
      okword okm;
      if constexpr (kKeysPerWave == 4) {
        // Eight waves of four keys: one nibble per byte, packed to 32 bits.
        uint64_t x = *reinterpret_cast<const uint64_t*>(s_ok[buf]) & 0x0F0F0F0F0F0F0F0Full;
        x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
        x = (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
        okm = (okword)(x | (x >> 16));
      } else {
        okm = *reinterpret_cast<const okword*>(s_ok[buf]);
      }
      const bool edge = k0 + kKeys - 1 > wfirst || okm != (okword)~(okword)0 ||
                        (p.window > 0 && k0 <= wlast - p.window);
      // x = score in units that exp2(x * c - m) turns into the weight: the
      // raw q.k with c = scale log2(e) when that is positive (the max of raw
      // scores gives the max of the scaled ones), else the scaled or
      // softcapped score in log2 units with c = 1.
      float x[16 * KB];
      if (p.softcap > 0.0f) {
#pragma unroll
        for (int v = 0; v < 16 * KB; ++v) {
          const float e = __builtin_amdgcn_exp2f(s[v / 16][v % 16] * p.cap_in);
          x[v] = (1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f)) * p.cap_out;
        }
      } else if (p.scale_log2 > 0.0f) {
#pragma unroll
        for (int v = 0; v < 16 * KB; ++v) x[v] = s[v / 16][v % 16];
      } else {
#pragma unroll
        for (int v = 0; v < 16 * KB; ++v) x[v] = s[v / 16][v % 16] * p.scale_log2;
      }
      if (edge) {
        // Key k0 + key is visible to this lane's query when usable,
        // <= qpos and > qlo.
        const okword okl = okm >> (4 * hh);
        const int hi = qpos - k0 - 4 * hh;  // largest visible key offset
        const int lo = qlo == INT32_MIN ? INT32_MIN : qlo - k0 - 4 * hh;
        const int ilo = img_lo - k0 - 4 * hh, ihi = img_hi - k0 - 4 * hh;  // image span
        // Bitwise operators, not && / ||: the short-circuit form compiled to
        // nested exec-mask branches, one of which dropped the restore of the
        // score for lanes visible through the image span only.
#pragma unroll
        for (int v = 0; v < 16 * KB; ++v) {
          const int key = 32 * (v / 16) + 8 * ((v % 16) / 4) + (v % 4);  // minus 4 hh
          const bool usable_key = ((okl >> key) & 1u) != 0;
          const bool causal = (key <= hi) & (key > lo);
          const bool image = (key >= ilo) & (key < ihi);
          x[v] = usable_key & (causal | image) ? x[v] : -INFINITY;
        }
      }
      // Lazy running max: rescale only when a score passes it by 2^8.
      // Returns whether this lane's max moved.
      auto lazy_max = [&]() -> bool {
        float top = x[0];
#pragma unroll
        for (int v = 1; v < 16 * KB; ++v) top = fmaxf(top, x[v]);
        top = fmaxf(top, __shfl_xor(top, 32)) * c;  // with the other half of this query's keys
        if (top > m + kSlack) {
          const float f = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - top);
          m = top;
          l *= f;
#pragma unroll
          for (int b = 0; b < kDW / 32; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[b][v] *= f;
          return true;
        }
        return false;
      };
      // P^T as the B operand: 16-key step ks holds values 8 ks .. 8 ks + 7,
      // i.e. keys 16 ks + 8 (t / 4) + 4 hh + t % 4. O^T += V^T P^T, A
      // operand of step ks for rows 32 b ..: keys 16 ks + 4 hh + 0..3 (first
      // read) and + 8 (second read).
      f16x8 pb[2 * KB];
      // The weights exp2(x c - mu) as 16-bit B operands, summed into `sum`.
      auto weights = [&](float mu, float& sum) {
#pragma unroll
        for (int ks = 0; ks < 2 * KB; ++ks) {
#pragma unroll
          for (int t2 = 0; t2 < 4; ++t2) {
            if constexpr (BF) {
              const bf16x2 pp = {(bf16)__builtin_amdgcn_exp2f(fmaf(x[8 * ks + 2 * t2], c, -mu)),
                                 (bf16)__builtin_amdgcn_exp2f(fmaf(x[8 * ks + 2 * t2 + 1], c, -mu))};
              sum = __builtin_amdgcn_fdot2_f32_bf16(pp, bf16x2{(bf16)1.0f, (bf16)1.0f}, sum, false);
              const f16x2 ph = __builtin_bit_cast(f16x2, pp);
              pb[ks][2 * t2] = ph[0];
              pb[ks][2 * t2 + 1] = ph[1];
            } else {
              const f16x2 ph = {(f16)__builtin_amdgcn_exp2f(fmaf(x[8 * ks + 2 * t2], c, -mu)),
                                (f16)__builtin_amdgcn_exp2f(fmaf(x[8 * ks + 2 * t2 + 1], c, -mu))};
              sum = __builtin_amdgcn_fdot2(ph, f16x2{(f16)1.0f, (f16)1.0f}, sum, false);
              pb[ks][2 * t2] = ph[0];
              pb[ks][2 * t2 + 1] = ph[1];
            }
          }
        }
      };
      // Optimistic weights (every width but 128): the weights against the
      // running max first. A weight past 2^8 (the lazy max's bound, which
      // keeps 16-bit weights finite) makes the lane's weights sum past 2^8;
      // only then, or while the lane's max is still -inf (every key so far
      // masked, or none seen), does the wave take the max, and weigh again
      // where it moved. (At D = 512 the four slices of a query block hold
      // the same scores, so they decide alike.) The max's reduction chain
      // leaves the common path: 3-7% faster at D = 64, 2-5% at D = 256, 2%
      // at D = 96, 1.3-2.4% at D = 512 (there against issuing each 16-key
      // step's products as soon as its probabilities exist, max first); at
      // D = 128 0-3% slower on causal prompts, so it keeps the max first.
      constexpr bool kOptimistic = D != 128;
      if constexpr (!kOptimistic) {
        lazy_max();
        // While every key so far is masked, m is -inf and so is every x.
        weights(m == -INFINITY ? 0.0f : m, l);
      } else {
        float lb = 0.0f;
        weights(m == -INFINITY ? 0.0f : m, lb);
        if (__ballot(m == -INFINITY || !(lb <= 256.0f)) != 0) {
          if (__ballot(lazy_max()) != 0) {
            lb = 0.0f;
            weights(m == -INFINITY ? 0.0f : m, lb);
          }
        }
        l += lb;
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int b = 0; b < kDW / 32; ++b) {
#pragma unroll
        for (int ks = 0; ks < 2 * KB; ++ks) {
          const f16* vp = sv + v_lane + 16 * ks * kVRow + 32 * b;
          const f16x4 lo4 = read_tr(vp);
          const f16x4 hi4 = read_tr(vp + 8 * kVRow);
          const f16x8 a = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
          o[b] = mfma16<BF>(a, pb[ks], o[b]);
        }
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (more) stash(buf ^ 1);
    __syncthreads();  // the next tile is in LDS; this one may be overwritten
  }

  finish<D, BF, GEN, ODD>(p, o, m, l, qi, h, split, hh, sl, q_live);
}

// ---------------------------------------------------------------------------
// The pipelined kernels: 16-bit K/V at head dims 64, 96, 128 and 256.
//
// The tile loop of prefill_body computes S, softmax and P V of a tile one
// after the other and moves K/V through registers on its way into LDS; the
// matrix cores were busy 31-34% of its cycles at D = 128. Here
//  * a step interleaves, instruction by instruction, the products of one
//    32-key block's V, the scores of a later block and the weights of the
//    block between them, so that one wave alone keeps the matrix core busy
//    while its exps run (`step`);
//  * K and V go from global memory straight into LDS (copies spread over the
//    slots of a step), in planes of 64 bytes per key whose reads touch each
//    bank once: V as it lies, K with its 16-byte chunks permuted by key;
//  * V runs one tile behind K, so that two LDS tiles of each serve the
//    pipeline with one barrier per tile;
//  * what only some tiles need (masks, softcap, the running max) sits behind
//    one wave-uniform test per step.
// What bounds it (counters): at D = 128 with one query block a wave (4096
// tokens at 0, 28/4 heads) the matrix cores are busy 39% of the cycles, the VALU
// 36% (6.4 of its instructions a product), no LDS bank conflicts, 38% of the
// waves' cycles waiting; with two blocks, which read K and V from LDS half as
// often (512 at 32256), 42%, 33% (5.4) and 27%. At D = 256 (16/8 heads, 2048 at
// 6144, window 1024) 23% and 16%: one wave per SIMD, masks and short ranges; at D =
// 64 (14/2 heads, 1531 at 389) 10% and 21%: 15 VALU instructions a product, a
// launch of a few tiles a workgroup.
// us a call, prefill_body / here: 4096 at 0 158 / 141; 512 at 32256, bf16, 279 /
// 227; 4096 at 32256 2220 / 1795; D = 64, 1531 at 389 30.8 / 26.0; D = 256,
// 2048 at 6144, window 1024 80 / 57.
//
// Short calls: the queries' loads, the table entries and the first tiles' copies
// are under way together, a 32-key block past a wave's last key is left out, and
// outputs that are still zeros are not rescaled. 16/8 heads of 256, 19 tokens at
// 0: 6.8 us; 9.6 with the loads in a row, both blocks always and the rescaling.
//
// Measured and not kept: the weights' sum on v_dot2 inside the step (it holds
// the matrix pipe; slower), fp32 adds of the rounded weights instead (level),
// operands read 2, 4 or 5 ahead instead of 3 (level), two query blocks a wave at
// D = 64 (31.7 us).
//
// QB: blocks of 32 queries per wave.
template <int D, int QB, bool BF>
__device__ __forceinline__ void prefill_pipe_body(const PrefillParams p) {
  constexpr int kKeys = 64;             // keys per tile: two 32-key blocks
  constexpr int kPlanes = D / 32;       // 64-byte planes of a row
  constexpr int kPlane = kKeys * 32;    // halves per plane of a tile
  constexpr int kTile = kPlanes * kPlane;
  // Outputs of 64 x 128 or 32 x 256 are 128 registers a lane: they live in
  // the accumulator registers, one wave per SIMD.
  constexpr bool kAcc = D * QB > 128;
  __shared__ __align__(1024) f16 s_k[2][kTile];
  __shared__ __align__(1024) f16 s_v[2][kTile];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int n = lane & 31;
  const int hh = lane >> 5;

  const int G = p.hq / p.hkv;
  int item = blockIdx.x;
  const int runs = p.tiles * p.splits * p.hkv;
  const int full = runs / kXcds * kXcds;
  if (item < full * G) {
    int x = item % kXcds;
    const int j = item / kXcds;
    // Where the XCDs hold several query tiles at once (fewer than 8 kv
    // heads), every other round hands them out in reverse, so that no XCD
    // gets the longer tile each time (us, in one direction / reversed: 28/4
    // heads of 128, 4096 tokens at 0 147.0 / 143.3; 14/2, 8192 at 0 278 / 255;
    // 14/2 of 64, 4096 at 0 60.7 / 59.2; where tiles are alike 0.2-0.4 us the
    // other way: 512 at 2048, 28/4 of 128 37.0 / 37.2).
    if ((j / G) & 1 && kXcds % p.hkv == 0) x = kXcds - p.hkv - x / p.hkv * p.hkv + x % p.hkv;
    item = ((j / G) * kXcds + x) * G + j % G;
  }
  const int run = item / G;
  const int h = (run % p.hkv) * G + (item - run * G);
  const int kvh = run % p.hkv;
  const int split = (run / p.hkv) % p.splits;
  const int tile = p.tiles - 1 - run / p.hkv / p.splits;

  // The wave's QB blocks of 32 queries; block j of a lane is query qi + 32 j.
  const int q0 = tile * (128 * QB);
  const int q1 = min(q0 + 128 * QB, p.count);
  const int wq0 = q0 + 32 * QB * w;
  const int qi = wq0 + n;
  const int qpos = p.start + qi;
  const bool wave_live = wq0 < p.count;
  const int wfirst = p.start + wq0;
  const int wlast = p.start + min(wq0 + 32 * QB - 1, p.count - 1);

  f16x8 qf[QB][D / 16];
#pragma unroll
  for (int j = 0; j < QB; ++j) {
    const bool live = qi + 32 * j < p.count;
    const f16* qp = p.q + ((int64_t)(live ? qi + 32 * j : 0) * p.hq + h) * D + 8 * hh;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      const f16x8 x = *reinterpret_cast<const f16x8*>(qp + 16 * c);
      qf[j][c] = live ? x : f16x8{};
    }
  }

  int last = p.start + q1 - 1;
  int kfirst = p.window > 0 ? max(0, p.start + q0 - p.window + 1) : 0;
  int img_lo[QB] = {}, img_hi[QB] = {}, wave_last = wlast;
  bool wave_img = false;
  for (int i = 0; i < p.num_images; ++i) {
    const int a = p.images[2 * i], b = min(p.images[2 * i + 1], p.start + p.count);
    if (a >= b) continue;
#pragma unroll
    for (int j = 0; j < QB; ++j)
      if (qpos + 32 * j >= a && qpos + 32 * j < b) img_lo[j] = a, img_hi[j] = b;
    if (a <= last && b > p.start + q0) {
      last = max(last, b - 1);
      kfirst = min(kfirst, a);
    }
    if (wave_live && a <= wlast && b > wfirst) {
      wave_last = max(wave_last, b - 1);
      wave_img = true;
    }
  }
  const int kbase = kfirst / kKeys * kKeys;
  const int ntile = (last - kbase) / kKeys + 1;
  const int t_begin = (int)((int64_t)ntile * split / p.splits);
  const int t_end = (int)((int64_t)ntile * (split + 1) / p.splits);
  // Tiles [wa, wb) of the range that this wave's queries see.
  int wa = t_begin, wb = wave_live ? min(t_end, (wave_last - kbase) / kKeys + 1) : t_begin;
  if (p.window > 0 && !wave_img) wa = max(wa, (max(0, wfirst - p.window + 1) - kbase) / kKeys);
  wa = uniform(wa);
  wb = uniform(wb);

  // Gather: thread tid moves key tid / 4 of a tile, 64-byte pieces.
  const int gk = tid >> 2;
  // Unsigned: the cursors run past the last key, which may be 2^31 - 2.
  const uint32_t page_size = p.page_size, table_len = p.table_len;
  uint32_t kp = (uint32_t)kbase + (uint32_t)(t_begin * kKeys) + gk;
  uint32_t pi = kp / page_size;
  uint32_t r = kp - pi * page_size;
  // 16-byte chunk of each 64-byte piece this lane fetches: K's are swizzled.
  const int kchunk = 8 * ((lane & 3) ^ ((lane >> 4) & 3));
  const int vchunk = 8 * (lane & 3);
  const uint32_t k_dst = uniform(lds_address(&s_k[0][0]) + 1024 * w);
  const uint32_t v_dst = uniform(lds_address(&s_v[0][0]) + 1024 * w);
  // The page of this thread's key is looked up one iteration before its rows
  // are copied (its K's; two for V's): the wait is that iteration's own, at its
  // end, with its copies'. Each wave looks up the pages of all 64 keys of the
  // tile as well (one per lane) for the mask of usable keys, which then needs
  // neither LDS nor a barrier.
  const uint32_t pages = (uint32_t)min(p.arena_pages, (int64_t)INT32_MAX);
  const uint32_t step_pages = kKeys / page_size, step_rows = kKeys % page_size;
  int page = 0, row_off = 0, page_m = 0;
  bool in = false, in_m = false;
  uint32_t kp_m = kp - gk + lane;
  uint32_t pi_m = kp_m / page_size;
  uint32_t r_m = kp_m - pi_m * page_size;
  auto lookup = [&]() {
    in = kp <= (uint32_t)last && pi < table_len;
    in_m = kp_m <= (uint32_t)last && pi_m < table_len;
    page = p.table[min(pi, table_len - 1)];
    page_m = p.table[min(pi_m, table_len - 1)];
    row_off = (int)r * p.row_elems + kvh * p.head_elems;
    kp += kKeys;
    kp_m += kKeys;
    r += step_rows;
    r_m += step_rows;
    pi += step_pages + (r >= page_size ? 1 : 0);
    pi_m += step_pages + (r_m >= page_size ? 1 : 0);
    r -= r >= page_size ? page_size : 0;
    r_m -= r_m >= page_size ? page_size : 0;
  };
  // This thread's rows of the tiles whose V and K are copied next, their
  // usable keys, and those of the tile after them.
  const f16* src_k = nullptr;
  const f16* src_v = nullptr;
  uint64_t at_k = 0;
  bool ok_k = false, ok_v = false;
  uint64_t ok_prev = 0, ok_now = 0, ok_next = 0;
  // Takes the looked-up tile as the next K to copy, the one before it as the
  // next V.
  auto advance = [&]() {
    src_v = static_cast<const f16*>(p.v) + at_k + vchunk;
    ok_v = ok_k;
    ok_prev = ok_now;
    ok_now = ok_next;
    ok_k = in && (uint32_t)page < pages;
    ok_next = __ballot(in_m && (uint32_t)page_m < pages);
    at_k = (uint64_t)(uint32_t)(ok_k ? page : 0) * (uint32_t)p.page_elems + (uint32_t)row_off;
    src_k = static_cast<const f16*>(p.k) + at_k + kchunk;
  };
  auto copy_k = [&](int buf, auto i) {
    copy_to_lds<64 * i.value, (2 * kPlane - 64) * i.value>(src_k, k_dst + buf * (2 * kTile));
  };
  auto copy_v = [&](int buf, auto i) {
    copy_to_lds<64 * i.value, (2 * kPlane - 64) * i.value>(src_v, v_dst + buf * (2 * kTile));
  };
  // After the copies have landed: rows of unusable keys become zeros (their
  // weight is 0; zero V keeps 0 * V finite whatever the arena holds there).
  auto clean_v = [&](int buf, bool ok) {
    if (!ok) {
#pragma unroll
      for (int i = 0; i < kPlanes; ++i)
        *reinterpret_cast<f16x8*>(&s_v[buf][kPlane * i + 32 * gk + 8 * (lane & 3)]) = f16x8{};
    }
  };

  f32x16 o[QB][D / 32];
  float m[QB], l[QB];
#pragma unroll
  for (int j = 0; j < QB; ++j) {
    m[j] = -INFINITY;
    l[j] = 0.0f;
#pragma unroll
    for (int b = 0; b < D / 32; ++b) o[j][b] = f32x16{};
  }
  f32x16 s0[QB] = {}, s1[QB] = {};  // scores of the even and the odd 32-key block
  f16x8 p0[QB][2] = {}, p1[QB][2] = {};  // and their weights

  const int g16 = lane >> 4, s16 = lane & 15;
  const int v_lane = (4 * (g16 >> 1) + (s16 >> 2)) * 32 + 16 * (g16 & 1) + 4 * (s16 & 3);
  const int ksw = (n >> 2) & 3;
  const int k_lane0 = 32 * n + 8 * (hh ^ ksw);
  const int k_lane1 = 32 * n + 8 * ((2 + hh) ^ ksw);
  const float c = p.softcap <= 0.0f && p.scale_log2 > 0.0f ? p.scale_log2 : 1.0f;

  // Bits 0 .. n - 1 (none for n <= 0, all from 32 on).
  auto below = [](int n) -> uint32_t {
    const uint32_t ones = n >= 32 ? 32u : n > 0 ? (uint32_t)n : 0u;
    return (uint32_t)((1ull << ones) - 1);
  };
  // Scores of a block in place: softcap or a scale that is not positive
  // (`special`), then the masks where the block has any.
  const bool special = p.softcap > 0.0f || !(p.scale_log2 > 0.0f);
  auto shape = [&](f32x16 (&xs)[QB], int k0, uint32_t okm, bool masks) {
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      f32x16& x = xs[j];
      if (p.softcap > 0.0f) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float e = __builtin_amdgcn_exp2f(x[v] * p.cap_in);
          x[v] = (1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f)) * p.cap_out;
        }
      } else if (!(p.scale_log2 > 0.0f)) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = x[v] * p.scale_log2;
      }
    }
    if (!masks) return;
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      f32x16& x = xs[j];
      // Keys k0 .. k0 + 31 this lane's query sees, one bit each: usable, and
      // not past its position, inside its window, or inside its image. Two
      // instructions per score then (bit to mask, select), where a test of
      // each key's position took nine: the diagonal tiles are most of a short
      // prompt.
      const int hi = qpos + 32 * j - k0;
      uint32_t see = below(hi + 1);
      if (p.window > 0) see &= ~below(hi - p.window + 1);
      if (wave_img) see |= below(img_hi[j] - k0) & ~below(img_lo[j] - k0);
      see = (see & okm) >> (4 * hh);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int bit = __builtin_amdgcn_sbfe((int)see, 8 * (v / 4) + (v % 4), 1);
        const float y = x[v];  // (a bit cast of x[v] itself takes element 0)
        x[v] = __builtin_bit_cast(float, (__builtin_bit_cast(int, y) & bit) |
                                             (~bit & (int)0xFF800000));
      }
    }
  };
  // Weights 2 i, 2 i + 1 of a block, rounded to 16 bits and packed.
  auto put_pair = [&](f16x8 (&pb)[2], int i, float e0, float e1) {
    f16x2 ph;
    if constexpr (BF)
      ph = __builtin_bit_cast(f16x2, bf16x2{(bf16)e0, (bf16)e1});
    else
      ph = f16x2{(f16)e0, (f16)e1};
    pb[i / 4][2 * (i % 4)] = ph[0];
    pb[i / 4][2 * (i % 4) + 1] = ph[1];
  };
  // Their sum, all of a block's at once: v_dot2 holds the matrix pipe, so none
  // goes between two products.
  auto total = [&](const f16x8 (&pb)[2], float sum) {
    float s2[2] = {sum, 0.0f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f16x2 ph = {pb[i / 4][2 * (i % 4)], pb[i / 4][2 * (i % 4) + 1]};
      if constexpr (BF)
        s2[i & 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, ph),
                                                    bf16x2{(bf16)1.0f, (bf16)1.0f}, s2[i & 1], false);
      else
        s2[i & 1] = __builtin_amdgcn_fdot2(ph, f16x2{(f16)1.0f, (f16)1.0f}, s2[i & 1], false);
    }
    return s2[0] + s2[1];
  };
  auto scores = [&](f32x16 (&x)[QB], const f16* kt) {
#pragma unroll
    for (int cc = 0; cc < D / 16; ++cc) {
      const f16x8 a = *reinterpret_cast<const f16x8*>(kt + (cc & 1 ? k_lane1 : k_lane0) +
                                                      kPlane * (cc >> 1));
#pragma unroll
      for (int j = 0; j < QB; ++j) x[j] = mfma16<BF>(a, qf[j][cc], cc == 0 ? f32x16{} : x[j]);
    }
  };
  auto accumulate = [&](const f16x8 (&pb)[QB][2], const f16* vt) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int b = 0; b < D / 32; ++b) {
        const f16* vp = vt + v_lane + kPlane * b + 512 * ks;
        const f16x4 lo4 = read_tr(vp);
        const f16x4 hi4 = read_tr(vp + 256);
        const f16x8 a = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
#pragma unroll
        for (int j = 0; j < QB; ++j) mfma_to<BF, kAcc>(a, pb[j][ks], o[j][b]);
      }
    }
  };
  // Between the re-weighing of a block and the first product that reads the
  // weights. (The outputs' rescaling lies before it. Weights that a step has
  // taken need no wait: their sum, pinned with them, comes after.)
  auto operands_done = [&](f16x8 (&pb)[QB][2]) {
    if constexpr (kAcc) {
#pragma unroll
      for (int j = 0; j < QB; ++j) asm volatile("" : "+v"(pb[j][0]), "+v"(pb[j][1]));
      asm volatile("s_nop 1");
    }
  };
  // Before the outputs are read by anything but a matrix-core instruction.
  auto outputs_done = [&]() {
    if constexpr (kAcc) {
      asm volatile("s_nop 15\n\ts_nop 7");
#pragma unroll
      for (int j = 0; j < QB; ++j)
#pragma unroll
        for (int b = 0; b < D / 32; ++b) asm volatile("" : "+a"(o[j][b]));
    }
  };
  // The weights of a block were taken against the running max and summed in
  // lb. A weight past 2^8 (which keeps 16-bit weights finite) makes lb pass
  // it; only then, or while no key was visible (lb then is infinite), the max
  // is taken and the block weighed again.
  auto settle = [&](const f32x16 (&xs)[QB], f16x8 (&pb)[QB][2], float (&lb)[QB]) {
    bool again = false;
#pragma unroll
    for (int j = 0; j < QB; ++j) again |= !(lb[j] <= 256.0f);
    if (__ballot(again) != 0) {
      outputs_done();
#pragma unroll
      for (int j = 0; j < QB; ++j) {
        const f32x16& x = xs[j];
        float top = x[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) top = fmaxf(top, x[v]);
        top = fmaxf(top, __shfl_xor(top, 32)) * c;
        if (top > m[j] + kSlack) {
          const bool seen = m[j] != -INFINITY;
          const float f = seen ? __builtin_amdgcn_exp2f(m[j] - top) : 0.0f;
          m[j] = top;
          // (Else the outputs are zeros. With two blocks the choice costs the loop
          // its registers' order and 1%.)
          if (QB == 2 || seen) {
            l[j] *= f;
#pragma unroll
            for (int b = 0; b < D / 32; ++b)
#pragma unroll
              for (int v = 0; v < 16; ++v) o[j][b][v] *= f;
          }
        }
        const float mu = m[j] == -INFINITY ? 0.0f : m[j];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          put_pair(pb[j], i, __builtin_amdgcn_exp2f(fmaf(x[2 * i], c, -mu)),
                   __builtin_amdgcn_exp2f(fmaf(x[2 * i + 1], c, -mu)));
        lb[j] = total(pb[j], 0.0f);
      }
      operands_done(pb);
    }
#pragma unroll
    for (int j = 0; j < QB; ++j) l[j] += lb[j];
  };
  // One step of the pipeline, QB x D / 8 matrix-core instructions in slots:
  // the products of a 32-key block's V (weights pv) alternate with the scores
  // of a later block (xn), and the weights of the block between them (x, into
  // pb, summed into lb) are spread over the slots, done two slots early.
  // Operands are read kAhead operands early.
  auto step = [&](const f32x16 (&x)[QB], f16x8 (&pb)[QB][2], const f16x8 (&pv)[QB][2],
                  f32x16 (&xn)[QB], float (&lb)[QB], const f16* kt, const f16* vt, auto beside) {
    constexpr int kOps = D / 8;  // operands: V and K fragments in turn
    constexpr int kSlots = QB * kOps;
    constexpr int kAhead = QB > 1 ? 3 : 4;
    constexpr int kScores = 16 * QB;
    float mu[QB], e[kScores];
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      mu[j] = m[j] == -INFINITY ? 0.0f : m[j];
      lb[j] = m[j] == -INFINITY ? INFINITY : 0.0f;
    }
    f16x8 a[kOps];
    auto read = [&](int i) {
      if (i & 1) {
        const int cc = i >> 1;
        a[i] = *reinterpret_cast<const f16x8*>(kt + (cc & 1 ? k_lane1 : k_lane0) +
                                               kPlane * (cc >> 1));
      } else {
        const int b = (i >> 1) % (D / 32), ks = (i >> 1) / (D / 32);
        const f16* vp = vt + v_lane + kPlane * b + 512 * ks;
        const f16x4 lo4 = read_tr(vp);
        const f16x4 hi4 = read_tr(vp + 256);
        a[i] = f16x8{lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
      }
    };
    auto pair = [&](int i) {
      put_pair(pb[i / 8], i % 8, e[2 * i], e[2 * i + 1]);
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) read(i);
    e[0] = fmaf(x[0][0], c, -mu[0]);
    __builtin_amdgcn_sched_barrier(0);
    auto slot = [&](auto sc) {
      constexpr int i = sc.value / QB, j = sc.value % QB;
      if constexpr (i & 1) {
        constexpr int cc = i >> 1;
        xn[j] = mfma16<BF>(a[i], qf[j][cc], cc == 0 ? f32x16{} : xn[j]);
      } else {
        constexpr int b = (i >> 1) % (D / 32), ks = (i >> 1) / (D / 32);
        mfma_to<BF, kAcc>(a[i], pv[j][ks], o[j][b]);
      }
      if constexpr (j == 0 && i + kAhead < kOps) read(i + kAhead);
      if constexpr (j == QB - 1) beside(std::integral_constant<int, i>{});
      constexpr int v0 = kScores * sc.value / (kSlots - 2);
      constexpr int v1 = kScores * (sc.value + 1) / (kSlots - 2);
#pragma unroll
      for (int v = v0 < kScores ? v0 : kScores; v < (v1 < kScores ? v1 : kScores); ++v) {
        // The argument of the next exp, this exp, the pair before.
        if (v + 1 < kScores) e[v + 1] = fmaf(x[(v + 1) / 16][(v + 1) % 16], c, -mu[(v + 1) / 16]);
        e[v] = __builtin_amdgcn_exp2f(e[v]);
        if ((v & 1) && v >= 3) pair((v - 3) / 2);
      }
      if constexpr (sc.value == kSlots - 2) pair(kScores / 2 - 1);
      __builtin_amdgcn_sched_barrier(0);
    };
    each(slot, std::make_integer_sequence<int, kSlots>{});
#pragma unroll
    for (int j = 0; j < QB; ++j) lb[j] = total(pb[j], lb[j]);
    // Keeps the products of the step in it (they would sink past the branch
    // of settle, away from the weights they are to overlap).
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      asm volatile("" : "+v"(xn[j]), "+v"(pb[j][0]), "+v"(pb[j][1]), "+v"(lb[j]));
#pragma unroll
      for (int b = 0; b < (kAcc ? 0 : D / 32); ++b) asm volatile("" : "+v"(o[j][b]));
    }
  };

  // Whether the blocks of an iteration (the odd one of the tile before and
  // the even one of this tile) need their masks, a softcap or an unusual scale.
  const int plain_hi = special ? INT32_MIN : wfirst - 31;
  const int plain_lo = p.window > 0 ? wlast - p.window : INT32_MIN;
  auto rough = [&](int k0) {
    return k0 > plain_hi || k0 - 32 <= plain_lo || ((ok_prev >> 32) & (uint32_t)ok_now) != 0xFFFFFFFFu;
  };
  // Whether a block needs its masks (every block of a softcapped call comes
  // through the test above; masked as well, whatever its keys, 4096 tokens at
  // 8192, 14/2 heads of 64, took 407 us instead of 367). One test in the loop:
  // a second beside it cost two query blocks 2%.
  auto masked = [&](int k0, uint32_t okm) {
    return !special || k0 > wfirst - 31 || k0 <= plain_lo || okm != 0xFFFFFFFFu;
  };
  // Iteration t of the workgroup: V of tile t and K of tile t + 1 are copied
  // beside the iteration's math and published by its barrier (close). The
  // looked-up rows move on (turn) once the copies are issued.
  auto each_plane = [&](auto f) { each(f, std::make_integer_sequence<int, kPlanes>{}); };
  auto turn = [&]() {
    advance();
    lookup();
  };
  auto copies = [&](int t) {
    const int buf = (t - t_begin) & 1;
    each_plane([&](auto i) { copy_v(buf, i); });
    each_plane([&](auto i) { copy_k(buf ^ 1, i); });
  };
  auto close = [&](int t, bool ok) {
    wait_vmem<0>();
    clean_v((t - t_begin) & 1, ok);
    __syncthreads();
  };
  int t = t_begin;
  lookup();
  __builtin_amdgcn_sched_barrier(0);
  // The queries are only ever matrix-core operands: into accumulator
  // registers, while the table entries are on their way. (Moved one by one as
  // they were loaded, each load waited for the one before.)
  if constexpr (kAcc) {
#pragma unroll
    for (int j = 0; j < QB; ++j)
#pragma unroll
      for (int c = 0; c < D / 16; ++c) asm volatile("" : "+a"(qf[j][c]));
  }
  advance();
  lookup();
  const f16* first_k = src_k;
  advance();
  // (The second entries are waited for here: a wait past the first copies
  // would wait for those as well.)
  asm volatile("" : "+v"(first_k), "+v"(src_v), "+v"(src_k), "+s"(ok_next));
  lookup();
  // K of the first tile, then its V and the second K: only the first is
  // waited for here, so a short call has one latency of K/V and not two.
  each_plane([&](auto i) {
    copy_to_lds<64 * i.value, (2 * kPlane - 64) * i.value>(first_k, k_dst);
  });
  copies(t);
  wait_vmem<2 * kPlanes>();
  __syncthreads();
  // Whether the odd block of the wave's last tile holds a key it sees.
  const bool odd_last = wave_last >= kbase + (wb - 1) * kKeys + 32;
  if (wa >= wb) wa = t_end;
  auto idle = [&]() {  // an iteration whose tile this wave's queries do not see
    const bool ok = ok_v;
    if (t > t_begin) copies(t);
    turn();
    close(t, ok);
  };
  for (; t < wa; ++t) idle();
  float lb[QB];
  auto unweighed = [&]() {
#pragma unroll
    for (int j = 0; j < QB; ++j) lb[j] = INFINITY;
  };
  if (t < t_end) {
    // First tile: scores of both blocks, weights of the first.
    {
      const bool ok = ok_v;
      if (t > t_begin) copies(t);
      const f16* kt = s_k[(t - t_begin) & 1];
      const int k0 = kbase + t * kKeys;
      scores(s0, kt);
      shape(s0, k0, (uint32_t)ok_now, true);
      if (wb - wa > 1 || odd_last) scores(s1, kt + 1024);
      unweighed();
      settle(s0, p0, lb);
      turn();
      close(t, ok);
    }
    // Scores of tile t, weights of its even block and of tile t - 1's odd
    // one, products of tile t - 1's V.
    for (++t; t < wb; ++t) {
      const int buf = (t - t_begin) & 1;
      const int k0 = kbase + t * kKeys;
      const f16* kt = s_k[buf];
      const f16* vt = s_v[buf ^ 1];
      const bool masks = rough(k0), ok = ok_v;
      const uint32_t ok_even = (uint32_t)ok_now, ok_odd = (uint32_t)(ok_prev >> 32);
      if (masks) shape(s1, k0 - 32, ok_odd, masked(k0 - 32, ok_odd));
      step(s1, p1, p0, s0, lb, kt, vt, [&](auto i) {
        if constexpr (i.value % 2 == 0) {
          constexpr int j = i.value / 2;
          if constexpr (j < kPlanes)
            copy_v(buf, std::integral_constant<int, j>{});
          else
            copy_k(buf ^ 1, std::integral_constant<int, j - kPlanes>{});
        }
      });
      settle(s1, p1, lb);
      if (masks) shape(s0, k0, ok_even, masked(k0, ok_even));
      step(s0, p0, p1, s1, lb, kt + 1024, vt + 1024, [&](auto i) {
        if constexpr (i.value == 1) turn();
      });
      settle(s0, p0, lb);
      close(t, ok);
    }
    // Past the last tile: weights of its odd block, products of its V.
    {
      const bool ok = ok_v;
      const uint32_t ok_odd = (uint32_t)(ok_prev >> 32);
      if (t < t_end) copies(t);
      const f16* vt = s_v[((t - t_begin) & 1) ^ 1];
      if (odd_last) shape(s1, kbase + (t - 1) * kKeys + 32, ok_odd, true);
      accumulate(p0, vt);
      if (odd_last) {
        unweighed();
        settle(s1, p1, lb);
        accumulate(p1, vt + 1024);
      }
      outputs_done();  // (here: copies of the outputs may follow on any way out)
      if (t < t_end) {
        turn();
        close(t, ok);
      }
    }
    for (++t; t < t_end; ++t) idle();
  }
  // (An empty range has waited for none but its first copies; the others have
  // to land before the LDS is another workgroup's.)
  wait_vmem<0>();
  // One block of outputs a wave leaves room for them in vector registers: moved
  // at once, not each before its store (0.4 us).
  if constexpr (kAcc && QB == 1) {
#pragma unroll
    for (int b = 0; b < D / 32; ++b) asm volatile("" : "+v"(o[0][b]));
  }
#pragma unroll
  for (int j = 0; j < QB; ++j)
    finish<D, BF, false, false>(p, o[j], m[j], l[j], qi + 32 * j, h, split, hh, 0,
                                qi + 32 * j < p.count);
}

template <int D, int QB, bool BF>
__global__ __launch_bounds__(256, QB == 1 ? occupancy_for(D) : 1) void paged_prefill_pipe_kernel(
    const PrefillParams p) {
  prefill_pipe_body<D, QB, BF>(p);
}

// The prefill kernel of every even head dim (template arguments as
// prefill_body's).
template <int D, bool Q8, bool BF, bool GEN>
__global__ __launch_bounds__(64 * waves_for(D)) void paged_prefill_kernel(const PrefillParams p) {
  prefill_body<D, Q8, BF, GEN, false>(p);
}

// Odd head dims (the reference's portable attention takes any): the generic
// kernel of width D with element-wise queries, gather and output.
template <int D, bool Q8, bool BF>
__global__ __launch_bounds__(64 * waves_for(D)) void paged_prefill_odd_kernel(const PrefillParams p) {
  prefill_body<D, Q8, BF, true, true>(p);
}

// Merge of the key ranges of a split prefill: for each (query, head),
// M = max_s m_s, w_s = 2^(m_s - M) (0 for an empty range), out =
// sum_s w_s o_s / sum_s w_s l_s (0 when nothing was visible). The same LSE
// merge as the reference's decode merge (metal_kernels.py:103-124), in the
// log2 domain. One thread per 4 dims, D / 4 threads per (query, head).
// GEN: output rows of hd (below D) elements, written one element at a time
// (an odd hd leaves rows 2-byte aligned); partials stay D wide.
template <int D, bool BF, bool GEN>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const float* __restrict__ part_o,
                                                            const float2* __restrict__ part_ml,
                                                            f16* __restrict__ out, int64_t pairs,
                                                            int splits, int hd) {
  constexpr int kT = D / 4;
  // 256 / kT pairs per block; at D = 96 the last 16 threads have none.
  if (threadIdx.x >= 256 / kT * kT) return;
  const int64_t pair = (int64_t)blockIdx.x * (256 / kT) + threadIdx.x / kT;
  if (pair >= pairs) return;
  const int d = 4 * (threadIdx.x % kT);
  float top = -INFINITY;
  for (int s = 0; s < splits; ++s) top = fmaxf(top, part_ml[s * pairs + pair].x);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  float sum = 0.0f;
  if (top != -INFINITY) {
    for (int s = 0; s < splits; ++s) {
      const float2 ml = part_ml[s * pairs + pair];
      if (ml.x == -INFINITY) continue;
      const float w = __builtin_amdgcn_exp2f(ml.x - top);
      const float4 x = *reinterpret_cast<const float4*>(part_o + (s * pairs + pair) * D + d);
      acc.x += w * x.x;
      acc.y += w * x.y;
      acc.z += w * x.z;
      acc.w += w * x.w;
      sum += w * ml.y;
    }
  }
  const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
  f16x4 y = {round16<BF>(acc.x * inv), round16<BF>(acc.y * inv), round16<BF>(acc.z * inv),
             round16<BF>(acc.w * inv)};
  if constexpr (GEN) {
    f16* row = out + pair * hd;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (d + j < hd) row[d + j] = y[j];
  } else {
    (void)hd;
    *reinterpret_cast<f16x4*>(out + pair * D + d) = y;
  }
}

using pda_internal::fail;
using pda_internal::ok;

template <bool Q8, bool BF, bool GEN>
const void* prefill_kernel_for(int kdim) {
  // 16-bit K/V at the narrower tuned head dims runs the pipelined kernels.
  if constexpr (!Q8 && !GEN)
    return reinterpret_cast<const void*>(paged_prefill_kernel<512, Q8, BF, GEN>);
  else
    return kdim == 64    ? reinterpret_cast<const void*>(paged_prefill_kernel<64, Q8, BF, GEN>)
         : kdim == 96  ? reinterpret_cast<const void*>(paged_prefill_kernel<96, Q8, BF, GEN>)
         : kdim == 128 ? reinterpret_cast<const void*>(paged_prefill_kernel<128, Q8, BF, GEN>)
         : kdim == 256 ? reinterpret_cast<const void*>(paged_prefill_kernel<256, Q8, BF, GEN>)
                       : reinterpret_cast<const void*>(paged_prefill_kernel<512, Q8, BF, GEN>);
}

template <bool Q8, bool BF>
const void* prefill_odd_kernel_for(int kdim) {
  return kdim == 64    ? reinterpret_cast<const void*>(paged_prefill_odd_kernel<64, Q8, BF>)
         : kdim == 96  ? reinterpret_cast<const void*>(paged_prefill_odd_kernel<96, Q8, BF>)
         : kdim == 128 ? reinterpret_cast<const void*>(paged_prefill_odd_kernel<128, Q8, BF>)
         : kdim == 256 ? reinterpret_cast<const void*>(paged_prefill_odd_kernel<256, Q8, BF>)
                       : reinterpret_cast<const void*>(paged_prefill_odd_kernel<512, Q8, BF>);
}

template <bool BF>
const void* pipe_kernel_for(int kdim, int blocks) {
  return kdim == 64   ? reinterpret_cast<const void*>(paged_prefill_pipe_kernel<64, 1, BF>)
         : kdim == 96 ? reinterpret_cast<const void*>(paged_prefill_pipe_kernel<96, 1, BF>)
         : kdim == 256 ? reinterpret_cast<const void*>(paged_prefill_pipe_kernel<256, 1, BF>)
         : blocks == 2 ? reinterpret_cast<const void*>(paged_prefill_pipe_kernel<128, 2, BF>)
                       : reinterpret_cast<const void*>(paged_prefill_pipe_kernel<128, 1, BF>);
}

template <bool Q8, bool BF>
const void* prefill_kernel_for(int kdim, bool gen, bool odd) {
  if (odd) return prefill_odd_kernel_for<Q8, BF>(kdim);
  return gen ? prefill_kernel_for<Q8, BF, true>(kdim) : prefill_kernel_for<Q8, BF, false>(kdim);
}

template <bool BF, bool GEN>
const void* merge_kernel_for(int kdim) {
  return kdim == 64    ? reinterpret_cast<const void*>(prefill_merge_kernel<64, BF, GEN>)
         : kdim == 96  ? reinterpret_cast<const void*>(prefill_merge_kernel<96, BF, GEN>)
         : kdim == 128 ? reinterpret_cast<const void*>(prefill_merge_kernel<128, BF, GEN>)
         : kdim == 256 ? reinterpret_cast<const void*>(prefill_merge_kernel<256, BF, GEN>)
                       : reinterpret_cast<const void*>(prefill_merge_kernel<512, BF, GEN>);
}

template <bool BF>
const void* merge_kernel_for(int kdim, bool gen) {
  return gen ? merge_kernel_for<BF, true>(kdim) : merge_kernel_for<BF, false>(kdim);
}

int prefill(const void* queries, const void* keys, const void* values, const void* key_scales,
            const void* value_scales, bool q8, bool bf16_elems, const int32_t* table,
            int32_t table_len,
            int32_t start, int32_t count, void* out, int32_t q_heads, int32_t kv_heads,
            int32_t head_dim, int32_t page_size, int64_t arena_rows, int32_t layout, float scale,
            int32_t window, float softcap, const int32_t* images, int32_t num_images,
            int32_t splits, void* workspace, size_t workspace_bytes, void* stream) {
  if (count < 0 || start < 0 || q_heads <= 0 || kv_heads <= 0 || page_size <= 0 ||
      table_len < 0 || window < 0 || splits < 0)
    return fail(PDA_ERR_INVALID_ARGUMENT,
                "count=%d start=%d q_heads=%d kv_heads=%d page_size=%d table_len=%d window=%d "
                "splits=%d",
                count, start, q_heads, kv_heads, page_size, table_len, window, splits);
  if (q_heads % kv_heads)
    return fail(PDA_ERR_HEAD_RATIO, "query heads must be a multiple of kv heads");
  const int kdim = prefill_dim(head_dim);
  if (kdim == 0)
    return fail(PDA_ERR_HEAD_DIM, "head_dim %d: prefill serves head dims 1..512", head_dim);
  const bool gen = kdim != head_dim;
  const bool odd = head_dim & 1;
  if (count == 0) return ok();
  if (table_len == 0)
    return fail(PDA_ERR_INVALID_ARGUMENT, "an empty page table holds no keys of the chunk");
  if ((int64_t)start + count > INT32_MAX)
    return fail(PDA_ERR_TOO_LONG, "start + count exceeds 2^31");
  if (!queries || !keys || !values || !table || !out || (q8 && (!key_scales || !value_scales)))
    return fail(PDA_ERR_INVALID_ARGUMENT, "null buffer pointer");
  if (num_images < 0 || (num_images > 0 && !images))
    return fail(PDA_ERR_INVALID_ARGUMENT, "num_images=%d needs an image span array",
                num_images);
  if ((uintptr_t)images & 3) return fail(PDA_ERR_ALIGNMENT, "image spans must be 4-byte aligned");
  if (layout != PDA_LAYOUT_ROWS && layout != PDA_LAYOUT_PAGES)
    return fail(PDA_ERR_INVALID_ARGUMENT, "unknown K/V layout %d", layout);
  if ((int64_t)page_size * kv_heads * head_dim > INT32_MAX)
    return fail(PDA_ERR_INVALID_ARGUMENT, "a page of one layer holds more than 2^31 elements");
  if (arena_rows < page_size)
    return fail(PDA_ERR_INVALID_ARGUMENT, "arena_rows %lld holds no whole page",
                (long long)arena_rows);
  if (!(scale == scale) || isinf(scale) || !(softcap >= 0.0f) || isinf(softcap))
    return fail(PDA_ERR_INVALID_ARGUMENT, "scale must be finite and softcap >= 0");
  const uintptr_t mis = (uintptr_t)queries | (uintptr_t)keys | (uintptr_t)values |
                        (uintptr_t)out;
  if (mis & 15)
    return fail(PDA_ERR_ALIGNMENT, "query, K/V and output buffers must be 16-byte aligned");
  if (q8 && (((uintptr_t)key_scales | (uintptr_t)value_scales) & 1))
    return fail(PDA_ERR_ALIGNMENT, "fp16 scale arenas must be 2-byte aligned");
  if ((uintptr_t)table & 3) return fail(PDA_ERR_ALIGNMENT, "the table must be 4-byte aligned");
  const bool pipe = pipelined(head_dim, q8);
  const int nsplit = prefill_splits(start, count, q_heads, kdim, window, splits);
  const int blocks =
      pipe ? query_blocks(start, count, q_heads, head_dim, window, softcap, nsplit) : 1;
  const int per_wg = blocks * queries_for(kdim);
  // (Counted with one query block a wave, whichever run.)
  if (((int64_t)count + queries_for(kdim) - 1) / queries_for(kdim) * q_heads * nsplit > INT32_MAX)
    return fail(PDA_ERR_INVALID_ARGUMENT, "query tiles x query heads x splits exceeds 2^31");
  const size_t need = prefill_workspace(nsplit, count, q_heads, kdim);
  if (need > 0 && (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)))
    return fail(PDA_ERR_WORKSPACE,
                "%d key ranges need a 256-byte aligned workspace of %zu bytes (got %zu)", nsplit,
                need, workspace ? workspace_bytes : (size_t)0);

  PrefillParams prm;
  prm.q = static_cast<const f16*>(queries);
  prm.k = keys;
  prm.v = values;
  prm.kscale = static_cast<const f16*>(key_scales);
  prm.vscale = static_cast<const f16*>(value_scales);
  // Scale arenas: [rows, kv_heads] beside the row arena, [pages, kv_heads,
  // page_size] beside page tiles (as the decode call's).
  prm.scale_page = (int64_t)page_size * kv_heads;
  prm.scale_row = layout == PDA_LAYOUT_ROWS ? kv_heads : 1;
  prm.scale_head = layout == PDA_LAYOUT_ROWS ? 1 : page_size;
  prm.table = table;
  prm.images = images;
  prm.num_images = num_images;
  prm.out = static_cast<f16*>(out);
  const size_t pairs = (size_t)count * q_heads;
  prm.part_o = nsplit > 1 ? static_cast<float*>(workspace) : nullptr;
  prm.part_ml = nsplit > 1 ? reinterpret_cast<float2*>(
                                 static_cast<char*>(workspace) +
                                 (((size_t)nsplit * pairs * kdim * 4 + 255) & ~(size_t)255))
                           : nullptr;
  prm.arena_pages = arena_rows / page_size;
  prm.page_elems = (int64_t)page_size * kv_heads * head_dim;
  if (layout == PDA_LAYOUT_ROWS) {
    prm.row_elems = kv_heads * head_dim;
    prm.head_elems = head_dim;
  } else {
    prm.row_elems = head_dim;
    prm.head_elems = page_size * head_dim;
  }
  prm.table_len = table_len;
  prm.start = start;
  prm.count = count;
  prm.tiles = (count + per_wg - 1) / per_wg;
  prm.splits = nsplit;
  const int tile_keys = kdim <= 128 ? 64 : 32;
  prm.page_step = tile_keys % page_size == 0 ? tile_keys / page_size : 0;
  prm.hq = q_heads;
  prm.hkv = kv_heads;
  prm.head_dim = head_dim;
  prm.page_size = page_size;
  prm.window = window;
  prm.scale_log2 = scale * kLog2e;
  prm.softcap = softcap;
  prm.cap_in = softcap > 0.0f ? 2.0f * kLog2e * scale / softcap : 0.0f;
  prm.cap_out = softcap * kLog2e;
  void* args[] = {&prm};
  const void* fn = pipe ? (bf16_elems ? pipe_kernel_for<true>(kdim, blocks)
                                      : pipe_kernel_for<false>(kdim, blocks))
                  : q8 ? prefill_kernel_for<true, false>(kdim, gen, odd)
                  : bf16_elems ? prefill_kernel_for<false, true>(kdim, gen, odd)
                               : prefill_kernel_for<false, false>(kdim, gen, odd);
  const hipStream_t hs = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((int64_t)prm.tiles * q_heads * nsplit));
  hipError_t err = hipLaunchKernel(fn, grid, dim3(64 * waves_for(kdim)), args, 0, hs);
  if (err != hipSuccess)
    return fail(PDA_ERR_HIP, "kernel launch failed: %s", hipGetErrorString(err));
  if (nsplit > 1) {
    const int64_t npairs = (int64_t)pairs;
    const int per_block = 256 / (kdim / 4);
    const float* po = prm.part_o;
    const float2* pml = prm.part_ml;
    f16* o16 = prm.out;
    int ns = nsplit;
    int hd = head_dim;
    void* margs[] = {&po, &pml, &o16, (void*)&npairs, &ns, &hd};
    const void* mfn = bf16_elems ? merge_kernel_for<true>(kdim, gen)
                                 : merge_kernel_for<false>(kdim, gen);
    err = hipLaunchKernel(mfn, dim3((unsigned)((npairs + per_block - 1) / per_block)),
                          dim3(256), margs, 0, hs);
    if (err != hipSuccess)
      return fail(PDA_ERR_HIP, "merge launch failed: %s", hipGetErrorString(err));
  }
  return ok();
}

}  // namespace

extern "C" {

int pda_prefill_workspace_bytes(int32_t start, int32_t count, int32_t q_heads,
                                int32_t head_dim, int32_t window, int32_t splits,
                                int32_t* splits_used, size_t* bytes) {
  if (count < 0 || start < 0 || q_heads <= 0 || window < 0 || splits < 0 || !bytes)
    return fail(PDA_ERR_INVALID_ARGUMENT, "count=%d start=%d q_heads=%d window=%d splits=%d",
                count, start, q_heads, window, splits);
  const int kdim = prefill_dim(head_dim);
  if (kdim == 0)
    return fail(PDA_ERR_HEAD_DIM, "head_dim %d: prefill serves head dims 1..512", head_dim);
  const int s = count == 0 ? 1 : prefill_splits(start, count, q_heads, kdim, window, splits);
  if (splits_used) *splits_used = s;
  *bytes = prefill_workspace(s, count, q_heads, kdim);
  return ok();
}

int pda_paged_prefill_attention(const void* queries, const void* keys, const void* values,
                                const int32_t* table, int32_t table_len, int32_t start,
                                int32_t count, void* out, int32_t q_heads, int32_t kv_heads,
                                int32_t head_dim, int32_t page_size, int64_t arena_rows,
                                int32_t layout, float scale, int32_t window, float softcap,
                                const int32_t* images, int32_t num_images, int32_t splits,
                                void* workspace, size_t workspace_bytes, void* stream) {
  return prefill(queries, keys, values, nullptr, nullptr, false, false, table, table_len, start,
                 count, out, q_heads, kv_heads, head_dim, page_size, arena_rows, layout, scale,
                 window, softcap, images, num_images, splits, workspace, workspace_bytes, stream);
}

int pda_paged_prefill_attention_bf16(const void* queries, const void* keys, const void* values,
                                     const int32_t* table, int32_t table_len, int32_t start,
                                     int32_t count, void* out, int32_t q_heads,
                                     int32_t kv_heads, int32_t head_dim, int32_t page_size,
                                     int64_t arena_rows, int32_t layout, float scale,
                                     int32_t window, float softcap, const int32_t* images,
                                     int32_t num_images, int32_t splits, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  return prefill(queries, keys, values, nullptr, nullptr, false, true, table, table_len, start,
                 count, out, q_heads, kv_heads, head_dim, page_size, arena_rows, layout, scale,
                 window, softcap, images, num_images, splits, workspace, workspace_bytes, stream);
}

int pda_paged_prefill_attention_q8(const void* queries, const void* keys, const void* values,
                                   const void* key_scales, const void* value_scales,
                                   const int32_t* table, int32_t table_len, int32_t start,
                                   int32_t count, void* out, int32_t q_heads, int32_t kv_heads,
                                   int32_t head_dim, int32_t page_size, int64_t arena_rows,
                                   int32_t layout, float scale, int32_t window, float softcap,
                                   const int32_t* images, int32_t num_images, int32_t splits,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  return prefill(queries, keys, values, key_scales, value_scales, true, false, table, table_len,
                 start, count, out, q_heads, kv_heads, head_dim, page_size, arena_rows, layout,
                 scale, window, softcap, images, num_images, splits, workspace, workspace_bytes,
                 stream);
}

}  // extern "C"
